"""Frames copied to the host in pieces through the pinned ring: below, at and
above its limits (no ring, one piece, a ragged last one, more pieces than
slots), the pixels in pageable and in pinned memory equal those of the same
frame left on the device, from a context's first frame on and where a frame is
replayed because its buffers had to grow."""
import ctypes as C

import numpy as np
import pytest

from rusterizer_amd import hostmath as hm
from rusterizer_amd import scenes

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("width,height", [
    (1, 1), (256, 128), (257, 128), (512, 512), (513, 512), (1024, 512), (1023, 1025), (1280, 1024), (3001, 1003)])
def test_read_back_equals_the_frame_on_the_device(width, height):
    import torch

    from rusterizer_amd.render import Context

    print(width, height, flush=True)
    npx = width * height
    dev = torch.zeros(npx, dtype=torch.int32, device="cuda")
    pin = torch.zeros(npx, dtype=torch.int32, pin_memory=True)
    eye = hm.identity()
    ctx = Context(width, height)
    try:
        ctx.set_uniforms(eye, eye, eye)
        for frame, n in enumerate((40, 300, 1, 30000)):
            rng = np.random.default_rng(frame)
            pos = rng.uniform(-1.2, 1.2, (3 * n, 3)).astype(np.float32)
            m = ctx.mesh(pos, rng.random((3 * n, 4)).astype(np.float32), None, np.arange(3 * n, dtype=np.uint32))
            ctx.draw(m, scenes.FS_COLOR)
            host = ctx.resolve()
            ctx.draw(m, scenes.FS_COLOR)
            ctx._check(ctx._L.rz_resolve(ctx.handle, C.c_void_p(pin.data_ptr())))
            ctx.draw(m, scenes.FS_COLOR)
            ctx.resolve_device(dev.data_ptr())
            want = dev.cpu().numpy().view(np.uint32).reshape(height, width)
            assert np.array_equal(host, want), frame
            assert np.array_equal(pin.numpy().view(np.uint32).reshape(height, width), want), frame
            m.destroy()
    finally:
        ctx.close()
