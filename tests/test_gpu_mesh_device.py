"""Meshes made from device arrays: the copy comes after the work on the null
stream that writes the arrays and before anything that the context does with the
mesh, so the frame equals the oracle's however late the arrays are written."""
import numpy as np
import pytest

from rusterizer_amd import scenes
from tests.harness import assert_parity, run_oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


@pytest.mark.parametrize("n", [1, 3000, 200_000])
def test_mesh_of_arrays_still_being_written(n):
    import torch

    from rusterizer_amd.render import Context, RzError

    sc = scenes.soup_scene(n, 320, 200, seed=n)
    src = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (sc.pos, sc.color, sc.idx.view(np.int32))]
    late = [torch.zeros_like(t) for t in src]
    busy = torch.zeros(1 << 28, device="cuda")
    ctx = Context(sc.width, sc.height)
    try:
        ctx.set_clear_depth(sc.clear_depth)
        ctx.set_uniforms(sc.world, sc.view, sc.proj)
        torch.cuda.synchronize()
        for _ in range(8):  # a few milliseconds of work before the arrays
            busy.add_(1.0)
        for d, s in zip(late, src):
            d.copy_(s)
        m = ctx.mesh_device(late[0], late[1], None, late[2])
        ctx.draw(m, sc.fs)
        img, col, dep = ctx.resolve_msaa()
        assert_parity(dict(img=img, col=col, dep=dep, flags=ctx.frame_flags()), run_oracle(sc), where=sc.name)
        m.destroy()
        bad = late[2].clone()
        bad[-1] = sc.pos.shape[0]
        with pytest.raises(RzError, match="index out of range"):
            ctx.mesh_device(late[0], late[1], None, bad)
    finally:
        ctx.close()
