"""Small jobs whose first pass outgrows a buffer: which one it was is in the
overflow bits, one larger pass follows (what the first one counted is the whole
job's need), and the images equal the oracle's."""
import numpy as np
import pytest

from rusterizer_amd import hostmath as hm
from rusterizer_amd import scenes
from tests.harness import assert_parity, run_batch, run_gpu, run_oracle

pytestmark = pytest.mark.gpu
F = np.float32
OVF_PRIMS, OVF_PAIRS, OVF_FINE = 1, 4, 16


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


def _column(n, width, height, seed):
    """n triangles as tall as the screen, at distinct depths: each is on the
    list of every 32-pixel tile of a narrow, high screen."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(-0.9, 0.9, (n, 1))
    corners = np.array([[0.0, -1.0], [0.1, 1.0], [-0.1, 1.0]])
    xy = corners[None] + np.stack([x, np.zeros_like(x)], -1)
    pos = np.concatenate([xy, rng.uniform(-0.9, 0.9, (n, 3, 1))], -1).clip(-1, 1)
    e1, e2 = pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0]
    back = e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0] > 0
    pos[back] = pos[back][:, [0, 2, 1]]
    eye = hm.identity()
    return scenes.Scene(f"column{n}_{width}x{height}", width, height, pos.reshape(-1, 3).astype(F),
                        rng.random((3 * n, 4)).astype(F), None, np.arange(3 * n, dtype=np.uint32), eye, eye, eye,
                        scenes.FS_COLOR)


def test_lists_of_a_batch_outgrow_their_first_estimate():
    """Eight scenes of 128 tiles and 256 triangles: 262,144 entries, where a
    new context has room for 174,080."""
    batch = [_column(256, 2, 4096, seed=s) for s in range(8)]
    out, stats = run_batch(batch)
    print(stats, flush=True)
    assert stats["replays"] == 1 and stats["overflow_bits"] == OVF_FINE
    for sc, g in zip(batch, out):
        assert_parity(g, run_oracle(sc), where=sc.name)


def test_lists_of_one_scene_outgrow_their_first_estimate():
    """512 tiles and 5,600 triangles: 2.87 million entries, neither placed side by
    side nor within the 2.62 million that a new context has room for."""
    sc = _column(5600, 3, 16384, seed=9)
    g = run_gpu(sc)
    print(g["stats"], flush=True)
    assert g["stats"]["replays"] == 1 and g["stats"]["overflow_bits"] == OVF_FINE
    assert_parity(g, run_oracle(sc), where=sc.name)


def test_prims_of_one_scene_outgrow_their_first_estimate():
    """1,400 triangles that clipping makes 9,559 of, where a new context has room
    for 7,840."""
    sc = scenes.nine_vertex_scene(1400)
    g = run_gpu(sc)
    print(g["stats"], flush=True)
    assert g["stats"]["prims"] == 9559
    assert g["stats"]["replays"] == 1 and g["stats"]["overflow_bits"] == OVF_PRIMS
    assert_parity(g, run_oracle(sc), where=sc.name)


@pytest.mark.parametrize("n,width,height,bits,tiles", [
    (17000, 3, 4096, OVF_PAIRS, {}),  # 256 bins of 16x16, room for 64,480 entries
    (20000, 256, 256, OVF_FINE, dict(coarse_bin=256, fine_tile=16))])  # one bin; room for 592,640 entries
def test_lists_of_the_two_level_binning_outgrow_their_first_estimate(n, width, height, bits, tiles):
    sc = _column(n, width, height, seed=n)
    g = run_gpu(sc, **tiles)
    print(g["stats"], flush=True)
    assert g["stats"]["replays"] == 1 and g["stats"]["overflow_bits"] == bits
    assert_parity(g, run_oracle(sc), where=sc.name)


@pytest.mark.parametrize("width,height", [(160, 96), (520, 520), (3001, 1003)])
def test_read_back_of_a_frame_that_outgrows_its_buffers(width, height):
    """Through the pinned ring (which a context's second frame starts): the pieces
    queued behind the first pass are copied again after the larger one."""
    import torch

    from rusterizer_amd.render import Context

    sc = scenes.nine_vertex_scene(1400, width, height)
    sc.idx = np.ascontiguousarray(sc.idx.reshape(-1, 3)[:, ::-1]).reshape(-1)  # (they face away as they are)
    print(width, height, flush=True)
    dev = torch.zeros(width * height, dtype=torch.int32, device="cuda")
    ctx = Context(width, height)
    try:
        ctx.set_uniforms(sc.world, sc.view, sc.proj)
        m = ctx.mesh(sc.pos, sc.color, sc.uv, sc.idx)
        one = ctx.mesh(sc.pos[:3], sc.color[:3], None, np.arange(3, dtype=np.uint32))
        ctx.draw(one, sc.fs)
        ctx.resolve()
        ctx.draw(m, sc.fs)
        host = ctx.resolve()
        stats = ctx.frame_stats()
        assert stats["replays"] >= 1 and stats["overflow_bits"] & OVF_PRIMS, stats
        ctx.draw(m, sc.fs)
        ctx.resolve_device(dev.data_ptr())
        assert ctx.frame_stats()["replays"] == 0
        assert np.array_equal(host, dev.cpu().numpy().view(np.uint32).reshape(height, width))
        assert np.unique(host).size > 100
        if width < 1000:
            assert np.array_equal(host, run_oracle(sc)["img"])
        m.destroy()
        one.destroy()
    finally:
        ctx.close()
