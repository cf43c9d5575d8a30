"""One-launch binning of small jobs (k_tile_bin): at the edges of its words of
64 prims, its rounds of 2048 list entries, its 32-pixel tiles and its limit of
16384 triangles a scene, the frame equals the oracle's and the one the two-level
binning gives (which a draw of 16385 culled triangles more selects), down to the
count of coarse entries that callers can read."""
import numpy as np
import pytest

from rusterizer_amd import hostmath as hm
from rusterizer_amd import scenes
from tests.harness import assert_parity, run_batch, run_gpu, run_oracle

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


def _frame(n, width, height, size, seed):
    """n front-facing triangles of about `size` pixels, at distinct depths."""
    rng = np.random.default_rng(seed)
    px = np.array([2.0 / width, 2.0 / height])
    xy = rng.uniform(-1, 1, (n, 1, 2)) + rng.uniform(-size, size, (n, 3, 2)) * px
    xy = xy.clip(-1, 1)
    z = rng.uniform(-0.9, 0.9, (n, 3))
    pos = np.concatenate([xy, z[..., None]], -1)
    e1, e2 = pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0]
    back = e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0] > 0
    pos[back] = pos[back][:, [0, 2, 1]]
    pos = pos.reshape(-1, 3).astype(F)
    eye = hm.identity()
    return scenes.Scene(f"tb{n}_{width}x{height}", width, height, pos, rng.random((3 * n, 4)).astype(F), None,
                        np.arange(3 * n, dtype=np.uint32), eye, eye, eye, scenes.FS_COLOR)


def _culled(sc):
    """16385 triangles without area, on the same screen."""
    n = 16385
    return scenes.Scene("culled", sc.width, sc.height, np.zeros((3, 3), F), np.zeros((3, 4), F), None,
                        np.zeros(3 * n, np.uint32), sc.world, sc.view, sc.proj, scenes.FS_COLOR)


@pytest.mark.parametrize("n,width,height,size", [
    (1, 1, 1, 4), (63, 31, 33, 9), (64, 32, 32, 9), (65, 95, 64, 9), (257, 64, 97, 200), (4000, 40, 70, 60),
    (16384, 100, 60, 3), (16385, 100, 60, 3), (700, 1000, 17, 30)])
def test_tile_bin_equals_two_level_binning(n, width, height, size):
    sc = _frame(n, width, height, size, seed=n)
    print(sc.name, flush=True)
    a, b = run_gpu(sc), run_gpu([sc, _culled(sc)])
    assert np.array_equal(a["img"], b["img"]) and np.array_equal(a["col"], b["col"])
    assert np.array_equal(a["dep"].view(np.uint32), b["dep"].view(np.uint32))
    for key in ("prims", "clipped", "bin_entries"):
        assert a["stats"][key] == b["stats"][key], (key, a["stats"], b["stats"])
    assert_parity(a, run_oracle(sc), where=sc.name)


@pytest.mark.parametrize("n,width,height", [(3840, 512, 512), (3841, 512, 512), (4096, 513, 512), (16384, 33, 31)])
def test_tile_bin_by_narrow_and_wide_workgroups(n, width, height):
    """Either side of the rule for 1024 threads (16 chunks of 256, 256 tiles)."""
    sc = _frame(n, width, height, 6, seed=n + width)
    print(sc.name, flush=True)
    for out in (run_gpu(sc, msaa=True), run_batch([sc])[0][0]):
        assert_parity(out, run_oracle(sc), where=sc.name)


def test_tile_bin_batches_switch_between_the_binnings():
    """Batches of small scenes, then with one scene too large, then small
    again, on one context (each binning keeps a graph of its own)."""
    from rusterizer_amd.render import Context

    small = [_frame(n, w, h, 20, seed=n) for n, w, h in ((5, 9, 9), (300, 70, 33), (1000, 64, 64), (1, 200, 3))]
    large = _frame(16400, 50, 40, 3, seed=9)
    want = {id(sc): run_oracle(sc) for sc in small + [large]}
    ctx = Context(64, 64)
    try:
        for batch in (small, small + [large], small, [large] + small):
            for sc, g in zip(batch, run_batch(batch, ctx=ctx)[0]):
                assert_parity(g, want[id(sc)], where=sc.name)
    finally:
        ctx.close()


@pytest.mark.parametrize("draws", [0, 64, 65])
def test_tile_bin_frames_of_many_draws(draws):
    """Each draw starts a chunk of 256 triangles of its own: 64 chunks are the
    most a frame's k_setup workgroups add up by themselves."""
    parts = [_frame(3 + i % 5, 90, 50, 25, seed=100 + i) for i in range(draws)]
    if not parts:
        parts = [_frame(1, 90, 50, 25, seed=1)]
        parts[0].idx = parts[0].idx[:0]
    assert_parity(run_gpu(parts), run_oracle(parts), where=f"{draws} draws")


@pytest.mark.parametrize("small", [1, 300, 16384])
def test_small_job_after_a_large_one_allocates_nothing(small):
    """A context that has run a large job runs a small one in the buffers it
    has: growing one waits for all work on the device (for a running raster
    service to go idle, a tenth of a second)."""
    from rusterizer_amd.render import Context

    ctx = Context(64, 64)
    try:
        run_batch([_frame(140000, 320, 240, 1, seed=3)], ctx=ctx)
        held = ctx.memory()["held"]
        run_batch([_frame(small, 320, 240, 4, seed=4)], ctx=ctx)
        assert ctx.memory()["held"] == held
    finally:
        ctx.close()
