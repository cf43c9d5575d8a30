"""A context keeps a captured graph for each launch sequence that its read-back
frames take (small scenes with and without k_scene_prep, either width of
k_tile_bin, two-level binning): frames of all kinds by turns, each several times,
equal the oracle's."""
import numpy as np
import pytest

from rusterizer_amd import hostmath as hm
from rusterizer_amd import scenes
from tests.harness import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu
F = np.float32
W, H = 90, 50


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


def _draw(n, size, seed):
    rng = np.random.default_rng(seed)
    px = np.array([2.0 / W, 2.0 / H])
    xy = (rng.uniform(-1, 1, (n, 1, 2)) + rng.uniform(-size, size, (n, 3, 2)) * px).clip(-1, 1)
    pos = np.concatenate([xy, rng.uniform(-0.9, 0.9, (n, 3, 1))], -1)
    eye = hm.identity()
    return scenes.Scene(f"kind{n}", W, H, pos.reshape(-1, 3).astype(F), rng.random((3 * n, 4)).astype(F), None,
                        np.arange(3 * n, dtype=np.uint32), eye, eye, eye, scenes.FS_COLOR)


def test_frames_of_every_kind_by_turns():
    from rusterizer_amd.render import Context

    few = [_draw(3 + i % 5, 20, 100 + i) for i in range(65)]  # 65 chunks: more than k_setup adds up by itself
    kinds = {"small": [_draw(300, 15, 1)], "small, wide": [_draw(6000, 4, 2)], "draws": few,
             "draws, wide": few + [_draw(6000, 4, 3)], "two-level": [_draw(16385, 3, 4)]}
    want = {k: run_oracle(v) for k, v in kinds.items()}
    ctx = Context(W, H)
    try:
        for order in (list(kinds), list(kinds)[::-1], list(kinds)[::2] + list(kinds)[1::2]):
            for kind in order:
                for _ in range(2):
                    print(kind, flush=True)
                    assert_parity(run_gpu(kinds[kind], ctx=ctx), want[kind], where=kind)
    finally:
        ctx.close()
