"""The raster's matrix path (one MFMA for a prim's edge values and depth at a
quadrant's 256 samples) against the oracle, bit for bit, where its margins
matter: edges through samples, depths within a few ulps of each other, slivers,
sub-pixel and screen-sized triangles, quadrants cut by the screen's border, and
clear depths that its arithmetic has to pass through unchanged."""
import numpy as np
import pytest

from rusterizer_amd import hostmath as hm
from rusterizer_amd import scenes
from tests.harness import assert_parity, run_gpu, run_oracle

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


def _frame(kind: str, width: int, height: int, seed: int) -> scenes.Scene:
    """Triangles in normalised device coordinates (identity matrices, w = 1)."""
    rng = np.random.default_rng(seed)
    n = 160
    px = np.array([2.0 / width, 2.0 / height])
    if kind == "screen":      # screen-sized planes that cut through each other
        xy = rng.uniform(-1, 1, (n, 3, 2))
        z = rng.uniform(-0.9, 0.9, (n, 3))
    elif kind == "tiny":      # about a sample apart
        xy = rng.uniform(-1, 1, (n, 1, 2)) + rng.uniform(-0.6, 0.6, (n, 3, 2)) * px
        z = rng.uniform(-0.9, 0.9, (n, 1)) + rng.uniform(-0.01, 0.01, (n, 3))
    elif kind == "sliver":    # as long as the screen, a fraction of a pixel wide
        a, b = rng.uniform(-1, 1, (n, 2)), rng.uniform(-1, 1, (n, 2))
        xy = np.stack([a, b, b + rng.uniform(-0.7, 0.7, (n, 2)) * px], 1)
        z = rng.uniform(-0.9, 0.9, (n, 3))
    elif kind == "ties":      # near-coplanar copies, 0 to 300 ulps (of 1.0) apart in depth
        xy = np.repeat(rng.uniform(-0.95, 0.95, (n // 8, 3, 2)), 8, axis=0)
        z = np.repeat(rng.uniform(0.2, 0.9, (n // 8, 3)), 8, axis=0)
        z = z + rng.choice([0, 1, -1, 3, -8, 20, -60, 300], (n, 1)) * 2.0 ** -23
    else:                     # lattice: vertices and edges on sample positions (eighths of a pixel)
        xy = (rng.integers(0, 8 * np.array([width, height]) + 1, (n, 3, 2)) * px / 8.0) - 1.0
        z = rng.integers(-8, 8, (n, 3)) / 16.0
    pos = np.concatenate([xy, z[..., None]], -1)
    # front-facing ones draw (y is down on the screen)
    e1, e2 = pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0]
    back = e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0] > 0
    pos[back] = pos[back][:, [0, 2, 1]]
    pos = pos.reshape(-1, 3).astype(F)
    eye = hm.identity()
    color = rng.random((len(pos), 4)).astype(F)
    return scenes.Scene(f"{kind}{width}x{height}", width, height, pos, color, None,
                        np.arange(len(pos), dtype=np.uint32), eye, eye, eye, scenes.FS_COLOR)


@pytest.mark.parametrize("size", [(7, 9), (8, 8), (33, 17), (251, 130)])
@pytest.mark.parametrize("kind", ["screen", "tiny", "sliver", "ties", "lattice"])
def test_matrix_walk_matches_oracle(kind, size):
    sc = _frame(kind, *size, seed=7 + size[0])
    print(sc.name, flush=True)
    assert_parity(run_gpu(sc), run_oracle(sc), where=sc.name)


@pytest.mark.parametrize("clear", [0.5, 1.0, -1.0, float("inf"), float("-inf"), float("nan"),
                                   -float(np.finfo(np.float32).max)])
def test_matrix_walk_clear_depths(clear):
    sc = _frame("screen", 61, 40, seed=3)
    sc.clear_depth = clear
    print(clear, flush=True)
    assert_parity(run_gpu(sc), run_oracle(sc), where=f"clear {clear}")
