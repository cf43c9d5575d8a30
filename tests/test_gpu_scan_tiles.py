"""The scans of count matrices above 2,048 tiles of 2,048 counts, which scan the
tiles' sums in a launch of their own: a frame of 4.5 million triangles on 256
coarse bins (4.5 million counts) equals the same frame on 4 bins (70,000)."""
import numpy as np
import pytest

from rusterizer_amd import hostmath as hm
from rusterizer_amd import scenes
from tests.harness import run_gpu

pytestmark = pytest.mark.gpu
F = np.float32


@pytest.fixture(scope="module", autouse=True)
def _need_gpu():
    from tests.conftest import gpu_available

    if not gpu_available():
        pytest.skip("no GPU")


def test_count_matrix_above_2048_scan_tiles():
    n, side = 4_500_000, 256
    rng = np.random.default_rng(8)
    xy = rng.uniform(-1, 1, (n, 1, 2)).astype(F) + rng.uniform(-1, 1, (n, 3, 2)).astype(F) * F(3.0 / side)
    pos = np.concatenate([xy.clip(-1, 1), rng.uniform(-0.9, 0.9, (n, 3, 1)).astype(F)], -1)
    e1, e2 = pos[:, 1] - pos[:, 0], pos[:, 2] - pos[:, 0]
    back = e1[:, 0] * e2[:, 1] - e1[:, 1] * e2[:, 0] > 0
    pos[back] = pos[back][:, [0, 2, 1]]
    eye = hm.identity()
    sc = scenes.Scene("scan_tiles", side, side, pos.reshape(-1, 3), rng.random((3 * n, 4), dtype=F), None,
                      np.arange(3 * n, dtype=np.uint32), eye, eye, eye, scenes.FS_COLOR)
    fine, coarse = run_gpu(sc, coarse_bin=16), run_gpu(sc, coarse_bin=128)
    assert fine["stats"]["prims"] == coarse["stats"]["prims"]
    chunks = (fine["stats"]["prims"] + 255) // 256
    print(fine["stats"], flush=True)
    assert chunks * 256 > 2048 * 2048 > chunks * 4
    for key in ("img", "col"):
        assert np.array_equal(fine[key], coarse[key])
    assert np.array_equal(fine["dep"].view(np.uint32), coarse["dep"].view(np.uint32))
