"""The scans of the binning's count matrices (by one workgroup, or by tiles that
add up the sums before them): frames whose matrices lie on either side of the
limit, by the number of triangles and the coarse bins' size, equal the oracle's
and each other."""
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


def _frame(n, width, height, seed):
    rng = np.random.default_rng(seed)
    px = np.array([2.0 / width, 2.0 / height])
    xy = (rng.uniform(-1, 1, (n, 1, 2)) + rng.uniform(-3, 3, (n, 3, 2)) * px).clip(-1, 1)
    pos = np.concatenate([xy, rng.uniform(-0.9, 0.9, (n, 3, 1))], -1)
    eye = hm.identity()
    return scenes.Scene(f"scan{n}", width, height, pos.reshape(-1, 3).astype(F), rng.random((3 * n, 4)).astype(F), None,
                        np.arange(3 * n, dtype=np.uint32), eye, eye, eye, scenes.FS_COLOR)


# chunks of 256 prims times coarse bins: about 300 to 400,000 counts
@pytest.mark.parametrize("n,side,bins", [(16500, 256, (128, 16)), (70000, 256, (128, 32, 16)), (400000, 256, (16,))])
def test_count_matrices_across_the_scans_limit(n, side, bins):
    sc = _frame(n, side, side, seed=n)
    print(sc.name, flush=True)
    runs = [run_gpu(sc, coarse_bin=cb) for cb in bins]
    for r in runs[1:]:
        assert np.array_equal(r["img"], runs[0]["img"]) and np.array_equal(r["dep"].view(np.uint32), runs[0]["dep"].view(np.uint32))
    assert_parity(runs[0], run_oracle(sc), where=sc.name)
