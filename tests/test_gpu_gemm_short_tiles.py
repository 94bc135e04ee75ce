"""Products with fewer rows or columns than the tile they run on, and empty ones: small integers, where any order of
summation is exact."""
import numpy as np
import pytest

from helpers import rng_for

pytestmark = pytest.mark.gpu

@pytest.fixture(scope="module")
def gt():
    import mcw_cppamp_torch_amd as pkg
    assert pkg._lib.lib.thgpu_init() == 0, pkg._lib.lib.thgpu_last_error()
    return pkg


def dev(gt, a):
    return gt.GPUTensor.from_numpy(np.ascontiguousarray(a, np.float32))


@pytest.mark.parametrize("n", [3, 70, 200])
def test_blas_product_of_an_empty_sum(gt, n):
    """alpha = 0: the tiled kernels' planner divides the reduction into steps, of which there are none."""
    rng = rng_for(500)
    a, c = np.full((n, 5), np.nan, np.float32), rng.integers(-3, 4, size=(n, n)).astype(np.float32)
    da, dc = dev(gt, a), dev(gt, c)
    gt.gputorch.gemm("n", "n", n, n, 5, 0.0, da, n, da, 5, 3.0, dc, n)
    assert np.array_equal(dc.float(), 3 * c)
