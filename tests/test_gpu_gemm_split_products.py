"""The tiled GEMM kernel forms its products from three bf16 parts of each operand: its error against 64 bits, and the
values that the parts cannot hold (infinities, NaN, numbers that round to infinity in bf16, results below the normal
range), which it multiplies in fp32 instead."""
import numpy as np
import pytest

from helpers import rng_for

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gt():
    import mcw_cppamp_torch_amd as pkg
    assert pkg._lib.lib.thgpu_init() == 0
    return pkg


def product(gt, A, B):
    """A (m x k) times B (k x n) through the BLAS entry point, each kept row-major."""
    m, k = A.shape
    n = B.shape[1]
    da, db = gt.FloatTensor(A).gpu(), gt.FloatTensor(B).gpu()
    dc = gt.FloatTensor(np.full((m, n), 7.0, np.float32)).gpu()
    gt.gputorch.gemm("n", "n", n, m, k, 1.0, db, n, da, k, 0.0, dc, n)
    return dc.float()


# m, n, k: one tile and one step; a step moved back; edge tiles moved back in both directions; long sums
SIZES = [(64, 64, 16), (64, 130, 17), (191, 257, 33), (129, 300, 255), (64, 64, 5000)]


@pytest.mark.parametrize("spread", [0.0, 4.0])
@pytest.mark.parametrize("m,n,k", SIZES)
def test_error_against_64_bits(gt, m, n, k, spread):
    """Each product loses at most 2^-24 (the three part products left out) and each of the 6 additions per 16 indices
    rounds a partial sum of at most S = sum |a||b| by 2^-24 S; split sums add one rounding per part."""
    rng = rng_for(301)
    draw = lambda *s: (rng.standard_normal(s) * np.exp(spread * rng.standard_normal(s))).astype(np.float32)
    A, B = draw(m, k), draw(k, n)
    got = product(gt, A, B).astype(np.float64)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    S = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    adds = 6 * ((k + 15) // 16) + 256
    assert np.all(np.abs(got - ref) <= (1 + adds) * 2.0 ** -24 * S)


@pytest.mark.parametrize("m,n,k", SIZES[:4])
def test_values_the_parts_cannot_hold(gt, m, n, k):
    rng = rng_for(302)
    A = rng.integers(-2, 3, size=(m, k)).astype(np.float32)
    B = rng.integers(-2, 3, size=(k, n)).astype(np.float32)
    A[0, 0], A[1, k - 1], A[m - 1, 3], A[5, 2] = np.inf, -np.inf, np.nan, 3.4e38  # 3.4e38 is infinite in bf16
    B[:, n - 1] = 0.0
    B[2, 1], B[2, n - 1], B[4, 40] = 0.5, 0.5, -np.inf
    with np.errstate(all="ignore"):
        # all finite sums are exact in 64 bits and, but for row 5, whole numbers; there 3.4e38 swallows the rest
        ref = (A.astype(np.float64) @ B.astype(np.float64)).astype(np.float32)
    got = product(gt, A, B)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = ~np.isnan(ref)
    assert np.array_equal(got[ok], ref[ok])


def test_results_below_the_normal_range(gt):
    """Eight products of 1.5 * 2^-130: the sum is a denormal that fp32 holds exactly."""
    m, n, k = 64, 96, 32
    A, B = np.zeros((m, k), np.float32), np.zeros((k, n), np.float32)
    A[:, ::4] = np.float32(1.5 * 2.0 ** -65)
    B[::4, :] = np.float32(2.0 ** -65)
    assert np.array_equal(product(gt, A, B), np.full((m, n), np.float32(8 * 1.5 * 2.0 ** -130)))
