"""Products with fewer rows or columns than the tile they run on, and empty ones: small integers, where any order of
summation is exact."""
import numpy as np
import pytest

from helpers import rng_for

pytestmark = pytest.mark.gpu

import oracle  # noqa: E402


@pytest.fixture(scope="module")
def gt():
    import mcw_cppamp_torch_amd as pkg
    assert pkg._lib.lib.thgpu_init() == 0, pkg._lib.lib.thgpu_last_error()
    return pkg


def dev(gt, a):
    return gt.GPUTensor.from_numpy(np.ascontiguousarray(a, np.float32))


def labels_of(gt, call, prefix):
    gt.gputorch.synchronize()
    gt.gputorch.prof_reset()
    gt.gputorch.prof_enable(True)
    try:
        call()
        gt.gputorch.synchronize()
        return [k for k in gt.gputorch.prof_report() if k.startswith(prefix)]
    finally:
        gt.gputorch.prof_enable(False)
        gt.gputorch.prof_reset()


@pytest.mark.parametrize("n", [3, 70, 200])
def test_blas_product_of_an_empty_sum(gt, n):
    """alpha = 0: the tiled kernels' planner divides the reduction into steps, of which there are none."""
    rng = rng_for(500)
    a, c = np.full((n, 5), np.nan, np.float32), rng.integers(-3, 4, size=(n, n)).astype(np.float32)
    da, dc = dev(gt, a), dev(gt, c)
    gt.gputorch.gemm("n", "n", n, n, 5, 0.0, da, n, da, 5, 3.0, dc, n)
    assert np.array_equal(dc.float(), 3 * c)


# tile -> (rows, columns); the BLAS entry point is column-major, so C's columns n are the kernels' rows
TILES = {"32x128": (32, 128), "64x64": (64, 64), "64x64k4": (64, 64), "64x128": (64, 128), "64x256": (64, 256)}
ROWS = [1, 31, 32, 33, 63, 64, 65]
COLS = [1, 63, 64, 65, 127, 128, 300]


@pytest.mark.parametrize("split", [1, 3])
@pytest.mark.parametrize("ta", "nt")
@pytest.mark.parametrize("tb", "nt")
@pytest.mark.parametrize("tile", sorted(TILES))
def test_blas_products_shorter_than_a_tile(gt, tile, ta, tb, split, switches):
    bm, bn = TILES[tile]
    switches("gemm_tile", tile)
    switches("gemm_split", str(split))
    rng = rng_for(501)
    k = 399 if split == 3 else 37  # a partial last step; eight steps and more to a part
    for n in ROWS:
        for m in COLS:
            # leading dimensions as small as BLAS allows: the first row or column that is not there is another's, or nobody's
            lda, ldb, ldc = (m if ta == "n" else k), (k if tb == "n" else n), m
            a = rng.integers(-3, 4, size=(k if ta == "n" else m, lda)).astype(np.float32)
            b = rng.integers(-3, 4, size=(n if tb == "n" else k, ldb)).astype(np.float32)
            c0 = rng.integers(-3, 4, size=(n + 1, ldc)).astype(np.float32)  # a guard column behind C
            op_a = a.astype(np.int64).T if ta == "n" else a.astype(np.int64)
            op_b = b.astype(np.int64).T if tb == "n" else b.astype(np.int64)
            ref = c0.copy()
            ref[:n] = (2 * (op_a @ op_b).T + 3 * c0[:n].astype(np.int64)).astype(np.float32)
            da, db, dc = dev(gt, a.ravel()), dev(gt, b.ravel()), dev(gt, c0.ravel())
            labels = labels_of(gt, lambda: gt.gputorch.gemm(ta, tb, m, n, k, 2.0, da, lda, db, ldb, 3.0, dc, ldc), "gemm_blas")
            assert np.array_equal(dc.float().reshape(c0.shape), ref), (n, m, labels)
            taken = (n >= bm or bm <= 64) and (m >= bn or bn <= 64) and not (tile == "32x128" and tb == "t")
            assert ("tile=%s " % (tile if taken else "generic")) in labels[0], (n, m, labels)


LAYERS = {  # B, C, H, W, M, kH, kW, pH, pW, sH, sW
    "rows_37_strided": (5, 3, 101, 77, 37, 5, 5, 0, 0, 3, 3),
    "rows_1": (7, 5, 20, 23, 1, 3, 3, 1, 1, 1, 1),
    "rows_31_quads": (7, 7, 16, 20, 31, 3, 3, 1, 1, 1, 1),     # image rows of whole quads
    "rows_32_taps_25": (10, 1, 24, 24, 32, 5, 5, 2, 2, 1, 1),
    "rows_33_one_image": (1, 48, 19, 17, 33, 3, 3, 1, 1, 1, 1),
    "rows_63_long": (6, 40, 12, 12, 63, 5, 5, 0, 0, 1, 1),
    "few_positions": (1, 64, 7, 7, 20, 4, 4, 0, 0, 1, 1),      # 16 positions
    "small_columns": (2, 7, 16, 20, 31, 3, 3, 1, 1, 1, 1),     # 158 KB of columns: they stay
    "strided_few_classes": (2, 3, 30, 41, 70, 5, 3, 1, 0, 2, 1),
}


@pytest.mark.parametrize("tile", [None] + sorted(TILES))
@pytest.mark.parametrize("name", sorted(LAYERS))
def test_layers_of_few_planes_without_columns(gt, name, tile, switches):
    """Forward, gradInput, gradWeight and gradBias of layers whose products have fewer rows than a tile, bit for bit, by the
    library's own choice and on every short tile; the guard row behind each parameter stays as it is."""
    B, C, H, W, M, kH, kW, pH, pW, sH, sW = LAYERS[name]
    geo, K = (kH, kW, pH, pW, sH, sW), C * kH * kW
    rng = rng_for(502)
    ints = lambda lo, hi, shape: rng.integers(lo, hi + 1, size=shape).astype(np.float32)
    x, w, b = ints(-2, 2, (B, C, H, W)), ints(-2, 2, (M, K)), ints(-3, 3, (M,))
    out, finput = oracle.conv_updateOutput(x, w, b, *geo)
    go = ints(-2, 2, out.shape)
    gi, _ = oracle.conv_updateGradInput(go, w, x.shape, *geo)
    gw0, gb0 = ints(-5, 5, (M, K)), ints(-5, 5, (M,))
    gw, gb = gw0.copy(), gb0.copy()
    oracle.conv_accGradParameters(go, finput, gw, gb, 2.0)
    if tile is not None:
        switches("gemm_tile", tile)
    m = gt.nn.SpatialConvolutionMM(C, M, kW, kH, sW, sH, 0, padW=pW, padH=pH)
    m._assign("weight", w)
    m._assign("bias", b)
    m.gpu()
    guard_w, guard_b = dev(gt, np.vstack([gw0, np.full((1, K), 9, np.float32)])), dev(gt, np.append(gb0, np.float32(9)))
    m.gradWeight, m.gradBias = guard_w.narrow(0, 0, M), guard_b.narrow(0, 0, M)
    dx, dgo = dev(gt, x), dev(gt, go)
    assert np.array_equal(m.forward(dx).float(), out)
    assert np.array_equal(m.updateGradInput(dx, dgo).float(), gi)
    labels = labels_of(gt, lambda: m.accGradParameters(dx, dgo, 2.0), ("gemm_conv", "im2col"))
    assert np.array_equal(guard_w.float(), np.vstack([gw, np.full((1, K), 9, np.float32)]))
    assert np.array_equal(guard_b.float(), np.append(gb, np.float32(9)))
    if tile is None:       # (a forced tile that gradWeight does not fit leaves the whole layer on columns)
        assert any(l.startswith("im2col") for l in labels) == (name == "small_columns"), labels
    if tile is None and name != "few_positions":
        assert not any("generic" in l for l in labels), labels


@pytest.mark.parametrize("at", [5, 150, 251, 398])  # a step of each of the four groups
@pytest.mark.parametrize("tile", ["32x128", "64x64k4"])
def test_values_that_bf16_parts_do_not_hold(gt, tile, at, switches):
    """A 24-bit number below 2^-110 against a large partner, an infinity and a NaN: multiplied in fp32, as on the other tiles
    (one product a result, so exact), wherever in the reduction they stand."""
    switches("gemm_tile", tile)
    switches("gemm_split", "1")
    m, n, k = 200, 40, 399
    a, b = np.zeros((k, m), np.float32), np.ones((n, k), np.float32)
    a[at, 3] = np.float32(2.0 ** -118 * (1 + 2.0 ** -23))
    a[at, 70], a[at, 71] = np.inf, np.nan
    b[:, at] = 2.0 ** 100
    b[7, at] = -(2.0 ** 100)
    c = gt.GPUTensor(n * m).fill(0)
    da, db = dev(gt, a.ravel()), dev(gt, b.ravel())
    labels = labels_of(gt, lambda: gt.gputorch.gemm("n", "n", m, n, k, 1.0, da, m, db, k, 0.0, c, m), "gemm_blas")
    assert "tile=%s " % tile in labels[0]
    got = c.float().reshape(n, m)
    ref = b[:, at:at + 1] * a[at]
    ref[:, 70], ref[:, 71] = np.copysign(np.inf, b[:, at]), np.nan
    assert np.array_equal(got, ref, equal_nan=True)
