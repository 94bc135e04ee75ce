"""The tiled GEMM kernel forms its products from three bf16 parts of each operand: its error against 64 bits, and the
values that the parts cannot hold (operands with bits below the smallest bf16 step, infinities, NaN, numbers that round to
infinity in bf16, results below the normal range), which it multiplies in fp32 instead.  Every tile and loader: the four
operand layouts through the BLAS entry point, the gathering loaders and reduction batching through convolution layers."""
import functools

import numpy as np
import pytest
import torch

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
def test_error_against_64_bits(gt, switches, m, n, k, spread):
    """Each product loses at most 2^-24 (the three part products left out).  The sum of a step of 16 indices is rounded
    twice by each of six instructions, and then once with the running sum of at most S = sum |a||b|, by 2^-24 S each."""
    switches("gemm_split", 1)
    rng = rng_for(301)
    draw = lambda *s: (rng.standard_normal(s) * np.exp(spread * rng.standard_normal(s))).astype(np.float32)
    A, B = draw(m, k), draw(k, n)
    got = product(gt, A, B).astype(np.float64)
    ref = A.astype(np.float64) @ B.astype(np.float64)
    S = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
    assert np.all(np.abs(got - ref) <= (1 + 12 + (k + 15) // 16) * 2.0 ** -24 * S)


@pytest.mark.parametrize("kind", ["uniform", "half of one operand zero", "positive"])
@pytest.mark.parametrize("k", [16, 48, 272, 1000])
def test_no_less_exact_than_sums_in_fp32(gt, switches, kind, k):
    """Against the same product summed index by index in fp32: no larger root mean square error, and no mean error either.
    (The matrix instruction cuts what lies far below the larger addend downwards; the sign it is given alternates.)  The
    mean of n errors of either sign is within six of its standard deviations; of each row, too, as the sums over pixels
    that follow a product meet it."""
    switches("gemm_split", 1)
    m, n = 192, 4096
    rng = rng_for(305)
    A, B = ((rng.random(shape, np.float32) * 2 - 1) for shape in ((m, k), (k, n)))
    if kind == "positive":
        A, B = np.abs(A), np.abs(B)
    elif kind != "uniform":
        B = np.maximum(B, 0)
    fp32 = np.zeros((m, n), np.float32)
    for r in range(k):
        fp32 += A[:, r:r + 1] * B[r]
    ref = A.astype(np.float64) @ B.astype(np.float64)
    err, err32 = product(gt, A, B) - ref, fp32 - ref
    rms = lambda e: np.sqrt(np.mean(np.square(e)))
    assert rms(err) <= rms(err32)
    assert abs(err.mean()) <= 6 * rms(err) / np.sqrt(err.size)
    assert np.all(np.abs(err.mean(1)) <= 6 * rms(err) / np.sqrt(n))


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


TILES = {"128x128": (128, 128), "192x128": (192, 128), "64x256": (64, 256), "128x256": (128, 256),
         "256x128": (256, 128), "64x64": (64, 64), "64x128": (64, 128), "96x128": (96, 128),
         "32x128": (32, 128), "64x64k4": (64, 64)}
LAYOUTS = [(tile, ta, tb) for tile in TILES for ta in "nt" for tb in "nt" if not (tile in ("96x128", "32x128") and ta == "t")]


def blas(gt, ta, tb, A, B):
    """C = A B (A m x k, B k x n) with either operand stored along k ('n' for A, 't' for B) or along its free index; the
    per-kernel timing labels of the product come with it."""
    (m, k), n = A.shape, B.shape[1]
    da = gt.FloatTensor(np.ascontiguousarray(A if ta == "n" else A.T)).gpu()
    db = gt.FloatTensor(np.ascontiguousarray(B if tb == "n" else B.T)).gpu()
    dc = gt.FloatTensor(np.full((m, n), 7.0, np.float32)).gpu()
    rec = gt.gputorch
    rec.synchronize()
    rec.prof_reset()
    rec.prof_enable(True)
    try:
        rec.gemm(tb, ta, n, m, k, 1.0, db, n if tb == "n" else k, da, k if ta == "n" else m, 0.0, dc, n)
        rec.synchronize()
        labels = [key for key in rec.prof_report() if key.startswith("gemm_blas")]
    finally:
        rec.prof_enable(False)
        rec.prof_reset()
    return dc.float(), labels


def columns64(x, geo):
    """im2col in 64 bits: (B, C*kH*kW, N)."""
    kH, kW, pH, pW, sH, sW = geo
    return torch.nn.functional.unfold(torch.from_numpy(x).double(), (kH, kW), padding=(pH, pW), stride=(sH, sW)).numpy()


def image64(cols, shape, geo):
    kH, kW, pH, pW, sH, sW = geo
    return torch.nn.functional.fold(torch.from_numpy(cols), shape[2:], (kH, kW), padding=(pH, pW), stride=(sH, sW)).numpy()


def conv64(x, w, go, geo):
    """Output, gradInput and gradWeight of a layer in 64 bits."""
    cols, g = columns64(x, geo), go.reshape(go.shape[0], go.shape[1], -1).astype(np.float64)
    W = w.astype(np.float64)
    return (np.matmul(W, cols).reshape(go.shape), image64(np.matmul(W.T, g), x.shape, geo),
            np.matmul(g, cols.transpose(0, 2, 1)).sum(0))


def conv(gt, x, w, go, geo):
    """The same of nn.SpatialConvolutionMM, bias zero; labels of its products."""
    kH, kW, pH, pW, sH, sW = geo
    m = gt.nn.SpatialConvolutionMM(x.shape[1], w.shape[0], kW, kH, sW, sH, 0, padW=pW, padH=pH)
    m._assign("weight", w)
    m.bias[...] = 0
    m.gradWeight[...] = 0
    m.gpu()
    dx, dgo = gt.FloatTensor(x).gpu(), gt.FloatTensor(go).gpu()
    rec = gt.gputorch
    rec.synchronize()
    rec.prof_reset()
    rec.prof_enable(True)
    try:
        out = m.forward(dx)
        gi = m.updateGradInput(dx, dgo)
        m.accGradParameters(dx, dgo, 1.0)
        rec.synchronize()
        labels = [key for key in rec.prof_report() if key.startswith("gemm_conv")]
    finally:
        rec.prof_enable(False)
        rec.prof_reset()
    return out.float(), gi.float(), m.gradWeight.float(), labels


def magnitudes(rng, shape, exponent):
    """Numbers of full precision (as far as fp32 has it there), 1 to 2 times a power of two, either sign."""
    return np.ldexp(rng.uniform(1, 2, shape), exponent).astype(np.float32) * rng.choice(np.float32([-1, 1]), shape)


# exponents of the small operand and of its partner: results from just above the normal range to ordinary numbers
SMALL = [(-112, 0), (-120, 0), (-126, 60), (-140, 120)]


@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("tile,ta,tb", LAYOUTS)
def test_small_operands(gt, switches, tile, ta, tb, split):
    """Operands with bits under the smallest bf16 step, either one, in every row (column) or in a single one, which few
    threads load: the bound of fp32 sums (k products and additions, each rounded; one more per part)."""
    switches("gemm_tile", tile)
    switches("gemm_split", split)
    (m, n), k = (d + 3 for d in TILES[tile]), 16 * 16 + 5
    rng = rng_for(303)
    for small, large in SMALL:
        for swap in (False, True):
            for everywhere in (False, True):
                rows, other = (n, m) if swap else (m, n)
                P, Q = magnitudes(rng, (rows, k), min(0, 100 - large)), magnitudes(rng, (k, other), large)
                some = np.s_[:] if everywhere else np.s_[rng.integers(rows)]
                P[some] = magnitudes(rng, P[some].shape, small)
                A, B = (Q.T, P.T) if swap else (P, Q)
                got, labels = blas(gt, ta, tb, A, B)
                assert len(labels) == 1 and "tile=%s split=%d" % (tile, split) in labels[0], labels
                ref = A.astype(np.float64) @ B.astype(np.float64)
                S = np.abs(A).astype(np.float64) @ np.abs(B).astype(np.float64)
                assert np.all(np.abs(got - ref) <= (k + split + 1) * 2.0 ** -24 * S), (small, large, swap, everywhere)


@functools.lru_cache(maxsize=6)
def small_layer(batch, width, small, large, which):
    rng = rng_for(304)
    C = M = 256
    x, w, go = (magnitudes(rng, shape, small if which == name else large)
                for name, shape in (("x", (batch, C, 32, width)), ("w", (M, C * 9)), ("go", (batch, M, 32, width))))
    geo = (3, 3, 1, 1, 1, 1)
    return x, w, go, geo, conv64(x, w, go, geo), conv64(np.abs(x), np.abs(w), np.abs(go), geo)


# width 8: image rows of whole quads (128-bit gathers in gradWeight); 9: not.  Two images and one.
@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("batch,width", [(2, 8), (2, 9), (1, 8), (1, 9)])
def test_small_operands_in_convolution_layers(gt, gathered_route, switches, tile, batch, width):
    switches("gemm_tile", tile)
    for small, large in ((-120, 20), (-130, 50)):
        for which in ("x", "w", "go"):
            x, w, go, geo, ref, S = small_layer(batch, width, small, large, which)
            *got, labels = conv(gt, x, w, go, geo)
            assert len(labels) == 3 and all("tile=%s " % tile in l for l in labels), labels
            # the longest sums: taps, gradients, pixels; at most 256 parts
            for g, r, s, terms in zip(got, ref, S, (w.shape[1], w.shape[0] * 9, batch * 32 * width)):
                assert np.all(np.abs(g.reshape(r.shape) - r) <= (terms + 258) * 2.0 ** -24 * s), (small, large, which, terms)


def whole_numbers(rng, shape, bits):
    """Odd numbers of exactly this many bits, either sign: one bf16 part up to 8, two up to 16, three up to 24."""
    top = rng.integers(2 ** (bits - 1), 2 ** bits, size=shape) | 1
    return (top * rng.choice([-1, 1], shape)).astype(np.float32)


BITS = [(24, 1), (1, 24), (12, 12), (16, 8), (8, 16)]


@pytest.mark.parametrize("tile,ta,tb", LAYOUTS)
def test_every_part_of_every_element_counts(gt, switches, tile, ta, tb):
    """Sums of one product of at most 24 bits are exact, and wrong if any part of either element, or any of the part
    products that reach 24 bits, is lost or misplaced.  One element of every row of the first operand, then of every column
    of the second, is not zero; every reduction index has its turn."""
    switches("gemm_tile", tile)
    (m, n), k = (d + 3 for d in TILES[tile]), 37
    rng = rng_for(306)
    for bits_a, bits_b in BITS:
        for sparse_first in (True, False):
            A, B = whole_numbers(rng, (m, k), bits_a), whole_numbers(rng, (k, n), bits_b)
            if sparse_first:
                A[np.arange(k) != (np.arange(m) % k)[:, None]] = 0
            else:
                B[np.arange(k)[:, None] != np.arange(n) % k] = 0
            got, labels = blas(gt, ta, tb, A, B)
            assert len(labels) == 1 and "tile=%s " % tile in labels[0], labels
            assert np.array_equal(got, A.astype(np.float64) @ B.astype(np.float64)), (bits_a, bits_b, sparse_first)


@functools.lru_cache(maxsize=1)
def one_product_layers(batch, width):
    """Layers of 256 planes whose sums hold one product each: weights of one tap per output plane (output and gradInput),
    one pixel per plane of the input or of gradOutput (gradWeight)."""
    rng = rng_for(307)
    C = M = 256
    shape, geo = (batch, C, 32, width), (3, 3, 1, 1, 1, 1)
    cases = []
    for bits, other in BITS:
        x, w, go = whole_numbers(rng, shape, bits), whole_numbers(rng, (M, C, 9), other), whole_numbers(rng, shape, bits)
        tap, plane = rng.integers(9, size=M), rng.permutation(C)
        keep = np.zeros((M, C, 9), bool)
        keep[np.arange(M), plane, tap] = True
        cases.append((x, (w * keep).reshape(M, -1), go, "both", None))
        for which in ("x", "go"):
            x, go = whole_numbers(rng, shape, bits), whole_numbers(rng, shape, other)
            sparse = x if which == "x" else go
            at = np.zeros(shape, bool)
            at[rng.integers(batch, size=C), np.arange(C), rng.integers(32, size=C), rng.integers(width, size=C)] = True
            sparse *= at
            cases.append((x, whole_numbers(rng, (M, C * 9), 1), go, "weight", None))
    return geo, [(x, w, go, what, conv64(x, w, go, geo)) for x, w, go, what, _ in cases]


@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("batch,width", [(2, 8), (2, 9), (1, 8), (1, 9)])
def test_every_part_of_every_element_counts_in_convolution_layers(gt, gathered_route, switches, tile, batch, width):
    switches("gemm_tile", tile)
    geo, cases = one_product_layers(batch, width)
    for x, w, go, what, (out, gi, gw) in cases:
        *got, labels = conv(gt, x, w, go, geo)
        assert len(labels) == 3 and all("tile=%s " % tile in l for l in labels), labels
        if what == "both":
            assert np.array_equal(got[0], out) and np.array_equal(got[1], gi)
        else:
            assert np.array_equal(got[2].reshape(gw.shape), gw)


def same(got, ref):
    """Equal, NaN where the reference is NaN."""
    ref = ref.astype(np.float32)
    return np.array_equal(np.isnan(got), np.isnan(ref)) and np.array_equal(got[~np.isnan(ref)], ref[~np.isnan(ref)])


@pytest.mark.parametrize("split", [1, 2])
@pytest.mark.parametrize("ta,tb", [("n", "n"), ("n", "t"), ("t", "n"), ("t", "t")])
def test_values_the_parts_cannot_hold_in_every_layout(gt, switches, ta, tb, split):
    """As above, whole numbers elsewhere, in either operand and in the second part of a split reduction."""
    switches("gemm_split", split)
    m, n, k = 131, 135, 261
    rng = rng_for(308)
    for swap in (False, True):
        P = rng.integers(-2, 3, size=(m, k)).astype(np.float32)
        Q = rng.integers(-1, 2, size=(k, n)).astype(np.float32)
        P[0, 0], P[1, k - 1], P[m - 1, 3], P[70, 200], P[100, 140] = np.inf, -np.inf, np.nan, 3.4e38, np.inf
        A, B = (Q.T, P.T) if swap else (P, Q)
        with np.errstate(all="ignore"):
            ref = (A.astype(np.float64) @ B.astype(np.float64))
        got, labels = blas(gt, ta, tb, A, B)
        assert len(labels) == 1 and "split=%d" % split in labels[0] and "generic" not in labels[0], labels
        assert same(got, ref), swap


@pytest.mark.parametrize("mode", [0, 2])
@pytest.mark.parametrize("batch,width", [(2, 8), (2, 9), (1, 8), (1, 9)])
def test_values_the_parts_cannot_hold_in_convolution_layers(gt, batch, width, mode):
    """Infinities, NaN and numbers that round to infinity in the input, the weights and gradOutput, on the column and the
    gathered route.  (gradInput of such weights is not compared: beyond the edge of gradOutput the routes
    multiply a weight with a padding zero or not at all.)"""
    rng = rng_for(309)
    C = M = 64
    shape, geo = (batch, C, 12, width), (3, 3, 1, 1, 1, 1)
    lib = gt._lib.lib
    before = lib.thgpu_conv_get_mode()
    assert lib.thgpu_conv_set_mode(mode) == 0
    try:
        for which in ("x", "w", "go"):
            x, go = (rng.integers(-1, 2, size=shape).astype(np.float32) for _ in range(2))
            w = rng.integers(-1, 2, size=(M, C * 9)).astype(np.float32)
            to = {"x": x, "w": w, "go": go}[which].reshape(-1)
            for value in (np.inf, -np.inf, np.nan, 3.4e38):
                to[rng.integers(to.size)] = value
            with np.errstate(all="ignore"):
                out, gi, gw = conv64(x, w, go, geo)
            *got, labels = conv(gt, x, w, go, geo)
            assert len(labels) == 3 and not any("generic" in l for l in labels), labels
            assert same(got[0], out), which
            assert same(got[2].reshape(gw.shape), gw), which
            if which != "w":
                assert same(got[1], gi), which
    finally:
        assert lib.thgpu_conv_set_mode(before) == 0
