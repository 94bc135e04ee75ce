"""Operators that stand for several launches: parameter updates of many tensors at once, nn.Linear's bias in the store of
its product and its bias gradient as one sum, the one-launch bias gradient of small convolution layers."""
import ctypes

import numpy as np
import pytest

from helpers import rng_for, uniform

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gt():
    import mcw_cppamp_torch_amd as pkg
    assert pkg._lib.lib.thgpu_init() == 0
    return pkg


def dev(gt, a):
    return gt.FloatTensor(np.ascontiguousarray(a, np.float32)).gpu()


def pointers(gt, tensors):
    return (gt._lib.TensorP * len(tensors))(*[t._p for t in tensors])


# ends of chunks, of 16-byte units and of a launch's 32 entries; offset 1 makes a pair unaligned
@pytest.mark.parametrize("sizes,offset", [([1, 3, 4095, 4096, 4097, 12289], 0), ([4096, 8192, 5], 1), ([7] * 33 + [4096], 0)])
def test_axpy_many_equals_add_bit_for_bit(gt, sizes, offset):
    rng = rng_for(401)
    hosts = [(rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32)) for n in sizes]
    place = lambda a: dev(gt, np.concatenate([np.full(offset, 9, np.float32), a])).narrow(0, offset, a.size)
    ys, xs = [place(y) for y, _ in hosts], [place(x) for _, x in hosts]
    gt._lib.check_status(gt._lib.lib.thgpu_axpy_many(pointers(gt, ys), pointers(gt, xs), len(ys), -0.37))
    for (y, x), got in zip(hosts, ys):
        assert np.array_equal(got.float(), y + np.float32(-0.37) * x)


def test_axpy_many_updates_a_shared_tensor_once_per_pair_and_rejects_bad_pairs(gt):
    rng = rng_for(402)
    y, a, b = (rng.integers(-8, 9, size=5000).astype(np.float32) for _ in range(3))
    dy, da, db = dev(gt, y), dev(gt, a), dev(gt, b)
    lib = gt._lib.lib
    assert lib.thgpu_axpy_many(pointers(gt, [dy, dy]), pointers(gt, [da, db]), 2, 2.0) == 0
    assert np.array_equal(dy.float(), y + 2 * a + 2 * b)
    short = dev(gt, b[:4])
    assert lib.thgpu_axpy_many(pointers(gt, [da, dy]), pointers(gt, [db, short]), 2, 1.0) != 0
    assert b"sizes" in lib.thgpu_last_error() and np.array_equal(da.float(), a)


# batch, inputs, outputs: below a tile (split and not), a tile and its edges, split tiles
@pytest.mark.parametrize("batch,inputs,outputs", [(1, 5, 2), (3, 4096, 10), (50, 300, 128), (64, 64, 64), (65, 130, 200),
                                                  (128, 2049, 333)])
def test_linear_integer_exact(gt, batch, inputs, outputs):
    rng = rng_for(403)
    ints = lambda *s: rng.integers(-3, 4, size=s).astype(np.float32)
    x, w, b, go = ints(batch, inputs), ints(outputs, inputs), ints(outputs), ints(batch, outputs)
    m = gt.nn.Linear(inputs, outputs)
    m._assign("weight", w)
    m._assign("bias", b)
    m.gradBias[...] = 1
    m.gpu()
    assert np.array_equal(m.forward(dev(gt, x)).float(), x @ w.T + b)
    m.accGradParameters(dev(gt, x), dev(gt, go), 2.0)
    assert np.array_equal(m.gradBias.float(), 1 + 2 * go.sum(0))
    wide = dev(gt, np.concatenate([x, x], 1)).narrow(1, 0, inputs)  # rows apart: the tensor library's own sequence
    assert np.array_equal(m.forward(wide).float(), x @ w.T + b)


@pytest.mark.parametrize("n", [2, 40, 300])
def test_axpy_many_finds_shared_memory_among_many_pairs(gt, n):
    """Results that meet one another or another pair's operand are updated in the order given: a pair's operand is another
    pair's result, results overlap by one element, and (not shared) an operand is its own pair's result."""
    rng = rng_for(405)
    host = rng.integers(-8, 9, size=40 * n).astype(np.float32)
    order = rng.permutation(n)
    for kind in ("operand", "overlap", "own", "apart"):
        whole, other = dev(gt, host), dev(gt, host[::-1])
        y0, x0 = host.copy(), host[::-1].copy()
        begin = [int(40 * i) for i in order]
        ys, xs = [whole.narrow(0, b, 40) for b in begin], [other.narrow(0, b, 40) for b in begin]
        hy, hx = [y0[b:b + 40] for b in begin], [x0[b:b + 40] for b in begin]
        if kind == "operand":
            xs[0], hx[0] = ys[n - 1], hy[n - 1]
        elif kind == "overlap":
            c = begin[n - 1] - 1 if begin[n - 1] > 0 else 1
            ys[n - 1], hy[n - 1] = whole.narrow(0, c, 40), y0[c:c + 40]
        elif kind == "own":
            xs[n - 1], hx[n - 1] = ys[n - 1], hy[n - 1]
        gt._lib.check_status(gt._lib.lib.thgpu_axpy_many(pointers(gt, ys), pointers(gt, xs), n, 2.0))
        for y, x in zip(hy, hx):
            y += 2 * x
        assert np.array_equal(whole.float(), y0), kind


def test_axpy_many_host_time_grows_with_the_number_of_pairs(gt):
    """Ten times the pairs take about ten times as long on the host (all pairs against all: a hundred)."""
    import time
    took = {}
    for n in (300, 3000):
        whole, other = gt.GPUTensor(8 * n).fill(1), gt.GPUTensor(8 * n).fill(1)
        pairs = [(whole.narrow(0, 8 * i, 8), other.narrow(0, 8 * i, 8)) for i in range(n)]
        ys, xs = pointers(gt, [y for y, _ in pairs]), pointers(gt, [x for _, x in pairs])
        times = []
        for _ in range(7):
            gt.gputorch.synchronize()
            start = time.perf_counter()
            assert gt._lib.lib.thgpu_axpy_many(ys, xs, n, 0.5) == 0
            times.append(time.perf_counter() - start)
        took[n] = min(times)
    assert took[3000] < 40 * took[300], took


def test_linear_gradients_with_scale_zero_stay_as_they_are(gt):
    m = gt.nn.Linear(7, 5)
    m.gradBias[...] = 3
    m.gradWeight[...] = 2
    m.gpu()
    go = np.full((4, 5), np.nan, np.float32)
    m.accGradParameters(dev(gt, np.full((4, 7), np.inf, np.float32)), dev(gt, go), 0.0)
    assert np.all(m.gradBias.float() == 3) and np.all(m.gradWeight.float() == 2)


def test_linear_bias_gradient_of_more_columns_than_a_launch_has_threads_for(gt):
    n = (1 << 28) + 70  # 64 columns to a workgroup of 1024: 2^32 threads and more
    go, gb = gt.GPUTensor(1, n).fill(2), gt.GPUTensor(n).fill(1)
    gt._lib.check_status(gt._lib.lib.thgpu_Linear_accGradBias(go._p, gb._p, 0.5))
    for at in (0, 1 << 27, n - 200):
        assert np.all(gb.narrow(0, at, 200).float() == 2), at


@pytest.mark.parametrize("batch,side", [(1, 1), (3, 7), (4, 64), (5, 64)])  # 5 * 64 * 64 > 16384: two stages
def test_bias_gradient_of_a_small_layer(gt, batch, side):
    rng = rng_for(404)
    m = gt.nn.SpatialConvolutionMM(2, 5, 1, 1)
    m.gradBias[...] = 3
    m.gpu()
    x, go = (rng.integers(-3, 4, size=(batch, c, side, side)).astype(np.float32) for c in (2, 5))
    m.forward(dev(gt, x))
    m.accGradParameters(dev(gt, x), dev(gt, go), 0.5)
    assert np.array_equal(m.gradBias.float(), 3 + 0.5 * go.sum((0, 2, 3)))


def test_bias_gradient_of_one_launch_allocates_nothing(gt):
    """A layer whose gradients take one launch each must not set up scratch memory: counted in a fresh process, whose
    library has none yet."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    code = """
import numpy as np, mcw_cppamp_torch_amd as gt
lib = gt._lib.lib
m = gt.nn.SpatialConvolutionMM(2, 5, 1, 1).gpu()
x, go = gt.GPUTensor(1, 2, 7, 7).fill(1), gt.GPUTensor(1, 5, 7, 7).fill(2)
m.forward(x)
gt.gputorch.synchronize()
before = lib.thgpu_device_alloc_calls()
m.accGradParameters(x, go, 1)
gt.gputorch.synchronize()
print("allocations", lib.thgpu_device_alloc_calls() - before)
"""
    out = subprocess.run([sys.executable, "-c", code], cwd=root, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True,
                         timeout=100)
    assert out.stdout.splitlines()[-1:] == ["allocations 0"], out.stdout


BACKWARD = {  # B, C, H, W, M, kH, kW, pH, pW, sH, sW
    "one_image": (1, 96, 13, 13, 70, 3, 3, 1, 1, 1, 1),       # 96 planes do not fill 64-row tiles: gradInput on columns
    "groups": (1, 128, 13, 13, 70, 3, 3, 1, 1, 1, 1),         # both products on the tile of four groups, both split
    "quads": (2, 64, 8, 12, 64, 3, 3, 1, 1, 1, 1),
    "few_rows": (3, 64, 10, 9, 20, 3, 3, 1, 1, 1, 1),
    "no_padding": (2, 64, 9, 9, 64, 3, 3, 0, 0, 1, 1),
    "strided": (2, 20, 17, 19, 66, 5, 5, 2, 2, 2, 2),
    "wide": (16, 64, 28, 28, 192, 3, 3, 1, 1, 1, 1),
    "columns": (2, 3, 12, 12, 64, 5, 5, 1, 1, 1, 1),          # gradInput of three planes goes through columns
}


@pytest.mark.parametrize("threshold", [None, 0.25])
@pytest.mark.parametrize("name", sorted(BACKWARD))
def test_backward_gives_what_its_two_passes_give(gt, name, threshold):
    """One call of the library for both passes against one after the other, bit for bit, twice (buffers new and kept)."""
    B, C, H, W, M, kH, kW, pH, pW, sH, sW = BACKWARD[name]
    rng = rng_for(405)
    made = []
    for _ in range(2):
        m = gt.nn.SpatialConvolutionMM(C, M, kW, kH, sW, sH, 0, padW=pW, padH=pH, rng=rng_for(406))
        m.gradWeight[...] = 0.5
        m.gradBias[...] = -0.5
        m.inputThreshold = threshold
        made.append(m.gpu())
    for _ in range(2):
        x = dev(gt, uniform(rng, (B, C, H, W)))
        outs = []
        for i, m in enumerate(made):
            o = m.forward(x)
            if i == 0:
                go = dev(gt, uniform(rng, o.size()))
                gi = m.backward(x, go, 0.75)
            else:
                gi = m.updateGradInput(x, go)
                m.accGradParameters(x, go, 0.75)
            outs.append([t.float() for t in (gi, m.gradWeight, m.gradBias)])
        for a, b in zip(*outs):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32))


def launches(gt, call):
    """{label's family: calls} of what a call enqueues."""
    gt.gputorch.synchronize()
    gt.gputorch.prof_reset()
    gt.gputorch.prof_enable(True)
    try:
        call()
        gt.gputorch.synchronize()
        found = {}
        for label, r in gt.gputorch.prof_report().items():
            family = label.split(" ")[0]
            found[family] = found.get(family, 0) + r["calls"]
        return found
    finally:
        gt.gputorch.prof_enable(False)
        gt.gputorch.prof_reset()


# name -> what one call enqueues and what the two passes do
_TWO = {"gemm_conv_gradinput": 1, "gemm_conv_gradweight": 1}
SHARED = {
    "groups": ({"pad_planes": 1, "gemm_conv_backward": 1, "gemm_split_reduce": 1}, {"pad_planes": 2, "gemm_split_reduce": 2, **_TWO}),
    "quads": ({"pad_planes": 1, "gemm_conv_backward": 1, "gemm_split_reduce": 1}, {"pad_planes": 2, "gemm_split_reduce": 2, **_TWO}),
    "no_padding": ({"pad_planes": 1, "gemm_conv_backward": 1, "gemm_split_reduce": 1}, {"pad_planes": 1, "gemm_split_reduce": 2, **_TWO}),
    "wide": ({"pad_planes": 1, "gemm_split_reduce": 1, **_TWO}, {"pad_planes": 2, "gemm_split_reduce": 2, **_TWO}),
    "columns": (None, None),
}


@pytest.mark.parametrize("name", sorted(SHARED))
def test_backward_shares_launches(gt, name):
    """What per-kernel timing sees is what runs without it, and where both products gather it is fewer launches than two passes
    make; a layer with columns in one of them makes the same."""
    B, C, H, W, M, kH, kW, pH, pW, sH, sW = BACKWARD[name]
    rng = rng_for(419)
    m = gt.nn.SpatialConvolutionMM(C, M, kW, kH, sW, sH, 0, padW=pW, padH=pH, rng=rng_for(420)).gpu()
    x = dev(gt, uniform(rng, (B, C, H, W)))
    go = dev(gt, uniform(rng, m.forward(x).size()))
    for _ in range(2):
        shared = launches(gt, lambda: m.backward(x, go))
        apart = launches(gt, lambda: (m.updateGradInput(x, go), m.accGradParameters(x, go)))
    print(name, shared, apart)
    want = SHARED[name]
    if want[0] is None:
        assert shared == apart and "col2im" in shared
    else:
        assert (shared, apart) == want


def test_backward_with_shared_or_strided_tensors(gt):
    """What the shared launches cannot take runs one pass after the other: a transposed gradOutput, a gradInput in the memory
    of the input, one buffer for finput and fgradInput, a class with its own updateGradInput."""
    B, C, H, W, M = 1, 64, 10, 10, 64
    rng = rng_for(407)
    x, go = uniform(rng, (B, C, H, W)), uniform(rng, (B, M, H, W))

    def module(cls=gt.nn.SpatialConvolutionMM):
        m = cls(C, M, 3, 3, 1, 1, 1, rng=rng_for(408))
        m.gradWeight[...] = 0
        m.gradBias[...] = 0
        return m.gpu()

    def results(m, dx, dgo, call):
        m.forward(dx)
        call(m, dx, dgo)
        return [t.float() for t in (m.gradInput, m.gradWeight, m.gradBias)]

    def passes(m, dx, dgo):
        m.updateGradInput(dx, dgo)
        m.accGradParameters(dx, dgo, 1)

    merged = lambda m, dx, dgo: m.backward(dx, dgo)
    ref = results(module(), dev(gt, x), dev(gt, go), passes)
    swapped = dev(gt, np.ascontiguousarray(go.transpose(0, 1, 3, 2))).transpose(2, 3)
    assert not swapped.isContiguous()
    assert all(np.array_equal(a, b) for a, b in zip(results(module(), dev(gt, x), swapped, merged), ref))
    one = module()
    one.fgradInput = one.finput
    assert all(np.array_equal(a, b) for a, b in zip(results(one, dev(gt, x), dev(gt, go), merged), ref))
    pair = []
    for call in (passes, merged):  # gradInput over the input: accGradParameters sees the gradient, as it did
        m, dx = module(), dev(gt, x)
        m.gradInput = dx
        pair.append(results(m, dx, dev(gt, go), call))
    assert all(np.array_equal(a, b) for a, b in zip(*pair))

    class Halved(gt.nn.SpatialConvolutionMM):
        def updateGradInput(self, input, gradOutput):
            return gt.nn.SpatialConvolutionMM.updateGradInput(self, input, gradOutput).mul(0.5)

    got = results(module(Halved), dev(gt, x), dev(gt, go), merged)
    assert np.array_equal(got[0], 0.5 * ref[0]) and np.array_equal(got[1], ref[1])


@pytest.mark.parametrize("shared", ["finput in the weight's memory", "second copy in gradOutput's memory"])
def test_backward_with_a_buffer_that_the_other_pass_reads(gt, shared):
    """Where one pass writes what the other reads, the two run in their order: gradInput is of the weight as it was, gradWeight
    of the gradOutput that the store of gradInput left."""
    lib, rng = gt._lib.lib, rng_for(421)
    x, go = uniform(rng, (1, 64, 10, 10)), uniform(rng, (1, 64, 10, 10))
    got = []
    for merged in (True, False):
        m = gt.nn.SpatialConvolutionMM(64, 64, 3, 3, 1, 1, 1, rng=rng_for(422)).gpu()
        m.zeroGradParameters()
        dx, dgo, twin = dev(gt, x), dev(gt, go), None
        m.forward(dx)
        if shared.startswith("finput"):
            m.finput = gt.GPUTensor().set(m.weight)
        else:
            twin = gt.GPUTensor().set(dgo)
        if merged:
            gt._lib.check_status(lib.thgpu_SpatialConvolutionMM_backward(
                dx._p, dgo._p, m.weight._p, m.gradWeight._p, m.gradBias._p, m.finput._p, m.fgradInput._p, m.gradInput._p,
                *(m._geom() + (1.0, 0, 0.0, twin._p if twin is not None else None, None))))
        else:
            m._updateGradInputTwin(dx, dgo, twin, False)
            m.accGradParameters(dx, dgo, 1)
        got.append([t.float() for t in (m.gradInput, m.gradWeight, m.gradBias)])
    assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(*got))


def test_backward_calls_a_pass_that_replaces_the_class_own(gt, monkeypatch):
    conv, seen = gt.nn.SpatialConvolutionMM, []
    for name in ("updateGradInput", "accGradParameters"):
        own = getattr(conv, name)
        monkeypatch.setattr(conv, name, lambda self, *args, own=own, name=name: (seen.append(name), own(self, *args))[1])
        m = conv(3, 64, 3, 3, 1, 1, 1).gpu()
        x = gt.GPUTensor(1, 3, 9, 9).fill(1)
        m.backward(x, m.forward(x))
        assert seen == (["updateGradInput"] if name == "updateGradInput" else ["updateGradInput", "updateGradInput", name])


@pytest.mark.parametrize("case", ["fused", "plain", "derived module"])
def test_container_backward_gives_what_its_two_passes_give(gt, case):
    """Against updateGradInput and then accGradParameters of the whole container, bit for bit."""
    nn = gt.nn

    class Noted(nn.ReLU):  # of another file
        def accGradParameters(self, input, gradOutput, scale=1):
            seen.append("accGradParameters")

        def updateGradInput(self, input, gradOutput):
            seen.append("updateGradInput")
            return nn.ReLU.updateGradInput(self, input, gradOutput)

    seen = []

    def stack():
        rng = rng_for(409)
        mods = [nn.SpatialConvolutionMM(3, 64, 5, 5, 2, 2, 2, rng=rng), nn.ReLU(), nn.SpatialMaxPooling(3, 3, 2, 2),
                nn.SpatialConvolutionMM(64, 96, 3, 3, 1, 1, 1, rng=rng), Noted() if case == "derived module" else nn.ReLU(),
                nn.SpatialConvolutionMM(96, 64, 3, 3, 1, 1, 1, rng=rng), nn.ReLU(),
                nn.SpatialMaxPooling(2, 2), nn.View(64 * 7 * 7), nn.Linear(64 * 7 * 7, 20, rng=rng), nn.LogSoftMax()]
        net = nn.Sequential()
        for m in mods:
            net.add(m)
        net.gpu()
        return net.fuse() if case == "fused" else net

    rng = rng_for(410)
    nets = [stack(), stack()]
    for _ in range(2):
        x, go = dev(gt, uniform(rng, (2, 3, 57, 57))), dev(gt, uniform(rng, (2, 20)))
        got = []
        for i, net in enumerate(nets):
            net.zeroGradParameters()
            net.forward(x)
            if i == 0:
                net.backward(x, go, 0.5)
            else:
                net.updateGradInput(x, go)
                net.accGradParameters(x, go, 0.5)
            got.append([net.gradInput.float()] + [g.float() for g in net.parameters()[1]])
        assert all(np.array_equal(a.view(np.uint32), b.view(np.uint32)) for a, b in zip(*got))
    assert seen == (["updateGradInput", "accGradParameters"] * 4 if case == "derived module" else [])


@pytest.mark.parametrize("where", ["outer", "nested"])
def test_container_backward_keeps_the_order_of_its_passes(gt, where):
    """gradInput of every module before the first accGradParameters, nested containers included: a module that changes its
    gradInput while it accumulates does not change what the modules in front of it receive."""
    nn = gt.nn

    class Cleared(nn.ReLU):
        def accGradParameters(self, input, gradOutput, scale=1):
            self.gradInput.zero()

    def stack(cls):
        rng = rng_for(412)
        net = nn.Sequential().add(nn.SpatialConvolutionMM(3, 64, 3, 3, 1, 1, 1, rng=rng))
        tail = [cls(), nn.View(64 * 36), nn.Linear(64 * 36, 5, rng=rng)]
        if where == "nested":
            inner = nn.Sequential()
            for m in tail:
                inner.add(m)
            net.add(inner)
        else:
            for m in tail:
                net.add(m)
        return net.gpu()

    rng = rng_for(413)
    x, go = dev(gt, uniform(rng, (2, 3, 6, 6))), dev(gt, uniform(rng, (2, 5)))
    got = []
    for cls in (Cleared, nn.ReLU):
        net = stack(cls)
        net.zeroGradParameters()
        net.forward(x)
        got.append(net.backward(x, go).float())
    assert np.any(got[1] != 0) and np.array_equal(got[0], got[1])


def test_container_backward_that_fails_accumulates_nothing(gt):
    """The first module meets an input of another size when every module behind it has its gradInput."""
    nn = gt.nn
    net = nn.Sequential().add(nn.SpatialConvolutionMM(3, 64, 3, 3, 1, 1, 1)).add(nn.ReLU())
    net.add(nn.SpatialConvolutionMM(64, 64, 3, 3, 1, 1, 1)).gpu()
    rng = rng_for(414)
    x, go = dev(gt, uniform(rng, (2, 3, 9, 9))), dev(gt, uniform(rng, (2, 64, 9, 9)))
    net.zeroGradParameters()
    net.forward(x)
    with pytest.raises(gt._lib.THGPUError):
        net.backward(dev(gt, uniform(rng, (2, 3, 8, 9))), go)
    assert all(np.all(g.float() == 0) for g in net.parameters()[1])
    net.backward(x, go)
    assert all(np.any(g.float() != 0) for g in net.parameters()[1])


def test_backward_with_a_second_copy_of_gradinput(gt):
    """thgpu_SpatialConvolutionMM_backward between two convolutions, as a caller that walks back module by module has it: gradOutput
    already in the layer's padded buffer, gradInput stored in the next one's too, against the two calls, bit for bit."""
    lib, nn = gt._lib.lib, gt.nn
    rng = rng_for(415)
    x, go = dev(gt, uniform(rng, (2, 64, 9, 9))), dev(gt, uniform(rng, (2, 64, 9, 9)))
    got = []
    for merged in (True, False):
        front = nn.SpatialConvolutionMM(64, 64, 3, 3, 1, 1, 1, rng=rng_for(416)).gpu()
        behind = nn.SpatialConvolutionMM(64, 64, 3, 3, 1, 1, 1, rng=rng_for(417)).gpu()
        for _ in range(2):
            behind.zeroGradParameters()
            mid = front.forward(x)
            behind.forward(mid)
            twin = front._gradOutputTwin(x)
            if merged:
                wrote = ctypes.c_int(-1)
                gt._lib.check_status(lib.thgpu_SpatialConvolutionMM_backward(
                    mid._p, go._p, behind.weight._p, behind.gradWeight._p, behind.gradBias._p, behind.finput._p,
                    behind.fgradInput._p, behind.gradInput._p, *(behind._geom() + (1.0, 0, 0.0, twin._p if twin is not None else None,
                                                                                  ctypes.byref(wrote)))))
                stored = wrote.value
            else:
                behind._updateGradInputTwin(mid, go, twin, False)
                stored = int(behind._wrote_twin)
                behind.accGradParameters(mid, go, 1)
            gi = front._updateGradInputTwin(x, behind.gradInput, None, stored == 1)
            got.append([stored] + [t.float() for t in (gi, behind.gradInput, behind.gradWeight, behind.gradBias)])
    for a, b in ((got[0], got[2]), (got[1], got[3])):
        assert a[0] == b[0] and all(np.array_equal(u.view(np.uint32), v.view(np.uint32)) for u, v in zip(a[1:], b[1:]))
    assert got[1][0] == 1


@pytest.mark.parametrize("shape,targets", [((1,), [1]), ((7,), [7]), ((3, 5), [0, 5, 6]), ((130, 3), None), ((2, 1000), [1000, 1])])
def test_criterion_gradient_of_one_launch(gt, shape, targets):
    """Every element, whatever gradInput held; targets outside 1..n are skipped."""
    frames, n = (shape if len(shape) == 2 else (1,) + shape)
    t = np.array(targets if targets is not None else rng_for(411).integers(1, n + 1, size=frames), np.float32)
    c = gt.nn.ClassNLLCriterion().gpu()
    c.gradInput = gt.GPUTensor(frames + 1, n).fill(np.nan)
    got = c.backward(gt.GPUTensor(*shape).fill(0), dev(gt, t)).float()
    ref = np.zeros((frames, n), np.float32)
    for i, k in enumerate(t.astype(int)):
        if 1 <= k <= n:
            ref[i, k - 1] = -1.0 / frames if len(shape) == 2 else -1.0
    assert np.array_equal(got, ref.reshape(shape))


# elements and targets a frame on either side of the lines between one launch and two
@pytest.mark.parametrize("frames,n,targets,launches", [(50, 10, 1, 1), (128, 1000, 100, 1), (64, 10000, 100, 2), (768, 4096, 1, 1),
                                                       (769, 4096, 1, 2), (1024, 2000, 4, 2), (4096, 1000, 8, 2)])
def test_criterion_gradient_takes_one_launch_where_that_is_less_work(gt, frames, n, targets, launches):
    rng = rng_for(418)
    t = rng.integers(0, n + 2, size=(frames, targets)).astype(np.float32)
    c, x, dt = gt.nn.ClassNLLCriterion().gpu(), gt.GPUTensor(frames, n).fill(0), dev(gt, t)
    c.gradInput = gt.GPUTensor(frames, n).fill(np.nan)
    gt.gputorch.synchronize()
    gt.gputorch.prof_reset()
    gt.gputorch.prof_enable(True)
    try:
        got = c.backward(x, dt)
        gt.gputorch.synchronize()
        report = gt.gputorch.prof_report()
    finally:
        gt.gputorch.prof_enable(False)
        gt.gputorch.prof_reset()
    ref = np.zeros((frames, n + 2), np.float32)
    np.put_along_axis(ref, t.astype(np.int64), np.float32(-1.0 / frames), 1)
    assert np.array_equal(got.float(), ref[:, 1:-1])
    assert sum(r["calls"] for r in report.values()) == launches, report
