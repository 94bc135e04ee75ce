"""What a user of this framework has it do, as cases that can be timed and compared: convolution stacks trained and
evaluated through nn.Sequential, single nn.SpatialConvolutionMM and nn.SpatialMaxPooling layers forward and backward,
and whole SGD steps with a classifier and a criterion.  Everything is fp32 NCHW on torch.GPUTensor, which is all the
framework computes in.

Kinds of case (the rest of a case's fields are its sizes and options):

  stack       a convolution stack of stacks.STACKS: "train" is zeroGradParameters, forward, backward (updateGradInput
              and accGradParameters of every module); "infer" takes a host batch, moves it with :gpu(), runs forward
              and brings the result back with :float(), as a program that serves requests does
  conv        one nn.SpatialConvolutionMM: zeroGradParameters, forward, backward
  pool        one nn.SpatialMaxPooling: forward, backward
  convnet     an SGD step of conv - ReLU - max-pool - conv - ReLU - sub-sampling - View - Linear - ReLU - Linear -
              LogSoftMax with ClassNLLCriterion (the call order of a Torch trainer), small images
  classifier  an SGD step of Linear - ReLU - Linear - ReLU - Linear - LogSoftMax with ClassNLLCriterion on features
"""
import math

import numpy as np
import torch

import mcw_cppamp_torch_amd as gt
from mcw_cppamp_torch_amd import nn, stacks

LEARNING_RATE = 1e-3


class Outputs(dict):
    """Results of a pass: GPUTensors by name, each handed out as a torch tensor on the same device memory."""

    def __getitem__(self, key):
        value = dict.__getitem__(self, key)
        return _as_torch(value) if isinstance(value, gt.GPUTensor) else value

    def values(self):
        return [self[k] for k in self]

    def items(self):
        return [(k, self[k]) for k in self]


class _Memory:
    """The CUDA array interface of a GPUTensor, which it keeps alive."""

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {
            "shape": tensor.size(), "strides": tuple(4 * s for s in tensor.stride()), "typestr": "<f4",
            "data": (tensor.data_ptr(), False), "version": 2}


def _as_torch(tensor):
    return torch.as_tensor(_Memory(tensor), device="cuda")


def _rng(seed, which):
    return np.random.Generator(np.random.PCG64([int(seed), which]))


def _uniform(rng, shape, bound=1.0):
    # uniform [-bound, bound) in fp32
    return (rng.random(size=shape, dtype=np.float32) * 2 - 1) * np.float32(bound)


# ---- the cases -------------------------------------------------------------------------------------------------------

def _stack(name, net, batch, mode, fused):
    return {"name": name, "kind": "stack", "net": net, "batch": batch, "mode": mode, "fused": fused}


def _conv(name, batch, C, M, kW, kH, dW, dH, padW, padH, W, H):
    return {"name": name, "kind": "conv", "batch": batch, "C": C, "M": M, "kW": kW, "kH": kH, "dW": dW, "dH": dH,
            "padW": padW, "padH": padH, "W": W, "H": H}


def listed():
    return [
        # The smallest call: one 13x13 layer on one image, a handful of launches.
        _conv("conv_one_image", 1, 384, 256, 3, 3, 1, 1, 1, 1, 13, 13),
        # A small image batch through a layer that fits no tile: 37 planes, stride 3, odd sizes.
        _conv("conv_odd_sizes", 5, 3, 37, 5, 5, 3, 3, 0, 0, 77, 101),
        # The usual first layer of an image net at a moderate batch.
        _conv("conv_first_layer", 16, 3, 64, 11, 11, 4, 4, 2, 2, 224, 224),
        # A kernel, stride and padding that differ between the two directions, on images that are not square.
        _conv("conv_not_square", 32, 3, 128, 7, 3, 2, 1, 3, 1, 96, 128),
        # A large kernel without padding: a layer of the framework's own per-layer benchmark.
        _conv("conv_large_kernel", 128, 64, 128, 9, 9, 1, 1, 0, 0, 64, 64),
        # Overlapping windows over activations with many equal values.
        {"name": "pool_overlapping", "kind": "pool", "batch": 128, "C": 256, "W": 27, "H": 27, "k": 3, "d": 2,
         "levels": 8},
        # One request of a program that serves images: host batch in, host features out.
        _stack("alexnet_infer_one", "alexnet", 1, "infer", True),
        # The training step of bench.py at its default batch, ReLUs fused.
        _stack("alexnet_train", "alexnet", 128, "train", True),
        # A stack as nn.Sequential leaves it (nothing fused), on the ragged last batch of an epoch.
        _stack("overfeat_train_ragged", "overfeat", 37, "train", False),
        # The largest step: deep 3x3 layers, large feature maps.
        _stack("vgg_a_train", "vgg_a", 64, "train", True),
        # A whole SGD step of a small net on small images: many short launches.
        {"name": "convnet_sgd", "kind": "convnet", "batch": 50, "planes1": 32, "planes2": 64, "size": 32,
         "hidden": 128, "classes": 10},
        # The three Linear layers behind the AlexNet-style stack, a step at its batch: large weight matrices.
        {"name": "classifier_sgd", "kind": "classifier", "batch": 128, "inputs": 9216, "hidden": 4096,
         "classes": 1000},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _draw_conv(rng):
    while True:
        k = rng.choice([1, 3, 3, 3, 5, 5, 7, 9, 11])
        kH = k if rng.random() < 0.8 else rng.choice([1, 3, 5, 7])
        d = rng.choice([1, 1, 1, 1, 2, 3, 4])
        dH = d if rng.random() < 0.8 else rng.choice([1, 2])
        pad = rng.choice([0, k // 2, k // 2, rng.randint(0, k - 1)])
        padH = min(pad, kH - 1) if kH != k else pad
        C = 3 if rng.random() < 0.2 else _log_int(rng, 4, 512)
        case = _conv("", _log_int(rng, 1, 128), C, _log_int(rng, 8, 512), k, kH, min(d, k), min(dH, kH), pad, padH,
                     _log_int(rng, 7, 128), _log_int(rng, 7, 128))
        del case["name"]
        if case["W"] + 2 * case["padW"] < k or case["H"] + 2 * case["padH"] < kH:
            continue
        Ho, Wo = _conv_out(case)
        columns = case["batch"] * C * k * kH * Ho * Wo
        planes = case["batch"] * max(C * case["W"] * case["H"], case["M"] * Ho * Wo)
        # no more work than the largest listed case, columns and images that fit three times over
        if 6.0 * columns * case["M"] <= 2e12 and columns <= 1 << 29 and planes <= 1 << 26 and Ho * Wo * columns > 0:
            return case


def draw(rng):
    kind = rng.choice(["conv", "conv", "conv", "conv", "stack", "stack", "stack", "pool", "convnet", "classifier"])
    if kind == "conv":
        return _draw_conv(rng)
    if kind == "stack":
        net = rng.choice(["alexnet", "overfeat", "vgg_a"])
        mode = rng.choice(["train", "train", "infer"])
        top = (60 if net == "vgg_a" else 128) if mode == "train" else 32
        return {"kind": "stack", "net": net, "batch": _log_int(rng, 2, top), "mode": mode,
                "fused": rng.random() < 0.6}
    if kind == "pool":
        k = rng.choice([2, 3, 3])
        return {"kind": "pool", "batch": _log_int(rng, 1, 128), "C": _log_int(rng, 16, 512),
                "W": _log_int(rng, 7, 64), "H": _log_int(rng, 7, 64), "k": k, "d": 2,
                "levels": rng.choice([0, 0, 8])}
    if kind == "convnet":
        return {"kind": "convnet", "batch": _log_int(rng, 8, 256), "planes1": 8 * rng.randint(1, 8),
                "planes2": 8 * rng.randint(1, 16), "size": 4 * rng.randint(4, 12), "hidden": _log_int(rng, 32, 512),
                "classes": rng.randint(2, 100)}
    return {"kind": "classifier", "batch": _log_int(rng, 1, 256), "inputs": _log_int(rng, 256, 9216),
            "hidden": _log_int(rng, 128, 4096), "classes": _log_int(rng, 10, 1000)}


# ---- inputs, modules and passes ----------------------------------------------------------------------------------------

def _conv_out(case):
    return ((case["H"] + 2 * case["padH"] - case["kH"]) // case["dH"] + 1,
            (case["W"] + 2 * case["padW"] - case["kW"]) // case["dW"] + 1)


def _pool_out(case):
    return (case["H"] - case["k"]) // case["d"] + 1, (case["W"] - case["k"]) // case["d"] + 1


def _convnet_features(case):
    return case["planes2"] * (case["size"] // 4) ** 2


def prepare(case, seed):
    kind = case["kind"]
    state = {"case": case}
    data = _rng(seed, 0)
    if kind == "stack":
        net = stacks.build(case["net"], seed_base=1000 * (int(seed) % 1000003)).gpu()
        if case["fused"]:
            net.fuse()
        state["net"] = net
        x = gt.FloatTensor(_uniform(data, (case["batch"],) + stacks.STACKS[case["net"]]["input"]))
        if case["mode"] == "infer":
            state["host"] = x
            return state
        state["x"] = x.gpu()
        state["go"] = gt.FloatTensor(_uniform(data, stacks.output_shape(case["net"], case["batch"]))).gpu()
        return state
    if kind == "conv":
        Ho, Wo = _conv_out(case)
        state["net"] = nn.SpatialConvolutionMM(case["C"], case["M"], case["kW"], case["kH"], case["dW"], case["dH"],
                                               padW=case["padW"], padH=case["padH"], rng=_rng(seed, 1)).gpu()
        state["x"] = gt.FloatTensor(_uniform(data, (case["batch"], case["C"], case["H"], case["W"]))).gpu()
        state["go"] = gt.FloatTensor(_uniform(data, (case["batch"], case["M"], Ho, Wo))).gpu()
        return state
    if kind == "pool":
        shape = (case["batch"], case["C"], case["H"], case["W"])
        x = data.integers(0, case["levels"], size=shape).astype(np.float32) if case["levels"] else _uniform(data, shape)
        state["net"] = nn.SpatialMaxPooling(case["k"], case["k"], case["d"], case["d"]).gpu()
        state["x"] = gt.FloatTensor(x).gpu()
        state["go"] = gt.FloatTensor(_uniform(data, shape[:2] + _pool_out(case))).gpu()
        return state
    weights = _rng(seed, 1)
    net = nn.Sequential()
    if kind == "convnet":
        p1, p2 = case["planes1"], case["planes2"]
        modules = [nn.SpatialConvolutionMM(3, p1, 5, 5, 1, 1, 2, rng=weights), nn.ReLU(), nn.SpatialMaxPooling(2, 2),
                   nn.SpatialConvolutionMM(p1, p2, 3, 3, 1, 1, 1, rng=weights), nn.ReLU(),
                   nn.SpatialSubSampling(p2, 2, 2, 2, 2, rng=weights), nn.View(_convnet_features(case)),
                   nn.Linear(_convnet_features(case), case["hidden"], rng=weights), nn.ReLU(),
                   nn.Linear(case["hidden"], case["classes"], rng=weights), nn.LogSoftMax()]
        x = _uniform(data, (case["batch"], 3, case["size"], case["size"]))
    else:
        h = case["hidden"]
        modules = [nn.Linear(case["inputs"], h, rng=weights), nn.ReLU(), nn.Linear(h, h, rng=weights), nn.ReLU(),
                   nn.Linear(h, case["classes"], rng=weights), nn.LogSoftMax()]
        # features behind a ReLU: none negative, about half of them zero
        x = np.maximum(_uniform(data, (case["batch"], case["inputs"])), 0)
    for m in modules:
        net.add(m)
    state["net"] = net.gpu()
    state["criterion"] = nn.ClassNLLCriterion().gpu()
    state["x"] = gt.FloatTensor(x).gpu()
    state["target"] = gt.FloatTensor(data.integers(1, case["classes"] + 1, size=case["batch"])).gpu()
    return state


def _with_gradients(out, net):
    _, grads = net.parameters()
    for i, g in enumerate(grads or []):
        out["grad %d" % i] = g
    return out


def run(state):
    case, net = state["case"], state["net"]
    if case.get("mode") == "infer":
        return net.forward(state["host"].gpu()).float()
    if "criterion" in state:
        criterion, x, target = state["criterion"], state["x"], state["target"]
        loss = criterion.forward(net.forward(x), target)
        net.zeroGradParameters()
        grad_input = net.backward(x, criterion.backward(net.output, target))
        net.updateParameters(LEARNING_RATE)
        params, _ = net.parameters()
        out = Outputs({"weight %d" % i: p for i, p in enumerate(params)})
        out["loss"], out["output"], out["gradInput"] = loss, net.output, grad_input
        return _with_gradients(out, net)
    x, go = state["x"], state["go"]
    if case["kind"] == "pool":
        return Outputs(output=net.forward(x), gradInput=net.backward(x, go), indices=net.indices)
    net.zeroGradParameters()
    output = net.forward(x)
    return _with_gradients(Outputs(output=output, gradInput=net.backward(x, go)), net)


# ---- what a pass cannot do without -------------------------------------------------------------------------------------

def work(case):
    """Each input read once, each result written once; multiply-adds of the convolutions and matrix products, as two
    operations each (three products per layer and training step: forward, gradInput, gradWeight)."""
    kind, B = case["kind"], case["batch"]
    if kind == "stack":
        cfg = stacks.STACKS[case["net"]]
        weights = sum(l[2] * (l[1] * l[3] * l[4] + 1) for l in cfg["layers"] if l[0] == "conv")
        image = int(np.prod(cfg["input"]))
        features = int(np.prod(stacks.output_shape(case["net"], 1)))
        flops = stacks.work(case["net"], B)["gemm_flops"]
        if case["mode"] == "infer":
            return {"bytes": 4.0 * (B * (image + features) + weights), "flops": flops / 3}
        return {"bytes": 4.0 * (2 * B * (image + features) + 2 * weights), "flops": flops}
    if kind == "conv":
        Ho, Wo = _conv_out(case)
        K = case["C"] * case["kW"] * case["kH"]
        planes = case["C"] * case["W"] * case["H"] + case["M"] * Ho * Wo
        return {"bytes": 4.0 * (2 * B * planes + 2 * case["M"] * (K + 1)), "flops": 6.0 * B * case["M"] * K * Ho * Wo}
    if kind == "pool":
        Ho, Wo = _pool_out(case)
        # input, output and both index planes; gradOutput, the index planes again, gradInput
        return {"bytes": 4.0 * B * case["C"] * (2 * case["W"] * case["H"] + 6 * Ho * Wo), "flops": 0.0}
    if kind == "convnet":
        s, p1, p2, h, c = case["size"], case["planes1"], case["planes2"], case["hidden"], case["classes"]
        f = _convnet_features(case)
        weights = p1 * 76 + p2 * (p1 * 9 + 1) + 2 * p2 + h * (f + 1) + c * (h + 1)
        macs = s * s * p1 * 75 + (s // 2) ** 2 * p2 * p1 * 9 + f * h + h * c
        return {"bytes": 4.0 * (2 * B * 3 * s * s + B * c + 3 * weights), "flops": 6.0 * B * macs}
    i, h, c = case["inputs"], case["hidden"], case["classes"]
    weights = h * (i + 1) + h * (h + 1) + c * (h + 1)
    # weights read, gradients written, weights written
    return {"bytes": 4.0 * (2 * B * i + B * c + 3 * weights), "flops": 6.0 * B * (i * h + h * h + h * c)}


def tolerance(case):
    """Four times the difference seen between two orders of summation (column buffers or not, reductions split three
    ways or not) and, for single layers, against the same layer in 64 bits.

    A training pass through ReLUs and max-pools is not continuous: where two activations agree to the last bits, or one
    lies at zero, another order of summation sends a gradient elsewhere.  Of the activations of a stack, of which there
    are up to 300 million, a few do, and its gradients differ by up to 5e-3 in all and 0.5 in one element; without such
    a tie the same gradients agree to 2e-6.  A smaller net meets a tie only now and then, which then weighs 2e-3."""
    if case["kind"] == "pool":
        return "exact"  # a maximum, its place, and sums of at most four gradients in a fixed order
    if case["kind"] == "conv":
        return {"rel": 3e-5, "max": 3e-4}
    if case.get("mode") == "infer":
        return {"rel": 5e-6, "max": 4e-5}
    return {"rel": 2e-2 if case["kind"] == "stack" else 1e-2, "max": 0.99}
