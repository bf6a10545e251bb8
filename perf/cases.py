"""Forward passes and weight updates of binary convolution layers, as a user's program makes
them through this package's public entry points.

A case is one layer and the way it is called:

    conv    xnor_nn_amd.Convolution.forward on device tensors, NCHW input and output
    nhwc    the same with NHWC input and output and HWIO weights
    module  xnor_nn_amd.torch_layer.XnorConv2d called on a device tensor (it allocates its output)
    train   one training iteration's share of that module: the weights have been written to, the
            forward pass, and sign(w) * mean(w) for the framework's backward pass
    host    Convolution.forward on host arrays, as a program written for the CPU library calls it
"""
import math

import numpy as np
import torch

from xnor_nn_amd import Convolution, capi
from xnor_nn_amd.torch_layer import XnorConv2d

WEIGHT_SIGMA = 0.05
# What a drawn case may cost at most: the traffic, and the binary operations with channels
# counted in whole 32-bit words, of the largest listed layer.
MOST_BYTES = 420e6
MOST_OPS = 2.4e11
MOST_HOST_BYTES = 32e6


def _case(name, kind, mb, ic, ih, iw, oc, k, stride=1, pad=0, zeros=False):
    return dict(name=name, kind=kind, mb=mb, ic=ic, ih=ih, iw=iw, oc=oc, k=k, stride=stride,
                pad=pad, zeros=zeros)


def listed():
    return [
        # one image at a time: the latency of a layer in an interactive program
        _case("conv4 mb 1", "conv", 1, 384, 13, 13, 256, 3, 1, 1),
        # the benchmark's layer: AlexNet's fourth convolution over a full batch
        _case("conv4 mb 256", "conv", 256, 384, 13, 13, 256, 3, 1, 1),
        # larger kernel, a channel count that is no multiple of 64, a plane of odd size
        _case("conv2 mb 128", "conv", 128, 96, 27, 27, 256, 5, 1, 2),
        # the largest layer: residual block on large planes
        _case("resnet 56 mb 64", "conv", 64, 256, 56, 56, 256, 3, 1, 1),
        # deep layer; its input comes from a rectifier, which leaves zeros
        _case("vgg 512 mb 32", "conv", 32, 512, 28, 28, 512, 3, 1, 1, zeros=True),
        # first layer of an image network: three channels, large strided kernel
        _case("conv1 mb 64", "conv", 64, 3, 227, 227, 96, 11, 4, 0),
        # bottleneck: many channels into few on a small plane, no neighbourhood
        _case("bottleneck 2048 mb 64", "conv", 64, 2048, 7, 7, 512, 1),
        # channels-last program
        _case("nhwc 128 mb 100", "nhwc", 100, 128, 32, 32, 256, 3, 1, 1),
        # a layer of a small image network called from torch
        _case("module 32-64 mb 100", "module", 100, 32, 32, 32, 64, 5, 1, 2),
        # nothing of it is round: an odd batch, plane, channel and filter count, a stride
        _case("module ragged mb 9", "module", 9, 130, 45, 51, 70, 3, 2, 1),
        # training: weights re-binarized on every iteration
        _case("train conv4 mb 64", "train", 64, 384, 13, 13, 256, 3, 1, 1),
        # drop-in use from a program that keeps its tensors in host memory
        _case("host conv4 mb 32", "host", 32, 384, 13, 13, 256, 3, 1, 1),
    ]


def _extent(n, c):
    return (n + 2 * c["pad"] - c["k"]) // c["stride"] + 1


def _in_bounds(n, c):
    """Kernel positions inside the image along one axis, summed over the output positions."""
    return sum(1 for o in range(_extent(n, c)) for t in range(c["k"])
               if 0 <= o * c["stride"] - c["pad"] + t < n)


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _too_much(c):
    w = work(c)
    words = -(-c["ic"] // 32) * 32
    return (w["bytes"] > (MOST_HOST_BYTES if c["kind"] == "host" else MOST_BYTES)
            or w["flops"] * words / c["ic"] > MOST_OPS)


def draw(rng):
    kind = rng.choice(["conv"] * 5 + ["nhwc", "module", "module", "train", "host"])
    k = rng.choice([1, 3, 3, 3, 3, 5, 5, 7, 11])
    stride = 4 if k == 11 else rng.choice([1, 1, 1, 2])
    ih = _log_int(rng, 7, 112) if k < 11 else _log_int(rng, 64, 227)
    iw = ih if rng.random() < 0.6 else max(7, ih + rng.randint(-5, 5))
    ic = _log_int(rng, 3, 2048 if k == 1 else 1024 if k == 3 else 256 if k == 5 else 48)
    oc = _log_int(rng, 16, 768)
    if rng.random() < 0.6:  # most networks' widths are multiples of 16 or 32
        ic = -(-ic // 16) * 16 if ic > 8 else ic
        oc = -(-oc // 32) * 32
    c = _case("", kind, _log_int(rng, 1, 256), ic, ih, iw, oc, k, stride,
              0 if rng.random() < 0.2 or k == 1 else k // 2, rng.random() < 0.3)
    del c["name"]
    c["pad"] = max(c["pad"], -(-max(0, k - min(ih, iw)) // 2))
    while _too_much(c) and c["mb"] > 1:
        c["mb"] = (c["mb"] + 1) // 2
    while _too_much(c):
        key = "oc" if c["oc"] >= c["ic"] else "ic"
        c[key] = (c[key] + 1) // 2
    return c


def _tensor(shape, seed, sigma=1.0, device="cuda"):
    g = torch.Generator(device=device)
    g.manual_seed(seed)
    t = torch.randn(shape, generator=g, device=device, dtype=torch.float32)
    return t.mul_(sigma) if sigma != 1.0 else t


def prepare(case, seed):
    c = dict(case)
    mb, ic, oc, k = c["mb"], c["ic"], c["oc"], c["k"]
    oh, ow = _extent(c["ih"], c), _extent(c["iw"], c)
    channels_last = c["kind"] == "nhwc"
    x_shape = (mb, c["ih"], c["iw"], ic) if channels_last else (mb, ic, c["ih"], c["iw"])
    y_shape = (mb, oh, ow, oc) if channels_last else (mb, oc, oh, ow)
    w_shape = (k, k, ic, oc) if channels_last else (oc, ic, k, k)
    weights = _tensor(w_shape, 2 * seed + 1, WEIGHT_SIGMA)
    if c["kind"] == "host":
        # normal deviates, like the device tensors of the other kinds
        rng = np.random.default_rng(2 * seed)
        x = rng.standard_normal(x_shape, dtype=np.float32)
        if c["zeros"]:
            x = np.maximum(x, np.float32(0))
        weights = weights.cpu().numpy()
        y = np.zeros(y_shape, np.float32)
    else:
        x = _tensor(x_shape, 2 * seed)
        if c["zeros"]:
            x = torch.relu_(x)
        y = None
    if c["kind"] in ("module", "train"):
        layer = XnorConv2d(ic, oc, k, c["stride"], c["pad"], weight=weights)
        return dict(kind=c["kind"], layer=layer, x=x)
    if y is None:
        y = torch.zeros(y_shape, device="cuda", dtype=torch.float32)
    src, wf = ((capi.FMT_NHWC, capi.FMT_HWIO) if channels_last
               else (capi.FMT_NCHW, capi.FMT_OIHW))
    conv = Convolution(capi.ALGORITHM_BCAST, src, wf, src, mb, oc, ic, c["ih"], c["iw"], k, k,
                       c["stride"], c["stride"], c["pad"], c["pad"], weights)
    return dict(kind=c["kind"], conv=conv, x=x, y=y)


def run(state):
    kind = state["kind"]
    if kind == "module":
        return state["layer"](state["x"])
    if kind == "train":
        layer = state["layer"]
        layer.weights_changed()
        y = layer(state["x"])
        return y, layer.binarized_weights()
    state["conv"].forward(state["x"], state["y"])
    return state["y"]


def work(case):
    c = case
    oh, ow = _extent(c["ih"], c), _extent(c["iw"], c)
    weights = c["oc"] * c["ic"] * c["k"] * c["k"]
    # the input once, the output once; an update reads the float weights and writes as many, a
    # plain forward pass needs their signs and one scale per filter only
    bytes_ = 4.0 * c["mb"] * (c["ic"] * c["ih"] * c["iw"] + c["oc"] * oh * ow)
    bytes_ += 8.0 * weights if c["kind"] == "train" else weights / 8.0 + 4.0 * c["oc"]
    # binary multiply-accumulates inside the image, two operations each
    ops = 2.0 * c["mb"] * c["oc"] * c["ic"] * _in_bounds(c["ih"], c) * _in_bounds(c["iw"], c)
    return {"bytes": bytes_, "flops": ops}


def tolerance(case):
    # integer dot products, scaled by means summed in 32 bits
    return {"rel": 1e-5}
