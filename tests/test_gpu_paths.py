"""Edges of the kernels and host paths that the size rules choose between, against the CPU
oracle bit for bit.  Everything goes through libxnor_nn.so."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_boundary import make, same_bits, second_table
from test_gpu_parity import run_and_compare
from util import oracle_shape
from xnor_nn_amd import capi, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("separate_k", [False, True])
@pytest.mark.parametrize("where", ["device", "asked", "host"])
def test_forward_pass_in_one_call(oracle, gpu, where, separate_k):
    """xnor_nn_hip_forward_pass: the three stages in one call, on a table whose K plane another
    call still owes, with a second table waiting for the same mean|x| plane."""
    import torch
    d, x1, w = synth.make_workload("alexnet_conv4_mb256", 3)
    x2 = (x1[::-1] * np.float32(-0.5)).copy()
    s = oracle_shape(oracle, d)
    want = oracle.forward(s, x2, w)
    owed = oracle.forward(s, x1, w)["k"]
    wt, x1t, x2t = (torch.from_numpy(v).to(gpu) for v in (w, x1, x2))
    conv = make(d, wt)
    other = second_table(conv, wt)
    own_a = other[capi.RES_A]
    try:
        other[capi.RES_A] = conv.res[capi.RES_A]
        for res in (other, conv.res): # both K planes are owed from x1's mean|x|
            res[capi.RES_USER_SRC] = x1t.data_ptr()
            assert conv.desc.binarize_data(C.byref(conv.desc), res) == capi.SUCCESS
            assert conv.desc.calculate_k(C.byref(conv.desc), res) == capi.SUCCESS
        conv.set_stage_fusion(not separate_k)
        if where == "host":
            dst = np.full(want["dst"].shape, np.nan, np.float32)
            conv.forward(x2, dst)
        else:
            yt = torch.full(want["dst"].shape, float("nan"), device=gpu)
            torch.cuda.synchronize()
            if where == "device":
                side = torch.cuda.Stream()
                conv.forward_on_stream(x2t, yt, side.cuda_stream)
            else:
                conv.forward(x2t.data_ptr(), yt.data_ptr())
            conv.synchronize()
            dst = yt.cpu().numpy()
        assert conv.res[capi.RES_USER_SRC] is None and conv.res[capi.RES_USER_DST] is None
        assert same_bits(dst, want["dst"])
        assert same_bits(conv.export_floats(capi.RES_A), want["a"])
        assert same_bits(conv.export_floats(capi.RES_K), want["k"])
        got = np.empty(owed.shape, np.float32)
        assert conv.lib.xnor_nn_hip_export_floats(C.byref(conv.desc), other, capi.RES_K,
                                                  got.ctypes.data, got.nbytes) == capi.SUCCESS
        assert same_bits(got, owed)
    finally:
        other[capi.RES_A] = own_a
        conv.lib.xnor_nn_free_resources(other)
        conv.close()


def problem(t, zeros=False):
    """Dimensions and synthetic tensors (NCHW, OIHW) of
    (mb, ic, oc, ih, iw, kh, kw, sh, sw, ph, pw)."""
    d = dict(zip(("mb", "ic", "oc", "ih", "iw", "kh", "kw", "sh", "sw", "ph", "pw"), t))
    x = synth.normal(77, d["mb"] * d["ic"] * d["ih"] * d["iw"])
    if zeros:
        x[synth.zero_mask(5, x.size, 3)] = np.float32(0)
    w = synth.normal(78, d["oc"] * d["ic"] * d["kh"] * d["kw"], 0.05)
    return d, x.reshape(d["mb"], d["ic"], d["ih"], d["iw"]), \
        w.reshape(d["oc"], d["ic"], d["kh"], d["kw"])


def in_layout(x, w, fmts):
    if fmts[0] == capi.FMT_NHWC:
        x = np.ascontiguousarray(x.transpose(0, 2, 3, 1))
    if fmts[1] == capi.FMT_HWIO:
        w = np.ascontiguousarray(w.transpose(2, 3, 1, 0))
    return x, w


NCHW = (capi.FMT_NCHW, capi.FMT_OIHW, capi.FMT_NCHW)
NHWC = (capi.FMT_NHWC, capi.FMT_HWIO, capi.FMT_NHWC)


@pytest.mark.parametrize("fmts,separate_k", [(NCHW, False), (NCHW, True), (NHWC, False)])
@pytest.mark.parametrize("t", [
    (1, 1, 1, 5, 5, 5, 5, 1, 1, 0, 0),       # one pixel, one filter
    (3, 1, 32, 28, 28, 5, 5, 1, 1, 0, 0),    # a byte of codes per kernel row
    (2, 3, 96, 61, 61, 11, 11, 4, 4, 0, 0),  # 33 products per kernel row
    (2, 16, 33, 9, 11, 5, 5, 1, 1, 2, 2),    # dword-aligned rows, filters past a block
    (5, 5, 70, 13, 13, 7, 7, 2, 2, 3, 3),    # uneven shifts, a tile's worth minus some
    (3, 11, 6, 7, 5, 5, 4, 1, 2, 2, 2),      # kernel nearly as large as the image, uneven
    (2, 8, 130, 10, 10, 7, 7, 1, 1, 3, 3),   # filters over several workgroups
    (3, 2, 8, 183, 183, 3, 3, 1, 1, 1, 1),   # tiles of 128 pixels, one step
    (12, 3, 32, 150, 150, 9, 9, 1, 1, 4, 4), # tiles of 128 pixels, eight waves
    (2, 16, 64, 40, 150, 9, 9, 1, 1, 4, 4),  # more than 64 KB of LDS
    (1, 16, 24, 20, 1600, 13, 13, 1, 1, 6, 6), # rows too many for the LDS: another kernel
], ids=str)
def test_few_channels(oracle, monkeypatch, t, fmts, separate_k):
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    run_and_compare(oracle, d, *in_layout(x, w, fmts), fmts)
