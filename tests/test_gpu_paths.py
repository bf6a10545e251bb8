"""Edges of the kernels and host paths that the size rules choose between, against the CPU
oracle bit for bit.  Everything goes through libxnor_nn.so."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_boundary import make, same_bits, second_table
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
