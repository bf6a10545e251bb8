"""Edges of the kernels and host paths that the size rules choose between, against the CPU
oracle bit for bit.  Everything goes through libxnor_nn.so."""
import ctypes as C

import numpy as np
import pytest

from test_gpu_boundary import make, same_bits, second_table
from test_gpu_parity import run_and_compare
from util import oracle_shape
from xnor_nn_amd import capi, synth
from xnor_nn_amd.convolution import XnorNNError

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


@pytest.mark.parametrize("t", [
    (22, 3, 70, 227, 227, 11, 11, 4, 4, 0, 0),  # mean|x| in the operands' place, eight waves
    (4, 3, 40, 33, 31, 5, 5, 1, 1, 2, 2),       # two bytes of codes per kernel row, rows left over
    (3, 3, 70, 60, 58, 7, 7, 2, 2, 3, 3),       # three
    (2, 4, 9, 40, 37, 7, 7, 1, 1, 3, 3),        # four
    (2, 8, 130, 64, 64, 7, 7, 1, 1, 3, 3),      # seven: stored one by one
    (2, 1, 8, 90, 90, 9, 9, 2, 2, 4, 4),        # a kernel width the sums of K are not unrolled for
    (40, 2, 20, 30, 30, 3, 3, 1, 1, 1, 1),      # 17 pixels reach into a dword of the string
], ids=str)
def test_few_channels_gathering(oracle, t):
    d, x, w = problem(t, zeros=True)
    assert make(d, w).kernel_name(0).startswith("conv_mfma_fp4_shallow_kernel")
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("t", [
    (40, 1, 20, 30, 30, 3, 3, 1, 1, 1, 1),      # a byte a kernel row, rows left over
    (6, 2, 70, 33, 31, 5, 4, 1, 1, 2, 2),
    (9, 5, 40, 90, 90, 6, 6, 4, 4, 2, 2),       # four bytes, stride four, six taps a row
    (9, 6, 40, 24, 22, 7, 7, 1, 1, 3, 3),       # six
    (5, 8, 33, 30, 30, 8, 8, 2, 2, 4, 4),       # eight
    (4, 9, 33, 70, 70, 9, 9, 2, 2, 4, 4),       # eleven
    (12, 10, 20, 40, 40, 7, 7, 1, 1, 3, 3),     # nine
    (12, 10, 20, 40, 40, 8, 8, 1, 1, 3, 3),     # ten
    (12, 12, 20, 40, 40, 8, 8, 1, 1, 4, 4),     # twelve
    (12, 10, 20, 40, 40, 10, 10, 1, 1, 4, 4),   # thirteen
    (12, 11, 20, 40, 40, 10, 10, 1, 1, 4, 4),   # fourteen
    (12, 10, 20, 40, 40, 12, 12, 1, 1, 5, 5),   # fifteen
    (12, 11, 20, 40, 40, 11, 11, 1, 1, 5, 5),   # sixteen
    (12, 10, 20, 40, 40, 13, 13, 1, 1, 6, 6),   # seventeen
    (12, 9, 20, 40, 40, 15, 16, 1, 1, 7, 7),    # eighteen: any number
    (12, 10, 20, 40, 40, 15, 15, 1, 1, 7, 7),   # nineteen
    (12, 10, 20, 40, 40, 17, 16, 1, 1, 7, 7),   # twenty, a single row left over
    (8, 3, 40, 61, 50, 7, 7, 3, 3, 3, 3),       # stride three
    (8, 3, 40, 61, 50, 7, 11, 1, 2, 5, 5),      # an odd width in pairs, another stride down
], ids=str)
def test_few_channels_rows_by_the_byte(oracle, t):
    """Kernel rows of every number of bytes that has code of its own, taps outside the image in every
    row of four; mean|x| read one, two and four at a time."""
    d, x, w = problem(t, zeros=True)
    assert make(d, w).kernel_name(0).startswith("conv_mfma_fp4_shallow_kernel")
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("oc,ic,k", [
    (1, 1, 3),        # most slices empty
    (1, 29, 3),       # the last slices cut short, none full
    (64, 1024, 4),    # every thread as many values as are under way together
    (64, 1025, 4),    # one more
    (321, 1111, 3),   # a slice that does not end with a wave
], ids=str)
def test_mean_of_weights_by_slices(gpu, oc, ic, k):
    """xnor_nn_binarize_weights_float adds 256 slices, 256 threads each, in a fixed order: the same
    sums here."""
    import torch
    d, _, w = problem((1, ic, oc, 8, 8, k, k, 1, 1, 0, 0))
    n = w.size
    per = -(-n // 256)
    rounds = -(-per // 256)

    def tree(v): # over the last axis
        half = 128
        while half:
            v = v[..., :half] + v[..., half:2 * half]
            half //= 2
        return v[..., 0]

    slices = np.zeros((256, rounds * 256), np.float32)
    flat = w.ravel()
    for p in range(256):
        part = flat[p * per:(p + 1) * per]
        slices[p, :part.size] = part
    sums = np.zeros((256, 256), np.float32)
    for r in range(rounds):
        sums += slices[:, r * 256:(r + 1) * 256]
    mean = tree(tree(sums)) * np.float32(np.float32(1) / np.float32(n))
    conv = make(d, w)
    got = torch.empty(w.shape, dtype=torch.float32, device=gpu)
    conv.binarizeWeightsFloat(torch.from_numpy(w).to(gpu), got)
    conv.close()
    assert same_bits(got.cpu().numpy(), np.where(w >= 0, mean, -mean))


@pytest.mark.parametrize("t", [
    (90, 1, 20, 3, 4, 5, 5, 1, 1, 2, 2),        # images shorter than a wave's step from row to row
    (40, 3, 40, 8, 9, 5, 5, 3, 1, 1, 2),        # image rows that no tap reaches
    (2, 3, 20, 30, 250, 5, 5, 1, 1, 3, 3),      # padded rows of 256 cells, and around that
    (2, 3, 20, 30, 251, 5, 5, 1, 1, 3, 3),
    (2, 2, 20, 30, 249, 5, 5, 1, 1, 3, 3),
    (1, 2, 8, 9, 700, 5, 7, 1, 2, 2, 3),        # three rounds of columns
], ids=str)
def test_few_channels_rows_of_mean_magnitudes(oracle, t):
    """mean|x| of a tile's padded rows is copied row by row, 256 cells at a time, from image to image."""
    d, x, w = problem(t, zeros=True)
    assert make(d, w).kernel_name(0).startswith("conv_mfma_fp4_shallow_kernel")
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("fmts,separate_k", [(NCHW, False), (NCHW, True), (NHWC, False)])
@pytest.mark.parametrize("t", [
    (4, 12, 40, 40, 40, 5, 5, 1, 1, 2, 2),      # as many channels as the kernel is given
    (2, 5, 130, 20, 20, 7, 7, 1, 1, 3, 3),      # filters over several workgroups
    (3, 11, 32, 150, 150, 9, 9, 1, 1, 4, 4),    # more than 64 KB of LDS
    (9, 8, 40, 24, 22, 5, 5, 1, 1, 2, 2),       # pixels that start on bytes
], ids=str)
def test_few_channels_in_their_kernel(oracle, monkeypatch, t, fmts, separate_k):
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    x, w = in_layout(x, w, fmts)
    assert make(d, w, fmts).kernel_name(0).startswith("conv_mfma_fp4_shallow_kernel")
    run_and_compare(oracle, d, x, w, fmts)


@pytest.mark.parametrize("t", [
    (1, 1, 1, 3, 3, 1, 1, 1, 1, 0, 0),        # one value
    (1, 7, 5, 4, 4, 3, 3, 1, 1, 1, 1),        # 63 values: one short of a row of the sum
    (1, 257, 33, 4, 4, 1, 1, 1, 1, 0, 0),     # 257: one more than it holds; channels past a word
    (1, 160, 40, 5, 5, 3, 3, 1, 1, 1, 1),     # paired taps, odd number of taps
    (1, 1100, 17, 4, 4, 3, 3, 1, 1, 1, 1),    # channel parts
    (1, 5000, 9, 3, 3, 1, 1, 1, 1, 0, 0),     # no matrix-core layout
    (1, 1612, 8, 4, 4, 2, 5, 1, 1, 2, 2),     # 16120 values: as many as fit
    (1, 1613, 8, 4, 4, 2, 5, 1, 1, 2, 2),     # too many for one launch
    (2, 6, 40, 40, 30, 5, 5, 1, 1, 0, 2),     # kernel rows back to back, many operation counts
], ids=str)
def test_weight_stage(oracle, t):
    d, x, w = problem(t)
    w[np.abs(w) < 0.01] = np.float32(-0.0)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("kind", ["ties", "zeros", "tiny", "huge", "mixed", "late"])
def test_scale_of_weights_the_sum_rounds_oddly(oracle, kind):
    """alpha is one chain of rounded additions: values halfway between two units of the running
    sum, sums that stay at or near zero, values that outgrow the sum and values it swallows."""
    d, x, w = problem((1, 64, 16, 3, 3, 4, 4, 1, 1, 1, 1))
    n = 1024
    flat = w.reshape(16, n)
    u = np.float32(2.0) ** np.arange(-14, 2, dtype=np.float32)
    if kind == "ties": # small multiples of a power of two: most additions end halfway
        flat[:] = (np.round(flat * 60) * 2.0 ** -11 + 2.0 ** -24).astype(np.float32)
        flat[:, 0] = u
    elif kind == "zeros":
        flat[:8] = 0
        flat[8:, :900] = 0
    elif kind == "tiny":
        flat *= np.float32(1e-38)
        flat[3:6, 700] = np.float32(1e-30)
    elif kind == "huge":
        flat *= np.float32(1e37)
    elif kind == "mixed":
        flat *= np.float32(2.0) ** (np.arange(n) % 37 - 18).astype(np.float32)
    else:
        flat[:, 1000] = np.float32(5000.0) * u
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("kind", ["normal", "ties", "mixed", "zeros"])
@pytest.mark.parametrize("n", [1, 255, 257, 4096, 4097, 8192, 8193, 16120])
def test_scale_of_weights_by_runs(oracle, n, kind):
    """Filters on either side of where a thread's run of values doubles, and the smallest and largest:
    runs that leave a binade, runs of ties for both parities of the sum, empty ones."""
    d, x, w = problem((1, n, 5, 2, 2, 1, 1, 1, 1, 0, 0))
    flat = w.reshape(5, n)
    if kind == "ties":
        flat[:] = (np.round(flat * 60) * 2.0 ** -11 + 2.0 ** -24).astype(np.float32)
        flat[:, 0] = np.float32(2.0) ** np.arange(-4, 1, dtype=np.float32)
    elif kind == "mixed":
        flat *= np.float32(2.0) ** (np.arange(n) % 37 - 18).astype(np.float32)
    elif kind == "zeros":
        flat[:, n // 3:n // 2] = 0
        flat[1:] = np.where(np.arange(n) % 3 == 0, flat[1:], np.float32(0))
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("kind", ["infinite", "late", "nan", "both", "outgrows"])
def test_scale_of_weights_that_is_not_finite(oracle, kind):
    """An infinite or NaN weight among the largest finite ones: the running sum stays what it has
    become, bit for bit where it is a number."""
    outgrows = kind == "outgrows" # 160 times the largest number, scaled by 1 / 160 and rounded
    d, _, w = problem((1, 160, 16, 3, 3, 1, 1, 1, 1, 0, 0) if outgrows
                      else (1, 64, 16, 3, 3, 4, 4, 1, 1, 1, 1))
    flat = w.reshape(16, -1)
    big = np.float32(2.0) ** np.arange(112, 128, dtype=np.float32) # scaled: 2^102 and up
    flat[:] = np.sign(flat) * big[:, None]
    rows = np.arange(16)
    if kind in ("infinite", "both"):
        flat[rows, rows] = np.float32(np.inf)
    if kind == "late":
        flat[rows, 900 + rows] = np.float32(-np.inf)
    if kind in ("nan", "both"):
        flat[rows[::2], 500 + rows[::2]] = np.float32(np.nan)
    if outgrows:
        flat[:] = np.finfo(np.float32).max
    _, want, _ = oracle.binarize_weights(oracle_shape(oracle, d), w)
    conv = make(d, w)
    try:
        got = conv.export_floats(capi.RES_ALPHA)
    finally:
        conv.close()
    assert not np.all(np.isfinite(want))
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert same_bits(got[~np.isnan(want)], want[~np.isnan(want)])


@pytest.mark.parametrize("n,shift", [(1, 0), (255, 0), (1025, 1), (4096, 0), (600001, 0),
                                     (600001, 3)])
def test_float_weights_at_any_length_and_alignment(oracle, gpu, n, shift):
    import torch
    d, _, _ = problem((1, n, 1, 1, 1, 1, 1, 1, 1, 0, 0))
    w = synth.normal(3, n, 0.05)
    conv = make(d, None)
    try:
        from_t = torch.zeros(n + shift, device=gpu)
        from_t[shift:] = torch.from_numpy(w).to(gpu)
        to_t = torch.full((n + 8,), 7.0, device=gpu)
        torch.cuda.synchronize()
        conv.binarizeWeightsFloat(from_t[shift:], to_t)
        conv.synchronize()
        got = to_t.cpu().numpy()
        assert np.all(got[n:] == 7.0)
        mean = float(np.mean(w.astype(np.float64)))
        assert np.array_equal(np.sign(got[:n]), np.sign(np.where(w >= 0, mean, -mean)))
        assert np.all(np.abs(np.abs(got[:n]) - abs(mean)) <= 1e-6 * np.mean(np.abs(w)))
    finally:
        conv.close()


@pytest.mark.parametrize("t", [
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0),        # four bytes each way
    (1, 3, 5, 7, 7, 3, 3, 1, 1, 1, 1),        # byte counts that are no multiples of 16
    (3, 31, 9, 47, 53, 3, 3, 1, 1, 1, 1),     # a little over a slice, one piece
    (5, 67, 70, 61, 59, 3, 3, 1, 1, 1, 1),    # several pieces both ways, helpers
    (2, 600, 8, 20, 20, 3, 3, 2, 2, 0, 0),    # much in, little out
    (2, 4200, 8, 5, 5, 1, 1, 1, 1, 0, 0),     # no matrix cores: through the executors
    (3, 67, 130, 191, 187, 3, 3, 1, 1, 1, 1), # more than the pinned blocks of a pass, both ways
], ids=str)
def test_host_tensors(oracle, t):
    """Forward passes between host arrays, twice in a row on other inputs, with the arrays at odd
    addresses."""
    d, x, w = problem(t)
    s = oracle_shape(oracle, d)
    conv = make(d, w)
    try:
        for scale in (1.0, -2.0):
            xs = x * np.float32(scale)
            want = oracle.forward(s, xs, w)
            held = np.full(xs.size + 1, np.float32(np.nan))[1:].reshape(xs.shape)
            held[:] = xs
            dst = np.full(want["dst"].size + 3, np.float32(7))
            conv.forward(held, dst[1:-2])
            assert same_bits(dst[1:-2], want["dst"].ravel())
            assert dst[0] == 7 and np.all(dst[-2:] == 7)
            assert same_bits(conv.export_floats(capi.RES_K), want["k"])
            # ... and stage by stage
            dst[:] = 7
            conv.stage("binarize_data", src=held, dst=dst[1:-2])
            conv.stage("calculate_k")
            conv.stage("forward")
            assert same_bits(dst[1:-2], want["dst"].ravel())
            assert dst[0] == 7 and np.all(dst[-2:] == 7)
    finally:
        conv.close()


def test_host_tensors_under_capture(oracle, gpu):
    """Nothing would arrive before the graph runs: refused, and the stream stays usable."""
    import torch
    d, x, w = problem((5, 67, 70, 61, 59, 3, 3, 1, 1, 1, 1))
    want = oracle.forward(oracle_shape(oracle, d), x, w)["dst"]
    conv = make(d, w)
    try:
        side = torch.cuda.Stream()
        conv.set_stream(side)
        dst = np.full(want.shape, np.nan, np.float32)
        conv.forward(x, dst)
        assert same_bits(dst, want)
        dst.fill(7)
        with torch.cuda.graph(torch.cuda.CUDAGraph(), stream=side):
            with pytest.raises(XnorNNError):
                conv.forward(x, dst)
        assert np.all(dst == 7)
        conv.forward(x, dst)
        assert same_bits(dst, want)
    finally:
        conv.close()


@pytest.mark.parametrize("which", ["src", "dst", "both"])
@pytest.mark.parametrize("t", [
    (1, 128, 40, 23, 21, 3, 3, 1, 1, 1, 1),   # small: through the library's buffers
    (5, 67, 70, 61, 59, 3, 3, 1, 1, 1, 1),    # in place, byte counts that are no multiples of 16
], ids=str)
def test_pinned_host_tensors(oracle, gpu, t, which):
    """Host tensors that the user has pinned, one or both, at odd addresses."""
    import torch
    d, x, w = problem(t)
    want = oracle.forward(oracle_shape(oracle, d), x, w)["dst"]
    pin = {n: which in (n, "both") for n in ("src", "dst")}
    src = torch.full((x.size + 1,), float("nan"), pin_memory=pin["src"])
    dst = torch.full((want.size + 3,), 7.0, pin_memory=pin["dst"])
    src[1:] = torch.from_numpy(x.ravel())
    conv = make(d, w)
    try:
        for stages in (False, True):
            dst.fill_(7)
            if stages:
                conv.stage("binarize_data", src=src[1:].numpy(), dst=dst[1:-2].numpy())
                conv.stage("calculate_k")
                conv.stage("forward")
            else:
                conv.forward(src[1:].numpy(), dst[1:-2].numpy())
            got = dst.numpy()
            assert same_bits(got[1:-2], want.ravel())
            assert got[0] == 7 and np.all(got[-2:] == 7)
    finally:
        conv.close()


@pytest.mark.parametrize("separate_k", [False, True])
@pytest.mark.parametrize("t", [
    (1, 33, 8, 1, 1, 1, 1, 1, 1, 0, 0),        # one pixel, a word and one channel
    (1, 128, 8, 4, 4, 1, 1, 1, 1, 0, 0),       # a set of words exactly, a tile exactly
    (3, 129, 8, 5, 7, 3, 3, 1, 1, 1, 1),       # one channel more, tiles across images
    (2, 1024, 8, 3, 3, 1, 1, 1, 1, 0, 0),      # one chunk, exactly
    (2, 1025, 8, 3, 3, 1, 1, 1, 1, 0, 0),      # two chunks
    (1, 3100, 8, 7, 7, 1, 1, 1, 1, 0, 0),      # four chunks, the last one ragged
    (16, 40, 8, 16, 16, 3, 3, 1, 1, 1, 1),     # 64 tiles of 64 pixels: the last that are few
    (16, 40, 8, 16, 17, 3, 3, 1, 1, 1, 1),     # 68: too many
], ids=str)
def test_few_input_pixels(oracle, monkeypatch, t, separate_k):
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("separate_k", [False, True])
@pytest.mark.parametrize("t", [
    (1, 2048, 8, 7, 7, 1, 1, 1, 1, 0, 0),      # both places of every loader once
    (3, 2049, 8, 5, 5, 1, 1, 1, 1, 0, 0),      # a third chunk, of one channel
    (5, 4095, 8, 9, 7, 1, 1, 1, 1, 0, 0),      # four, all places twice
    (2, 8160, 8, 3, 11, 1, 1, 1, 1, 0, 0),     # eight: as deep as tiles go
    (17, 511, 8, 16, 16, 1, 1, 1, 1, 0, 0),    # 68 tiles of 64 pixels, a channel short
    (17, 512, 8, 16, 16, 1, 1, 1, 1, 0, 0),    # ... and deep enough for tiles of 16
    (32, 1025, 8, 16, 16, 1, 1, 1, 1, 0, 0),   # 128 tiles: the last that are few
    (33, 1025, 8, 16, 16, 1, 1, 1, 1, 0, 0),   # 132: too many
], ids=str)
def test_deep_input_of_few_pixels(oracle, monkeypatch, t, separate_k):
    """Parts of chunks are handed to the adding wave and their places given back one by one."""
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("small", ["0", "1"])
@pytest.mark.parametrize("kh,kw", [(1, 2), (2, 1), (4, 3), (3, 4), (6, 6), (5, 8), (9, 9), (2, 10),
                                   (11, 11), (11, 1), (3, 12), (12, 12)])
@pytest.mark.parametrize("mb,ic,ih,iw", [(1, 16, 1, 1), (1, 16, 2, 1), (2, 40, 1, 3), (3, 70, 13, 12)])
def test_sums_of_mean_magnitudes_of_any_width(oracle, monkeypatch, mb, ic, ih, iw, kh, kw, small):
    """K of kernels that are narrower than the rows their sums read, down to images of one pixel."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", small)
    pad = max(kh, kw) // 2
    d, x, w = problem((mb, ic, 40, ih, iw, kh, kw, 1, 1, pad, pad), zeros=True)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("separate_k", [False, True])
@pytest.mark.parametrize("t,small", [
    ((1, 256, 112, 41, 61, 5, 5, 1, 1, 2, 2), True),       # 316 pairs of blocks (256 compute units), 100 steps
    ((1, 256, 192, 42, 60, 5, 5, 1, 1, 2, 2), False),      # 474
    ((2, 300, 96, 56, 60, 3, 3, 1, 1, 1, 1), False),       # 630, as many steps of nine taps
    ((1, 64, 40, 47, 45, 5, 5, 1, 1, 2, 2), True),         # 25 steps, two launches of 134
    ((1, 50, 40, 29, 31, 5, 5, 1, 1, 2, 2), True),         # no more than 1024 words to pack
    ((1, 1, 33, 24, 25, 11, 11, 1, 1, 5, 5), False),       # (a kernel for few channels)
    ((1, 70, 33, 9, 9, 9, 9, 1, 1, 4, 4), True),           # the summing wave has no steps
    ((1, 70, 33, 9, 9, 1, 3, 1, 1, 0, 1), True),           # six steps in four waves
], ids=str)
def test_sums_of_k_beside_the_steps(oracle, gpu, t, small, separate_k, monkeypatch):
    """One wave of the kernel for few tiles sums K and has fewer steps, or none."""
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    conv = make(d, w)
    try:
        assert ("small_kernel" in conv.kernel_name(0)) == small
    finally:
        conv.close()
    run_and_compare(oracle, d, x, w, NCHW, True, gpu)


@pytest.mark.parametrize("separate_k", [False, True])
@pytest.mark.parametrize("t,name", [
    ((1, 32, 8, 9, 8, 1, 1, 1, 1, 0, 0), "tiled_kernel"),            # whole pieces, one slice
    ((2, 6, 8, 9, 8, 3, 3, 1, 1, 1, 1), "generic_kernel"),
    ((2, 7, 8, 9, 8, 3, 3, 1, 1, 1, 1), "tiled_kernel<RAGGED>"),     # one ragged slice
    ((1, 31, 8, 13, 5, 1, 1, 1, 1, 0, 0), "tiled_kernel<RAGGED>"),   # 65 pixels
    ((1, 31, 8, 8, 8, 1, 1, 1, 1, 0, 0), "generic_kernel"),          # 64
    ((1, 33, 8, 1, 1, 1, 1, 1, 1, 0, 0), "tiled_kernel<RAGGED>"),    # one pixel
    ((3, 130, 8, 9, 7, 3, 3, 1, 1, 1, 1), "tiled_kernel<RAGGED>"),   # tiles across images
    ((2, 383, 8, 8, 16, 1, 1, 1, 1, 0, 0), "tiled_kernel<RAGGED>"),  # twelve waves, whole tiles
    ((1, 385, 8, 9, 9, 1, 1, 1, 1, 0, 0), "tiled_kernel<RAGGED>"),   # two rounds of seven
    ((1, 1502, 8, 6, 11, 1, 1, 1, 1, 0, 0), "tiled_kernel<RAGGED>"), # above 64 KB of LDS
    ((1, 13535, 1, 9, 8, 1, 1, 1, 1, 0, 0), "tiled_kernel<RAGGED>"), # as deep as LDS goes
    ((1, 13537, 1, 9, 8, 1, 1, 1, 1, 0, 0), "generic_kernel"),
    ((1, 2048, 8, 8, 8, 1, 1, 1, 1, 0, 0), "binarize_nhwc_kernel"),  # 64 pixels
    ((1, 2048, 8, 13, 5, 1, 1, 1, 1, 0, 0), "tiled_kernel"),         # 65
    ((1, 13536, 1, 9, 8, 1, 1, 1, 1, 0, 0), "tiled_kernel"),
    ((1, 13540, 1, 9, 8, 1, 1, 1, 1, 0, 0), "binarize_nhwc_kernel"),
], ids=str)
def test_channels_last_of_any_count(oracle, gpu, monkeypatch, t, name, separate_k):
    """Pixels that begin anywhere in a line, and the rule that chooses their kernel on either side of
    each line."""
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    x, w = in_layout(x, w, NHWC)
    conv = make(d, w, NHWC)
    try:
        assert conv.kernel_name(2).endswith(name)
    finally:
        conv.close()
    run_and_compare(oracle, d, x, w, NHWC, True, gpu)


@pytest.mark.parametrize("fmts,separate_k", [(NCHW, False), (NCHW, True), (NHWC, False)])
@pytest.mark.parametrize("t", [
    (1, 1, 1, 1, 1, 1, 1, 1, 1, 0, 0),         # one value
    (1, 32, 33, 4, 8, 3, 3, 1, 1, 1, 1),       # a word, a tile exactly; paired taps
    (2, 31, 70, 5, 7, 3, 3, 1, 1, 1, 1),       # ragged word, filters and tiles across images
    (3, 32, 8, 9, 11, 1, 1, 2, 2, 0, 0),       # input pixels that no output reads
    (2, 8, 40, 13, 12, 2, 3, 5, 4, 0, 1),      # the same, between and behind the tiles
    (1, 33, 32, 6, 6, 3, 3, 1, 1, 2, 2),       # two words, ragged
    (9, 64, 64, 7, 7, 3, 3, 1, 1, 1, 1),       # two words, many tiles
    (1, 64, 96, 19, 40, 5, 3, 2, 1, 2, 0),     # a span of several rows a lane
    (1, 24, 16, 12, 12, 7, 7, 1, 1, 3, 3),     # eight waves, paired taps
    (1, 64, 16, 12, 12, 5, 5, 1, 1, 2, 2),     # eight waves, two words
    (1, 20, 8, 200, 3, 3, 3, 1, 1, 0, 0),      # one pixel a row
], ids=str)
def test_one_launch_forward(oracle, gpu, monkeypatch, t, fmts, separate_k):
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    run_and_compare(oracle, d, *in_layout(x, w, fmts), fmts, True, gpu)


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("t", [
    (9, 64, 64, 7, 7, 3, 3, 1, 1, 1, 1),       # one launch where input and output lie apart
    (2, 96, 96, 9, 9, 3, 3, 1, 1, 1, 1),
    (40, 40, 40, 30, 30, 3, 3, 1, 1, 1, 1),
], ids=str)
def test_output_over_the_input(oracle, gpu, t, shift):
    """In place, and into a buffer that begins some images on: all of the input is read first."""
    import torch
    d, x, w = problem(t, zeros=True)
    want = oracle.forward(oracle_shape(oracle, d), x, w)
    conv = make(d, torch.from_numpy(w).to(gpu))
    try:
        buf = torch.zeros(x.size + shift * x[0].size, device=gpu)
        for _ in range(3):
            buf[:x.size] = torch.from_numpy(x).to(gpu).ravel()
            y = buf[shift * x[0].size:][:x.size]
            torch.cuda.synchronize()
            conv.forward(buf.data_ptr(), y.data_ptr())
            conv.synchronize()
            assert same_bits(y.cpu().numpy().reshape(x.shape), want["dst"])
            assert same_bits(conv.export_floats(capi.RES_K), want["k"])
    finally:
        conv.close()


@pytest.mark.parametrize("t,launches", [
    ((1, 32, 33, 4, 8, 3, 3, 1, 1, 1, 1), 1),
    ((3, 64, 512, 16, 16, 3, 3, 1, 1, 1, 1), 1),   # 64 channels, 1.5 workgroups per compute unit
    ((1, 65, 33, 4, 8, 3, 3, 1, 1, 1, 1), 2),      # a third word
    ((3, 64, 513, 16, 16, 3, 3, 1, 1, 1, 1), 2),   # more workgroups
    ((64, 3, 96, 227, 227, 11, 11, 4, 4, 0, 0), 2),
], ids=str)
def test_launches_of_a_forward_pass(gpu, t, launches):
    """Counted as the nodes of a captured pass."""
    import torch
    d, x, w = problem(t)
    conv = make(d, torch.from_numpy(w).to(gpu))
    try:
        xt = torch.from_numpy(x).to(gpu)
        yt = torch.empty(d["mb"], d["oc"], conv.desc.oh, conv.desc.ow, device=gpu)
        side = torch.cuda.Stream()
        conv.set_stream(side)
        conv.forward(xt, yt)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph, stream=side):
            conv.forward(xt, yt)
        nodes = C.c_size_t()
        assert conv.lib.hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None,
                                         C.byref(nodes)) == 0
        assert nodes.value == launches
    finally:
        conv.close()


@pytest.mark.parametrize("t", [
    (1, 160, 40, 12, 12, 5, 5, 1, 1, 2, 2),    # paired taps, 65 steps
    (1, 96, 32, 9, 9, 5, 5, 1, 1, 2, 2),       # 39 steps
    (1, 128, 70, 9, 9, 1, 1, 1, 1, 0, 0),      # two steps for four waves
    (1, 384, 33, 5, 6, 1, 2, 1, 1, 0, 0),      # twelve steps for eight waves
    (1, 384, 33, 5, 6, 1, 1, 1, 1, 0, 0),      # six steps
    (2, 1030, 64, 7, 7, 3, 3, 1, 1, 1, 1),     # more than a ring per wave
], ids=str)
def test_steps_shared_by_waves(oracle, t):
    d, x, w = problem(t, zeros=True)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("separate_k", [False, True])
@pytest.mark.parametrize("t", [
    (1, 64, 70, 9, 9, 1, 1, 1, 1, 0, 0),       # one step for four waves
    (1, 64, 70, 9, 9, 1, 2, 1, 1, 0, 0),       # two
    (2, 1000, 64, 7, 7, 3, 3, 1, 1, 1, 1),     # 144 for eight: more than a ring each
], ids=str)
def test_few_tiles_in_their_kernel(oracle, monkeypatch, t, separate_k):
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    assert make(d, w).kernel_name(0).startswith("conv_mfma_fp4_small_kernel")
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("kw", [1, 2, 3, 5, 7, 8])
@pytest.mark.parametrize("blocks", ["small", "1", "2", "3", "4"])
def test_k_sums_by_kernel_width(oracle, monkeypatch, blocks, kw):
    """Rows of one, three, five and seven taps are read whole, others tap by tap; taps outside the
    image on every side, tiles across images, an odd number of pixel blocks."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", "1" if blocks == "small" else "0")
    if blocks != "small":
        monkeypatch.setenv("XNOR_NN_HIP_MFMA_PS", blocks)
    d, x, w = problem((3, 70, 200, 8, 6, 3, kw, 1, 1, kw // 2, kw // 2), zeros=True)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("blocks", [1, 2, 3, 4])
@pytest.mark.parametrize("ic", [20, 64, 70, 128, 192, 700])
def test_short_and_long_walks(oracle, monkeypatch, ic, blocks):
    """Walks of one to fifteen groups of weight fragments, with and without paired taps: fewer than
    are under way at once, and every remainder of what the loop takes together."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_PS", str(blocks))
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", "0")
    for kh, kw in [(1, 1), (1, 2), (1, 3), (2, 2), (1, 5), (2, 3), (1, 7), (2, 4), (3, 3), (2, 5),
                   (1, 11), (3, 4), (1, 13), (2, 7), (3, 5)]:
        d, x, w = problem((2, ic, 70, 5, 14, kh, kw, 1, 1, kh // 2, kh // 2), zeros=True)
        run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("t", [
    (1, 70, 33, 3, 200, 3, 3, 1, 1, 1, 1),      # rows longer than a tile, taps above and below
    (2, 20, 40, 9, 61, 1, 1, 2, 2, 0, 0),       # one tap, rows and pixels that nothing reads
    (2, 64, 40, 9, 61, 2, 2, 3, 3, 0, 0),       # gaps between the taps
    (3, 40, 40, 5, 37, 3, 5, 1, 2, 2, 4),       # taps left and right of the image
    (2, 96, 300, 1, 90, 1, 7, 1, 1, 3, 3),      # one row; most kernel rows outside
    (1, 130, 30, 12, 150, 5, 5, 2, 1, 2, 2),
    (1, 1100, 40, 4, 70, 3, 3, 1, 1, 1, 1),     # channel parts
    (1, 864, 40, 5, 83, 3, 3, 1, 1, 1, 1),      # more than the LDS if whole rows were staged
    (2, 96, 40, 9, 32, 3, 3, 1, 1, 1, 1),       # the widest rows that are staged whole,
    (2, 96, 40, 9, 33, 3, 3, 1, 1, 1, 1),       # one column more,
    (2, 96, 40, 9, 32, 3, 3, 2, 1, 1, 1),       # and a stride either way
    (2, 96, 40, 9, 32, 3, 3, 1, 2, 1, 1),
], ids=str)
@pytest.mark.parametrize("small", ["0", "1"])
def test_tiles_that_begin_inside_a_row(oracle, monkeypatch, t, small):
    """The input of a tile runs from its first pixel's first tap to its last pixel's last one."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", small)
    d, x, w = problem(t, zeros=True)
    assert make(d, w).kernel_name(0).startswith("conv_mfma_fp4")
    for blocks in ("1", "2", "3"):
        if small == "0":
            monkeypatch.setenv("XNOR_NN_HIP_MFMA_PS", blocks)
        run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("blocks", [1, 2, 3, 4])
@pytest.mark.parametrize("ic", [20, 64, 70, 128, 192])
def test_walks_with_several_groups_under_way(oracle, monkeypatch, ic, blocks):
    """... whatever their length: fewer groups than are under way, every remainder, and the lengths on
    either side of where the rule takes them."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_PS", str(blocks))
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", "0")
    for long_walk, kernels in (("1", [(1, 1), (1, 2), (2, 2), (1, 5), (2, 3), (1, 7), (2, 4), (3, 3), (2, 5),
                                      (1, 11), (3, 4), (1, 13), (2, 7)]),
                               (None, [(1, 7), (2, 4), (3, 5), (3, 6), (4, 5), (3, 13), (5, 8), (6, 13),
                                       (8, 10), (11, 11)])):
        if long_walk:
            monkeypatch.setenv("XNOR_NN_HIP_MFMA_LONG", long_walk)
        else:
            monkeypatch.delenv("XNOR_NN_HIP_MFMA_LONG")
        for kh, kw in kernels:
            for oc in (70,) if long_walk else (33, 70, 140): # four, two and one pixel groups
                d, x, w = problem((2, ic, oc, 5, 14, kh, kw, 1, 1, kh // 2, kh // 2), zeros=True)
                run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("groups", ["1", "2", "4"])
@pytest.mark.parametrize("t", [
    (4, 64, 64, 64, 64, 1, 1, 1, 1, 0, 0),      # 128 workgroups of four groups, 256 of two
    (1, 70, 33, 46, 45, 3, 3, 1, 1, 1, 1),      # a last tile of a few pixels
    (1, 130, 128, 31, 33, 3, 3, 1, 1, 1, 1),
    (3, 288, 24, 19, 23, 3, 3, 2, 2, 1, 1),
], ids=str)
def test_pixel_groups_of_few_workgroups(oracle, monkeypatch, t, groups):
    """A layer of few filters and pixels with every number of pixel groups; 1 is what the plan takes."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", "0")
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_GROUPS", groups)
    d, x, w = problem(t, zeros=True)
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("t", [
    (1, 3000, 33, 28, 28, 3, 3, 1, 1, 1, 1),    # one tile to a compute unit's LDS
    (1, 4096, 8, 14, 14, 3, 3, 1, 1, 1, 1),     # four channel parts
    (1, 2048, 8, 15, 28, 5, 5, 1, 1, 2, 2),
    (3, 1024, 40, 10, 10, 3, 3, 1, 1, 1, 1),    # tiles across images
    (9, 1100, 40, 7, 7, 1, 1, 1, 1, 0, 0),      # a tile's pixels and no more
], ids=str)
@pytest.mark.parametrize("separate_k", [False, True])
def test_deep_narrow_images(oracle, monkeypatch, t, separate_k):
    """Tiles that begin inside a row of a narrow image."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", "0")
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    assert make(d, w).kernel_name(0).startswith("conv_mfma_fp4_kernel<")
    run_and_compare(oracle, d, x, w)


@pytest.mark.parametrize("t,joined", [
    ((26, 384, 40, 13, 13, 3, 3, 1, 1, 1, 1), True),
    ((26, 70, 8, 13, 13, 15, 15, 4, 4, 7, 7), True),      # long filters, few tiles
    ((75, 64, 8, 88, 88, 3, 3, 4, 4, 1, 1), True),        # 9075 tiles, short filters
    ((72, 40, 8, 64, 64, 19, 19, 4, 4, 9, 9), False),     # 4608, long filters, few channels
], ids=str)
def test_new_weights_join_the_binarize_launch(gpu, t, joined):
    """Where the filters' LDS leaves the tiles enough workgroups; the same result either way."""
    import torch
    d, x, w = problem(t)
    wt, xt = torch.from_numpy(w).to(gpu), torch.from_numpy(x).to(gpu)
    conv = make(d, -2 * wt)
    try:
        assert conv.kernel_name(0).startswith("conv_mfma_fp4")
        yt = torch.empty(d["mb"], d["oc"], conv.desc.oh, conv.desc.ow, device=gpu)
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        conv.forward_on_stream(xt, yt, side.cuda_stream, wt)
        torch.cuda.synchronize()
        first = yt.clone()
        graph = torch.cuda.CUDAGraph(keep_graph=True)
        with torch.cuda.graph(graph, stream=side):
            conv.forward_on_stream(xt, yt, side.cuda_stream, wt)
        nodes = C.c_size_t()
        assert conv.lib.hipGraphGetNodes(C.c_void_p(graph.raw_cuda_graph()), None,
                                         C.byref(nodes)) == 0
        assert nodes.value == (2 if joined else 3)
        conv.change_weights(wt)
        yt.fill_(float("nan"))
        torch.cuda.synchronize()
        conv.forward(xt, yt)
        torch.cuda.synchronize()
        assert torch.equal(first, yt)
    finally:
        conv.close()


@pytest.mark.parametrize("fmts,separate_k", [(NCHW, False), (NCHW, True), (NHWC, False)])
@pytest.mark.parametrize("t", [
    (26, 384, 40, 13, 13, 3, 3, 1, 1, 1, 1),    # in one launch with twelve waves of input
    (9, 40, 300, 30, 30, 3, 3, 1, 1, 1, 1),     # two waves of input, filters past a chunk
    (5, 1612, 33, 30, 30, 2, 5, 1, 1, 2, 2),    # the longest filters, several rounds of input
    (5, 1613, 3, 30, 30, 2, 5, 1, 1, 2, 2),     # too long
    (70, 130, 9, 9, 9, 1, 1, 1, 1, 0, 0),       # one tap
    (2, 384, 40, 13, 13, 3, 3, 1, 1, 1, 1),     # few input pixels: a launch of its own
    (2, 64, 64, 7, 7, 3, 3, 1, 1, 1, 1),        # a pass of one launch
    (4, 3, 32, 40, 40, 11, 11, 4, 4, 0, 0),     # few channels
], ids=str)
def test_pass_with_new_weights(oracle, gpu, monkeypatch, t, fmts, separate_k):
    import torch
    if separate_k:
        monkeypatch.setenv("XNOR_NN_HIP_SEPARATE_K", "1")
    d, x, w = problem(t, zeros=True)
    x, w = in_layout(x, w, fmts)
    s = oracle_shape(oracle, d, fmts)
    want = oracle.forward(s, x, w)
    wt, xt = torch.from_numpy(w).to(gpu), torch.from_numpy(x).to(gpu)
    conv = make(d, -2 * wt, fmts)
    try:
        yt = torch.full(want["dst"].shape, float("nan"), device=gpu)
        side = torch.cuda.Stream()
        torch.cuda.synchronize()
        for _ in range(2):
            conv.forward_on_stream(xt, yt, side.cuda_stream, wt)
        conv.synchronize()
        assert same_bits(yt.cpu().numpy(), want["dst"])
        for slot, name in ((capi.RES_ALPHA, "alpha"), (capi.RES_A, "a"), (capi.RES_K, "k")):
            assert same_bits(conv.export_floats(slot), want[name])
        assert np.array_equal(conv.export_bin_src(), want["bin_src"])
        assert np.array_equal(conv.export_operations_count(), want["opc"])
        if d["oc"] % oracle.default_oci(s) == 0:
            assert np.array_equal(conv.export_bin_weights(), want["bin_weights"])
        assert np.array_equal(conv.forward_popcount(), want["popc"])
    finally:
        conv.close()


@pytest.mark.parametrize("t", [
    (26, 384, 64, 13, 13, 3, 3, 1, 1, 1, 1),    # weights join the binarize launch
    (2, 64, 64, 7, 7, 3, 3, 1, 1, 1, 1),        # a pass of one launch
], ids=str)
@pytest.mark.parametrize("tensors", ["device", "host", "mixed", "timed"])
@pytest.mark.parametrize("weights", ["device", "host"])
def test_new_weights_wherever_they_lie(oracle, gpu, t, tensors, weights):
    """XNOR_NN_HIP_NEW_WEIGHTS and nothing vouched for; "timed": with kernel timing on."""
    import torch
    d, x, w = problem(t, zeros=True)
    s = oracle_shape(oracle, d)
    want = oracle.forward(s, x, w)
    conv = make(d, torch.from_numpy(-2 * w).to(gpu))
    try:
        xt, wt = (torch.from_numpy(v).to(gpu) for v in (x, w))
        yt = torch.full(want["dst"].shape, float("nan"), device=gpu)
        dst = np.full(want["dst"].shape, np.nan, np.float32)
        torch.cuda.synchronize()
        src = capi.as_pointer(x if tensors == "host" else xt)
        to = capi.as_pointer(dst if tensors in ("host", "mixed") else yt)
        call = lambda src: conv.lib.xnor_nn_hip_forward_pass(
            C.byref(conv.desc), conv.res, src, to, None, capi.NEW_WEIGHTS)
        conv.res[capi.RES_USER_WEIGHTS] = None
        assert call(src) == capi.ERROR_INVALID_INPUT
        conv.res[capi.RES_USER_WEIGHTS] = capi.as_pointer(wt if weights == "device" else w)
        assert call(None) == capi.ERROR_INVALID_INPUT
        if tensors == "timed":
            conv.time_kernels(8)
        for _ in range(2):
            assert call(src) == capi.SUCCESS
        conv.synchronize()
        if tensors == "timed":
            for stage in (capi.OP_BINARIZE_DATA, capi.OP_CONVOLUTION_FORWARD):
                assert len(conv.kernel_times(stage)) == 2
        got = dst if tensors in ("host", "mixed") else yt.cpu().numpy()
        assert same_bits(got, want["dst"])
        assert same_bits(conv.export_floats(capi.RES_ALPHA), want["alpha"])
        assert np.array_equal(conv.export_bin_weights(), want["bin_weights"])
    finally:
        conv.close()


def test_new_weights_in_host_memory_on_a_stream(oracle, gpu):
    import torch
    d, x, w = problem((26, 384, 64, 13, 13, 3, 3, 1, 1, 1, 1))
    want = oracle.forward(oracle_shape(oracle, d), x, w)
    xt = torch.from_numpy(x).to(gpu)
    conv = make(d, torch.from_numpy(-2 * w).to(gpu))
    try:
        side = torch.cuda.Stream()
        for weights in (w, torch.from_numpy(w)):
            yt = torch.full(want["dst"].shape, float("nan"), device=gpu)
            torch.cuda.synchronize()
            conv.forward_on_stream(xt, yt, side.cuda_stream, weights)
            conv.synchronize()
            assert same_bits(yt.cpu().numpy(), want["dst"])
    finally:
        conv.close()
