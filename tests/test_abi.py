"""The C-ABI boundary without a GPU: the library loads, exports every function that
include/*.h declares, the descriptor has the layout a C compiler gives it, and the host-only
entry points behave like the reference's."""
import ctypes as C
import os
import re
import subprocess

import numpy as np
import pytest

from xnor_nn_amd import capi

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
INCLUDE = os.path.join(ROOT, "include")


def declared_functions():
    names = set()
    for header in ("xnor_nn.h", "xnor_nn_hip.h"):
        text = open(os.path.join(INCLUDE, header)).read()
        text = re.sub(r"/\*.*?\*/", "", text, flags=re.S)
        names.update(re.findall(r"\b(xnor_nn_\w+)\s*\(", text))
    return sorted(names)


def test_every_declared_symbol_is_exported():
    lib = C.CDLL(capi.library_path())
    names = declared_functions()
    assert len(names) >= 16
    for name in names:
        assert hasattr(lib, name), name
    # and the ctypes tables cover exactly the declared set
    assert set(names) == set(capi.CORE_SYMBOLS) | set(capi.HIP_SYMBOLS)


def test_descriptor_layout_matches_a_c_compiler(tmp_path):
    src = tmp_path / "layout.c"
    src.write_text(r'''
#include <stdio.h>
#include <stddef.h>
#include "xnor_nn.h"
#include "xnor_nn_hip.h"
int main(void) {
    printf("%zu %zu %zu %zu %zu %zu %zu %zu\n", sizeof(xnor_nn_convolution_t),
        offsetof(xnor_nn_convolution_t, mb), offsetof(xnor_nn_convolution_t, src_format),
        offsetof(xnor_nn_convolution_t, resource_size),
        offsetof(xnor_nn_convolution_t, binarize_weights),
        offsetof(xnor_nn_convolution_t, forward), offsetof(xnor_nn_convolution_t, state),
        sizeof(xnor_nn_resources_t));
    printf("%d %d %d %d %d %d\n", xnor_nn_unimplemented, xnor_nn_algorithm_bcast,
        xnor_nn_resource_operations_count, xnor_nn_resource_number,
        xnor_nn_weights_format_hwio, xnor_nn_operation_calculate_k);
    return 0;
}''')
    exe = tmp_path / "layout"
    subprocess.check_call(["gcc", "-std=c11", "-Wall", "-Werror", "-I", INCLUDE,
                           str(src), "-o", str(exe)])
    out = subprocess.check_output([str(exe)]).decode().split()
    D = capi.ConvolutionDesc
    want = [C.sizeof(D), D.mb.offset, D.src_format.offset, D.resource_size.offset,
            D.binarize_weights.offset, D.forward.offset, D.state.offset,
            C.sizeof(capi.Resources)]
    assert [int(v) for v in out[:8]] == want
    assert [int(v) for v in out[8:]] == [3, 1, 8, 9, 3, 3]


def test_cpp_wrapper_header_compiles(tmp_path):
    src = tmp_path / "wrap.cpp"
    src.write_text('#include "xnor_nn.hpp"\n'
                   'int use(const void *w) { xnor_nn::Convolution c{xnor_nn_algorithm_bcast,'
                   ' xnor_nn_data_format_nchw, xnor_nn_weights_format_oihw,'
                   ' xnor_nn_data_format_nchw, 1, 16, 8, 5, 5, 3, 3, 1, 1, 1, 1, w};'
                   ' return 0; }\n')
    subprocess.check_call(["g++", "-std=c++14", "-Wall", "-Werror", "-fsyntax-only",
                           "-I", INCLUDE, str(src)])


def test_status_messages():
    """reference src/status.cpp:3-15"""
    lib = capi.load()
    assert [capi.status_message(lib, s) for s in range(4)] == [
        "success", "memory_error", "bad_input", "unimplemented"]


def test_init_fills_descriptor_like_the_reference():
    """reference src/common_convolution.cpp:9-63: every field set, oh AND ow from pw,
    always success; plus this library's device buffer sizes."""
    lib = capi.load()
    c = capi.ConvolutionDesc()
    st = lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, capi.FMT_NCHW,
                                      capi.FMT_OIHW, capi.FMT_NCHW,
                                      4, 256, 96, 27, 27, 5, 5, 1, 1, 2, 2)
    assert st == capi.SUCCESS
    assert (c.mb, c.ic, c.ih, c.iw, c.oc, c.oh, c.ow) == (4, 96, 27, 27, 256, 27, 27)
    assert (c.kh, c.kw, c.sh, c.sw, c.ph, c.pw) == (5, 5, 1, 1, 2, 2)
    assert c.state and all((c.binarize_weights, c.binarize_data, c.calculate_k, c.forward))
    assert c.resource_size[capi.RES_BIN_SRC] == 4 * 27 * 27 * 3 * 4
    # packed sign words [OC/16][taps][words][16], then the same signs as FP4 matrix-core
    # fragments [OC/32][units][steps][64 lanes][16 bytes]; IC = 96 is three 32-channel words,
    # an odd number, so a unit is a pair of taps (13 for 25 taps) of 3 steps
    assert c.resource_size[capi.RES_BIN_WEIGHTS] == 16 * 25 * 3 * 16 * 4 + 8 * 13 * 3 * 64 * 16
    assert c.resource_size[capi.RES_A] == c.resource_size[capi.RES_K] == 4 * 27 * 27 * 4
    assert c.resource_size[capi.RES_ALPHA] == 256 * 4
    assert c.resource_size[capi.RES_OPERATIONS_COUNT] == 27 * 27 * 4
    # oh uses pw, not ph (reference src/common_convolution.cpp:16)
    lib.xnor_nn_destroy_convolution(C.byref(c))
    assert not c.state
    lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, 0, 2, 0,
                                 1, 16, 8, 10, 10, 3, 3, 1, 1, 0, 1)
    assert (c.oh, c.ow) == (10, 10)
    lib.xnor_nn_destroy_convolution(C.byref(c))
    lib.xnor_nn_destroy_convolution(C.byref(c))  # idempotent


def test_null_and_format_checks_of_the_executors():
    """Same status codes as the reference for missing slots
    (reference src/bcast_binarize_data.cpp:15-19, src/bcast_calculate_k.cpp:15-20,
    src/bcast_binarize_weights.cpp:15-21, src/default/bcast_convolution_default.cpp:25-33)
    and unknown formats (reference src/bcast_binarize_data.cpp:36-38).  No GPU needed: the
    checks come before any device work."""
    lib = capi.load()
    c = capi.ConvolutionDesc()
    lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, capi.FMT_NCHW,
                                 capi.FMT_OIHW, capi.FMT_NCHW, 1, 16, 8, 5, 5, 3, 3, 1, 1, 1, 1)
    res = capi.Resources()
    for stage in ("binarize_data", "calculate_k", "binarize_weights", "forward"):
        assert getattr(c, stage)(C.byref(c), res) == capi.ERROR_INVALID_INPUT, stage
    lib.xnor_nn_free_resources(res)  # safe on a zeroed table
    lib.xnor_nn_destroy_convolution(C.byref(c))

    dummy = (C.c_float * 4)()
    for i in range(capi.RES_NUMBER):
        res[i] = C.addressof(dummy)
    lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, 7, 9, 11,
                                 1, 16, 8, 5, 5, 3, 3, 1, 1, 1, 1)
    for stage in ("binarize_data", "calculate_k", "binarize_weights", "forward"):
        assert getattr(c, stage)(C.byref(c), res) == capi.UNIMPLEMENTED, stage
    lib.xnor_nn_destroy_convolution(C.byref(c))


def test_reference_algorithm_has_no_gpu_path():
    lib = capi.load()
    c = capi.ConvolutionDesc()
    st = lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_REFERENCE, 0, 2, 0,
                                      1, 16, 8, 5, 5, 3, 3, 1, 1, 1, 1)
    assert st == capi.SUCCESS and not c.state
    res = capi.Resources()
    assert c.forward(C.byref(c), res) == capi.UNIMPLEMENTED
    lib.xnor_nn_destroy_convolution(C.byref(c))


def test_word_size_of_the_exported_layout():
    """The export helpers hand out the reference's CPU layout, whose packed words are 16 bits
    wide while IC*KH*KW < 32767 and 32 bits wide from there on (reference
    src/implementation.cpp:17-22, src/convolution_traits.hpp:29-56)."""
    lib = capi.load()
    for ic, want in ((384, 2), (3640, 2), (3641, 4), (4000, 4)):
        c = capi.ConvolutionDesc()
        lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, 0, 2, 0,
                                     1, 16, ic, 5, 5, 3, 3, 1, 1, 1, 1)
        assert lib.xnor_nn_hip_canonical_bici(C.byref(c)) == want, ic
        lib.xnor_nn_destroy_convolution(C.byref(c))


def test_package_does_not_touch_the_oracle():
    """The oracle is test infrastructure: nothing under xnor_nn_amd/ may name it."""
    pkg = os.path.join(ROOT, "xnor_nn_amd")
    for base, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".hip", ".hpp", ".h", ".cpp")):
                text = open(os.path.join(base, f)).read()
                assert "oracle" not in text.lower(), os.path.join(base, f)


@pytest.mark.skipif(not os.path.isdir("/root/reference/example"),
                    reason="upstream sources not mounted")
@pytest.mark.parametrize("name,cc", [("simple_convolution.c", "gcc"),
                                     ("simple_convolution.cpp", "g++")])
def test_upstream_examples_compile_and_link_unchanged(tmp_path, name, cc):
    """The reference's own example programs (reference example/simple_convolution.c,
    .cpp) build against include/ and link to libxnor_nn.so without edits."""
    exe = tmp_path / "example"
    libdir = os.path.dirname(capi.library_path())
    subprocess.check_call([cc, "-I", INCLUDE, os.path.join("/root/reference/example", name),
                           "-L", libdir, "-lxnor_nn", "-Wl,-rpath," + libdir,
                           "-Wl,-rpath-link,/opt/rocm/lib", "-o", str(exe)])


def test_forward_popcount_needs_only_the_two_packed_tensors():
    """xnor_nn_hip_forward_popcount checks exactly the slots its header names: bin_src,
    bin_weights and the output pointer (host-only: the checks come before device work)."""
    lib = capi.load()
    c = capi.ConvolutionDesc()
    lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, capi.FMT_NCHW,
                                 capi.FMT_OIHW, capi.FMT_NCHW, 1, 16, 8, 5, 5, 3, 3, 1, 1, 1, 1)
    res = capi.Resources()
    out = (C.c_int32 * (16 * 25))()
    assert lib.xnor_nn_hip_forward_popcount(C.byref(c), res, out) == capi.ERROR_INVALID_INPUT
    dummy = (C.c_float * 4)()
    res[capi.RES_BIN_SRC] = C.addressof(dummy)
    assert lib.xnor_nn_hip_forward_popcount(C.byref(c), res, out) == capi.ERROR_INVALID_INPUT
    res[capi.RES_BIN_WEIGHTS] = C.addressof(dummy)
    assert lib.xnor_nn_hip_forward_popcount(C.byref(c), res, None) == capi.ERROR_INVALID_INPUT
    lib.xnor_nn_destroy_convolution(C.byref(c))
    # a descriptor without the bcast state has no popcount path
    assert lib.xnor_nn_hip_forward_popcount(C.byref(c), res, out) == capi.ERROR_INVALID_INPUT
    assert lib.xnor_nn_hip_set_stage_fusion(C.byref(c), 0) == capi.ERROR_INVALID_INPUT


def test_stage_fusion_switch_and_table_bookkeeping_without_a_gpu():
    """The switch is per descriptor; freeing a zeroed or hand-filled table and destroying a
    descriptor that never ran are safe (the hand-over bookkeeping is keyed on buffers)."""
    lib = capi.load()
    c = capi.ConvolutionDesc()
    lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, capi.FMT_NCHW,
                                 capi.FMT_OIHW, capi.FMT_NCHW, 1, 16, 8, 5, 5, 3, 3, 1, 1, 1, 1)
    assert lib.xnor_nn_hip_set_stage_fusion(C.byref(c), 0) == capi.SUCCESS
    assert lib.xnor_nn_hip_set_stage_fusion(C.byref(c), 1) == capi.SUCCESS
    res = capi.Resources()
    lib.xnor_nn_free_resources(res)
    lib.xnor_nn_destroy_convolution(C.byref(c))


def kernel_names(shape, fmts=(capi.FMT_NCHW, capi.FMT_OIHW, capi.FMT_NCHW),
                 stages=(capi.OP_BINARIZE_DATA, capi.OP_CONVOLUTION_FORWARD)):
    """(binarize kernel, convolution kernel) or those of other stages that the library plans for a
    shape (mb, oc, ic, ih, iw, kh, kw, sh, sw, ph, pw); planning needs no GPU (256 CUs assumed)."""
    lib = capi.load()
    c = capi.ConvolutionDesc()
    assert lib.xnor_nn_init_convolution(C.byref(c), capi.ALGORITHM_BCAST, *fmts, *shape) \
        == capi.SUCCESS
    buf = C.create_string_buffer(96)
    out = []
    for stage in stages:
        lib.xnor_nn_hip_kernel_name(C.byref(c), stage, buf, len(buf))
        out.append(buf.value.decode())
    lib.xnor_nn_destroy_convolution(C.byref(c))
    return tuple(out)


def test_kernel_variants_planned_for_known_shapes(monkeypatch):
    """The counterpart of the reference's dispatcher (reference src/bcast_convolution.hpp:13-38,
    src/bcast_convolution.cpp:14-43: exact-match table of shapes -> unrolled kernel, else the
    runtime-shape kernel): which kernel variant each of the five benchmark workloads and the
    boundary shapes get, decided at init from the shape alone."""
    for key in ("XNOR_NN_HIP_CONV", "XNOR_NN_HIP_MFMA_PS", "XNOR_NN_HIP_MFMA_MIX",
                "XNOR_NN_HIP_MFMA_PAIR", "XNOR_NN_HIP_NHWC", "XNOR_NN_HIP_STREAM_DST",
                "XNOR_NN_HIP_MFMA_PERSIST", "XNOR_NN_HIP_MFMA_SMALL", "XNOR_NN_HIP_MFMA_GROUPS"):
        monkeypatch.delenv(key, raising=False)
    conv4 = (256, 384, 13, 13, 3, 3, 1, 1, 1, 1)
    # 6 pixel blocks x 8 filter blocks: fewer (block, block) pairs than compute units
    assert kernel_names((1,) + conv4) == ("binarize_nchw_split_kernel",
                                          "conv_mfma_fp4_small_kernel<KS=6>")
    assert kernel_names((8,) + conv4)[1] == "conv_mfma_fp4_small_kernel<KS=6>"
    # up to two pairs per compute unit when a wave would walk 48 steps or more (here 54)
    assert kernel_names((12,) + conv4)[1] == "conv_mfma_fp4_small_kernel<KS=6>"
    assert kernel_names((16,) + conv4)[1] == "conv_mfma_fp4_kernel<KS=6,PS=1>"
    # 36 steps: the large-launch kernel from 1.5 pairs per compute unit
    assert kernel_names((8, 256, 256, 14, 14, 3, 3, 1, 1, 1, 1))[1] == "conv_mfma_fp4_kernel<KS=4,PS=1>"
    # 5.3 pixel blocks per compute unit: two tile sizes in one launch
    assert kernel_names((256,) + conv4)[1] == "conv_mfma_fp4_kernel<KS=6,PS=4+2>"
    assert kernel_names((1024,) + conv4)[1] == "conv_mfma_fp4_kernel<KS=6,PS=4>"
    # 96 channels = three words: two taps share three steps; several rounds of tiles with at
    # most four steps per tap: tiles of two blocks, three workgroups to a compute unit
    assert kernel_names((128, 256, 96, 27, 27, 5, 5, 1, 1, 2, 2))[1] \
        == "conv_mfma_fp4_kernel<KS=3,PS=2,PAIR>"
    assert kernel_names((64, 256, 256, 56, 56, 3, 3, 1, 1, 1, 1))[1] \
        == "conv_mfma_fp4_kernel<KS=4,PS=2>"
    # 64 filters are one wave's worth: the other three waves take further pixel blocks; 128
    # filters: two pixel groups
    assert kernel_names((64, 64, 64, 56, 56, 3, 3, 1, 1, 1, 1))[1] \
        == "conv_mfma_fp4_kernel<KS=1,PS=2,GROUPS=4>"
    assert kernel_names((64, 128, 128, 56, 56, 3, 3, 1, 1, 1, 1))[1] \
        == "conv_mfma_fp4_kernel<KS=2,PS=2,GROUPS=2>"
    # their one-block tiles are cheaper than the weight stream makes others, up to 47 steps
    assert kernel_names((39, 96, 64, 30, 30, 3, 3, 1, 1, 1, 1))[1] \
        == "conv_mfma_fp4_kernel<KS=1,PS=1,GROUPS=2>"
    assert kernel_names((30, 96, 192, 24, 24, 5, 5, 1, 1, 2, 2))[1] \
        == "conv_mfma_fp4_kernel<KS=3,PS=2,GROUPS=2>"
    # 98 blocks for 32 slots per XCD and filter chunk: 2 tiles of four, 30 of three
    assert kernel_names((32, 512, 512, 28, 28, 3, 3, 1, 1, 1, 1))[1] \
        == "conv_mfma_fp4_kernel<KS=8,PS=4+3>"
    # more than 1024 channels: channel parts; more than 4096: no matrix cores
    assert re.fullmatch(r"conv_mfma_fp4_kernel<KS=1[26],PS=\d,PARTS=\d>",
                        kernel_names((2, 64, 2048, 8, 8, 3, 3, 1, 1, 1, 1))[1])
    deep = kernel_names((1, 32, 8200, 4, 4, 1, 1, 1, 1, 0, 0))
    assert deep[0] == "binarize_generic_kernel" and deep[1] == "conv_xnor_popc_kernel<XW=0,Q=16>"  # XW=0: word count at run time
    # kernels wider than 32 taps keep their tap masks in 32 bits: XNOR/popcount kernel
    assert kernel_names((1, 16, 32, 40, 40, 33, 33, 1, 1, 0, 0))[1].startswith("conv_xnor_popc")
    # input layouts
    nhwc = (capi.FMT_NHWC, capi.FMT_OIHW, capi.FMT_NCHW)
    assert kernel_names((4,) + conv4, nhwc)[0] == "binarize_nhwc_tiled_kernel"
    assert kernel_names((1, 32, 2048, 6, 6, 3, 3, 1, 1, 1, 1), nhwc)[0] == "binarize_nhwc_kernel"
    assert kernel_names((1, 32, 30, 6, 6, 3, 3, 1, 1, 1, 1), nhwc)[0] == "binarize_generic_kernel"
    # the switch that forces the XNOR/popcount kernel (used to profile the two side by side)
    monkeypatch.setenv("XNOR_NN_HIP_CONV", "valu")
    assert kernel_names((256,) + conv4)[1] == "conv_xnor_popc_kernel<XW=12,Q=16>"


def test_deep_narrow_images_run_on_the_matrix_cores():
    """A tile stages its taps' span however few columns the image has: with whole rows the tiles of these
    layers do not fit the LDS, or only one by one."""
    for t, steps in (((4, 128, 3000, 28, 28, 3, 3, 1, 1, 1, 1), 16), ((8, 128, 4096, 14, 14, 3, 3, 1, 1, 1, 1), 16),
                     ((2, 128, 2048, 28, 28, 5, 5, 1, 1, 2, 2), 16), ((4, 128, 3000, 28, 33, 3, 3, 1, 1, 1, 1), 16)):
        assert kernel_names(t)[1].startswith("conv_mfma_fp4_kernel<KS=%d,PS=" % steps), t


def test_small_tiles_of_long_walks_are_not_chosen_for_their_number():
    """The spans that tiles stage let small tiles lie in the LDS by fours; where the weight stream bounds
    them they are slower all the same, by 12 to 35 % for these layers, and so is a tile that has the LDS for
    itself where a smaller one leaves room for a second."""
    for t, ps in (((163, 306, 877, 13, 13, 3, 3, 1, 1, 1, 1), 2), ((120, 544, 1024, 13, 16, 3, 3, 1, 1, 1, 1), 2),
                  ((157, 64, 80, 63, 63, 5, 5, 1, 1, 2, 2), 2), ((49, 32, 80, 65, 65, 5, 5, 1, 1, 2, 2), 2),
                  ((27, 224, 336, 71, 75, 3, 3, 1, 1, 0, 0), 2), ((66, 320, 272, 56, 56, 3, 3, 2, 2, 1, 1), 1)):
        assert "PS=%d" % ps in kernel_names(t)[1], (t, kernel_names(t)[1])


def test_pixel_groups_leave_no_half_of_the_chip_idle(monkeypatch):
    """Few filters: the waves without filters take pixel blocks of their own, but not where that leaves half
    of the 256 compute units without a workgroup."""
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_SMALL", "0")
    for t, groups in (((2, 64, 416, 103, 103, 1, 1, 2, 2, 0, 0), 1),   # 44 workgroups of four groups
                      ((4, 64, 64, 64, 64, 1, 1, 1, 1, 0, 0), 2),      # 128
                      ((1, 64, 64, 113, 145, 1, 1, 1, 1, 0, 0), 4),    # 129
                      ((2, 64, 64, 64, 64, 1, 1, 1, 1, 0, 0), 1),      # 64, 128 of two groups
                      ((1, 64, 64, 91, 91, 1, 1, 1, 1, 0, 0), 2),      # 65, 130
                      ((2, 128, 64, 64, 64, 1, 1, 1, 1, 0, 0), 1), ((1, 128, 64, 91, 91, 1, 1, 1, 1, 0, 0), 2)):
        name = kernel_names(t)[1]
        assert ("GROUPS=%d" % groups in name) if groups > 1 else "GROUPS" not in name, (t, name)


def test_inputs_that_reach_the_dropped_offset_take_the_generic_kernel():
    """The tiled binarize kernels read a channel past the end of a ragged slice through the
    byte offset 0xFFFFFFF0, which the hardware drops only while it lies outside the buffer.
    An input that ends at or beyond that offset (but below 4 GiB) must not run them."""
    # 1 x 3 x 21 x 17043521 floats = 0xFFFFFFFC bytes: inside the gap
    assert kernel_names((1, 4, 3, 21, 17043521, 1, 1, 1, 1, 0, 0))[0] == "binarize_generic_kernel"
    nhwc = (capi.FMT_NHWC, capi.FMT_OIHW, capi.FMT_NCHW)
    # 1 x 4 x 1 x 268435455 floats = 0xFFFFFFF0 bytes, channels a multiple of four
    assert kernel_names((1, 4, 4, 1, 268435455, 1, 1, 1, 1, 0, 0), nhwc)[0] \
        == "binarize_generic_kernel"
    # just below: 0xFFFFFFEC bytes
    assert kernel_names((1, 4, 1, 1, 1073741819, 1, 1, 1, 1, 0, 0))[0] == "binarize_nchw_kernel"
    assert kernel_names((1, 4, 4, 1, 268435454, 1, 1, 1, 1, 0, 0), nhwc)[0] \
        == "binarize_nhwc_tiled_kernel"


def test_channels_last_input_is_streamed_by_size():
    """Not where the L2s may hold it, nor where it is large."""
    nhwc = (capi.FMT_NHWC, capi.FMT_OIHW, capi.FMT_NHWC)
    for t, streams in (((2, 8, 1024, 64, 64, 1, 1, 1, 1, 0, 0), False),      # 32 MB
                       ((13, 8, 100, 81, 80, 3, 3, 1, 1, 1, 1), True),       # a little more
                       ((100, 256, 128, 32, 32, 3, 3, 1, 1, 1, 1), True),
                       ((1, 8, 1040, 161, 160, 1, 1, 1, 1, 0, 0), True),     # 102 MB
                       ((1, 8, 1040, 162, 162, 1, 1, 1, 1, 0, 0), False)):   # 104 MB and a little
        assert kernel_names(t, nhwc)[0] \
            == "binarize_nhwc_tiled_kernel" + ("<STREAM>" if streams else ""), t


def test_persistent_workgroups_are_planned_on_request_only(monkeypatch):
    """XNOR_NN_HIP_MFMA_PERSIST=N: N workgroups per XCD that walk over the tiles; without it a
    workgroup per tile, whatever the size (measured faster)."""
    resnet = (64, 256, 256, 56, 56, 3, 3, 1, 1, 1, 1)
    monkeypatch.delenv("XNOR_NN_HIP_MFMA_PERSIST", raising=False)
    assert kernel_names(resnet)[1] == "conv_mfma_fp4_kernel<KS=4,PS=2>"
    monkeypatch.setenv("XNOR_NN_HIP_MFMA_PERSIST", "64")
    assert kernel_names(resnet)[1] == "conv_mfma_fp4_persistent_kernel<KS=4,PS=4+3>"
    # sixteen steps per tap have no four-block tile: never persistent
    assert kernel_names((8, 256, 1024, 14, 14, 3, 3, 1, 1, 1, 1))[1].startswith(
        "conv_mfma_fp4_kernel<KS=16")


@pytest.mark.parametrize("t,small", [
    ((2, 512, 128, 16, 16, 3, 3, 1, 1, 1, 1), True),    # one workgroup per compute unit (256)
    ((2, 513, 128, 16, 16, 3, 3, 1, 1, 1, 1), False),   # a few more
    ((8, 512, 256, 8, 8, 3, 3, 1, 1, 1, 1), True),      # 36 steps
    ((8, 512, 384, 8, 8, 3, 3, 1, 1, 1, 1), True),      # 54 steps
    ((16, 512, 384, 8, 8, 3, 3, 1, 1, 1, 1), True),     # ... two workgroups per compute unit
    ((16, 513, 384, 8, 8, 3, 3, 1, 1, 1, 1), False),
    ((1, 256, 384, 32, 64, 3, 3, 1, 1, 1, 1), False),   # ... a block touches 3 rows of 64
    ((3, 512, 64, 16, 16, 3, 3, 1, 1, 1, 1), True),     # one launch a pass: 1.5
    ((3, 513, 64, 16, 16, 3, 3, 1, 1, 1, 1), False),
    ((3, 512, 64, 16, 16, 5, 5, 1, 1, 2, 2), False),    # ... not with 25 steps
    ((1, 64, 256, 16, 16, 1, 1, 1, 1, 0, 0), False),    # four steps
    ((1, 64, 384, 16, 16, 1, 1, 1, 1, 0, 0), True),     # six
], ids=str)
def test_where_the_kernel_for_few_tiles_begins(monkeypatch, t, small):
    """Its size rule, on either side of each line (256 compute units)."""
    for key in ("XNOR_NN_HIP_CONV", "XNOR_NN_HIP_MFMA_PS", "XNOR_NN_HIP_MFMA_MIX",
                "XNOR_NN_HIP_MFMA_PAIR", "XNOR_NN_HIP_MFMA_PERSIST", "XNOR_NN_HIP_MFMA_SMALL"):
        monkeypatch.delenv(key, raising=False)
    assert kernel_names(t)[1].startswith("conv_mfma_fp4_small_kernel") == small


@pytest.mark.parametrize("t,shallow", [
    ((5, 64, 12, 32, 32, 5, 5, 1, 1, 2, 2), True),      # five steps, thirteen pairs of taps
    ((5, 64, 13, 32, 32, 5, 5, 1, 1, 2, 2), False),     # six
    ((4, 600, 11, 150, 150, 11, 11, 4, 4, 0, 0), True), # 22 of 61
    ((4, 600, 12, 150, 150, 11, 11, 4, 4, 0, 0), False),
    ((33, 32, 3, 32, 32, 3, 3, 1, 1, 1, 1), True),      # 264 tiles of 128 pixels
    ((32, 32, 3, 32, 32, 3, 3, 1, 1, 1, 1), False),
    ((132, 32, 3, 32, 32, 3, 3, 2, 2, 1, 1), False),
    ((8, 32, 6, 32, 32, 7, 7, 1, 1, 3, 3), True),       # few tiles: six steps of 25, one launch
    ((8, 32, 7, 32, 32, 7, 7, 1, 1, 3, 3), False),      # seven
    ((9, 32, 7, 32, 32, 7, 7, 1, 1, 3, 3), True),       # ... not few
    ((49, 97, 5, 8, 8, 7, 7, 2, 2, 3, 3), False),       # many padded rows to 64 pixels
], ids=str)
def test_where_the_kernel_for_few_channels_is_taken(monkeypatch, t, shallow):
    """Its rule, on either side of each line (256 compute units)."""
    for key in ("XNOR_NN_HIP_CONV", "XNOR_NN_HIP_MFMA_PS", "XNOR_NN_HIP_MFMA_MIX",
                "XNOR_NN_HIP_MFMA_PAIR", "XNOR_NN_HIP_MFMA_PERSIST", "XNOR_NN_HIP_MFMA_SMALL",
                "XNOR_NN_HIP_MFMA_GROUPS"):
        monkeypatch.delenv(key, raising=False)
    assert kernel_names(t)[1].startswith("conv_mfma_fp4_shallow_kernel") == shallow


@pytest.mark.parametrize("t,name", [
    ((16, 8, 40, 16, 16, 3, 3, 1, 1, 1, 1), "binarize_nchw_split_kernel"), # 64 tiles of 64 pixels
    ((16, 8, 40, 16, 17, 3, 3, 1, 1, 1, 1), "binarize_nchw_kernel"),       # 68
    ((1, 8, 33, 1, 1, 1, 1, 1, 1, 0, 0), "binarize_nchw_split_kernel"),
    ((1, 8, 32, 1, 1, 1, 1, 1, 1, 0, 0), "binarize_nchw_shallow_kernel"),
    ((1, 8, 8160, 7, 7, 1, 1, 1, 1, 0, 0), "binarize_nchw_split_kernel"),  # as deep as tiles go
    ((1, 8, 8161, 7, 7, 1, 1, 1, 1, 0, 0), "binarize_generic_kernel"),
], ids=str)
def test_where_the_binarize_kernel_for_few_pixels_is_taken(t, name):
    """Its rule, on either side of each line (256 compute units)."""
    assert kernel_names(t)[0] == name


def test_weight_stage_kernel_names():
    """The whole stage in one launch for OIHW filters that fit, four kernels otherwise."""
    name = lambda t, w=capi.FMT_OIHW: kernel_names(
        t, (capi.FMT_NCHW, w, capi.FMT_NCHW), (capi.OP_BINARIZE_WEIGHTS,))[0]
    assert name((1, 8, 1612, 4, 4, 2, 5, 1, 1, 2, 2)) == "binarize_filter_kernel"  # 16120 values
    assert name((1, 8, 1613, 4, 4, 2, 5, 1, 1, 2, 2)) == "pack_weights_kernel"
    assert name((1, 8, 64, 4, 4, 3, 3, 1, 1, 1, 1), capi.FMT_HWIO) == "pack_weights_kernel"


def test_only_new_weights_on_the_gpu_are_vouched_for():
    """forward_on_stream: weights in host memory must not reach a kernel as they are."""
    import torch

    from xnor_nn_amd.convolution import Convolution

    class OnGpu:
        is_cuda = True
        data_ptr = staticmethod(lambda: 64)

    calls = []
    conv = Convolution.__new__(Convolution)
    conv.lib, conv.res, conv._desc_at, conv._res_at = None, capi.Resources(), 1, 2
    conv._forward_pass = lambda *args: calls.append(args) or capi.SUCCESS
    for weights in (None, OnGpu(), torch.zeros(4), np.zeros(4, np.float32), 4096):
        conv.forward_on_stream(OnGpu(), OnGpu(), 3, weights)
    new, vouched = capi.NEW_WEIGHTS | capi.ON_STREAM, capi.DEVICE_POINTERS
    assert [c[:5] for c in calls] == [(1, 2, 64, 64, 3)] * 5
    assert [c[5] for c in calls] == [vouched | capi.ON_STREAM, vouched | new, new, new, new]
