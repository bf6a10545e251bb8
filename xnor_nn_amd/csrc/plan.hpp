// Launch plan and per-descriptor state of the gfx950 implementation.
//
// Takes the place of the reference's Implementation object behind c->state
// (reference src/implementation.hpp:11-27, src/bcast_convolution.cpp:58-117): instead of
// CPU blocking factors (BIC/ABIC/ICO/OCI/OCO) it records the device word layout, the
// launch geometry, the stream and the staging buffers used when the caller hands over
// host pointers.
#pragma once

#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <stdint.h>

#include <atomic>
#include <mutex>
#include <vector>

#include "host_io.hpp"
#include "xnor_nn.h"

// Byte offset that the kernels give a buffer access they want the hardware to drop (a channel
// past the end, a dead pixel): it has to lie outside every buffer it is used with, so the
// kernels that use it take buffers below this size only.
#define XNOR_HIP_DROPPED_OFFSET 0xFFFFFFF0ull

namespace xnor_hip {

// n / d for 32-bit n by multiply-high and shifts; d is fixed on the host.
struct FastDiv {
    uint32_t mul, sh1, sh2, d;
    __host__ static FastDiv make(uint32_t d) {
        FastDiv f{0u, 0u, 0u, d};
        if (d <= 1) return f;
        uint32_t L = 0;
        while ((1ull << L) < d) L++;
        f.mul = (uint32_t)(((1ull << 32) * ((1ull << L) - d)) / d + 1);
        f.sh1 = 1;
        f.sh2 = L - 1;
        return f;
    }
    __host__ __device__ __forceinline__ uint32_t div(uint32_t n) const {
#if defined(__HIP_DEVICE_COMPILE__)
        const uint32_t t = __umulhi(n, mul);
#else
        const uint32_t t = (uint32_t)(((uint64_t)n * mul) >> 32);
#endif
        return (t + ((n - t) >> sh1)) >> sh2;
    }
};

// Geometry shared by all kernels.  Device layouts:
//   bin_src      uint32 [MB*IH*IW][XW]          word j, bit (31-b) = channel 32j+b has its
//                                               sign bit clear; channels >= IC are 0
//   bin_weights  uint32 [OCB][KH*KW][XW][Q]     same bit order; channels >= IC and
//                                               filters >= OC are all ones; followed (at
//                                               wfrag_offset) by the same signs as FP4
//                                               matrix-core fragments when use_mfma is set
//   alpha        float  [OC]
//   a            float  [MB*IH*IW]
//   k            float  [MB*OH*OW]
//   op count     int32  [OH*OW]
struct Geometry {
    int mb, ic, ih, iw, oc, oh, ow, kh, kw, sh, sw, ph, pw;
    int src_fmt, w_fmt, dst_fmt;
    int xw;       // 32-bit words per pixel = ceil(ic/32)
    int q;        // filters per wave in the convolution kernel
    int ocb;      // ceil(oc/q)
    int ihw, ohw; // ih*iw, oh*ow
    uint32_t npix_in, npix_out; // mb*ihw, mb*ohw
    int mfma_groups;            // pixel groups per tile (1, 2, 4): with 128 / 64 filters or fewer
                                // the waves without filters take further pixel blocks instead
    int stream_dst;             // 1: the matrix-core kernel stores its output with the nt bit
    FastDiv div_ihw, div_iw, div_ohw, div_ow;
};

// What the kernel for few tiles needs beside it (kernels_conv_small.hip).
struct SmallPlan {
    int max_rows;     // input pixels a block stages at most
    int ks, nsteps;   // steps per tap (or pair of taps), and in all
    int k_steps;      // what the sums of K count for where the steps are dealt out
    int subs;         // 32-filter blocks
    int row_bytes;    // of an input pixel's FP4 row in LDS
    uint32_t blocks, wfrag_bytes; // 32-pixel blocks
    FastDiv div_xw, div_ks, div_kw, div_subs;
};

// What the kernel for few input channels needs (kernels_conv_shallow.hip), in place of Geometry: less
// to copy per launch.
struct ShallowPlan {
    uint32_t npix_out, npix_in;
    int ic, ih, iw, oc, oh, ow, ohw, kh, kw, sh, sw, ph, pw;
    int prows, pcols;            // rows and columns of an image with the padding its taps reach
    int row_codes, steps;        // bytes of sign bits per kernel row; 64-product steps in all
    int max_rows;                // padded rows a tile stages at most
    int row_words;               // dwords of a padded row's bit string (two spare ones included)
    int row_pixels;              // pixels that share one of them at most
    int row_bytes;               // of a pixel's FP4 row: steps * 32 + 16
    int blocks, blocks_per_wg;   // 32-filter blocks: all, and of one workgroup
    int a_pitch;                 // cells of a padded row's mean|x|, a multiple of the stride
    int a_shares_rows;           // 1: its LDS is that of the operands, which are gathered after it
    int gathers;                 // waves that share the kernel rows of 64 pixels, four rows each
    uint32_t tiles, chunks, units, units_per_xcd; // chunks: of the filters; a unit is a tile with one
    uint32_t wfrag_bytes;
    int nchw, stream;
    FastDiv div_ohw, div_ow, div_prows, div_words, div_ic, div_chunks;
};

// The arguments a kernel begins with, fetched in one go.  Left alone the compiler fetches what an
// early exit compares, waits, and fetches the rest behind it, which is another miss for each cache line
// of the argument block (36 layers 1.4 % faster on average; 32 -> 64 channels 3x3 on 33x33, minibatch
// 20, 8.1 -> 7.8 us a pass, 3 channels 7x7 on 224x224 9.05 -> 8.6, AlexNet conv4 minibatch 64 16.4 -> 16.05).
template <class T> __device__ __forceinline__ void fetch_one(const T v) { asm volatile("" : : "s"(v)); }
template <class... T> __device__ __forceinline__ void fetch_together(const T... v) { (fetch_one(v), ...); }
__device__ __forceinline__ void fetch_together(const FastDiv &d) { fetch_together(d.mul, d.sh1, d.sh2); }

// Mask that keeps the n most significant bits of a word (n in 1..32).
__device__ __forceinline__ uint32_t top_bits(int n) {
    return n >= 32 ? 0xFFFFFFFFu : ~(0xFFFFFFFFu >> n);
}

// FP4 codes of 32 sign bits (set: +1 -> 0x2, clear: -1 -> 0xA): nibble n of dword d is bit 4n + 3 - d.
// Weights are packed in the same order, so any order would do; with this one a word takes eight vector
// instructions, where a table in LDS (one dword per byte of the word) took eight and four reads that
// conflict at random.
__device__ __forceinline__ uint32_t fp4_codes(uint32_t word, int d) {
    return ((~word << d) & 0x88888888u) | 0x22222222u;
}
// The same, zero where `valid` is clear.
__device__ __forceinline__ uint32_t fp4_codes(uint32_t word, uint32_t valid, int d) {
    return (((~word & valid) << d) & 0x88888888u) | ((valid << d) & 0x88888888u) >> 2;
}
// The channel of a packed word (first channel in the highest bit) that nibble stands for.
__host__ __device__ inline int fp4_channel(int d, int n) { return 28 - 4 * n + d; }

// The product that nibble n of dword j of a pixel's operand stands for in that kernel: bit b of
// kernel row kh.  Four kernel rows of row_codes bytes make row_codes words, a word four dwords, and
// nibble n of dword d is the word's bit 4n + 3 - d.
__host__ __device__ inline void shallow_product(int j, int n, int row_codes, int &kh, int &b) {
    const int part = j / (4 * row_codes), i = j - part * 4 * row_codes;
    const int bit = 4 * n + 3 - (i & 3), byte = 4 * (i >> 2) + (bit >> 3), row = byte / row_codes;
    kh = 4 * part + row;
    b = (byte - row * row_codes) * 8 + (bit & 7);
}

// What the host adds to it when a descriptor is initialised: which kernels run and with what
// tiles.  Kernels get the Geometry part (geometry() below) and their own: the argument block is
// copied on every launch and read by every workgroup.
struct Plan : Geometry {
    int bin_waves;              // waves per workgroup of the binarize kernel at most
    int bin_nhwc_lane;          // 1: NHWC input by the one-lane-per-pixel kernel
    int cus;                    // compute units of the device (256 if it cannot be asked)
    int use_mfma;               // 1: stage 3 runs the FP4 matrix-core kernel
    int mfma_ps;                // its tile size in 32-pixel blocks (1..4)
    int mfma_ps_small;          // > 0: a launch with two tile sizes; the later workgroups of an
                                // XCD take this many blocks (see the kernel)
    uint32_t mfma_big_per_xcd;  // ... after this many workgroups with mfma_ps blocks,
    uint32_t mfma_blocks_per_xcd; // out of this many pixel blocks per XCD
    int mfma_persist;           // 1: two workgroups per CU stay and walk over the tiles, taking
    uint32_t mfma_tiles_per_round; // every mfma_tiles_per_round-th tile of their XCD
    uint32_t mfma_rounds;       // rounds of tiles a persistent workgroup walks at most
    int mfma_reverse;           // 1: the second workgroup of a CU walks its tiles last to first
    uint32_t mfma_stagger;      // ... and starts this many sleep periods late
    size_t wfrag_offset;        // byte offset of the FP4 weight fragments in bin_weights
    // the matrix-core kernel's variant and sizes, fixed once by mfma_plan: steps per tap (or
    // per pair of taps), tap pairing, channel parts, input pixels a tile stages at most, LDS
    // bytes per workgroup, bytes of the weight fragments
    int mfma_steps, mfma_pair, mfma_parts, mfma_rows;
    int mfma_long_walk;         // 1: the variant with several groups of weight fragments under way
    int mfma_small;             // 1: few tiles: the small-problem kernel (kernels_conv_small.hip),
    SmallPlan small;            // its part of the plan
    uint32_t mfma_small_lds;    // and its LDS bytes per workgroup
    int one_launch;             // 1: a forward pass on device buffers is that kernel alone
    int mfma_shallow;           // > 0: few channels: the kernel of kernels_conv_shallow.hip with
                                // tiles of this many output pixels,
    ShallowPlan shallow;        // and its part of the plan
    uint32_t mfma_lds, mfma_wbytes;
};
inline const Geometry &geometry(const Plan &p) { return p; }

// First and last input pixel (flattened index) that a tile of the output pixels
// [p_first, p_end) can touch with an in-bounds tap, by whole input rows: from the start of the first
// input row of its first pixel to the end of the last input row of its last pixel (with a stride above 1
// the span also holds the input pixels the stride skips).  What it takes to work out is on the way to the
// first load; the kernel for few tiles, which is bound by that way, takes this one.
__host__ __device__ inline void row_span(const Geometry &g, uint32_t p_first, uint32_t p_end,
        int &lo, int &hi) {
    const uint32_t p_last = p_end - 1;
    const uint32_t i0 = g.div_ohw.div(p_first), i1 = g.div_ohw.div(p_last);
    const int oh0 = (int)g.div_ow.div(p_first - i0 * g.ohw);
    const int oh1 = (int)g.div_ow.div(p_last - i1 * g.ohw);
    int r0 = oh0 * g.sh - g.ph, r1 = oh1 * g.sh - g.ph + g.kh - 1;
    if (r0 < 0) r0 = 0;
    if (r0 > g.ih - 1) r0 = g.ih - 1;
    if (r1 > g.ih - 1) r1 = g.ih - 1;
    if (r1 < 0) r1 = 0;
    lo = (int)(i0 * g.ihw) + r0 * g.iw;
    hi = (int)(i1 * g.ihw) + r1 * g.iw + g.iw - 1;
    if (hi < lo) hi = lo;
}

// The same from the first tap of the first pixel to the last tap of the last pixel.  A first pixel whose
// taps begin above the image has none there, but a pixel of the next row may reach the image's first row
// further left: the span then begins with that row; likewise at the end.  Whole rows are a sixth to a
// third more to stage (64 pixels of a 3x3 kernel on 56x56: up to 280 input pixels instead of 178), and
// wide rows of many channels more than the LDS holds.  Kernel alone, whole rows / this, us: 130 to 70
// channels 3x3 stride 2 on 45x51 6.9 / 6.4 (a pass 11.4 / 11.0), 256 to 128 channels 1x1 stride 2 on
// 56x56 15.9 / 10.7, 224 channels 5x5 on 78x78 16.0 / 15.2, 156 channels on 101x101 39.7 / 37.8, 864 on
// 83x83 226 (the popcount kernel) / 65.  Narrow images without a stride alike, us a pass, whole rows /
// this: 3000 to 128 channels 3x3 on 28x28, minibatch 4, 276.8 (the popcount kernel) / 47.1, 4096 on 14x14,
// 8, 378.6 / 62.5, 2048 to 512 1x1 on 13x13, 96, 60.7 / 55.6, 1024 to 128 3x3 on 10x10, 256, 51.4 / 47.5,
// on 28x28, 8, 26.8 / 24.7; where a tile fits either way there is little between them (512 on 28x28, 32,
// behind a rectifier 38.8 / 38.6; of 155 layers of up to 32 columns one is slower by more than 1.5 %).
__host__ __device__ inline void tile_span(const Geometry &g, uint32_t p_first, uint32_t p_end,
        int &lo, int &hi) {
    const uint32_t p_last = p_end - 1;
    const uint32_t i0 = g.div_ohw.div(p_first), i1 = g.div_ohw.div(p_last);
    const int rem0 = (int)(p_first - i0 * g.ohw), rem1 = (int)(p_last - i1 * g.ohw);
    const int oh0 = (int)g.div_ow.div((uint32_t)rem0), oh1 = (int)g.div_ow.div((uint32_t)rem1);
    int r0 = oh0 * g.sh - g.ph, r1 = oh1 * g.sh - g.ph + g.kh - 1;
    int c0 = (rem0 - oh0 * g.ow) * g.sw - g.pw, c1 = (rem1 - oh1 * g.ow) * g.sw - g.pw + g.kw - 1;
    if (r0 < 0 || c0 < 0) c0 = 0;
    if (r1 > g.ih - 1 || c1 > g.iw - 1) c1 = g.iw - 1;
    if (c0 > g.iw - 1) c0 = g.iw - 1;
    if (c1 < 0) c1 = 0;
    if (r0 < 0) r0 = 0;
    if (r0 > g.ih - 1) r0 = g.ih - 1;
    if (r1 > g.ih - 1) r1 = g.ih - 1;
    if (r1 < 0) r1 = 0;
    lo = (int)(i0 * g.ihw) + r0 * g.iw + c0;
    hi = (int)(i1 * g.ihw) + r1 * g.iw + c1;
    if (hi < lo) hi = lo;
}

// Optional timing of one launch: when both events are set the kernel is launched with them
// attached to its own dispatch, and their difference is the kernel's duration on the GPU (no
// marker packets on the stream, which would cost more than a short kernel takes).
struct KernelEvents {
    hipEvent_t start = nullptr, stop = nullptr;
};

template <class K, class... A>
inline void launch_kernel(K kernel, dim3 grid, dim3 block, size_t lds, hipStream_t s,
        const KernelEvents &ev, A... args) {
    if (ev.start != nullptr && ev.stop != nullptr)
        hipExtLaunchKernelGGL(kernel, grid, block, (uint32_t)lds, s, ev.start, ev.stop, 0,
                args...);
    else
        hipLaunchKernelGGL(kernel, grid, block, lds, s, args...);
}

// More than 64 KB of dynamic LDS has to be asked for: once per kernel, device and size.  One
// static object per kernel remembers what has been granted; the attribute and the record of it
// change together, under the lock, and only grow.
struct LdsGrant {
    std::atomic<size_t> have[64];
    std::mutex mu;
    hipError_t ask(const void *kernel, size_t lds) {
        if (lds <= 64 * 1024) return hipSuccess;
        int dev = 0;
        if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return hipErrorInvalidDevice;
        if (lds <= have[dev].load(std::memory_order_acquire)) return hipSuccess;
        std::lock_guard<std::mutex> lock(mu);
        if (lds <= have[dev].load(std::memory_order_relaxed)) return hipSuccess;
        const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
                (int)lds);
        if (e == hipSuccess) have[dev].store(lds, std::memory_order_release);
        return e;
    }
};

// Event pairs for xnor_nn_hip_time_kernels: one ring per timed stage.
struct KernelTimer {
    std::vector<KernelEvents> ring;
    size_t launches = 0; // since timing was switched on
    KernelEvents next() {
        if (ring.empty()) return KernelEvents{};
        return ring[launches++ % ring.size()];
    }
};

struct State {
    Plan g;
    hipStream_t stream = nullptr;
    // Held for the length of every executor call: two host threads may share one descriptor
    // (each with a resource table of its own), and the staging buffers below, the stream and
    // the order in which a call's launches and copies are enqueued belong to one call at a
    // time.  Recursive: xnor_nn_hip_forward_pass holds it over the executors it calls.
    std::recursive_mutex mu;
    // staging buffers for host-side user tensors (allocated on first use, a multiple of 16 bytes)
    // and what moves the bytes
    void *stage_src = nullptr, *stage_weights = nullptr, *stage_dst = nullptr;
    HostIo io;
    // partial sums of xnor_nn_binarize_weights_float (allocated on first use)
    float *float_parts = nullptr;
    // Stage fusion (xnor_nn_hip_set_stage_fusion): binarize_data hands mean|x| to the
    // calculate_k that follows it, and calculate_k leaves its box filter to the matrix-core
    // convolution.  What is handed over is recorded per resource table, not here (api.hip).
    bool fuse_stages = true;
    bool verbose = false;
    // Orders this descriptor's stream with another one (a box filter owed by a descriptor
    // that runs on another stream); created on first use, under mu.
    hipEvent_t order_before = nullptr, order_after = nullptr;
    KernelTimer time_binarize, time_convolution; // empty unless timing is switched on
};

inline State *state_of(const xnor_nn_convolution_t *c) {
    return reinterpret_cast<State *>(c->state);
}

// Kernel launchers (one per stage); each returns the hipError_t of the launch.
void binarize_plan(Plan &g); // bin_waves, bin_nhwc_lane
hipError_t launch_binarize_data(const Plan &g, const float *x, uint32_t *bits,
        float *a_or_null, hipStream_t s, const KernelEvents &ev = KernelEvents{});
hipError_t launch_mean_abs(const Plan &g, const float *x, float *a, hipStream_t s);
// Whether it can be done together with the weight stage, and that.
bool weights_join_binarize(const Plan &g);
hipError_t launch_binarize_data_and_weights(const Plan &g, const float *x, uint32_t *bits, float *a,
        const float *w, uint32_t *wbits, uint32_t *frag_or_null, float *alpha, int32_t *opc,
        hipStream_t s);
hipError_t launch_box_filter(const Plan &g, const float *a, float *k, hipStream_t s);
// calibration: one pass of plain 16-byte reads over bytes / 16 * 16 bytes of device memory
hipError_t launch_plain_read(const void *buf, size_t bytes, hipStream_t s,
        const KernelEvents &ev = KernelEvents{});
// (frag_or_null: where the matrix-core kernel's fragments go, when it applies)
hipError_t launch_binarize_weights(const Plan &g, const float *w, uint32_t *bits,
        uint32_t *frag_or_null, float *alpha, int32_t *opc, hipStream_t s);
hipError_t launch_convolution(const Plan &g, const uint32_t *xbits,
        const uint32_t *wbits, const float *alpha, const float *k, const int32_t *opc,
        float *dst, int32_t *popc_or_null, hipStream_t s,
        const KernelEvents &ev = KernelEvents{});
// sign(w) * mean(w); parts: weights_float_parts() floats of device memory for partial sums
int weights_float_parts();
hipError_t launch_weights_float(const float *from, float *to, size_t n, float *parts,
        hipStream_t s);
// device address of the library's own partial-sum array on the current GPU (static device
// memory: nothing is allocated)
hipError_t weights_float_scratch(float **out);
// Decides whether the matrix-core kernel takes the problem and fills use_mfma, mfma_ps and
// the mfma_* fields and the kernels' own plans (everything the launch needs: a forward call takes
// its arguments from here).
void mfma_plan(Plan &g);
const char *mfma_kernel_name(const Plan &g);
size_t mfma_weight_bytes(const Plan &g);
hipError_t launch_pack_weights_fp4(const Plan &g, const float *w, uint32_t *frag,
        hipStream_t s);
// With a_or_null set, the kernel ignores k, computes the K plane itself from mean|x| (the
// box filter of stage 2) and also stores it to k_out.
hipError_t launch_convolution_mfma(const Plan &g, const uint32_t *xbits,
        const uint32_t *wfrag, const float *alpha, const float *k,
        float *dst, int32_t *popc_or_null, const float *a_or_null, float *k_out,
        hipStream_t s, const KernelEvents &ev = KernelEvents{});
// calibration: `workgroups` x 4 waves, each issuing 8 * iterations FP4 matrix instructions
// (32x32x64) on register-resident +-1 operands
hipError_t launch_mfma_only(int workgroups, int iterations, hipStream_t s);
const char *convolution_kernel_name(const Plan &g);
// The matrix-core kernel for launches of few tiles (filled in by mfma_plan: g.mfma_small).
bool small_kernel_applies(const Plan &g, int *rows, uint32_t *lds);
SmallPlan small_plan(const Plan &g, int rows);
bool one_launch_applies(const Plan &g);
hipError_t launch_forward_small(const Plan &g, const float *x, uint32_t *bits_out, float *a_out,
        const uint32_t *wfrag, const float *alpha, float *k_out, float *dst, hipStream_t s);
hipError_t launch_convolution_small(const Plan &g, const uint32_t *xbits,
        const uint32_t *wfrag, const float *alpha, const float *k, float *dst,
        const float *a_or_null, float *k_out, hipStream_t s,
        const KernelEvents &ev = KernelEvents{});
// The matrix-core kernel for few input channels (chosen by mfma_plan: g.mfma_shallow).
bool shallow_plan(Plan &g); // mfma_shallow, shallow and the sizes that depend on them
hipError_t launch_pack_weights_shallow(const Plan &g, const float *w, uint32_t *frag,
        hipStream_t s);
hipError_t launch_convolution_shallow(const Plan &g, const uint32_t *xbits,
        const uint32_t *wfrag, const float *alpha, const float *k, float *dst, int32_t *popc,
        const float *a_or_null, float *k_out, hipStream_t s,
        const KernelEvents &ev = KernelEvents{});
const char *binarize_kernel_name(const Plan &g);
const char *weights_kernel_name(const Plan &g); // the first of four, or the only one

int pick_q(int oc, int xw);

} // namespace xnor_hip
