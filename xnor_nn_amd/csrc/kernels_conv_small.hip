// Stage 3 on the matrix cores for launches of few tiles (small batches): the same FP4
// implicit GEMM as kernels_conv_mfma.hip, cut the other way; and, for inputs of few channels, the
// whole forward pass in one launch.
// Semantics: reference src/default/bcast_convolution_default.cpp:60-105.
//
// The large-launch kernel gives a workgroup 32*PS pixels x 256 filters and every wave all
// taps of its 64 filters: at minibatch 1 of AlexNet conv4 that is 6 workgroups on a chip of
// 256 compute units, each wave walking 54 steps one behind the other with the latency of a
// weight fetch between the groups.  Here a workgroup is one block of 32 pixels x ONE block of
// 32 filters, and its waves split the (tap, channel step) sequence between them: 48
// workgroups for that problem, 6 or 7 matrix instructions per wave.  The partial sums are
// exact integers in FP32, so the waves' accumulators add up to the same bits in any order; they
// meet in LDS and every wave scales and stores an eighth of the block.
//
// Nothing is hand-scheduled: a wave asks for the input and then for its first eight weight fragments
// (they arrive while the input is staged; with eight waves they are usually all it needs; asked for
// first they held the input up, whose words can be waited for only after them), reads an operand
// while the step before is multiplied, and the waits are the compiler's.  What bounds it is one
// latency after the other: arguments, input, barrier, operands, barrier, stores.  That order, us a
// pass: AlexNet conv4, minibatch 1, 9.6 -> 9.5; 64 channels on 56x56 7.9 -> 7.4; 512 -> 1000 filters
// on one pixel 10.1 -> 9.4; eight images of conv4 as before (12.0).
//
// FUSED (up to 64 channels): the workgroup starts from the float input.  A lane takes a pixel of
// the tile's span: sign words straight to FP4 rows in LDS, mean|x| (in channel order, the
// reference's) beside them.  Workgroups of the first filter block also store the packed words and
// mean|x| of their share of the input, so that the pass leaves behind what the separate stages
// leave.  Every filter block repeats the packing, which costs less than a second launch as long
// as the launch is small: a pass is then bound by the host's 2.8 us per launch no more than by
// the GPU.
#include <cstdlib>
#include <type_traits>

#include "box_sum.hpp"
#include "plan.hpp"
#include "tap_walk.hpp"

namespace xnor_hip {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int SMALL_RING = 8;         // weight fragments in flight per wave
constexpr uint32_t SMALL_DROP = 0xFFFFFFF0u;

__device__ __forceinline__ v16f small_mfma_fp4(const v4i a, const v4i b, const v16f c) {
    const v8i a8 = {a.x, a.y, a.z, a.w, 0, 0, 0, 0};
    const v8i b8 = {b.x, b.y, b.z, b.w, 0, 0, 0, 0};
    // cbsz = blgp = 4: FP4 (E2M1) operands; zero scale operands select the unscaled form
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a8, b8, c, 4, 4, 0, 0, 0, 0);
}

__device__ __forceinline__ v4i small_codes(const uint32_t word) {
    return v4i{(int)fp4_codes(word, 0), (int)fp4_codes(word, 1), (int)fp4_codes(word, 2),
        (int)fp4_codes(word, 3)};
}

// LDS: [rows: zero row + max_rows rows of row_bytes][mean|x| of the staged
// pixels + one slot of zero][partial sums]
// PAIR: the weight fragments of kernels_conv_mfma.hip's paired taps (an odd number KS of words
// per pixel: two taps share KS steps, and the two halves of a wave may be at different taps).
// WORDS: words per pixel that FUSED takes (0: from the packed input).
template <int WAVES, int WORDS, bool PAIR>
__global__ __launch_bounds__(64 * WAVES)
void conv_mfma_fp4_small_kernel(const uint32_t *__restrict__ xbits, const v4i *__restrict__ wfrag,
        const float *__restrict__ alpha, const float *__restrict__ kplane,
        float *__restrict__ dst, const Geometry g, const SmallPlan s,
        const float *__restrict__ a_plane, float *__restrict__ k_out, const float inv_khw,
        const float *__restrict__ x, uint32_t *__restrict__ bits_out, float *__restrict__ a_out,
        const float inv_ic) {
    constexpr bool FUSED = WORDS > 0;
    constexpr int THREADS = 64 * WAVES, KEEP = 16 / WAVES; // accumulator registers a wave finishes
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char *rows = smem;
    float *a_lds = reinterpret_cast<float *>(rows + (size_t)(1 + s.max_rows) * s.row_bytes);
    float *parts = a_lds + ((s.max_rows + 1 + 3) & ~3);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int half = lane >> 5;
    const uint32_t block = s.subs == 1 ? blockIdx.x : s.div_subs.div(blockIdx.x);
    const int sub = (int)(blockIdx.x - block * (uint32_t)s.subs); // 32-filter block
    const uint32_t p_first = block * 32u, p_limit = g.npix_out;
    const bool fuse_k = FUSED || a_plane != nullptr; // uniform
    // this wave's share of the steps; the last wave sums K as well
    const int share = s.nsteps + (fuse_k ? s.k_steps : 0);
    const int s_lo = min((wave * share) / WAVES, s.nsteps);
    const int s_hi = min(((wave + 1) * share) / WAVES, s.nsteps);

    // ---- the input: which pixels the tile touches; their words and mean|x| are asked for first (a
    // buffer ends with the tile's run: with a branch around each load the compiler would wait for one
    // after the other)
    int lo, hi;
    row_span(g, p_first, min(p_first + 32u, p_limit), lo, hi);
    const int nrows = min(hi - lo + 1, s.max_rows), nitems = nrows * g.xw;
    const uint32_t *run = xbits + (size_t)lo * g.xw;
    [[maybe_unused]] uint32_t word[4];
    [[maybe_unused]] float a_early = 0.f;
    if constexpr (!FUSED) {
        auto load = [&](const void *from, int dwords, int i) {
            return __builtin_amdgcn_raw_buffer_load_b32(__builtin_amdgcn_make_buffer_rsrc(
                    const_cast<void *>(from), 0, dwords * 4, 0x00020000), i * 4, 0, 0);
        };
#pragma unroll
        for (int u = 0; u < 4; u++) word[u] = load(run, nitems, u * THREADS + tid);
        if (fuse_k) a_early = __uint_as_float(load(a_plane + lo, nrows, tid));
    }

    // ---- weight fragments: [32-filter block][tap][step][lane]; the first ring is asked for now
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<v4i *>(wfrag), 0, (int)s.wfrag_bytes, 0x00020000);
    const uint32_t wvoff = (uint32_t)lane * 16u;
    const uint32_t wbase = (uint32_t)sub * (uint32_t)s.nsteps * 1024u;
    auto fragment = [&](int st) { // a step past the wave's share reads outside the buffer: zeros
        return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf,
                st < s_hi ? wvoff : SMALL_DROP, st < s_hi ? wbase + (uint32_t)st * 1024u : 0u, 0));
    };
    v4i ring[SMALL_RING];
#pragma unroll
    for (int i = 0; i < SMALL_RING; i++) ring[i] = fragment(s_lo + i);

    // the alphas of the filters this lane will scale (register i of the block is filter
    // 8*(i/4) + 4*half + i%4), asked for now so that the epilogue does not wait
    const int i0 = KEEP * wave, f0 = sub * 32 + 8 * (i0 >> 2) + 4 * half + (i0 & 3);
    float al[KEEP];
#pragma unroll
    for (int ii = 0; ii < KEEP; ii++)
        al[ii] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(alpha), 0, g.oc * 4, 0x00020000),
                (f0 + ii) * 4, 0, 0));

    // ---- the block's pixels, one per lane (both halves of the wave hold the same 32)
    const uint32_t pix = p_first + (lane & 31);
    const bool live = pix < p_limit;
    const uint32_t pc = live ? pix : p_limit - 1;
    const uint32_t img = g.div_ohw.div(pc), rem = pc - img * g.ohw;
    const int oh = (int)g.div_ow.div(rem), ow = (int)rem - oh * g.ow;
    const int ih0 = oh * g.sh - g.ph, iw0 = ow * g.sw - g.pw; // input pixel of tap (0,0)
    const int in0 = (int)(img * g.ihw) + ih0 * g.iw + iw0 - lo;
    const uint32_t rowmask = live ? taps_inside(ih0, g.ih, g.kh) : 0u;
    const uint32_t colmask = taps_inside(iw0, g.iw, g.kw);
    // byte offsets into `rows` of the row of tap (0,0) of the lane's pixel; row 0 is zero
    const int base_off = (1 + in0) * s.row_bytes;

    // ---- staging: zero row, mean|x|, FP4 rows
    const float k_read = fuse_k ? 0.f : kplane[live ? pix : 0]; // asked for early
    for (int i = tid; i < s.row_bytes / 4; i += THREADS) reinterpret_cast<uint32_t *>(rows)[i] = 0;
    if (tid == 0) a_lds[s.max_rows] = 0.f;
    if constexpr (FUSED) {
        // The input pixels this workgroup packs: the tile's span and, in the first filter block,
        // all from here to where the next tile's span begins (every input pixel is in exactly one
        // such stretch).
        const bool writes = sub == 0; // uniform
        int from = lo, to = lo + nrows, w_from = 0, w_to = 0;
        if (writes) {
            int nlo, nhi;
            w_from = block == 0 ? 0 : lo;
            if (block + 1 < s.blocks) row_span(g, p_first + 32u, min(p_first + 64u, p_limit), nlo, nhi);
            else nlo = (int)g.npix_in;
            w_to = nlo;
            from = min(from, w_from);
            to = max(to, w_to);
        }
        const bool planar = g.src_fmt == xnor_nn_data_format_nchw;
        const uint32_t step = planar ? (uint32_t)g.ihw * 4u : 4u; // bytes from a channel to the next
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(x), 0, (int)(g.npix_in * (uint32_t)g.ic * 4u), 0x00020000);
        for (int p0 = from; p0 < to; p0 += THREADS) {
            const int p = p0 + tid;
            const uint32_t q = p < to ? (uint32_t)p : (uint32_t)(to - 1);
            const uint32_t im = g.div_ihw.div(q);
            const uint32_t off = (planar ? im * (uint32_t)(g.ic * g.ihw) + (q - im * g.ihw)
                                         : q * (uint32_t)g.ic) * 4u;
            float v[WORDS * 32];
#pragma unroll
            for (int c = 0; c < WORDS * 32; c++)
                v[c] = c < g.ic ? __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        src, off, (uint32_t)c * step, 0)) : 0.f; // (uniform) |+0| adds nothing
            float acc = 0.f;
            uint32_t word[WORDS];
#pragma unroll
            for (int j = 0; j < WORDS; j++) {
                uint32_t neg = 0; // sign bits, first channel ends up in the MSB
#pragma unroll
                for (int i = 0; i < 32; i++) {
                    const float t = v[32 * j + i];
                    neg = __builtin_amdgcn_alignbit(neg, __float_as_uint(t), 31);
                    acc = __fadd_rn(acc, __fmul_rn(__builtin_fabsf(t), inv_ic));
                }
                const int left = g.ic - 32 * j;
                word[j] = ~neg & (left >= 32 ? 0xFFFFFFFFu : ~(0xFFFFFFFFu >> left));
            }
            if (p >= to) continue;
            if (p >= lo && p < lo + nrows) {
                a_lds[p - lo] = acc;
#pragma unroll
                for (int j = 0; j < WORDS; j++)
                    *reinterpret_cast<v4i *>(rows + (size_t)(1 + p - lo) * s.row_bytes + j * 16)
                        = small_codes(word[j]);
            }
            if (writes && p >= w_from && p < w_to) {
                a_out[p] = acc;
#pragma unroll
                for (int j = 0; j < WORDS; j++) bits_out[(size_t)p * WORDS + j] = word[j];
            }
        }
    } else {
        auto expand = [&](int i, uint32_t w) { // item i of the run -> 32 FP4 codes of its row
            const int r = (int)s.div_xw.div((uint32_t)i), j = i - r * g.xw;
            *reinterpret_cast<v4i *>(rows + (size_t)(1 + r) * s.row_bytes + j * 16) = small_codes(w);
        };
#pragma unroll
        for (int u = 0; u < 4; u++)
            if (u * THREADS + tid < nitems) expand(u * THREADS + tid, word[u]);
        for (int i = 4 * THREADS + tid; i < nitems; i += THREADS) expand(i, run[i]);
        if (fuse_k) {
            if (tid < nrows) a_lds[tid] = a_early;
            for (int i = THREADS + tid; i < nrows; i += THREADS) a_lds[i] = a_plane[lo + i];
        }
    }
    __syncthreads();

    // ---- this wave's steps: two accumulators in turn (the sums are exact, any order).  The lane's
    // operand of step st: word 2*(st % KS) + half of the words of its tap (PAIR: of the 2*KS words
    // of a pair of taps).
    v16f acc0, acc1;
#pragma unroll
    for (int i = 0; i < 16; i++) acc0[i] = acc1[i] = 0.f;
    auto row_of_tap = [&](int t) { // a tap outside the image: the zero row
        const int kh = (int)s.div_kw.div((uint32_t)t), kw = t - kh * g.kw;
        const uint32_t ok = (rowmask >> kh) & (colmask >> kw) & 1u;
        return ok ? base_off + (kh * g.iw + kw) * s.row_bytes : 0;
    };
    const int taps = g.kh * g.kw;
    const int unit0 = (int)s.div_ks.div((uint32_t)s_lo);
    int unit = unit0, cs = s_lo - unit0 * s.ks; // uniform
    int first_row = 0, second_row = 0;
    auto enter_unit = [&]() {
        if constexpr (PAIR) {
            first_row = 2 * unit < taps ? row_of_tap(2 * unit) : 0;
            second_row = 2 * unit + 1 < taps ? row_of_tap(2 * unit + 1) : 0;
        } else {
            first_row = row_of_tap(unit < taps ? unit : 0);
        }
    };
    enter_unit();
    auto operand = [&]() {
        const int w = 2 * cs + half;
        const int at = PAIR ? (w < s.ks ? first_row + w * 16 : second_row + (w - s.ks) * 16)
                            : first_row + w * 16;
        return *reinterpret_cast<const v4i *>(rows + at);
    };
    v4i ahead = operand(); // read while the step before is multiplied
    for (int st = s_lo; st < s_hi; st += SMALL_RING) {
#pragma unroll
        for (int i = 0; i < SMALL_RING; i++) {
            if (st + i < s_hi) { // uniform
                const v4i b = ahead;
                if (++cs == s.ks) {
                    cs = 0;
                    unit++;
                    enter_unit(); // (past the last: some row of the tile, not used)
                }
                ahead = operand();
                if (i & 1) acc1 = small_mfma_fp4(ring[i], b, acc1);
                else acc0 = small_mfma_fp4(ring[i], b, acc0);
                ring[i] = fragment(st + i + SMALL_RING);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) acc0[i] += acc1[i];

    // ---- the partial sums meet in LDS: a wave keeps KEEP registers and gets the other waves'
    // values for them
#pragma unroll
    for (int i = 0; i < 16; i++)
        if (i / KEEP != wave) parts[(wave * 16 + i) * 64 + lane] = acc0[i]; // uniform
    // ---- K of the lane's pixel (box_sum.hpp): the last wave's, where it keeps registers itself
    float kv = k_read;
    float *k_lds = parts + (WAVES - 1) * (16 + KEEP) * 64;
    if (fuse_k && wave == WAVES - 1) {
        kv = box_sum<true>(a_lds, in0, s.max_rows, rowmask, colmask, g.kh, g.kw, g.iw, inv_khw);
        k_lds[lane] = kv;
        if (sub == 0 && lane < 32 && live) k_out[pix] = kv;
    }

    __syncthreads();
    if (fuse_k) kv = k_lds[lane];
    float sum[KEEP];
#pragma unroll
    for (int ii = 0; ii < KEEP; ii++) {
        float v = 0.f;
#pragma unroll
        for (int q = 0; q < WAVES; q++)
            if (q == wave) v = acc0[KEEP * q + ii]; // uniform
#pragma unroll
        for (int q = 0; q < WAVES; q++)
            if (q != wave) v += parts[(q * 16 + i0 + ii) * 64 + lane]; // uniform
        sum[ii] = v; // = 2*popc - n, exactly
    }

    // ---- epilogue: dst = fl(fl((float)(2*popc - n) * alpha) * k), every product rounded
    const bool nchw = g.dst_fmt == xnor_nn_data_format_nchw;
#pragma unroll
    for (int ii = 0; ii < KEEP; ii++) {
        const int f = f0 + ii;
        if (f < g.oc && live) {
            const float out = __fmul_rn(__fmul_rn(sum[ii], al[ii]), kv);
            const size_t at = nchw ? ((size_t)img * g.oc + f) * g.ohw + rem
                                   : (size_t)pix * g.oc + f;
            dst[at] = out;
        }
    }
}

// Waves per workgroup: eight from twelve steps on (kernel plus binarize kernel, us with 4 / 8 waves:
// 384 channels 3x3 (54 steps) 10.8 / 10.2, 48 channels 7x7 (49) 12.5 / 11.1, 128 channels 3x3 (18)
// 9.5 / 8.8, 64 channels 3x3 (9) 8.1 / 8.4).
int small_waves(const Plan &g) {
    const int nsteps = (g.mfma_pair ? (g.kh * g.kw + 1) / 2 : g.kh * g.kw) * g.mfma_steps;
    return nsteps >= 12 ? 8 : 4;
}

int small_row_bytes(const Plan &g) {
    // an odd number of 16-byte words per row spreads the fragment reads over the banks
    return g.mfma_pair ? g.xw * 16 : g.mfma_steps * 32 + 16;
}

} // namespace

// (once the rest of the plan is made)
SmallPlan small_plan(const Plan &g, int rows) {
    SmallPlan s{};
    s.max_rows = rows;
    s.ks = g.mfma_steps;
    s.nsteps = (g.mfma_pair ? (g.kh * g.kw + 1) / 2 : g.kh * g.kw) * g.mfma_steps;
    // The last wave sums K besides its steps, so it gets fewer: by half a step's time per tap, at most by
    // all that the others can take evenly.  us of the kernel with all waves summing it / one, with as many
    // steps / one, with fewer: 11x11 stride 4, 16 channels on 85x86, minibatch 3, 10.1 / 8.5 / 7.2; 7x7 of 19
    // on 36x39 6.2 / 6.3 / 5.5; 5x5 of 208 on 59x59, minibatch 1, 6.4 / 6.6 / 6.0; 3x3 of 384 on 13x13,
    // minibatch 1, 5.1 / 5.2 / 4.9 (a quarter 5.0, a whole step 4.8), 512 on 28x28 7.5 / 7.3 / 7.0.
    const int waves = small_waves(g), even = (s.nsteps + waves - 2) / (waves - 1);
    s.k_steps = (g.kh * g.kw + 1) / 2 < even ? (g.kh * g.kw + 1) / 2 : even;
    s.subs = (g.oc + 31) / 32;
    s.row_bytes = small_row_bytes(g);
    s.blocks = (g.npix_out + 31) / 32;
    s.wfrag_bytes = g.mfma_wbytes;
    s.div_xw = FastDiv::make((uint32_t)g.xw);
    s.div_ks = FastDiv::make((uint32_t)g.mfma_steps);
    s.div_subs = FastDiv::make((uint32_t)s.subs);
    s.div_kw = FastDiv::make((uint32_t)g.kw);
    return s;
}

// Every filter block repeats the packing of what its pixels touch, `rows` input pixels: in one launch up
// to 1024 words.  us a pass, one launch / two, on the device and through the torch module, whose host part
// is 3 us for two launches more than for one (on a machine where two launches are bound by 3.7 and 5.4):
//   448 words  64 channels 3x3 on 56x56                4.3 / 3.9
//   588        64 3x3 stride 2 on 42x42, minibatch 4   4.7 / 3.8   4.7 / 5.5
//   850        64 3x3 stride 2 on 85x85                5.0 / 3.9   5.0 / 5.6
//   1530       64 7x7 stride 2 on 85x85                5.6 / 4.2   5.6 / 5.5
//   1932       64 11x11 stride 4 on 42x42, 4           6.7 / 5.0   6.8 / 5.4
//   3360       64 11x11 stride 4 on 112x112, 4        11.0 / 6.7  10.9 / 6.7
static bool one_launch_pays(const Plan &g, int rows) { return rows * g.xw <= 1024; }

// Which problems take this kernel: one channel part and so few (pixel block, filter block) pairs,
// a workgroup each, that the large-launch kernel would leave most of the chip idle.  Both were
// timed on 150 problems (0.2 to 3 pairs per compute unit, 1x1 to 5x5, 17 to 1024 channels, 16 to
// 768 filters; us a pass, large-launch / this):
//   up to one pair per compute unit this kernel is ahead, by 1.06 to 1.55 (544 channels 3x3
//   24.1 / 15.5), beyond it a second workgroup waits for the first and the large tiles are ahead
//   (64 channels 5x5 on 12x12, 1.4 pairs: 10.8 / 12.6; 128 channels 3x3 on 22x22, 1.2: 9.4 / 10.4);
//   with 48 steps or more in a walk, where the large-launch kernel is one long chain, two per
//   compute unit while a block stages 112 input pixels at most (1000 channels 3x3 on 17x17, 2.0
//   pairs: 17.7 / 15.5; conv4 of AlexNet, minibatch 12: 7.6 / 7.2 in the kernel; with more to stage
//   2.0 pairs of 602 channels on 26x26: 19.7 / 20.6, 1.75 of 660 on 45x45: 27.3 / 30.8);
//   with 48 steps of 25 taps or more 1.75 per compute unit, whatever a block stages: the other waves do
//   not wait for the sums of K here (us in the kernel, 1.7 pairs: 256 channels 7x7 on 28x28 17.5 / 10.4,
//   100 on 28x28 10.5 / 8.4, 256 channels 5x5 on 50x50 11.2 / 8.7, 40 channels 11x11 stride 4 on 150x150
//   19.0 / 16.0, 24 on 227x227 19.4 / 16.4, 48 on 110x110 17.3 / 15.9; 2.2 pairs: 48 channels 7x7 on 19x19
//   7.8 / 9.7, 100 10.2 / 10.9, 200 channels 5x5 10.6 / 10.5);
//   with up to 64 channels and a short walk the pass is one launch here, which saves the host
//   more than the kernel loses (1.1 pairs: 8.6 / 9.4 on the device, 11.4 / 8.5 through the torch
//   module): 1.5 pairs;
//   walks of up to four steps are not worth splitting (104 channels 1x1, 0.7 pairs: 7.8 / 8.3).
// XNOR_NN_HIP_MFMA_SMALL=0|1 overrides the size rule (for measurements).
bool small_kernel_applies(const Plan &g, int *rows_out, uint32_t *lds_out) {
    if (!g.use_mfma || g.mfma_parts > 1) return false;
    const uint32_t blocks = (g.npix_out + 31) / 32;
    const uint32_t subs = (uint32_t)(g.oc + 31) / 32;
    const uint64_t pairs = (uint64_t)blocks * subs, cus = (uint64_t)g.cus;
    const int walk = (g.mfma_pair ? (g.kh * g.kw + 1) / 2 : g.kh * g.kw) * g.mfma_steps;
    // input pixels a block of 32 output pixels touches at most (blocks start at multiples of 32)
    int most = g.kw > 7 ? 2 : 1; // (the sums of K read up to ten floats ahead of mean|x|: rows lie there)
    const uint32_t look = blocks < (uint32_t)g.ohw + 1 ? blocks : (uint32_t)g.ohw + 1;
    auto see = [&](uint32_t b) {
        int lo, hi;
        row_span(g, b * 32u, b * 32u + 32u < g.npix_out ? b * 32u + 32u : g.npix_out, lo, hi);
        if (hi - lo + 1 > most) most = hi - lo + 1;
    };
    for (uint32_t b = 0; b < look; b++) see(b);
    see(blocks - 1);
    const bool one_launch = g.xw <= 2 && walk < 16 && one_launch_pays(g, most);
    bool take = one_launch ? 2 * pairs <= 3 * cus
        : walk >= 48 && most <= 112 ? pairs <= 2 * cus
        : walk >= 48 && g.kh * g.kw >= 25 ? 4 * pairs <= 7 * cus : walk > 4 && pairs <= cus;
    // paired taps: from packed words only on long walks (160 channels 5x5, 65 steps: 11.2 us a pass
    // against 13.5; 96 channels 3x3, 15 steps: 9.1 against 8.7 in the large kernel)
    if (g.mfma_pair && g.xw > 1 && walk < 24) take = false;
    // a tile size, tap pairing, tile mix or persistent workgroups asked for by name mean the
    // other kernel
    if (getenv("XNOR_NN_HIP_MFMA_PS") || getenv("XNOR_NN_HIP_MFMA_MIX")
            || getenv("XNOR_NN_HIP_MFMA_PERSIST") || getenv("XNOR_NN_HIP_MFMA_PAIR"))
        take = false;
    if (const char *e = getenv("XNOR_NN_HIP_MFMA_SMALL")) take = e[0] == '1';
    if (!take) return false;
    const size_t lds = (1 + (size_t)most) * small_row_bytes(g)
        + (((size_t)most + 1 + 3) & ~(size_t)3) * 4 + small_waves(g) * (size_t)(16 * 64 * 4);
    if (lds > 160 * 1024) return false;
    if (rows_out) *rows_out = most;
    if (lds_out) *lds_out = (uint32_t)lds;
    return true;
}

// Whether a forward pass on device buffers may run the one-launch form: up to 64 channels, not too much to
// pack, 32-bit offsets into the input (with room for the dropped one).  Measured per pass, device-bound: 32
// channels 3x3 on 14x14, minibatch 1: 7.0 us against 8.2 for two launches, 64 channels on 56x56:
// 8.1 against 8.5; called from Python through the torch module 8.5 against 11.4 (the host's part).
bool one_launch_applies(const Plan &g) {
    return g.mfma_small && g.xw <= 2 && one_launch_pays(g, g.small.max_rows)
        && (uint64_t)g.npix_in * (uint64_t)g.ic * 4u < XNOR_HIP_DROPPED_OFFSET;
}

#define XNOR_SMALL(WAVES_, WORDS_, PAIR_) \
    do { \
        static LdsGrant grant; \
        const auto kernel = conv_mfma_fp4_small_kernel<WAVES_, WORDS_, PAIR_>; \
        const hipError_t e = grant.ask((const void *)kernel, g.mfma_small_lds); \
        if (e != hipSuccess) return e; \
        launch_kernel(kernel, dim3(s.blocks * (uint32_t)s.subs), dim3(64 * WAVES_), \
                (size_t)g.mfma_small_lds, stream, ev, xbits, wf, alpha, k, dst, geometry(g), s, \
                a_or_null, k_out, 1.f / g.kh / g.kw, x, bits_out, a_out, 1.f / g.ic); \
    } while (0)

hipError_t launch_convolution_small(const Plan &g, const uint32_t *xbits,
        const uint32_t *wfrag, const float *alpha, const float *k, float *dst,
        const float *a_or_null, float *k_out, hipStream_t stream, const KernelEvents &ev) {
    const SmallPlan &s = g.small;
    const v4i *wf = reinterpret_cast<const v4i *>(wfrag);
    const float *x = nullptr;
    uint32_t *bits_out = nullptr;
    float *a_out = nullptr;
    if (small_waves(g) == 8) {
        if (g.mfma_pair) XNOR_SMALL(8, 0, true);
        else XNOR_SMALL(8, 0, false);
    } else {
        if (g.mfma_pair) XNOR_SMALL(4, 0, true);
        else XNOR_SMALL(4, 0, false);
    }
    return hipGetLastError();
}

// A whole forward pass (one_launch_applies): from the float input, leaving packed words, mean|x|
// and K behind like the separate stages.
hipError_t launch_forward_small(const Plan &g, const float *x, uint32_t *bits_out, float *a_out,
        const uint32_t *wfrag, const float *alpha, float *k_out, float *dst, hipStream_t stream) {
    const SmallPlan &s = g.small;
    const v4i *wf = reinterpret_cast<const v4i *>(wfrag);
    const uint32_t *xbits = nullptr;
    const float *k = nullptr, *a_or_null = nullptr;
    const KernelEvents ev{};
    if (small_waves(g) == 8) {
        if (g.mfma_pair) XNOR_SMALL(8, 1, true);
        else if (g.xw == 1) XNOR_SMALL(8, 1, false);
        else XNOR_SMALL(8, 2, false);
    } else {
        if (g.mfma_pair) XNOR_SMALL(4, 1, true);
        else if (g.xw == 1) XNOR_SMALL(4, 1, false);
        else XNOR_SMALL(4, 2, false);
    }
    return hipGetLastError();
}
#undef XNOR_SMALL

} // namespace xnor_hip
