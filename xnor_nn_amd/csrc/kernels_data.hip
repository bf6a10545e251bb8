// Stage 1 and stage 2 of the forward pass: sign-bit packing of the input, mean |x| over
// channels (the "A" plane) and its box filter (the "K" plane).
//
// Semantics follow reference src/bcast_binarize_data.cpp:43-73 and
// src/bcast_calculate_k.cpp:42-85.  Both float reductions are evaluated in exactly the
// reference's order with separately rounded products and sums (no FMA contraction), so
// a and k come out bit-identical to the CPU library.
#include <cstdlib>

#include "filter_stage.hpp"
#include "plan.hpp"

namespace xnor_hip {

namespace {

constexpr int TILE = 64;       // pixels per workgroup = lanes per wave
constexpr int MAX_WAVES = 12;  // waves per workgroup
constexpr int TURN_ROW = 36;   // floats per pixel row of the NHWC turn-around buffer (32 + 4)
// Cache policy of the NHWC input: the "nt" bit, or none (nhwc_streams)
constexpr int LOAD_STREAMING = 2;
typedef uint32_t v4u __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t fbits(float v) { return __float_as_uint(v); }

// NCHW input.  A tile is 64 consecutive pixels of the flattened (mb, ih, iw) index; wave w of
// the workgroup owns the 32-channel slices w, w + NW, ... of it.  A lane is a pixel, so every
// load instruction reads 64 consecutive floats of one channel plane.  All 32 loads of a slice
// are issued before the first use.  Sign bits are shifted into the lane's word with one
// funnel shift per element (a ballot would produce pixel-major masks of one channel, i.e.
// the transpose of what is stored).
//
// mean|x| must be summed over channels in order.  The waves therefore hand the running
// sum from one to the next through LDS: wave w adds its terms after wave w-1 has published
// its result.  The packed words of the tile are staged in LDS and written as one
// contiguous run.
//
// One workgroup per tile.  (A persistent grid that issues the loads of its next tile before
// it processes the current one was measured and is not used: at these sizes the kernel is
// bound by the transfer plus one pass of the sum through the waves, and the hardware's own
// workgroup scheduling does as well as the hand-made pipeline.)
//
// Workgroups are dealt to the eight XCDs round-robin.  XCD x owns the contiguous range of
// tiles [x * tiles_per_xcd, (x+1) * tiles_per_xcd): the cache lines that straddle two
// neighbouring tiles (a channel plane is rarely a multiple of 128 bytes) are fetched into
// one L2 instead of two.  Workgroup b takes local tile b / 8 of XCD b % 8.
//
// NHWC input runs the same tile: the 32 values of a slice are then 128 contiguous bytes of a
// pixel.  A wave fetches them eight lanes to a pixel, so that
// every load instruction reads eight whole cache lines, and turns the block around through
// LDS into the lane = pixel layout (one lane per pixel straight from memory, 64 partial
// cache lines per instruction, took 19.7 us where this takes 13.5 us, the NCHW kernel 13.3).
// RAGGED: a channel count that is no multiple of 4.  Its whole slices are read the same way, from
// wherever a pixel begins; in the last one a lane is a channel, since 16 bytes would run into
// the next pixel (111 channels on 40x40, minibatch 60: 89.8 -> 10.7 us, 4.0 TB/s).  An instantiation of
// its own, since that slice takes 36 registers more (128 channels on 32x32, minibatch 100: 10.5 -> 11.7),
// and without the "nt" bit: neighbouring pixels share lines (130 on 40x40, minibatch 60: 18.1, 19.4 with).
template <bool NHWC, bool STREAM, bool RAGGED, bool WRITE_BITS, bool WRITE_A>
__device__ __forceinline__
void binarize_tile(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const Geometry &g, const float inv_ic, const int rounds,
        const uint32_t ntiles, const uint32_t tiles_per_xcd, const uint32_t block) {
    extern __shared__ uint32_t lds[];
    float *chain = reinterpret_cast<float *>(lds); // [TILE]
    uint32_t *stage = lds + TILE;                  // [TILE][xw]
    // NHWC: [waves][32 pixels][TURN_ROW floats], 16-byte aligned
    float *turn = reinterpret_cast<float *>(lds + ((TILE + TILE * g.xw + 3) & ~3));

    const int lane = threadIdx.x & (TILE - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nw = blockDim.x >> 6;
    const uint32_t tile = (block & 7) * tiles_per_xcd + (block >> 3);
    fetch_together(x, g.ic, g.ihw, g.npix_in, g.xw, inv_ic, rounds);
    fetch_together(g.div_ihw);
    if (tile >= ntiles) return;

    // the whole input as one raw buffer (the host side checks that it is below 4 GiB)
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(x), 0, (int)((uint32_t)g.npix_in * (uint32_t)g.ic * 4u),
            0x00020000);
    // slice (r * nw + wave) of a tile: 32 channel values of this lane's pixel
    auto load_slice = [&](float (&t)[32], uint32_t tile, int r) {
        const uint32_t p = tile * TILE + lane;
        const uint32_t pc = p < g.npix_in ? p : g.npix_in - 1;
        const uint32_t img = g.div_ihw.div(pc);
        const uint32_t hw = pc - img * g.ihw;
        const int c0 = (r * nw + wave) * 32; // wave-uniform
        if (c0 >= g.ic) return;
        if constexpr (NHWC) {
            // Load i of the wave reads the slice of pixels 8i .. 8i+7 of the tile: eight
            // lanes per pixel, 16 bytes each, i.e. eight whole cache lines per instruction.
            // The wave then turns the 64 x 128 bytes around through its own piece of LDS
            // (32 pixels at a time, rows of 144 bytes so that neither side has bank
            // conflicts) to end up with the lane = pixel layout of the rest of the kernel.
            typedef float v4f __attribute__((ext_vector_type(4)));
            float *mine = turn + wave * (32 * TURN_ROW);
            // rows of 32 pixels to lane = pixel
            auto turn_around = [&](int half) {
                if ((lane >> 5) != half) return;
#pragma unroll
                for (int u = 0; u < 8; u++) {
                    const v4f r = *reinterpret_cast<const v4f *>(
                            mine + (lane & 31) * TURN_ROW + 4 * u);
#pragma unroll
                    for (int e = 0; e < 4; e++) t[4 * u + e] = r[e];
                }
            };
            if (RAGGED && c0 + 32 > g.ic) { // uniform
                // The last slice of a channel count that is no multiple of 4: a channel to a lane, two
                // pixels per load.
                const int c = c0 + (lane & 31);
                // (a pixel past the last one lies outside the buffer, or where nothing is written from)
                const uint32_t off = ((tile * TILE + (lane >> 5)) * (uint32_t)g.ic + (uint32_t)c) * 4u;
                float v[32];
#pragma unroll
                for (int i = 0; i < 32; i++) v[i] = 0.f;
                if (c < g.ic) {
#pragma unroll
                    for (int i = 0; i < 32; i++)
                        v[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                src, off + (uint32_t)i * (8u * (uint32_t)g.ic), 0, 0));
                }
#pragma unroll
                for (int half = 0; half < 2; half++) {
#pragma unroll
                    for (int i = 0; i < 16; i++)
                        mine[(2 * i + (lane >> 5)) * TURN_ROW + (lane & 31)] = v[16 * half + i];
                    turn_around(half);
                }
                return;
            }
            const int piece = lane & 7;
            const int c = c0 + 4 * piece; // a piece is inside or outside
            v4f v[8];
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const uint32_t q = tile * TILE + 8 * i + (lane >> 3);
                const uint32_t qc = q < g.npix_in ? q : g.npix_in - 1;
                // a piece past the last channel gets an offset outside the buffer: reads +0
                const uint32_t off = c < g.ic ? qc * (uint32_t)g.ic * 4u + (uint32_t)c * 4u
                                              : 0xFFFFFFF0u;
                v[i] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                        src, off, 0, STREAM ? LOAD_STREAMING : 0));
            }
#pragma unroll
            for (int half = 0; half < 2; half++) {
#pragma unroll
                for (int i = 0; i < 4; i++)
                    *reinterpret_cast<v4f *>(mine + (8 * i + (lane >> 3)) * TURN_ROW + 4 * piece)
                        = v[4 * half + i];
                turn_around(half);
            }
            return;
        }
        // Buffer loads: one VGPR holds the lane's byte offset for all 32 loads, the channel
        // plane is a scalar offset (no 64-bit address arithmetic per load, fewer VGPRs).
        const uint32_t lane_off = (img * (uint32_t)(g.ic * g.ihw) + hw) * 4u;
        const uint32_t plane_bytes = (uint32_t)g.ihw * 4u;
        if (c0 + 32 <= g.ic) {
#pragma unroll
            for (int i = 0; i < 32; i++)
                t[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        src, lane_off, (uint32_t)(c0 + i) * plane_bytes, 0));
        } else {
            // last, ragged slice: a channel past the end gets an offset outside the buffer and
            // reads +0 (no branch per load); its bit is masked out of the word below and |+0|
            // leaves the running sum as it is
#pragma unroll
            for (int i = 0; i < 32; i++)
                t[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        src, c0 + i < g.ic ? lane_off : 0xFFFFFFF0u,
                        c0 + i < g.ic ? (uint32_t)(c0 + i) * plane_bytes : 0u, 0));
        }
    };

    // everything after the loads of the first pass over the slices (r = 0); t holds them
    auto process = [&](float (&t)[32], uint32_t tile) {
        const uint32_t p = tile * TILE + lane;
        if (wave == 0) chain[lane] = 0.f;
        for (int r = 0; r < rounds; r++) {
            if (r > 0) load_slice(t, tile, r);
            const int slice = r * nw + wave; // wave-uniform
            const int c0 = slice * 32;
            const bool has = c0 < g.ic;
            if (has) {
                uint32_t neg = 0; // sign bits, first channel ends up in the MSB
#pragma unroll
                for (int i = 0; i < 32; i++) {
                    neg = __builtin_amdgcn_alignbit(neg, fbits(t[i]), 31);
                    t[i] = __fmul_rn(__builtin_fabsf(t[i]), inv_ic);
                }
                if (WRITE_BITS) stage[lane * g.xw + slice] = (~neg) & top_bits(g.ic - c0);
            }
            // ordered hand-over of the running sum: wave s goes after wave s-1
            for (int s = 0; s < nw; s++) {
                if (s == wave && has) {
                    float acc = chain[lane];
#pragma unroll
                    for (int i = 0; i < 32; i++) acc = __fadd_rn(acc, t[i]);
                    chain[lane] = acc;
                }
                __syncthreads();
            }
        }
        const size_t tile_words = (size_t)TILE * g.xw;
        const size_t first = (size_t)tile * tile_words;
        const size_t total = (size_t)g.npix_in * g.xw;
        if (WRITE_BITS)
            for (uint32_t i = threadIdx.x; i < tile_words; i += blockDim.x)
                if (first + i < total) bits[first + i] = stage[i];
        if (WRITE_A && wave == 0 && p < g.npix_in) a[p] = chain[lane];
    };

    float t[32];
    load_slice(t, tile, 0);
    process(t, tile);
}

template <bool WRITE_BITS, bool WRITE_A>
__global__ __launch_bounds__(TILE * 16)
void binarize_nchw_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const Geometry g, const float inv_ic, const int rounds,
        const uint32_t ntiles, const uint32_t tiles_per_xcd) {
    binarize_tile<false, false, false, WRITE_BITS, WRITE_A>(x, bits, a, g, inv_ic, rounds, ntiles,
            tiles_per_xcd, blockIdx.x);
}

// The same and the weight stage in one launch, for a pass that brings new weights: neither needs
// anything of the other, and the weight stage by itself leaves most of the chip waiting (a filter to a
// workgroup, most of whose time is one wave putting an ordered sum together).  The first
// `weight_blocks` workgroups (a multiple of eight, so that tiles keep their XCDs) are filters, by
// their first FILTER_THREADS threads.
// conv4 of AlexNet, minibatch 64: the two kernels took 8.6 and 5.4 us one after the other.
__global__ __launch_bounds__(TILE * 16)
void binarize_nchw_and_weights_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const Geometry g, const float inv_ic, const int rounds,
        const uint32_t ntiles, const uint32_t tiles_per_xcd, const uint32_t weight_blocks,
        const float *__restrict__ w, uint32_t *__restrict__ wbits, uint32_t *__restrict__ frag,
        float *__restrict__ alpha, int32_t *__restrict__ opc, const FilterPlan f) {
    extern __shared__ __attribute__((aligned(16))) float row[];
    __shared__ Runs runs;
    if (blockIdx.x >= weight_blocks) {
        binarize_tile<false, false, false, true, true>(x, bits, a, g, inv_ic, rounds, ntiles, tiles_per_xcd,
                blockIdx.x - weight_blocks);
        return;
    }
    // (the other waves are through before the first barrier, which counts those that are left)
    if (threadIdx.x >= FILTER_THREADS || blockIdx.x >= f.workgroups) return;
    filter_stage(w, wbits, frag, alpha, opc, g, f, row, runs, blockIdx.x);
}

template <bool STREAM, bool RAGGED, bool WRITE_BITS, bool WRITE_A>
__global__ __launch_bounds__(TILE * 16)
void binarize_nhwc_tiled_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const Geometry g, const float inv_ic, const int rounds,
        const uint32_t ntiles, const uint32_t tiles_per_xcd) {
    binarize_tile<true, STREAM, RAGGED, WRITE_BITS, WRITE_A>(x, bits, a, g, inv_ic, rounds, ntiles,
            tiles_per_xcd, blockIdx.x);
}

// NCHW input with few tiles of 64 pixels: tiles of T = 16 pixels, and a wave of its own for the
// ordered sum.
// The tiled kernel above walks the running sum from wave to wave, with a barrier at every
// hand-over, and gives a tile's whole transfer to one compute unit: 2048 channels on 7x7,
// minibatch 64, were 49 workgroups of 11 waves that took six rounds, 23.6 us.  Here a wave loads
// four words (128 channels) of 16 pixels at a time, lane = (pixel, word); the loaders pack and store
// the sign words and leave the magnitudes in LDS, channel by channel along a pixel's row, and the
// last wave of the workgroup adds them, reading 32 values ahead, while the loaders fetch the next
// chunk.  What bounds it is that chain: one addition per eight cycles and channel, 7 us for 2048
// channels.  It must not stand still: no barrier, every loader says by itself that its part of a
// chunk lies there, and the adding wave takes as many parts in a row as it finds (a part at a time,
// with the first read of each exposed: 13.9 and 10.6 us below), and frees their places one by one.
// us for 2048 channels on 7x7, minibatch 64 / 1, and 3000 channels, minibatch 8, with a barrier per
// chunk of all loaders: 16.3 / 11.6 and 17.5, now 13.4 / 10.0 and 15.0.  Both of the first two
// chunks asked for at once make the first one come later: 17.0 / 12.3 and 18.7.
struct SplitPlan {
    uint32_t npix, ihw, ntiles, tiles_per_xcd;
    int ic, xw, loaders, chunks;
    FastDiv div_ihw;
};
constexpr int SPLIT_TILE = 16, SPLIT_WORDS = 64 / SPLIT_TILE, SPLIT_LOADERS = 8;

template <int T, bool WRITE_BITS, bool WRITE_A>
__global__ __launch_bounds__(64 * (SPLIT_LOADERS + 1))
void binarize_nchw_split_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const SplitPlan s, const float inv_ic) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    constexpr int G = 64 / T; // words a wave loads together
    extern __shared__ __attribute__((aligned(16))) float split_lds[];
    // a pixel's row in floats: 4 mod 64, so that the 16-byte accesses of both sides spread over
    // the banks
    const int chunk_words = s.loaders * G, row = chunk_words * 32 + 4;
    // [one or two buffers][T pixels][row], then the loaders' chunks that lie there, then the number of
    // loaders' chunks that have been added
    uint32_t *there = reinterpret_cast<uint32_t *>(split_lds + (s.chunks > 1 ? 2 : 1) * T * row);
    uint32_t *added = there + SPLIT_LOADERS;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = (blockIdx.x & 7) * s.tiles_per_xcd + (blockIdx.x >> 3);
    fetch_together(x, a, bits, s.npix, s.ihw, s.ic, s.xw, s.loaders, s.chunks, inv_ic);
    fetch_together(s.div_ihw);
    if (tile >= s.ntiles) return;
    const int lp = lane & (T - 1), lg = lane / T;
    const uint32_t p = tile * T + lp;
    if (WRITE_A && wave == s.loaders && lane <= SPLIT_LOADERS) there[lane] = 0; // (`added` as well)
    auto load_of = [](uint32_t *flag) {
        return __hip_atomic_load(flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    // (what this wave read or wrote in LDS before is done)
    auto say = [](uint32_t *flag, uint32_t value) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __hip_atomic_store(flag, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    };
    auto flags_are_clear = [] { // loads from memory stay under way
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    if (wave < s.loaders) {
        const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float *>(x), 0, (int)(s.npix * (uint32_t)s.ic * 4u), 0x00020000);
        const uint32_t pc = p < s.npix ? p : s.npix - 1, img = s.div_ihw.div(pc);
        const uint32_t plane = s.ihw * 4u;
        const uint32_t pixel = (img * (uint32_t)s.ic * s.ihw + (pc - img * s.ihw)) * 4u;
        float t[32];
        auto load = [&](int k) { // this lane's word of chunk k
            const int set = k * s.loaders + wave, j = set * G + lg, left = s.ic - 32 * j;
            const uint32_t off = pixel + (uint32_t)(32 * j) * plane;
            if (32 * (set + 1) * G <= s.ic) { // uniform: whole words
#pragma unroll
                for (int i = 0; i < 32; i++)
                    t[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            src, off, (uint32_t)i * plane, 0));
            } else { // a channel past the end: an offset outside the buffer, which reads +0
#pragma unroll
                for (int i = 0; i < 32; i++)
                    t[i] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                            src, i < left ? off + (uint32_t)i * plane : 0xFFFFFFF0u, 0, 0));
            }
        };
        load(0);
        if (WRITE_A) flags_are_clear();
        for (int k = 0; k < s.chunks; k++) {
            const int j = (k * s.loaders + wave) * G + lg;
            uint32_t neg = 0; // sign bits, first channel ends up in the MSB
            v4f *to = reinterpret_cast<v4f *>(split_lds + ((k & 1) * T + lp) * row
                    + (wave * G + lg) * 32);
#pragma unroll
            for (int i = 0; i < 32; i++) {
                neg = __builtin_amdgcn_alignbit(neg, fbits(t[i]), 31);
                t[i] = __fmul_rn(__builtin_fabsf(t[i]), inv_ic);
            }
            if (WRITE_A) {
                // what chunk k - 2 left here has been added (chunks are added in order, a chunk loader by
                // loader)
                if (k >= 2) {
                    while (load_of(added) < (uint32_t)((k - 2) * s.loaders + wave + 1))
                        __builtin_amdgcn_s_sleep(1);
                    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
                }
#pragma unroll
                for (int i = 0; i < 8; i++)
                    to[i] = v4f{t[4 * i], t[4 * i + 1], t[4 * i + 2], t[4 * i + 3]};
                say(there + wave, k + 1);
            }
            // (sixteen bytes of a pixel; they meet the next wave's in L2)
            if (WRITE_BITS && j < s.xw && p < s.npix)
                bits[(size_t)p * s.xw + j] = (~neg) & top_bits(s.ic - 32 * j);
            if (k + 1 < s.chunks) load(k + 1);
        }
        return;
    }
    if (!WRITE_A) return;
    // the chain is what the workgroup waits for: ahead of the loaders' packing on its SIMD (2048
    // channels on 7x7, a pass at minibatch 1 / 64: 17.7 / 24.5 -> 17.0 / 23.7 us)
    flags_are_clear();
    __builtin_amdgcn_s_setprio(3);
    float sum = 0.f;
    v4f u[8], v[8];
    auto read = [&](v4f (&to)[8], int k, int word) {
        const v4f *at = reinterpret_cast<const v4f *>(split_lds + ((k & 1) * T + lp) * row) + 8 * word;
#pragma unroll
        for (int i = 0; i < 8; i++) to[i] = at[i];
    };
    auto add = [&](const v4f (&from)[8]) {
#pragma unroll
        for (int i = 0; i < 8; i++)
#pragma unroll
            for (int e = 0; e < 4; e++) sum = __fadd_rn(sum, from[i][e]);
    };
    for (int k = 0; k < s.chunks; k++) {
        const int words = min(chunk_words, s.xw - k * chunk_words); // uniform
        for (int w = 0; w < words;) {
            // the loaders whose chunks lie there, in the order of their channels (a flag that no loader has
            // stays 0)
            const uint64_t lie_there = __ballot(load_of(there + (lane & (SPLIT_LOADERS - 1))) > (uint32_t)k);
            const int ready = __builtin_ctz(~((uint32_t)lie_there & ((1u << SPLIT_LOADERS) - 1)));
            const int end = min(words, ready * G);
            if (w >= end) {
                __builtin_amdgcn_s_sleep(1);
                continue;
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
            read(u, k, w);
            for (; w < end; w += 2) {
                if (w + 1 < end) read(v, k, w + 1);
                add(u);
                if (w + 1 < end) {
                    if (w + 2 < end) read(u, k, w + 2);
                    add(v);
                }
            }
            if (k + 2 < s.chunks) say(added, k * s.loaders + ready);
        }
    }
    if (lane < T && p < s.npix) a[p] = sum;
}

// NCHW input of at most 32 channels (one packed word per pixel): a lane takes all channels of U
// pixels 256 apart, so nothing is handed over between waves and nothing goes through LDS.  CH is
// the channel count rounded up to a power of two (4 to 32), U = 32 / CH, so that a lane has up to
// 32 loads in flight whatever the channel count: with one wave per 64 pixels and three channels
// the tiled kernel above kept 768 bytes in flight per wave and was bound by the rate at which
// workgroups start (AlexNet's first layer, minibatch 64: 40 MB in 32 us, here 17).
template <int CH, int U, bool WRITE_BITS, bool WRITE_A>
__global__ __launch_bounds__(256)
void binarize_nchw_shallow_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const uint32_t npix, const int ic, const uint32_t ihw,
        const FastDiv div_ihw, const float inv_ic, const uint32_t groups,
        const uint32_t groups_per_xcd) {
    // each XCD takes one contiguous range of the pixels (shared cache lines meet in one L2)
    const uint32_t group = (blockIdx.x & 7) * groups_per_xcd + (blockIdx.x >> 3);
    fetch_together(x, a, bits, npix, ic, ihw, inv_ic);
    fetch_together(div_ihw);
    if (group >= groups) return;
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(x), 0, (int)(npix * (uint32_t)ic * 4u), 0x00020000);
    const uint32_t p0 = group * (256u * U) + threadIdx.x;
    float t[U][CH];
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t p = p0 + u * 256u, pc = p < npix ? p : npix - 1;
        const uint32_t img = div_ihw.div(pc);
        const uint32_t off = (img * ((uint32_t)ic * ihw) + (pc - img * ihw)) * 4u;
#pragma unroll
        for (int c = 0; c < CH; c++)
            if (c < ic) // uniform
                t[u][c] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                        src, off, (uint32_t)c * ihw * 4u, 0));
            else
                t[u][c] = 0.f; // bit masked out below, |+0| leaves the sum as it is
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
        const uint32_t p = p0 + u * 256u;
        uint32_t neg = 0; // sign bits, first channel ends up in the MSB of CH bits
        float acc = 0.f;
#pragma unroll
        for (int c = 0; c < CH; c++) {
            neg = __builtin_amdgcn_alignbit(neg, fbits(t[u][c]), 31);
            acc = __fadd_rn(acc, __fmul_rn(__builtin_fabsf(t[u][c]), inv_ic));
        }
        if (p < npix) {
            if (WRITE_BITS) bits[p] = (~(neg << (32 - CH))) & top_bits(ic);
            if (WRITE_A) a[p] = acc;
        }
    }
}

// Any source layout, one lane per pixel, channels visited in order (reference src/bcast_binarize_data.cpp:56-57, src/bcast_calculate_k.cpp:59-60).
template <bool WRITE_BITS, bool WRITE_A>
__global__ __launch_bounds__(256)
void binarize_generic_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const Geometry g, const float inv_ic) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= g.npix_in) return;
    const uint32_t img = g.div_ihw.div(p);
    const uint32_t hw = p - img * g.ihw;
    size_t idx, step;
    if (g.src_fmt == xnor_nn_data_format_nchw) {
        idx = (size_t)img * g.ic * g.ihw + hw;
        step = g.ihw;
    } else {
        idx = (size_t)p * g.ic;
        step = 1;
    }
    float acc = 0.f;
    for (int j = 0; j < g.xw; j++) {
        uint32_t neg = 0;
        const int n = min(32, g.ic - 32 * j);
        for (int i = 0; i < n; i++) {
            const float v = x[idx];
            idx += step;
            neg = __builtin_amdgcn_alignbit(neg, fbits(v), 31);
            acc = __fadd_rn(acc, __fmul_rn(__builtin_fabsf(v), inv_ic));
        }
        if (WRITE_BITS) bits[(size_t)p * g.xw + j] = (~(neg << (32 - n))) & top_bits(n);
    }
    if (WRITE_A) a[p] = acc;
}

// NHWC input with IC a multiple of 4 that the tiled kernel does not take (nhwc_tiled): a lane
// is a pixel and walks over its channels, which are contiguous, in order, 32 at a time (one packed word): eight 16-byte buffer loads per
// word, the loads of the next three words in flight while the current one is folded into
// the sign word and the running mean|x| (reference src/bcast_binarize_data.cpp:56-57,
// src/bcast_calculate_k.cpp:59-60).  The lanes of a wave read addresses IC*4 bytes apart,
// so every load touches 64 cache lines, but each line is used completely by the loads that
// follow, and HBM traffic is the algorithmic minimum.
template <bool WRITE_BITS, bool WRITE_A>
__global__ __launch_bounds__(256)
void binarize_nhwc_kernel(const float *__restrict__ x, uint32_t *__restrict__ bits,
        float *__restrict__ a, const Geometry g, const float inv_ic) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t pc = p < g.npix_in ? p : g.npix_in - 1;
    const __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(x), 0, (int)((uint32_t)g.npix_in * (uint32_t)g.ic * 4u),
            0x00020000);
    const uint32_t lane_off = pc * (uint32_t)g.ic * 4u;
    // 32 channels starting at c0; channels >= IC read as +0 (sign bit clear, |x| = 0: they
    // are masked out of the word and add nothing to the sum)
    auto fetch = [&](v4f (&v)[8], int c0) {
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const int c = c0 + 4 * u; // uniform
            v[u] = c < g.ic ? __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                      src, lane_off, (uint32_t)c * 4u, 0))
                            : v4f{0.f, 0.f, 0.f, 0.f};
        }
    };
    float acc = 0.f;
    auto fold = [&](const v4f (&v)[8], int j) { // word j: sign bits and the running sum
        if (j >= g.xw) return; // uniform
        uint32_t neg = 0; // sign bits, first channel ends up in the MSB
        const int n = min(32, g.ic - 32 * j);
#pragma unroll
        for (int u = 0; u < 8; u++)
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const float val = v[u][e];
                neg = __builtin_amdgcn_alignbit(neg, fbits(val), 31);
                if (4 * u + e < n) // uniform; a sum must not see the padding's +0 terms
                    acc = __fadd_rn(acc, __fmul_rn(__builtin_fabsf(val), inv_ic));
            }
        if (WRITE_BITS && p < g.npix_in) bits[(size_t)p * g.xw + j] = (~neg) & top_bits(n);
    };
    // four register sets used in turn: three words are in flight while one is folded
    v4f b0[8], b1[8], b2[8], b3[8];
    fetch(b0, 0);
    fetch(b1, 32);
    fetch(b2, 64);
    for (int j = 0; j < g.xw; j += 4) {
        fetch(b3, 32 * (j + 3));
        fold(b0, j);
        fetch(b0, 32 * (j + 4));
        fold(b1, j + 1);
        fetch(b1, 32 * (j + 5));
        fold(b2, j + 2);
        fetch(b2, 32 * (j + 6));
        fold(b3, j + 3);
    }
    if (WRITE_A && p < g.npix_in) a[p] = acc;
}

// K plane: k = sum over in-bounds taps, row-major, of fl(a * KHW)
// (reference src/bcast_calculate_k.cpp:69-85).  One lane per output pixel.
__global__ __launch_bounds__(256)
void box_filter_kernel(const float *__restrict__ a, float *__restrict__ k,
        const Geometry g, const float inv_khw) {
    const uint32_t p = blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= g.npix_out) return;
    const uint32_t img = g.div_ohw.div(p);
    const uint32_t rem = p - img * g.ohw;
    const int oh = (int)g.div_ow.div(rem);
    const int ow = (int)rem - oh * g.ow;
    const float *plane = a + (size_t)img * g.ihw;
    float acc = 0.f;
    for (int kh = 0; kh < g.kh; kh++) {
        const int ih = oh * g.sh - g.ph + kh;
        if (ih < 0 || ih >= g.ih) continue;
        for (int kw = 0; kw < g.kw; kw++) {
            const int iw = ow * g.sw - g.pw + kw;
            if (iw < 0 || iw >= g.iw) continue;
            acc = __fadd_rn(acc, __fmul_rn(plane[ih * g.iw + iw], inv_khw));
        }
    }
    k[p] = acc;
}

// Calibration only: reads a buffer once, 16 bytes per lane and load, four loads in flight per
// lane, and keeps nothing.  What this takes is what the memory system allows a kernel that
// does no work at all on the same bytes.
__global__ __launch_bounds__(256)
void plain_read_kernel(const v4u *__restrict__ x, const size_t n16) {
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * 256;
    v4u acc = {0u, 0u, 0u, 0u};
    for (; i + 3 * stride < n16; i += 4 * stride) {
        const v4u v0 = x[i], v1 = x[i + stride], v2 = x[i + 2 * stride], v3 = x[i + 3 * stride];
        acc ^= v0 ^ v1 ^ v2 ^ v3;
    }
    for (; i < n16; i += stride) acc ^= x[i];
    asm volatile("" : : "v"(acc)); // the loads have a use
}

// Waves of a workgroup of the tiled kernels, and the rounds in which they take the slices.
int tiled_waves(const Plan &g, int *rounds) {
    *rounds = (g.xw + g.bin_waves - 1) / g.bin_waves;
    return (g.xw + *rounds - 1) / *rounds;
}

// Whether the tiled kernel reads its NHWC input with the "nt" bit: every line is read once and whole, so
// it need not push out what waits in the caches to be written back.  It pays for inputs above the 32 MB
// of the eight L2s and up to 104 MB.  Smaller ones may still lie in the L2s, where the bit lets them go;
// larger ones lose where they have just been written, which is how a network's layers find them.  us a
// pass with / without it, on changing inputs, on the same one, on one that a kernel has just written, on
// changing ones just written:
//   13 MB   256 channels 14x14   14.5 / 14.6   14.0 / 13.0   24.2 / 22.8   19.6 / 19.0
//   26 MB   64 on 56x56          16.0 / 16.8   14.7 / 13.9   31.0 / 32.4   26.2 / 25.4
//   38 MB   64 on 56x56          21.6 / 22.6   19.1 / 20.9   35.1 / 38.0   35.7 / 34.3
//   52 MB   128 on 32x32         37.9 / 39.8   35.6 / 38.1   55.7 / 56.1   56.6 / 55.1
//   103 MB  128 on 56x56         32.0 / 35.2   29.6 / 30.9   60.0 / 60.4   64.2 / 62.6
//   128 MB  100 on 40x40         62.4 / 65.9   59.8 / 55.4  112.2 / 100.6 112.6 / 112.8
//   154 MB  192 on 56x56         57.3 / 62.0   55.9 / 54.5  106.6 / 101.9 110.0 / 103.8
//   205 MB  256 on 56x56         97.6 / 104.8  94.7 / 90.3  152.4 / 150.1 152.5 / 152.8
// Not for NCHW, where neighbouring tiles share lines: 384 channels on 13x13 44.9 / 41.7 (without / with)
// on changing inputs, but 35.8 / 39.6 on the same one and 56.2 / 65.1 on one just written.
bool nhwc_streams(const Plan &g) {
    const uint64_t bytes = (uint64_t)g.npix_in * (uint64_t)g.ic * 4u;
    return bytes > (32u << 20) && bytes <= (104u << 20);
}

// At most twelve waves per workgroup, the slices split evenly over the rounds: with more
// waves the hand-over chain of one workgroup gets long and too few workgroups are
// resident to cover it (512 input channels: 14.1 us with 16 waves, 10.4 us with 2 x 8;
// 384 channels: 12 x 1 and 6 x 2 are equal at MB 256, 12 x 1 is 5% faster at MB 1024).
template <bool WRITE_BITS, bool WRITE_A>
void launch_tiled(const Plan &g, const float *x, uint32_t *bits, float *a, hipStream_t s,
        const KernelEvents &ev) {
    int rounds;
    const int nw = tiled_waves(g, &rounds);
    const uint32_t ntiles = (g.npix_in + TILE - 1) / TILE;
    const uint32_t per_xcd = (ntiles + 7) / 8;
    launch_kernel(binarize_nchw_kernel<WRITE_BITS, WRITE_A>, dim3(per_xcd * 8),
            dim3(nw * TILE), sizeof(uint32_t) * (TILE + (size_t)TILE * g.xw), s, ev, x, bits, a,
            geometry(g), 1.f / g.ic, rounds, ntiles, per_xcd);
}

// LDS of the tiled NHWC kernel: chain, packed words, turn-around rows.
size_t nhwc_tiled_lds_bytes(const Plan &g, int waves) {
    const size_t words = sizeof(uint32_t) * (TILE + (size_t)TILE * g.xw);
    return ((words + 15) & ~(size_t)15) + sizeof(float) * waves * 32 * TURN_ROW;
}

template <bool WRITE_BITS, bool WRITE_A>
hipError_t launch_nhwc_tiled(const Plan &g, const float *x, uint32_t *bits, float *a, hipStream_t s,
        const KernelEvents &ev) {
    int rounds;
    const int nw = tiled_waves(g, &rounds);
    const uint32_t ntiles = (g.npix_in + TILE - 1) / TILE;
    const uint32_t per_xcd = (ntiles + 7) / 8;
    const size_t lds = nhwc_tiled_lds_bytes(g, nw);
    const bool ragged = (g.ic & 3) != 0, streams = nhwc_streams(g);
    const auto kernel = ragged ? binarize_nhwc_tiled_kernel<false, true, WRITE_BITS, WRITE_A>
        : streams ? binarize_nhwc_tiled_kernel<true, false, WRITE_BITS, WRITE_A>
                          : binarize_nhwc_tiled_kernel<false, false, WRITE_BITS, WRITE_A>;
    static LdsGrant grants[3];
    const hipError_t e = grants[ragged ? 2 : streams ? 1 : 0].ask((const void *)kernel, lds);
    if (e != hipSuccess) return e;
    launch_kernel(kernel, dim3(per_xcd * 8), dim3(nw * TILE), lds, s, ev, x, bits, a, geometry(g),
            1.f / g.ic, rounds, ntiles, per_xcd);
    return hipSuccess;
}

size_t split_lds_bytes(const Plan &g, int *loaders, int *chunks) {
    const int sets = (g.xw + SPLIT_WORDS - 1) / SPLIT_WORDS; // of words that a wave loads together
    *loaders = sets < SPLIT_LOADERS ? sets : SPLIT_LOADERS;
    *chunks = (sets + *loaders - 1) / *loaders;
    return sizeof(float) * ((*chunks > 1 ? 2 : 1) * SPLIT_TILE * (*loaders * SPLIT_WORDS * 32 + 4)
            + SPLIT_LOADERS + 1);
}

template <bool WRITE_BITS, bool WRITE_A>
hipError_t launch_split(const Plan &g, const float *x, uint32_t *bits, float *a, hipStream_t s,
        const KernelEvents &ev) {
    SplitPlan p{};
    p.npix = g.npix_in;
    p.ihw = (uint32_t)g.ihw;
    p.ntiles = (g.npix_in + SPLIT_TILE - 1) / SPLIT_TILE;
    p.tiles_per_xcd = (p.ntiles + 7) / 8;
    p.ic = g.ic;
    p.xw = g.xw;
    p.div_ihw = g.div_ihw;
    const size_t lds = split_lds_bytes(g, &p.loaders, &p.chunks);
    const auto kernel = binarize_nchw_split_kernel<SPLIT_TILE, WRITE_BITS, WRITE_A>;
    static LdsGrant grant;
    const hipError_t e = grant.ask((const void *)kernel, lds);
    if (e != hipSuccess) return e;
    launch_kernel(kernel, dim3(p.tiles_per_xcd * 8), dim3(64 * (p.loaders + 1)), lds, s, ev, x, bits,
            a, p, 1.f / g.ic);
    return hipSuccess;
}

template <int CH, bool WRITE_BITS, bool WRITE_A>
void launch_shallow(const Plan &g, const float *x, uint32_t *bits, float *a, hipStream_t s,
        const KernelEvents &ev) {
    constexpr int U = 32 / CH;
    // several pixels per lane only where that still leaves every compute unit two workgroups
    const bool many = U > 1 && g.npix_in >= 2u * (uint32_t)g.cus * 256u * U;
    const uint32_t groups = (g.npix_in + 256u * (many ? U : 1) - 1) / (256u * (many ? U : 1));
    const uint32_t per_xcd = (groups + 7) / 8;
    const auto kernel = many ? binarize_nchw_shallow_kernel<CH, U, WRITE_BITS, WRITE_A>
                             : binarize_nchw_shallow_kernel<CH, 1, WRITE_BITS, WRITE_A>;
    launch_kernel(kernel, dim3(per_xcd * 8), dim3(256), 0, s, ev, x, bits, a, g.npix_in, g.ic,
            (uint32_t)g.ihw, g.div_ihw, 1.f / g.ic, groups, per_xcd);
}

template <bool WRITE_BITS, bool WRITE_A>
void launch_shallow_any(const Plan &g, const float *x, uint32_t *bits, float *a,
        hipStream_t s, const KernelEvents &ev) {
    if (g.ic <= 4) launch_shallow<4, WRITE_BITS, WRITE_A>(g, x, bits, a, s, ev);
    else if (g.ic <= 8) launch_shallow<8, WRITE_BITS, WRITE_A>(g, x, bits, a, s, ev);
    else if (g.ic <= 16) launch_shallow<16, WRITE_BITS, WRITE_A>(g, x, bits, a, s, ev);
    else launch_shallow<32, WRITE_BITS, WRITE_A>(g, x, bits, a, s, ev);
}

} // namespace

// The tiled kernel addresses the input with 32-bit byte offsets and stages the packed words
// of a tile in LDS (64 KB at most: up to 8160 channels); deeper or larger inputs run the
// generic kernel.  A channel past the end of a ragged slice is read through the byte offset
// 0xFFFFFFF0, which has to lie outside the buffer for the load to return +0: the input must
// end below that offset.
static bool tiled_nchw(const Plan &g) {
    return g.src_fmt == xnor_nn_data_format_nchw
        && (uint64_t)g.npix_in * (uint64_t)g.ic * 4u < XNOR_HIP_DROPPED_OFFSET
        && sizeof(uint32_t) * (TILE + (size_t)TILE * g.xw) <= 64 * 1024;
}

// Few channels: pixel numbers (rounded up to a workgroup's) and byte offsets stay below 2^31.
static bool shallow_nchw(const Plan &g) {
    return g.ic <= 32 && tiled_nchw(g)
        && (uint64_t)g.npix_in * (uint64_t)g.ic * 4u < (1ull << 31);
}

static uint32_t pixel_tiles(const Plan &g) { return (g.npix_in + TILE - 1) / TILE; }

// Up to one tile of 64 pixels for every four compute units, one for every two from 512 channels on:
// us here / by the tiled kernel
//   384 channels   13x13, minibatch 1 / 8 / 24 (3 / 22 / 64 tiles): 4.1 / 4.3 / 4.7 and 4.6 / 4.7 / 5.0
//                  9x9, 13x13, 14x14, 27x27, about 85 tiles: 5.4, 5.9, 5.1, 5.4 and 5.6, 5.6, 5.4, 5.5
//   512 channels   the same: 7.2, 7.0, 6.2, 7.3 and 7.3, 7.3, 7.0, 7.0; 125 tiles 6.4 to 7.2 and 7.2 to 7.7
//   1024 channels  the same: 10.6, 11.6, 10.4, 10.8 and 11.6, 11.7, 11.6, 11.7; 125 tiles 11.3 to 12.8 and
//                  13.8 to 15.4
//   2048 channels  7x7, minibatch 64 / 128 / 160 (49 / 98 / 123 tiles): 13.4 / 24.3 / 27.3 and
//                  23.0 / 30.8 / 31.6
//   4000 channels  14x14, 74 / 120 tiles: 38.7 / 43.6 and 55.1 / 57.3
// With more tiles a compute unit gets a third one of 16 pixels and has LDS for one or two, and the tiled
// kernel's whole cache lines count for more than the shorter walk: 200 tiles on 14x14, 512 / 1024 / 2048
// channels 8.6 / 19.6 / 44.7 and 8.2 / 17.3 / 32.7.
static bool split_nchw(const Plan &g) {
    int loaders, chunks;
    return tiled_nchw(g) && pixel_tiles(g) <= (uint32_t)g.cus / (g.ic < 512 ? 4 : 2)
        && split_lds_bytes(g, &loaders, &chunks) <= 160 * 1024;
}

// The NHWC kernels read at 32-bit byte offsets (and drop what lies past the last channel the same
// way).
static bool vector_nhwc(const Plan &g) {
    return g.src_fmt == xnor_nn_data_format_nhwc
        && (uint64_t)g.npix_in * (uint64_t)g.ic * 4u < XNOR_HIP_DROPPED_OFFSET;
}

// The tiled kernel takes NHWC input that its LDS can hold: about 13500 channels.  us here / where it
// does not run, a lane to a pixel:
//   channels a multiple of 4: binarize_nhwc_kernel, whose loads touch 64 lines each
//     1500 on 7x7, minibatch 100: 19.3 / 84.0; 28x28, minibatch 60: 61.1 / 160;  2048 on 7x7, minibatch
//     8 / 64: 19.0 / 84.5 and 21.4 / 86.2;  4000 on 14x14, minibatch 2: 33.4 / 167
//     (a single tile of more than 64 KB, 2048 channels on 6x6, would be 18.0 / 42.0; that choice is fixed
//     by the names that the interface reports for it)
//   others: binarize_generic_kernel, one channel per load
//     minibatch 64 on 100x100, 6 / 7 / 9 / 13 / 30 / 33 channels: 7.9 / 7.9, 8.0 / 9.7, 8.6 / 13.6,
//     9.8 / 23.8, 16.1 / 246, 21 / 290; on 224x224, 6 / 7 channels: 33.9 / 29.4, 34.3 / 36.1
//     minibatch 18 on 23x23, 33 / 111 / 254 / 1023 channels: 4.2 / 6.5, 4.1 / 28.8, 5.4 / 59.7, 16.2 / 447
//     one tile, 30 / 33 / 65 / 401 channels: 4.2 / 4.2, 4.2 / 4.2, 4.0 / 7.4, 5.2 / 45.1
static bool nhwc_tiled(const Plan &g) {
    if (!vector_nhwc(g) || g.bin_nhwc_lane) return false;
    int rounds;
    const size_t lds = nhwc_tiled_lds_bytes(g, tiled_waves(g, &rounds));
    const bool one_tile = g.npix_in <= (uint32_t)TILE;
    if (g.ic & 3) return g.ic > (one_tile ? 32 : 6) && lds <= 160 * 1024;
    return lds <= (one_tile ? 64 : 160) * 1024;
}

// A lane to a pixel, 16 bytes per load.
static bool nhwc_by_lane(const Plan &g) { return vector_nhwc(g) && (g.ic & 3) == 0 && !nhwc_tiled(g); }

// The measurement switches of this stage, read once when a descriptor is initialised (a launch
// asks the environment for nothing): XNOR_NN_HIP_BIN_WAVES caps the waves of a workgroup,
// XNOR_NN_HIP_NHWC=lane forces the one-lane-per-pixel kernel for NHWC input.
void binarize_plan(Plan &g) {
    g.bin_waves = MAX_WAVES;
    if (const char *e = getenv("XNOR_NN_HIP_BIN_WAVES")) {
        const int v = atoi(e);
        if (v >= 1 && v <= 16) g.bin_waves = v;
    }
    const char *e = getenv("XNOR_NN_HIP_NHWC");
    g.bin_nhwc_lane = e && e[0] == 'l' ? 1 : 0;
}

const char *binarize_kernel_name(const Plan &g) {
    return shallow_nchw(g) ? "binarize_nchw_shallow_kernel"
        : split_nchw(g) ? "binarize_nchw_split_kernel"
        : tiled_nchw(g) ? "binarize_nchw_kernel"
        : nhwc_by_lane(g) ? "binarize_nhwc_kernel"
        : !nhwc_tiled(g) ? "binarize_generic_kernel"
        : g.ic & 3 ? "binarize_nhwc_tiled_kernel<RAGGED>"
        : nhwc_streams(g) ? "binarize_nhwc_tiled_kernel<STREAM>" : "binarize_nhwc_tiled_kernel";
}

hipError_t launch_binarize_data(const Plan &g, const float *x, uint32_t *bits,
        float *a_or_null, hipStream_t s, const KernelEvents &ev) {
    const float inv_ic = 1.f / g.ic;
    if (shallow_nchw(g)) {
        if (a_or_null) launch_shallow_any<true, true>(g, x, bits, a_or_null, s, ev);
        else launch_shallow_any<true, false>(g, x, bits, nullptr, s, ev);
    } else if (split_nchw(g)) {
        const hipError_t e = a_or_null ? launch_split<true, true>(g, x, bits, a_or_null, s, ev)
                                       : launch_split<true, false>(g, x, bits, nullptr, s, ev);
        if (e != hipSuccess) return e;
    } else if (tiled_nchw(g)) {
        if (a_or_null) launch_tiled<true, true>(g, x, bits, a_or_null, s, ev);
        else launch_tiled<true, false>(g, x, bits, nullptr, s, ev);
    } else if (nhwc_tiled(g)) {
        const hipError_t e = a_or_null ? launch_nhwc_tiled<true, true>(g, x, bits, a_or_null, s, ev)
                                       : launch_nhwc_tiled<true, false>(g, x, bits, nullptr, s, ev);
        if (e != hipSuccess) return e;
    } else if (nhwc_by_lane(g)) {
        const unsigned blocks = (g.npix_in + 255) / 256;
        if (a_or_null)
            launch_kernel(binarize_nhwc_kernel<true, true>, dim3(blocks), dim3(256), 0, s, ev,
                    x, bits, a_or_null, geometry(g), inv_ic);
        else
            launch_kernel(binarize_nhwc_kernel<true, false>, dim3(blocks), dim3(256), 0, s, ev,
                    x, bits, a_or_null, geometry(g), inv_ic);
    } else {
        const unsigned blocks = (g.npix_in + 255) / 256;
        if (a_or_null)
            launch_kernel(binarize_generic_kernel<true, true>, dim3(blocks), dim3(256), 0, s,
                    ev, x, bits, a_or_null, geometry(g), inv_ic);
        else
            launch_kernel(binarize_generic_kernel<true, false>, dim3(blocks), dim3(256), 0, s,
                    ev, x, bits, a_or_null, geometry(g), inv_ic);
    }
    return hipGetLastError();
}

namespace {

// The grid of binarize_nchw_and_weights_kernel: tiles, and filters ahead of them.
struct JoinedGrid {
    int rounds, tile_waves, waves; // of a tile; of any workgroup
    uint32_t ntiles, per_xcd, weight_blocks;
    FilterPlan filters;
    size_t lds;                    // dynamic; every workgroup has `Runs` beside it
};
JoinedGrid joined_grid(const Plan &g, bool fragments) {
    JoinedGrid j{};
    j.tile_waves = tiled_waves(g, &j.rounds);
    j.waves = j.tile_waves < FILTER_WAVES ? FILTER_WAVES : j.tile_waves;
    j.ntiles = (g.npix_in + TILE - 1) / TILE;
    j.per_xcd = (j.ntiles + 7) / 8;
    j.filters = filter_plan(g, fragments);
    j.weight_blocks = (j.filters.workgroups + 7) / 8 * 8;
    const size_t tile = sizeof(uint32_t) * (TILE + (size_t)TILE * g.xw);
    j.lds = tile > j.filters.lds ? tile : j.filters.lds;
    return j;
}

} // namespace

// A tile of the joined launch takes the LDS of a filter and four waves at least.  Where long filters leave
// a compute unit fewer workgroups than its 32 waves allow, what the tiles lose grows with their number
// and what the launch saves does not: joined while there are at most seven tiles for every 32 channels
// that are under way on a unit.  us of a pass with new weights, joined / in two launches, beside the tiles
// up to which they are joined (64 filters, planes of 64x64, stride 4):
//   40 channels 19x19   4480 tiles   4096: 106.4 / 110.2   8192: 124.6 / 119.4   12288: 204.8 / 182.1
//   64 channels 15x15   7168         4096:  74.9 /  81.2   8192:  99.2 /  99.6   12288: 152.9 / 147.6
//   96 channels 12x12  10752         4096:  64.3 /  70.6   8192: 119.6 / 122.4   12288: 146.1 / 143.7
//   128 channels 11x11 14336         8192: 133.3 / 134.4  12288: 186.5 / 196.5   24576: 361.2 / 353.0
// Nowhere else was joining slower, on 60 layers: 384 channels 3x3 on 13x13, minibatch 64, 20.9 / 26.6, 256
// channels 7x7 on 14x14, minibatch 128, 54.8 / 58.8, 64 channels 3x3 on 224x224, minibatch 64 (50176
// tiles, as many workgroups as the waves allow), 273 / 280.
// Input of at most one tile for every four compute units is left to its own kernel.
bool weights_join_binarize(const Plan &g) {
    if (!tiled_nchw(g) || shallow_nchw(g) || pixel_tiles(g) <= (uint32_t)g.cus / 4
            || !filter_kernel_applies(g))
        return false;
    const JoinedGrid j = joined_grid(g, g.use_mfma != 0);
    const int by_waves = 32 / j.waves, by_lds = (int)(160 * 1024 / (j.lds + sizeof(Runs)));
    return by_lds >= by_waves
        || (uint64_t)j.ntiles * 32 <= (uint64_t)7 * by_lds * g.ic * g.cus;
}

hipError_t launch_binarize_data_and_weights(const Plan &g, const float *x, uint32_t *bits, float *a,
        const float *w, uint32_t *wbits, uint32_t *frag, float *alpha, int32_t *opc, hipStream_t s) {
    const JoinedGrid j = joined_grid(g, frag != nullptr);
    static LdsGrant grant;
    const hipError_t e = grant.ask((const void *)binarize_nchw_and_weights_kernel,
            j.lds + sizeof(Runs));
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(binarize_nchw_and_weights_kernel, dim3(j.weight_blocks + j.per_xcd * 8),
            dim3(j.waves * TILE), j.lds, s, x, bits, a, geometry(g), 1.f / g.ic, j.rounds, j.ntiles,
            j.per_xcd, j.weight_blocks, w, wbits, frag, alpha, opc, j.filters);
    return hipGetLastError();
}

hipError_t launch_mean_abs(const Plan &g, const float *x, float *a, hipStream_t s) {
    const float inv_ic = 1.f / g.ic;
    if (shallow_nchw(g)) {
        launch_shallow_any<false, true>(g, x, nullptr, a, s, KernelEvents{});
    } else if (split_nchw(g)) {
        const hipError_t e = launch_split<false, true>(g, x, nullptr, a, s, KernelEvents{});
        if (e != hipSuccess) return e;
    } else if (tiled_nchw(g)) {
        launch_tiled<false, true>(g, x, nullptr, a, s, KernelEvents{});
    } else if (nhwc_tiled(g)) {
        const hipError_t e = launch_nhwc_tiled<false, true>(g, x, nullptr, a, s, KernelEvents{});
        if (e != hipSuccess) return e;
    } else if (nhwc_by_lane(g)) {
        const unsigned blocks = (g.npix_in + 255) / 256;
        hipLaunchKernelGGL((binarize_nhwc_kernel<false, true>), dim3(blocks), dim3(256), 0, s,
                x, nullptr, a, geometry(g), inv_ic);
    } else {
        const unsigned blocks = (g.npix_in + 255) / 256;
        hipLaunchKernelGGL((binarize_generic_kernel<false, true>), dim3(blocks), dim3(256),
                0, s, x, nullptr, a, geometry(g), inv_ic);
    }
    return hipGetLastError();
}

hipError_t launch_plain_read(const void *buf, size_t bytes, hipStream_t s,
        const KernelEvents &ev) {
    launch_kernel(plain_read_kernel, dim3(2048), dim3(256), 0, s, ev,
            static_cast<const v4u *>(buf), bytes / 16);
    return hipGetLastError();
}

hipError_t launch_box_filter(const Plan &g, const float *a, float *k, hipStream_t s) {
    const float inv_khw = 1.f / g.kh / g.kw; // two divisions, like the reference
    const unsigned blocks = (g.npix_out + 255) / 256;
    hipLaunchKernelGGL(box_filter_kernel, dim3(blocks), dim3(256), 0, s, a, k, geometry(g), inv_khw);
    return hipGetLastError();
}

} // namespace xnor_hip
