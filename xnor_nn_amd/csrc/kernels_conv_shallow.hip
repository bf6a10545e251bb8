// Stage 3 on the matrix cores for inputs of few channels (first layers of image networks): the
// FP4 implicit GEMM of kernels_conv_mfma.hip with the (tap, channel) pairs of a pixel packed
// back to back.
// Semantics: reference src/default/bcast_convolution_default.cpp:60-105.
//
// The large-launch kernel walks the taps one by one (or two by two), 32 channels wide at least:
// with three channels 29 of every 32 products are zeros, and AlexNet's first layer (3 channels,
// 11x11) is 61 steps of 64 where its 363 products fill six.  Here the products of one kernel row
// are packed back to back (33 bits there, rounded up to bytes): seven steps.  What bounds the
// kernel then is its output and the instructions and cache lines it takes to gather the operands,
// so these are kept few: a first version that collected a pixel's operand tap by tap issued 2000
// scalar and 1200 vector instructions per wave and took 84 us on that layer (minibatch 64), the
// large-launch kernel 160 us; with rows as strings 34 us; with four pixels to a load of the
// strings, two instructions to a pixel of them, 16-byte stores of the gathered codes and mean|x|
// laid out by the stride (LDS bank conflicts 4.3 -> 1.2 million cycles) 31 us (the pass 53.4 -> 50.3).
//
// Workgroup = P consecutive output pixels (flattened mb, oh, ow) x a run of 32-filter blocks:
//   1. rows: every input row the tile touches goes to LDS as one string of sign bits (IC bits per
//      pixel, first channel lowest, zeros for the padding left and right), mean|x| beside it.
//   2. gather: a lane is an output pixel.  The bits a kernel row multiplies are consecutive in the
//      row's string: one funnel shift per 32 of them, whatever the stride and channel count.
//      They are expanded to FP4 through a 256-entry table (a second table clears the codes of
//      taps outside the image) and stored as one LDS row per pixel.  One wave per 64 pixels sums
//      K meanwhile (box filter of mean|x|, the reference's order), or ahead of it where mean|x|
//      shares the operands' LDS.
//   3. multiply and store: a wave takes 32 filters x 64 pixels at a time; a pixel's row is read
//      from front to back, there are no taps left.
#include <cstdlib>
#include <type_traits>

#include "plan.hpp"

namespace xnor_hip {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_word;

constexpr int SHALLOW_CHANNELS = 12;          // (13 and up never meet the rule of shallow_plan)
constexpr int SHALLOW_TABLES = 2 * 256 * 4;   // codes and validity masks
constexpr uint32_t SHALLOW_DROP = 0xFFFFFFF0u;
constexpr size_t SHALLOW_LDS = 160 * 1024;     // of a compute unit
constexpr int SHALLOW_AHEAD = 4;              // weight fragments asked for together

__device__ __forceinline__ v16f shallow_mfma_fp4(const v4i a, const v4i b, const v16f c) {
    const v8i a8 = {a.x, a.y, a.z, a.w, 0, 0, 0, 0};
    const v8i b8 = {b.x, b.y, b.z, b.w, 0, 0, 0, 0};
    // cbsz = blgp = 4: FP4 (E2M1) operands; zero scale operands select the unscaled form
    return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a8, b8, c, 4, 4, 0, 0, 0, 0);
}

// First and last padded row (image * prows + row) that the output pixels [p0, p1) reach.
__host__ __device__ inline void padded_rows(const ShallowPlan &s, uint32_t p0, uint32_t p1,
        uint32_t &r0, uint32_t &r1) {
    const uint32_t i0 = s.div_ohw.div(p0), i1 = s.div_ohw.div(p1 - 1);
    const uint32_t y0 = s.div_ow.div(p0 - i0 * s.ohw), y1 = s.div_ow.div(p1 - 1 - i1 * s.ohw);
    r0 = i0 * s.prows + y0 * s.sh;
    r1 = i1 * s.prows + y1 * s.sh + s.kh - 1;
}

// LDS of the gathered operands and of mean|x|, in one place or one after the other.
__host__ __device__ inline int operand_bytes(const ShallowPlan &s, int pixels, int rows) {
    const int operands = pixels * s.row_bytes, cells = (rows * s.a_cols * s.sw * 4 + 15) & ~15;
    return !s.a_shares_rows ? operands + cells : operands > cells ? operands : cells;
}

template <int P, int WAVES, bool RAW>
__global__ __launch_bounds__(64 * WAVES, WAVES == 8 ? 6 : 1) // three workgroups of eight waves
void conv_mfma_fp4_shallow_kernel(const uint32_t *__restrict__ xbits,
        const v4i *__restrict__ wfrag, const float *__restrict__ alpha,
        const float *__restrict__ kplane, float *__restrict__ dst, int32_t *__restrict__ popc,
        const float *__restrict__ a_plane, float *__restrict__ k_out, const float inv_khw,
        const ShallowPlan s) {
    constexpr int PB = P / 64, THREADS = 64 * WAVES; // PB: groups of 64 pixels
    extern __shared__ unsigned char smem[];
    uint32_t *codes = reinterpret_cast<uint32_t *>(smem);
    uint32_t *masks = codes + 256;
    float *k_lds = reinterpret_cast<float *>(smem + SHALLOW_TABLES);
    float *alpha_lds = k_lds + P;
    unsigned char *rows = reinterpret_cast<unsigned char *>(alpha_lds + s.blocks_per_wg * 32);
    const int a_pitch = s.a_cols * s.sw; // floats of mean|x| per padded row
    float *a_cells = reinterpret_cast<float *>(s.a_shares_rows ? rows : rows + P * s.row_bytes);
    uint32_t *strings = reinterpret_cast<uint32_t *>(rows
            + operand_bytes(s, P, s.max_rows));

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // each XCD takes one contiguous range of (tile, filter chunk) units: neighbouring tiles
    // share input rows and output lines in one L2
    const uint32_t unit = (blockIdx.x & 7) * s.units_per_xcd + (blockIdx.x >> 3);
    if (unit >= s.units) return;
    const uint32_t chunks = s.units / s.tiles;
    const uint32_t tile = chunks == 1 ? unit : unit / chunks;
    const int chunk = (int)(unit - tile * chunks);
    const uint32_t p_first = tile * P, p_end = min(p_first + P, s.npix_out);
    const bool fuse_k = !RAW && a_plane != nullptr; // uniform

    // ---- rows ------------------------------------------------------------------------------
    uint32_t r0, r1;
    padded_rows(s, p_first, p_end, r0, r1);
    const int nrows = min((int)(r1 - r0 + 1), s.max_rows);
    const uint32_t in_bytes = s.npix_in * 4u;
    const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<uint32_t *>(xbits), 0, (int)in_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t abuf = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<float *>(a_plane), 0, fuse_k ? (int)in_bytes : 0, 0x00020000);
    // mean|x|: copied straight to LDS (nothing waits here and no register is held), a wave takes
    // a row at a time, 64 pixels per instruction; outside the image the copy reads zero.  Columns
    // that differ by the stride lie side by side: neighbouring output pixels then read
    // neighbouring banks (with stride 4 a plain row had four lanes on every bank in use).
    if (fuse_k) {
        for (int r = wave; r < nrows; r += WAVES) {
            const uint32_t R = r0 + r, img = s.div_prows.div(R); // uniform
            const int y = (int)(R - img * s.prows) - s.ph;
            const bool row_ok = (unsigned)y < (unsigned)s.ih;
            const uint32_t at = ((img * s.ih + y) * s.iw - s.pw) * 4u;
            for (int c0 = 0; c0 < a_pitch; c0 += 64) {
                const int phase = (int)s.div_acols.div((uint32_t)(c0 + lane));
                const int c = (c0 + lane - phase * s.a_cols) * s.sw + phase;
                if (c0 + lane < a_pitch)
                    __builtin_amdgcn_raw_ptr_buffer_load_lds(abuf,
                            (lds_word *)(a_cells + r * a_pitch + c0), 4,
                            row_ok && (unsigned)(c - s.pw) < (unsigned)s.iw ? at + 4u * c
                                                                            : SHALLOW_DROP,
                            0, 0, 0);
            }
        }
    }
    { // codes: bit i of the index = nibble i, +1 -> 0x2, -1 -> 0xA; masks: set -> 0xF
        uint32_t x = (uint32_t)tid & 0xFFu; // bit i -> bit 4i
        x = (x | x << 12) & 0x000F000Fu;
        x = (x | x << 6) & 0x03030303u;
        x = (x | x << 3) & 0x11111111u;
        if (tid < 256) {
            codes[tid] = 0xAAAAAAAAu ^ (x << 3);
            masks[tid] = 15u * x;
        }
    }
    if (!RAW)
        for (int i = tid; i < s.blocks_per_wg * 32; i += THREADS) {
            const int f = chunk * s.blocks_per_wg * 32 + i;
            alpha_lds[i] = f < s.oc ? alpha[f] : 0.f;
        }
    // bit strings: a lane is a dword of one; it reads the pixels that reach into it, last one
    // first, and shifts the string along by a pixel's bits for each (two vector instructions a
    // pixel).  Pixels outside the image are masked at the end: what was read for them is another
    // pixel of the input, or zero outside the buffer.
    for (int i = tid; i < nrows * s.row_words; i += THREADS) {
        const int r = (int)s.div_words.div((uint32_t)i), d = i - r * s.row_words;
        const uint32_t R = r0 + r, img = s.div_prows.div(R);
        const int y = (int)(R - img * s.prows) - s.ph;
        const int first = (int)s.div_ic.div(32u * d), x = first - s.pw; // may begin in the dword before
        const int pos = first * s.ic - 32 * d;  // bit its first channel would have: -IC < pos <= 0
        const uint32_t pixel = (img * s.ih + y) * s.iw + x, at = pixel * 4u;
        uint32_t out = 0;
        auto collect = [&](auto batch) { // all loads of a batch are under way together
            constexpr int N = decltype(batch)::value;
            // Four pixels a load: a wave's lanes are a dword of string apart and every load
            // touches as many cache lines as four would, which is what these loads cost.  Only
            // where all of them lie in the buffer: one that begins outside may be dropped whole.
            const uint32_t reach = (uint32_t)((s.row_pixels + N - 1) / N * N) * 4u;
            const bool wide = __all(reach <= in_bytes && at <= in_bytes - reach);
            for (int k0 = (s.row_pixels - 1) / N * N; k0 >= 0; k0 -= N) { // uniform
                uint32_t w[N];
                if (wide) {
#pragma unroll
                    for (int k = 0; k < N; k += 4) {
                        const v4i v = __builtin_bit_cast(v4i,
                                __builtin_amdgcn_raw_buffer_load_b128(xbuf, at + 4u * (k0 + k), 0, 0));
#pragma unroll
                        for (int n = 0; n < 4; n++) w[k + n] = (uint32_t)v[n];
                    }
                } else {
                    // One by one, each inside the buffer or dropped: loads at neighbouring offsets
                    // are merged into a wide one by the compiler, and one that begins ahead of the
                    // first pixel then loses the pixels behind it as well.
#pragma unroll
                    for (int k = 0; k < N; k++) {
                        const uint32_t q = pixel + (uint32_t)(k0 + k);
                        w[k] = __builtin_amdgcn_raw_buffer_load_b32(xbuf,
                                q < s.npix_in ? q * 4u : SHALLOW_DROP, 0, 0);
                    }
                }
#pragma unroll
                for (int k = N - 1; k > 0; k--) // first channel lowest
                    out = out << s.ic | __brev(w[k]);
                if (k0 > 0) out = out << s.ic | __brev(w[0]);
                else out = out << (s.ic + pos) | __brev(w[0]) >> -pos;
            }
        };
        if (s.row_pixels <= 4) collect(std::integral_constant<int, 4>{});
        else collect(std::integral_constant<int, 12>{});
        // bits of pixels inside the image: [lo, hi) of the dword
        const int lo = max(max(-x, 0) * s.ic + pos, 0), hi = min((s.iw - x) * s.ic + pos, 32);
        const bool some = (unsigned)y < (unsigned)s.ih && lo < hi;
        strings[i] = some ? out & 0xFFFFFFFFu << lo & 0xFFFFFFFFu >> (32 - hi) : 0u;
    }
    __syncthreads();

    // ---- gather ----------------------------------------------------------------------------
    auto gather_job = [&](const int job) {
        const int pb = job % PB, part = job / PB; // uniform
        const uint32_t p = p_first + pb * 64 + lane;
        const bool live = p < s.npix_out;
        const uint32_t pc = live ? p : s.npix_out - 1;
        const uint32_t img = s.div_ohw.div(pc), rem = pc - img * s.ohw;
        const uint32_t oy = s.div_ow.div(rem), ox = rem - oy * s.ow;
        // a dead lane takes the tile's first row: that of the last pixel may lie outside the tile
        const uint32_t row0 = live ? img * s.prows + oy * s.sh - r0 : 0u, col0 = ox * s.sw;
        if (part == 0) {
            float sum = 0.f;
            if (fuse_k) { // in-bounds taps in row-major order, each product rounded, then added;
                          // a cell outside the image holds +0, which changes no sum
                const float *row = a_cells + row0 * a_pitch + ox;
                auto add_rows = [&](auto width) { // a row is asked for while the last one is added
                    constexpr int KW = decltype(width)::value;
                    int at[KW]; // uniform
#pragma unroll
                    for (int x = 0, phase = 0, q = 0; x < KW; x++) {
                        at[x] = phase * s.a_cols + q;
                        if (++phase == s.sw) phase = 0, q++;
                    }
                    float t[KW];
#pragma unroll
                    for (int x = 0; x < KW; x++) t[x] = row[at[x]];
                    for (int y = 1; y <= s.kh; y++) {
                        float next[KW];
                        row += y < s.kh ? a_pitch : 0;
#pragma unroll
                        for (int x = 0; x < KW; x++) next[x] = row[at[x]];
#pragma unroll
                        for (int x = 0; x < KW; x++) t[x] = __fmul_rn(t[x], inv_khw);
#pragma unroll
                        for (int x = 0; x < KW; x++) {
                            sum = __fadd_rn(sum, t[x]);
                            t[x] = next[x];
                        }
                    }
                };
                switch (s.kw) { // uniform
                case 3: add_rows(std::integral_constant<int, 3>{}); break;
                case 5: add_rows(std::integral_constant<int, 5>{}); break;
                case 7: add_rows(std::integral_constant<int, 7>{}); break;
                case 11: add_rows(std::integral_constant<int, 11>{}); break;
                default:
                    for (int y = 0; y < s.kh; y++, row += a_pitch)
                        if (s.sw == 1)
                            for (int x = 0; x < s.kw; x++) sum = __fadd_rn(sum, __fmul_rn(row[x], inv_khw));
                        else
                            for (int x = 0, phase = 0, q = 0; x < s.kw; x++) {
                                sum = __fadd_rn(sum, __fmul_rn(row[phase * s.a_cols + q], inv_khw));
                                if (++phase == s.sw) phase = 0, q++;
                            }
                }
                if (chunk == 0 && live) k_out[p] = sum;
            } else if (!RAW) {
                sum = kplane[pc];
            } else { // operation count of the pixel (reference src/bcast_binarize_weights.cpp:126-142)
                const int y0 = (int)oy * s.sh - s.ph, x0 = (int)ox * s.sw - s.pw;
                const int ny = min(y0 + s.kh, s.ih) - max(y0, 0), nx = min(x0 + s.kw, s.iw) - max(x0, 0);
                sum = (float)(ny > 0 && nx > 0 ? ny * nx * s.ic : 0);
            }
            k_lds[pb * 64 + lane] = sum;
            return;
        }
        const int ya = (part - 1) * 4, yb = min(ya + 4, s.kh); // gathers * 4 >= kh
        const uint32_t bit0 = col0 * s.ic; // where the pixel's products begin in a row's string
        const uint32_t shift = bit0 & 31u;
        const uint32_t *string = strings + row0 * s.row_words + (bit0 >> 5);
        uint32_t *out = reinterpret_cast<uint32_t *>(rows + (pb * 64 + lane) * s.row_bytes);
        const int iy = (int)oy * s.sh - s.ph, ix = (int)ox * s.sw - s.pw;
        // products outside the image in this pixel's kernel rows: all but [in_a, in_b)
        const int in_a = max(0, -ix) * s.ic, in_b = min(s.kw, s.iw - ix) * s.ic;
        // The codes of the four rows are 4 * row_codes consecutive dwords of the pixel's operand, a
        // whole number of 16-byte units: with the number known to the compiler they are stored as
        // such (16-byte stores an odd number of units apart touch every bank, 4-byte stores a
        // quarter of them).  What the units hold past the last kernel row meets weights of zero.
        auto gather = [&](auto edges, auto width) { // edges: some lane has taps outside its image
            constexpr bool EDGES = decltype(edges)::value;
            constexpr int RC = decltype(width)::value; // row_codes, 0: any
            const int row_codes = RC ? RC : s.row_codes;
            const uint32_t *at[4];
            uint32_t lo[4];
            bool row_in[4];
            [[maybe_unused]] uint32_t unit[RC ? 4 * RC : 1];
#pragma unroll
            for (int k = 0; k < 4; k++) { // past the last: the last one again
                const int yk = min(ya + k, yb - 1);
                at[k] = string + yk * s.row_words;
                row_in[k] = (unsigned)(iy + yk) < (unsigned)s.ih;
                lo[k] = at[k][0];
            }
            auto word = [&](const int c) { // codes c to c + 3
                uint32_t bits[4];
#pragma unroll
                for (int k = 0; k < 4; k++) {
                    const uint32_t hi = at[k][c / 4 + 1];
                    bits[k] = __builtin_amdgcn_alignbit(hi, lo[k], shift);
                    lo[k] = hi;
                }
                uint32_t columns = 0;
                if constexpr (EDGES) {
                    const int va = max(in_a - 8 * c, 0), vb = min(in_b - 8 * c, 32);
                    if (va < vb) columns = (0xFFFFFFFFu << va) & (0xFFFFFFFFu >> (32 - vb));
                }
#pragma unroll
                for (int i = 0; i < 4; i++)
                    if (c + i < row_codes) { // uniform
                        uint32_t q[4];
#pragma unroll
                        for (int k = 0; k < 4; k++) q[k] = codes[(bits[k] >> (8 * i)) & 0xFF];
                        if constexpr (EDGES) {
                            const uint32_t in = masks[(columns >> (8 * i)) & 0xFF];
#pragma unroll
                            for (int k = 0; k < 4; k++) q[k] = row_in[k] ? q[k] & in : 0u;
                        }
#pragma unroll
                        for (int k = 0; k < 4; k++) {
                            if constexpr (RC > 0) unit[k * RC + c + i] = q[k];
                            else if (ya + k < yb) out[(ya + k) * row_codes + c + i] = q[k]; // uniform
                        }
                    }
            };
            if constexpr (RC > 0) {
#pragma unroll
                for (int c = 0; c < RC; c += 4) word(c);
            } else {
                for (int c = 0; c < row_codes; c += 4) word(c); // uniform
            }
            if constexpr (RC > 0) {
                v4i *to = reinterpret_cast<v4i *>(out + ya * RC);
#pragma unroll
                for (int u = 0; u < RC; u++)
                    if (ya * RC + 4 * u < s.kh * RC) // uniform
                        to[u] = v4i{(int)unit[4 * u], (int)unit[4 * u + 1], (int)unit[4 * u + 2],
                                (int)unit[4 * u + 3]};
            }
        };
        auto gather_rows = [&](auto edges) {
            switch (s.row_codes) { // uniform
            case 2: gather(edges, std::integral_constant<int, 2>{}); break;
            case 3: gather(edges, std::integral_constant<int, 3>{}); break;
            case 4: gather(edges, std::integral_constant<int, 4>{}); break;
            case 5: gather(edges, std::integral_constant<int, 5>{}); break;
            default: gather(edges, std::integral_constant<int, 0>{});
            }
        };
        const bool inside = !live || (iy >= 0 && iy + s.kh <= s.ih && ix >= 0
                && ix + s.kw <= s.iw);
        if (__all(inside)) gather_rows(std::false_type{});
        else gather_rows(std::true_type{});
    };
    // jobs of one wave over 64 pixels; part 0 sums K, parts 1.. take kernel rows, after all of part
    // 0 where mean|x| lies in the operands' place
    for (int job = 0, end = s.a_shares_rows ? PB : PB * (1 + s.gathers);;) {
        for (job += wave; job < end; job += WAVES) gather_job(job);
        if (end > PB) break;
        __syncthreads();
        job = PB;
        end = PB * (1 + s.gathers);
    }
    __syncthreads();

    // ---- multiply: (32-filter block, 64 pixels) at a time ------------------------------------
    const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(
            const_cast<v4i *>(wfrag), 0, (int)s.wfrag_bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t outbuf = __builtin_amdgcn_make_buffer_rsrc(
            RAW ? static_cast<void *>(popc) : static_cast<void *>(dst), 0,
            (int)(s.npix_out * (uint32_t)s.oc * 4u), 0x00020000);
    const int lane_hi = lane >> 5;
    const bool nchw = RAW || s.nchw != 0;
    const uint32_t fstep = nchw ? (uint32_t)s.ohw * 4u : 4u; // bytes from a filter to the next
    const int first_block = chunk * s.blocks_per_wg;
    const int nblocks = min(s.blocks_per_wg, s.blocks - first_block);
    for (int job = wave; job < nblocks * PB; job += WAVES) {
        const int b = job / PB, pb = job - b * PB; // uniform
        const unsigned char *row0 = rows + (pb * 64 + (lane & 31)) * s.row_bytes + lane_hi * 16;
        const unsigned char *row1 = row0 + 32 * s.row_bytes;
        const uint32_t wbase = (uint32_t)(first_block + b) * (uint32_t)s.steps * 1024u;
        v16f acc[2];
#pragma unroll
        for (int i = 0; i < 16; i++) acc[0][i] = acc[1][i] = 0.f;
        auto fragment = [&](int st) { // past the last step: the last one again, not used
            return __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(wbuf,
                    (uint32_t)lane * 16u, wbase + (uint32_t)min(st, s.steps - 1) * 1024u, 0));
        };
        v4i w[SHALLOW_AHEAD];
#pragma unroll
        for (int u = 0; u < SHALLOW_AHEAD; u++) w[u] = fragment(u);
        for (int st = 0; st < s.steps; st += SHALLOW_AHEAD) {
#pragma unroll
            for (int u = 0; u < SHALLOW_AHEAD; u++)
                if (st + u < s.steps) { // uniform
                    const v4i b0 = *reinterpret_cast<const v4i *>(row0 + (st + u) * 32);
                    const v4i b1 = *reinterpret_cast<const v4i *>(row1 + (st + u) * 32);
                    acc[0] = shallow_mfma_fp4(w[u], b0, acc[0]);
                    acc[1] = shallow_mfma_fp4(w[u], b1, acc[1]);
                    w[u] = fragment(st + u + SHALLOW_AHEAD);
                }
        }

        // register i of a block holds filter 8*(i/4) + 4*(lane/32) + i%4, pixel lane%32
        const float kv[2] = {k_lds[pb * 64 + (lane & 31)], k_lds[pb * 64 + 32 + (lane & 31)]};
        const uint32_t p64 = p_first + pb * 64;
        const bool all = (first_block + b + 1) * 32 <= s.oc; // uniform
        auto value = [&](int q, int i, float al) -> uint32_t {
            const float d = acc[q][i]; // = 2*popc - n, exactly
            if constexpr (RAW) return (uint32_t)(((int)d + (int)kv[q]) / 2);
            // dst = fl(fl((float)(2*popc - n) * alpha) * k), rounded per product
            else return __float_as_uint(__fmul_rn(__fmul_rn(d, al), kv[q]));
        };
        auto store_planes = [&](auto policy, auto whole) { // NCHW: 64 consecutive pixels of a filter
            constexpr int AUX = decltype(policy)::value;
            constexpr bool ALL = decltype(whole)::value; // no filter past the last
            const uint32_t p = p64 + lane, pc = p < s.npix_out ? p : s.npix_out - 1;
            const uint32_t im = s.div_ohw.div(pc);
            const uint32_t off = p < s.npix_out
                ? (im * (uint32_t)s.oc * (uint32_t)s.ohw + (pc - im * s.ohw)) * 4u : SHALLOW_DROP;
#pragma unroll
            for (int i4 = 0; i4 < 4; i4++) {
                const v4f al = *reinterpret_cast<const v4f *>(alpha_lds + b * 32 + 8 * i4
                        + 4 * lane_hi);
#pragma unroll
                for (int ii = 0; ii < 4; ii++) {
                    const int f = (first_block + b) * 32 + 8 * i4 + ii;
                    const auto r = __builtin_amdgcn_permlane32_swap(value(0, 4 * i4 + ii, al[ii]),
                            value(1, 4 * i4 + ii, al[ii]), false, false);
                    // r[0]: filter f, pixels lane; r[1]: filter f + 4
                    if (ALL || f < s.oc)
                        __builtin_amdgcn_raw_buffer_store_b32(r[0], outbuf, off,
                                (uint32_t)f * fstep, AUX);
                    if (ALL || f + 4 < s.oc)
                        __builtin_amdgcn_raw_buffer_store_b32(r[1], outbuf, off,
                                (uint32_t)(f + 4) * fstep, AUX);
                }
            }
        };
        if (nchw) {
            auto store = [&](auto policy) {
                if (all) store_planes(policy, std::true_type{});
                else store_planes(policy, std::false_type{});
            };
            if (s.stream) store(std::integral_constant<int, 2>{}); // nt
            else store(std::integral_constant<int, 0>{});
        } else { // a lane holds four consecutive filters of a pixel
#pragma unroll
            for (int q = 0; q < 2; q++) {
                const uint32_t p = p64 + q * 32 + (lane & 31);
#pragma unroll
                for (int i4 = 0; i4 < 4; i4++) {
                    const int f = (first_block + b) * 32 + 8 * i4 + 4 * lane_hi;
                    const v4f al = *reinterpret_cast<const v4f *>(alpha_lds + b * 32 + 8 * i4
                            + 4 * lane_hi);
                    v4i v;
#pragma unroll
                    for (int ii = 0; ii < 4; ii++) v[ii] = (int)value(q, 4 * i4 + ii, al[ii]);
                    const uint32_t at = (p * (uint32_t)s.oc + (uint32_t)f) * 4u;
                    if ((s.oc & 3) == 0) {
                        __builtin_amdgcn_raw_buffer_store_b128(v, outbuf,
                                p < s.npix_out && f < s.oc ? at : SHALLOW_DROP, 0, 0);
                    } else {
#pragma unroll
                        for (int ii = 0; ii < 4; ii++)
                            __builtin_amdgcn_raw_buffer_store_b32((uint32_t)v[ii], outbuf,
                                    p < s.npix_out && f + ii < s.oc ? at + 4u * ii : SHALLOW_DROP,
                                    0, 0);
                    }
                }
            }
        }
    }
}

// One thread per dword of the fragments [32-filter block][step][lane][4 dwords]: lane l holds
// filter l % 32 and dwords 8*step + 4*(l / 32) + 0..3 of the inner dimension, eight products per
// dword, low nibble first; dword j is byte j % row_codes of kernel row j / row_codes, whose bit b
// is channel b % IC of tap column b / IC.  Whatever lies past a kernel row's end, past the last
// kernel row or past the last filter is FP4 zero.
__global__ __launch_bounds__(256)
void pack_weights_shallow_kernel(const float *__restrict__ w, uint32_t *__restrict__ frag,
        const Geometry g, const int steps, const int row_codes, const uint32_t total) {
    const uint32_t i = blockIdx.x * 256u + threadIdx.x;
    if (i >= total) return;
    const int dw = (int)(i & 3), lane = (int)((i >> 2) & 63);
    const int f = (int)(i >> 8), step = f % steps, oc = (f / steps) * 32 + (lane & 31);
    const int j = 8 * step + 4 * (lane >> 5) + dw, kh = j / row_codes;
    uint32_t out = 0;
    for (int n = 0; n < 8; n++) {
        const int b = (j - kh * row_codes) * 8 + n, kw = b / g.ic, c = b - kw * g.ic;
        if (kh < g.kh && kw < g.kw && oc < g.oc) {
            const size_t at = g.w_fmt == xnor_nn_weights_format_oihw
                ? (((size_t)oc * g.ic + c) * g.kh + kh) * g.kw + kw
                : (((size_t)kh * g.kw + kw) * g.ic + c) * g.oc + oc;
            out |= ((__float_as_uint(w[at]) >> 31) ? 0xAu : 0x2u) << (4 * n);
        }
    }
    frag[i] = out;
}

int row_codes_of(const Plan &g) { return (g.kw * g.ic + 7) / 8; }

ShallowPlan make_plan(const Plan &g) {
    ShallowPlan s{};
    s.npix_out = g.npix_out; s.npix_in = g.npix_in;
    s.ic = g.ic; s.ih = g.ih; s.iw = g.iw; s.oc = g.oc; s.oh = g.oh; s.ow = g.ow; s.ohw = g.ohw;
    s.kh = g.kh; s.kw = g.kw; s.sh = g.sh; s.sw = g.sw; s.ph = g.ph; s.pw = g.pw;
    s.prows = (g.oh - 1) * g.sh + g.kh;
    s.pcols = (g.ow - 1) * g.sw + g.kw;
    s.row_codes = row_codes_of(g);
    s.steps = (s.kh * s.row_codes + 7) / 8;
    // (the last pixel's kernel row begins in the string and reads one dword past its last one)
    s.row_words = (s.pcols * g.ic + 31) / 32 + 2;
    s.row_pixels = 31 / g.ic + 2;
    s.a_cols = (s.pcols + s.sw - 1) / s.sw;
    s.gathers = (s.kh + 3) / 4;
    s.div_acols = FastDiv::make((uint32_t)s.a_cols);
    s.row_bytes = s.steps * 32 + 16; // 4 mod 8 dwords: fragment reads spread over the banks
    s.blocks = (g.oc + 31) / 32;
    s.nchw = g.dst_fmt == xnor_nn_data_format_nchw ? 1 : 0;
    s.stream = g.stream_dst;
    s.div_ohw = g.div_ohw; s.div_ow = g.div_ow;
    s.div_prows = FastDiv::make((uint32_t)s.prows);
    s.div_words = FastDiv::make((uint32_t)s.row_words);
    s.div_ic = FastDiv::make((uint32_t)g.ic);
    s.wfrag_bytes = (uint32_t)s.blocks * (uint32_t)s.steps * 1024u;
    return s;
}

// Padded rows a tile of `pixels` output pixels stages at most: where in an image a tile starts
// repeats after at most OHW tiles.
int most_rows(const ShallowPlan &s, int pixels) {
    const uint32_t tiles = (s.npix_out + pixels - 1) / pixels;
    uint32_t most = 1;
    auto see = [&](uint32_t t) {
        uint32_t r0, r1;
        const uint32_t p0 = t * pixels;
        padded_rows(s, p0, p0 + pixels < s.npix_out ? p0 + pixels : s.npix_out, r0, r1);
        if (r1 - r0 + 1 > most) most = r1 - r0 + 1;
    };
    const uint32_t look = tiles < (uint32_t)s.ohw + 1 ? tiles : (uint32_t)s.ohw + 1;
    for (uint32_t t = 0; t < look; t++) see(t);
    see(tiles - 1);
    return (int)most;
}

// The rest of the plan for tiles of `pixels` with `rows` padded rows at most and `per_wg` filter
// blocks per workgroup; returns the LDS bytes.
size_t set_tile(ShallowPlan &s, int pixels, int per_wg, int rows, int cus) {
    s.tiles = (s.npix_out + pixels - 1) / pixels;
    s.blocks_per_wg = per_wg;
    const uint32_t chunks = (uint32_t)(s.blocks + per_wg - 1) / per_wg;
    s.units = s.tiles * chunks;
    s.units_per_xcd = (s.units + 7) / 8;
    s.max_rows = rows;
    auto lds = [&](int shares) {
        s.a_shares_rows = shares;
        return SHALLOW_TABLES + ((size_t)pixels + 32 * per_wg) * 4
            + (size_t)operand_bytes(s, pixels, rows) + (size_t)rows * s.row_words * 4;
    };
    // A place of its own for mean|x| lets K be summed beside the gathering; sharing one lets more
    // workgroups fit a compute unit, which is worth more where there are more of them (8 images of
    // 227x227, 3 channels, 11x11, 379 tiles: 15.1 us a pass with its own, 17.9 shared).
    const size_t own = lds(0), shared = lds(1), fit = SHALLOW_LDS / own;
    return SHALLOW_LDS / shared > fit && fit < 4 && s.units > fit * (uint32_t)cus ? shared : lds(0);
}

// Output pixels per tile and filter blocks per workgroup.
size_t choose_tile(const Plan &g, ShallowPlan &s, int *pixels) {
    for (int p : {128, 64}) {
        // below two tiles of 128 per compute unit the smaller ones fill the chip better (100 images
        // of 32x32, 3 channels, 5x5: 12.2 us with 800 tiles of 128, 14.0 with 1600 of 64; 82 images
        // of 17x18 outputs, 4 channels, 11x11: 22 us with 196 tiles of 128, 16 with 392 of 64)
        if (p == 128 && (s.npix_out + 127) / 128 < 2u * (uint32_t)g.cus) continue;
        const uint32_t tiles = (s.npix_out + p - 1) / p;
        // few tiles: the filters are split over workgroups, which repeat the gathering
        uint32_t chunks = (2u * (uint32_t)g.cus + tiles - 1) / tiles;
        if (chunks > (uint32_t)s.blocks) chunks = (uint32_t)s.blocks;
        const int per_wg = (s.blocks + (int)chunks - 1) / (int)chunks;
        const size_t lds = set_tile(s, p, per_wg, most_rows(s, p), g.cus);
        if (lds <= (p == 128 ? SHALLOW_LDS / 2 : SHALLOW_LDS)) { *pixels = p; return lds; }
    }
    return 0;
}

} // namespace

// Up to 12 input channels, where the large-launch kernel's pairs of taps are mostly padding.  Timed
// beside it and beside the kernel for few tiles on 110 problems (us a pass, other / this):
//   20 taps or more (5x5 and up) and at most 5/13 as many steps as pairs: ahead throughout, 5x5 of
//   3 channels on 27x27 22.5 / 19.6, 7x7 of 5 channels on 46x46 34.2 / 19.2, 11x11 stride 4 of 3
//   channels 28.3 / 13.1; with more steps the operands fill the LDS and the gathering costs what
//   the shorter walk saves (16 channels 5x5 stride 2 on 24x24 10.4 / 13.2, on 94x94 17.9 / 14.9; 12
//   channels 11x11 33.8 / 38.1);
//   fewer taps: a quarter of the steps, stride 1 and a tile of 128 pixels per compute unit (3x3 of 3
//   channels on 47x47 12.4 / 9.4; smaller or strided 6.5 / 7.5, 7.6 / 9.6);
//   where the kernel for few tiles makes the pass one launch it stays ahead if the steps are more
//   than a quarter, or a tile of 64 pixels reaches over many padded rows (7x7 of 7 channels on
//   12x12 9.1 / 9.7, stride 2 on 7x7 8.9 / 12.9; 11x11 of 5 channels on 128x128 15.9 / 11.9).
// Only where a tile's padded input rows fit the LDS; a tile shape or variant of another kernel
// asked for by name means that kernel.
bool shallow_plan(Plan &g) {
    for (const char *e : {"XNOR_NN_HIP_CONV", "XNOR_NN_HIP_MFMA_PS", "XNOR_NN_HIP_MFMA_PAIR",
                 "XNOR_NN_HIP_MFMA_MIX", "XNOR_NN_HIP_MFMA_SMALL", "XNOR_NN_HIP_MFMA_GROUPS",
                 "XNOR_NN_HIP_MFMA_PERSIST"})
        if (getenv(e)) return false;
    if (g.ic > SHALLOW_CHANNELS || g.kh * g.kw < 2 || g.oh < 1 || g.ow < 1) return false;
    // 32-bit byte offsets, with room for the dropped one, and padded row numbers below 2^31
    if ((uint64_t)g.npix_out * g.oc * 4u >= XNOR_HIP_DROPPED_OFFSET
            || (uint64_t)g.npix_in * 4u >= XNOR_HIP_DROPPED_OFFSET
            || (uint64_t)g.mb * ((g.oh - 1) * g.sh + g.kh) >= 0x7FFFFFFFull)
        return false;
    ShallowPlan s = make_plan(g);
    const int taps = g.kh * g.kw, pairs = (taps + 1) / 2;
    if (taps < 20 ? 4 * s.steps > pairs || g.sh > 1 || g.sw > 1
                || g.npix_out <= 128u * (uint32_t)g.cus
                  : 13 * s.steps > 5 * pairs)
        return false;
    if ((uint64_t)s.blocks * s.steps * 1024u >= XNOR_HIP_DROPPED_OFFSET) return false;
    int pixels = 0;
    const size_t lds = choose_tile(g, s, &pixels);
    if (lds == 0) return false;
    if ((uint64_t)((g.npix_out + 31) / 32) * (uint64_t)s.blocks <= (uint64_t)g.cus
            && (4 * s.steps > pairs || s.max_rows > 40))
        return false;
    g.mfma_shallow = pixels;
    g.shallow = s;
    g.mfma_lds = (uint32_t)lds;
    g.mfma_steps = s.steps;
    g.mfma_wbytes = s.wfrag_bytes;
    return true;
}

hipError_t launch_convolution_shallow(const Plan &g, const uint32_t *xbits,
        const uint32_t *wfrag, const float *alpha, const float *k, float *dst, int32_t *popc,
        const float *a_or_null, float *k_out, hipStream_t stream, const KernelEvents &ev) {
    const ShallowPlan &s = g.shallow;
    const dim3 grid(s.units_per_xcd * 8);
    const v4i *wf = reinterpret_cast<const v4i *>(wfrag);
    const float inv_khw = 1.f / g.kh / g.kw;
#define XNOR_SHALLOW(P_, W_, RAW_) \
    do { \
        static LdsGrant grant; \
        const auto kernel = conv_mfma_fp4_shallow_kernel<P_, W_, RAW_>; \
        const hipError_t e = grant.ask((const void *)kernel, g.mfma_lds); \
        if (e != hipSuccess) return e; \
        launch_kernel(kernel, grid, dim3(64 * W_), g.mfma_lds, stream, ev, xbits, wf, alpha, k, \
                dst, popc, a_or_null, k_out, inv_khw, s); \
    } while (0)
    if (g.mfma_shallow == 128 && s.blocks_per_wg > 2 && g.mfma_lds > SHALLOW_LDS / 8) {
        // with three filter blocks or more there are jobs for eight waves (us a pass with four and
        // eight: AlexNet's first layer, minibatch 64, 48.9 / 43.0; 100 filters 16.6 / 15.1; with 64
        // filters, 8 channels 7x7 on 112x112, 19.6 / 22.6), unless many workgroups fit
        if (popc) XNOR_SHALLOW(128, 8, true);
        else XNOR_SHALLOW(128, 8, false);
    } else if (g.mfma_shallow == 128) {
        if (popc) XNOR_SHALLOW(128, 4, true);
        else XNOR_SHALLOW(128, 4, false);
    } else {
        if (popc) XNOR_SHALLOW(64, 4, true);
        else XNOR_SHALLOW(64, 4, false);
    }
#undef XNOR_SHALLOW
    return hipGetLastError();
}

hipError_t launch_pack_weights_shallow(const Plan &g, const float *w, uint32_t *frag,
        hipStream_t s) {
    const uint32_t dwords = g.mfma_wbytes / 4;
    hipLaunchKernelGGL(pack_weights_shallow_kernel, dim3((dwords + 255) / 256), dim3(256), 0, s,
            w, frag, geometry(g), g.mfma_steps, row_codes_of(g), dwords);
    return hipGetLastError();
}

} // namespace xnor_hip
