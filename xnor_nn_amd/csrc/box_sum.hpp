// K of one output pixel per lane from mean|x| of the staged input pixels: the box filter of stage 2
// as the convolution kernels sum it (in-bounds taps in row-major order, each product rounded, then
// added: reference src/bcast_calculate_k.cpp:69-85).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xnor_hip {

// a: mean|x| of the staged pixels in LDS, `limit` of them at most; first: index of tap (0,0), which
// may lie outside; bits kh of rowmask and kw of colmask: taps inside the image.
// A row's KW values are read from neighbouring addresses whether their taps lie inside or not, and
// those that do not are replaced by +0, which leaves a sum of non-negative terms (and a NaN) as it is:
// an address per row and three vector instructions per tap, with a row's reads under way while the
// row ahead of it is added.  (An address selected per tap took eight.)  A row that has a valid tap
// begins at -(KW-1) at least and limit-1 at most; others are moved there, so reads reach from
// KW-1 floats ahead of a to KW-1 floats past a[limit]: LDS of the same workgroup on both sides.
// A kernel of fewer columns runs the next wider one: a column past its last has no bit in the mask.
// MASKS: the columns' bits are kept as a lane mask each, two scalar registers: 22 with 11 columns, for which
// the convolution kernels with two tile sizes spilled 20 to 42 of theirs.  Those test a bit where it is used, two
// vector instructions more per tap: us a pass with the masks / without, two tile sizes, 384 channels on 13x13,
// minibatch 256, 43.2 / 42.9, 512 on 28x28, minibatch 32, 36.7 / 36.8 (two runs of one side differ by 0.5 %);
// one tile size, 11x11 stride 4, 32 to 192 channels on 170x174, 4, 16.9 / 17.5, 41 to 64 on 208x207, 5,
// 40.7 / 41.9, 48 to 512 on 225x225, 8, 125.6 / 127.9.
// What it bounds: the end of a tile's staging, which the waves that sum K reach last.  32 to 64
// channels 5x5 on 32x32, minibatch 100: 3.6 -> 1.1 us of a tile's 10.2 (a pass 17.2 -> 15.3); 3x3: a
// pass of 64 channels on 56x56, minibatch 4, 9.9 -> 8.6.  Rows of 11 and of even widths (the loop at
// the end before), us of the kernel: 11x11 stride 4, 16 channels on 83x83, minibatch 64, 20.0 -> 17.2,
// 48 on 120x120, 30, 44.1 -> 37.4, 16 on 85x86, 3, 12.6 -> 10.1; 8x8, 6x6, 4x4 and 2x2 of 16 channels on
// 22x22, 3: 8.2 -> 7.0, 7.4 -> 6.2, 5.5 -> 4.9, 4.8 -> 4.5.
template <int KW, bool MASKS>
__device__ __forceinline__ float box_sum_rows(const float *a, const int first, const int limit,
        const uint32_t rowmask, const uint32_t colmask, const int kh_n, const int iw,
        const float inv_khw) {
    [[maybe_unused]] bool col[KW];
    if constexpr (MASKS)
#pragma unroll
        for (int x = 0; x < KW; x++) col[x] = (colmask >> x) & 1u;
    auto fetch = [&](float (&t)[KW], int kh) {
        const float *row = a + max(min(first + kh * iw, limit), 1 - KW);
#pragma unroll
        for (int x = 0; x < KW; x++) t[x] = row[x];
    };
    float t[KW], sum = 0.f;
    fetch(t, 0);
    for (int kh = 0; kh < kh_n; kh++) {
        float next[KW];
        fetch(next, kh + 1); // (past the last row: read and not used)
        const bool in_row = (rowmask >> kh) & 1u;
        const uint32_t inside = in_row ? colmask : 0u;
#pragma unroll
        for (int x = 0; x < KW; x++) {
            bool in;
            if constexpr (MASKS) in = in_row && col[x];
            else in = (inside >> x) & 1u;
            sum = __fadd_rn(sum, __fmul_rn(in ? t[x] : 0.f, inv_khw));
        }
#pragma unroll
        for (int x = 0; x < KW; x++) t[x] = next[x];
    }
    return sum;
}

template <bool MASKS>
__device__ __forceinline__ float box_sum(const float *a, const int first, const int limit,
        const uint32_t rowmask, const uint32_t colmask, const int kh_n, const int kw_n, const int iw,
        const float inv_khw) {
    if (kw_n == 1) return box_sum_rows<1, MASKS>(a, first, limit, rowmask, colmask, kh_n, iw, inv_khw);
    if (kw_n <= 3) return box_sum_rows<3, MASKS>(a, first, limit, rowmask, colmask, kh_n, iw, inv_khw);
    if (kw_n <= 5) return box_sum_rows<5, MASKS>(a, first, limit, rowmask, colmask, kh_n, iw, inv_khw);
    if (kw_n <= 7) return box_sum_rows<7, MASKS>(a, first, limit, rowmask, colmask, kh_n, iw, inv_khw);
    if (kw_n <= 11) return box_sum_rows<11, MASKS>(a, first, limit, rowmask, colmask, kh_n, iw, inv_khw);
    // four taps per round, all reads of a round issued before its first addition; a tap outside
    // the image reads the slot past the last pixel, which holds zero
    float sum = 0.f;
    for (int kh = 0; kh < kh_n; kh++)
        for (int kw0 = 0; kw0 < kw_n; kw0 += 4) {
            float term[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int kw = kw0 + u;
                const bool ok = kw < kw_n && ((rowmask >> kh) & (colmask >> (kw & 31)) & 1u);
                term[u] = __fmul_rn(a[ok ? first + kh * iw + kw : limit], inv_khw);
            }
#pragma unroll
            for (int u = 0; u < 4; u++) sum = __fadd_rn(sum, term[u]);
        }
    return sum;
}

} // namespace xnor_hip
