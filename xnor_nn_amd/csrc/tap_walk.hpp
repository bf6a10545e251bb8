// Which LDS row the matrix-core kernels read for each kernel tap of an output pixel.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace xnor_hip {

// Kernel positions t, 0 <= t < taps, with first + t inside an axis of n input pixels, as bits t
// (taps <= 32).
__host__ __device__ __forceinline__ uint32_t taps_inside(const int first, const int n, const int taps) {
    const int from = first < 0 ? -first : 0, to = (n - first < taps ? n - first : taps) - 1;
    return to < from ? 0u : (0xFFFFFFFFu >> (31 - to)) & (0xFFFFFFFFu << from);
}

// The taps of PS pixels one after the other, row by row (PARTS: every tap as many times as it has
// channel parts, which lie one behind the other in a row).  next() gives each pixel's row of the
// coming tap, or the zero row when the tap falls outside the image, as it does for every pixel behind
// the last tap: the kernels ask for up to two taps more than there are.
// The masks are kept reversed, so that a tap is valid if the top bit of both, shifted to it, is set, and
// the address moves along: six instructions per tap and block (an address computed from (kh, kw) took
// fifteen, most of the loop where a tap is one step).
template <int PS, bool PARTS>
struct TapWalk {
    uint32_t row[PS], rowbits[PS], colbits[PS];
    int column = 0, part = 0; // of the next tap

    // row: address of the row of tap (0,0); masks: taps_inside, of the kernel's rows and columns
    __host__ __device__ __forceinline__ void begin(const int ps, const uint32_t first_row,
            const uint32_t rowmask, const uint32_t colmask) {
        row[ps] = first_row;
        rowbits[ps] = __builtin_bitreverse32(rowmask);
        colbits[ps] = __builtin_bitreverse32(colmask);
    }
    // to_next_row: from the tap in a kernel row's last column to the first one of the row below
    __host__ __device__ __forceinline__ void next(uint32_t (&out)[PS], const uint32_t zero_row,
            const uint32_t row_bytes, const uint32_t to_next_row, const int kw, const int parts,
            const uint32_t part_bytes) {
#pragma unroll
        for (int ps = 0; ps < PS; ps++)
            out[ps] = (int)(rowbits[ps] & (colbits[ps] << column)) < 0
                ? row[ps] + (PARTS ? (uint32_t)part * part_bytes : 0u) : zero_row;
        if constexpr (PARTS) {
            if (++part < parts) return;
            part = 0;
        }
        const bool next_row = ++column == kw; // uniform
        column = next_row ? 0 : column;
#pragma unroll
        for (int ps = 0; ps < PS; ps++) {
            rowbits[ps] <<= next_row ? 1 : 0;
            row[ps] += next_row ? to_next_row : row_bytes;
        }
    }
};

} // namespace xnor_hip
