// The rows that the matrix-core kernels read (xnor_nn_amd/csrc/tap_walk.hpp), walked on the CPU over
// every pixel of every tile of a range of layers: a tap inside the image reads its input pixel, which
// the tile has staged; any other tap, and the two that the kernels ask for behind the last one, read
// the zero row.
#include <cstdio>
#include <random>

#include "plan.hpp"
#include "tap_walk.hpp"

using namespace xnor_hip;

namespace {

template <bool PARTS>
bool walk(const Geometry &g, uint32_t p, int lo, int staged, int parts) {
    const uint32_t row_bytes = 48, part_bytes = 16, zero = 1000;
    const int img = (int)(p / g.ohw), rem = (int)(p % g.ohw), oh = rem / g.ow, ow = rem % g.ow;
    const int ih0 = oh * g.sh - g.ph, iw0 = ow * g.sw - g.pw;
    const int first = img * g.ihw + ih0 * g.iw + iw0 - lo;
    TapWalk<1, PARTS> w;
    w.begin(0, zero + (uint32_t)(1 + first) * row_bytes, taps_inside(ih0, g.ih, g.kh),
            taps_inside(iw0, g.iw, g.kw));
    for (int t = 0; t < g.kh * g.kw + 2; t++) {
        const int kh = t / g.kw, kw = t % g.kw, y = ih0 + kh, x = iw0 + kw;
        const bool inside = kh < g.kh && y >= 0 && y < g.ih && x >= 0 && x < g.iw;
        for (int part = 0; part < parts; part++) {
            uint32_t at[1];
            w.next(at, zero, row_bytes, (uint32_t)(g.iw - g.kw + 1) * row_bytes, g.kw, parts, part_bytes);
            const int input = img * g.ihw + y * g.iw + x - lo; // of the rows that are staged
            const uint32_t want = inside
                ? zero + (uint32_t)(1 + input) * row_bytes + (PARTS ? part * part_bytes : 0) : zero;
            if (at[0] == want && (!inside || (input >= 0 && input < staged))) continue;
            printf("%dx%d kernel %dx%d stride %dx%d padding %dx%d: pixel %u, tap %d of %d, row %d, not %d "
                    "(%d are staged)\n", g.ih, g.iw, g.kh, g.kw, g.sh, g.sw, g.ph, g.pw, p, t,
                    g.kh * g.kw, (int)(at[0] - zero) / (int)row_bytes - 1, inside ? input : -1, staged);
            return false;
        }
    }
    return true;
}

bool layer(int mb, int ih, int iw, int kh, int kw, int sh, int sw, int ph, int pw, uint32_t tile) {
    Geometry g{};
    g.mb = mb; g.ih = ih; g.iw = iw; g.kh = kh; g.kw = kw; g.sh = sh; g.sw = sw; g.ph = ph; g.pw = pw;
    g.oh = (ih + 2 * pw - kh) / sh + 1; // (the reference takes pw for both)
    g.ow = (iw + 2 * pw - kw) / sw + 1;
    if (ih + 2 * pw < kh || iw + 2 * pw < kw) return true;
    g.ihw = ih * iw;
    g.ohw = g.oh * g.ow;
    g.npix_out = (uint32_t)(mb * g.ohw);
    g.div_ohw = FastDiv::make((uint32_t)g.ohw);
    g.div_ow = FastDiv::make((uint32_t)g.ow);
    for (uint32_t from = 0; from < g.npix_out; from += tile) {
        const uint32_t end = from + tile < g.npix_out ? from + tile : g.npix_out;
        // what the large kernel stages, and whole rows, as the one for few tiles does
        for (const auto span : {tile_span, row_span}) {
            int lo, hi;
            span(g, from, end, lo, hi);
            if (lo < 0 || hi < lo || (uint32_t)hi >= (uint32_t)(mb * g.ihw)) {
                printf("%dx%d kernel %dx%d: a tile stages %d to %d\n", ih, iw, kh, kw, lo, hi);
                return false;
            }
            for (uint32_t p = from; p < end; p++)
                if (!walk<false>(g, p, lo, hi - lo + 1, 1) || !walk<true>(g, p, lo, hi - lo + 1, 3))
                    return false;
        }
    }
    return true;
}

// A launch reads the descriptor's plan from any thread: nothing in it may be written through a const one (a
// plan with a mutable member is no constant to copy from).
constexpr Plan PLANNED{};
[[maybe_unused]] constexpr Plan READ_BY_A_LAUNCH = PLANNED;

} // namespace

int main() {
    bool ok = layer(2, 14, 14, 3, 3, 1, 1, 1, 1, 128) && layer(1, 27, 27, 5, 5, 1, 1, 2, 2, 96)
        && layer(3, 7, 7, 1, 1, 1, 1, 0, 0, 32) && layer(1, 40, 40, 32, 32, 1, 1, 3, 3, 64)
        && layer(1, 8, 9, 32, 31, 2, 1, 15, 15, 32) && layer(2, 13, 17, 2, 4, 2, 3, 0, 1, 64);
    std::mt19937 random(1);
    auto from = [&](int lo, int hi) { return lo + (int)(random() % (uint32_t)(hi - lo + 1)); };
    for (int i = 0; ok && i < 400; i++) {
        const int k = from(0, 3) ? from(1, 7) : from(8, 32), p = from(0, k);
        ok = layer(from(1, 2), from(1, 24), from(1, 24), k, from(0, 1) ? k : from(1, 9), from(1, 3),
                from(1, 3), from(0, 2) ? p : from(0, 3), p, 32u * from(1, 4));
    }
    // wide images, whose tiles begin and end inside a row: without a stride between columns, and with one
    for (int i = 0; ok && i < 200; i++) {
        const int k = from(0, 3) ? from(1, 7) : from(8, 32);
        ok = layer(from(1, 2), from(1, 12), from(25, 130), from(0, 1) ? k : from(1, 9), k, from(1, 3),
                i % 4 ? 1 : from(2, 3), from(0, 3), from(0, k), 32u * from(1, 4));
    }
    if (ok) printf("ok\n");
    return ok ? 0 : 1;
}
