// Host build of the tracers' tile order (sirius_amd/csrc/geodesic.hpp) for images as large as a batch may
// be, of few rows and of few columns among them: positions at the ends of the image, of its bands and
// of its tiles, and some in between, map to the pixel that 64-bit arithmetic gives. Prints "OK".
#include "../../sirius_amd/csrc/geodesic.hpp"

#include <cstdio>

using namespace sirius;

// The order in 64 bits: bands of 64 >> lw rows, tiles of 1 << lw columns, row by row inside a tile.
static int64_t pixel64(int64_t w, int64_t h, int lw, int64_t t) {
    const int64_t tw = 1LL << lw, th = 64LL >> lw, band = t / (th * w), y0 = band * th;
    const int64_t bh = h - y0 < th ? h - y0 : th, in = t - y0 * w;
    const int64_t x0 = in / (tw * bh) * tw, cw = w - x0 < tw ? w - x0 : tw, q = in - x0 * bh;
    return (y0 + q / cw) * w + x0 + q % cw;
}

int main() {
    const int64_t most = 2147483647LL - (1 << 20);  // rays of a batch
    const int64_t sides[] = {1, 2, 3, 5, 7, 8, 9, 64, 65, 1000, 46340, 131071, 1LL << 20, 268435456, 268435457, 536870911,
                             536870912, 536870913, 600000000, 1073741824, most};
    long images = 0;
    for (int lw : {TILE_SQUARE, TILE_ROW})
        for (int64_t w : sides)
            for (int64_t hh : sides) {
                const int64_t h = hh < most / w ? hh : most / w, n = w * h;  // as many rows as fit
                if (h < 1) continue;
                ++images;
                auto check = [&](int64_t t) {
                    if (t < 0 || t >= n) return true;
                    const int64_t p = tile_pixel((int)w, (int)h, lw, t), r = pixel64(w, h, lw, t);
                    if (p != r) std::printf("%lld x %lld lw %d position %lld: %lld, not %lld\n", (long long)w, (long long)h, lw, (long long)t, (long long)p, (long long)r);
                    return p == r;
                };
                const int64_t band = (64LL >> lw) * w;
                const int64_t at[] = {0, 64, n / 3, n / 2, n - 1, band, n / band * band, n / 2 / band * band + band, 505032704};
                for (int64_t t : at)
                    for (int64_t d = -1; d <= 1; ++d)
                        if (!check(t + d)) return 1;
                for (int64_t k = 0; k < 1000; ++k)
                    if (!check((int64_t)((unsigned long long)k * 0x9E3779B97F4A7C15ull % (unsigned long long)n))) return 1;
            }
    std::printf("%ld images\n", images);
    std::puts("OK");
    return 0;
}
