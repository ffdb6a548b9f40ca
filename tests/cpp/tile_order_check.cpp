// Host build of the tracers' tile order (sirius_amd/csrc/geodesic.hpp): for images from 1 x 1 to wider
// and taller than several tiles, in rows and in squares, every position maps to one pixel and every
// pixel is taken once, and 64 consecutive positions from a multiple of 64 inside a full band of
// tiles are one tile. Prints "OK".
#include "../../sirius_amd/csrc/geodesic.hpp"

#include <cstdio>
#include <vector>

using namespace sirius;

int main() {
    const int sides[] = {1, 2, 7, 8, 9, 63, 64, 65, 100, 131};
    for (int lw : {TILE_SQUARE, TILE_ROW})
        for (int w : sides)
            for (int h : sides) {
                std::vector<char> seen((size_t)w * h, 0);
                const int tw = 1 << lw, th = 64 >> lw;
                for (int64_t t = 0; t < (int64_t)w * h; ++t) {
                    const int64_t p = tile_pixel(w, h, lw, t);
                    if (p < 0 || p >= (int64_t)w * h || seen[p]) return std::printf("%d x %d lw %d at %lld\n", w, h, lw, (long long)t), 1;
                    seen[p] = 1;
                    const int64_t band = t / ((int64_t)th * w), in = t - band * th * w;
                    if (band * th + th <= h && in / 64 * tw + tw <= w)
                        if (p / w / th != band || p % w / tw != in / 64) return std::printf("tile %d x %d lw %d at %lld\n", w, h, lw, (long long)t), 1;
                }
            }
    // the largest batches: 2^31 pixels
    if (tile_pixel(46340, 46340, TILE_SQUARE, 46340LL * 46340 - 1) != 46340LL * 46340 - 1) return std::puts("largest"), 1;
    std::puts("OK");
    return 0;
}
