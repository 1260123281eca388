// Host-side check of which kernel takes a product of f32 weight rows over many rows of x (csrc/gemv_rows_plan.h): over the
// shapes of routers of a few dozen to two thousand experts and chunks of up to 4,096 rows, no second launch where the small
// tiles are the faster (up to four a CU), no large tiles where a CU has at most two small ones, and none where they cannot be had.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "gemv_rows_plan.h"

using namespace fnx;

static long checked = 0;
static void require(bool ok, const char* what, int rows, int n, int T) {
    ++checked;
    if (ok) return;
    std::printf("FAILED %s: %d weight rows of %d, %d rows of x\n", what, rows, n, T);
    std::exit(1);
}

int main() {
    const int cus = 256;
    // measured to be the faster as small tiles: 33, 65, 129, 300 and 1,000 weight rows, whose last rows would want a launch of their own
    const int faster[][2] = {{33, 2900}, {33, 4000}, {65, 1633}, {65, 2048}, {129, 897}, {129, 1136}, {129, 1300}, {300, 432}, {300, 512}, {300, 800}, {1000, 130}, {1000, 240}};
    for (const auto& f : faster) require(gemv_rows_form(f[0], 2048, f[1], cus) == GemvRows::small_tiles, "small tiles are the faster", f[0], 2048, f[1]);
    // and as large ones: 257 and 513 weight rows, whose last row rides along, and whole tiles
    const int large[][2] = {{257, 482}, {513, 249}, {513, 4096}, {2048, 80}};
    for (const auto& f : large) require(gemv_rows_form(f[0], 2048, f[1], cus) == GemvRows::large_tiles, "large tiles are the faster", f[0], 2048, f[1]);
    for (int n : {2048, 4096, 6144})
        for (int rows = 1; rows <= 2100; rows += rows < 600 ? 1 : 37)
            for (int T = 17; T <= 4096; T += 13) {
                const GemvRows f = gemv_rows_form(rows, n, T, cus);
                const long tiles = gemv_small_tiles(rows, T);
                const int net = rows / RM_TILE, left = rows % RM_TILE;
                require(f != GemvRows::many, "tiles of either kind", rows, n, T);
                if (tiles <= 2 * cus || T < 2 * RM_TILE || rows < RM_TILE) require(f == GemvRows::small_tiles, "small tiles", rows, n, T);
                if (f == GemvRows::large_rest) require(left > 0 && tiles > 4 * cus, "a launch for the rest", rows, n, T);
                if (f == GemvRows::large_tiles) require(RM_TILE * left <= 4 * net, "a wave an item of the rest", rows, n, T);
            }
    for (int n : {256, 768, 1280}) require(gemv_rows_form(513, n, 300, cus) == GemvRows::many, "no tiles", 513, n, 300);
    std::printf("ok %ld\n", checked);
    return 0;
}
