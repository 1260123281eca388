// Host-side check of the kernel that a product of f32 weight rows over many rows of x runs (gemv_rows_route in csrc/gemv_rows_plan.h): what
// gemv_rows_form says, except where the left weight rows' items are spread over the waves of all CUs beside the large tiles. There the large
// tiles can be had, a wave has four items at most, no form of fewer launches and whole rounds is passed by, and the shapes measured to be
// faster so are among them.
#include <cstdio>
#include <cstdlib>
#include <initializer_list>

#include "gemv_rows_plan.h"

using namespace fnx;

static long checked = 0;
static void require(bool ok, const char* what, int rows, int n, int T, int cus) {
    ++checked;
    if (ok) return;
    std::printf("FAILED %s: %d weight rows of %d, %d rows of x, %d CUs\n", what, rows, n, T, cus);
    std::exit(1);
}

int main() {
    const int faster[][2] = {{33, 2900}, {65, 1633}, {65, 4000}, {97, 2330}, {129, 918}, {129, 1820}, {129, 4096}, {161, 770}, {258, 500}, {258, 1500}, {1000, 500}};
    for (const auto& f : faster) require(gemv_rows_route(f[0], 2048, f[1], 256) == GemvRows::large_spread, "spread items are the faster", f[0], 2048, f[1], 256);
    // as many small tiles as two a CU, a last row that rides along, whole tiles, more than four items a wave
    const int other[][2] = {{129, 512}, {65, 1000}, {513, 512}, {513, 4096}, {512, 4096}, {257, 482}, {33, 8192}, {129, 4097}};
    for (const auto& f : other) require(gemv_rows_route(f[0], 2048, f[1], 256) != GemvRows::large_spread, "not spread", f[0], 2048, f[1], 256);
    long spread = 0;
    for (int cus : {64, 256, 304})
        for (int n : {2048, 4096, 6144, 1024})
            for (int rows = 1; rows <= 2100; rows += rows < 600 ? 1 : 37)
                for (int T = 17; T <= 9000; T += 23) {
                    const GemvRows f = gemv_rows_route(rows, n, T, cus), g = gemv_rows_form(rows, n, T, cus);
                    if (f != GemvRows::large_spread) {
                        require(f == g, "the form", rows, n, T, cus);
                        continue;
                    }
                    ++spread;
                    const int left = rows % RM_TILE;
                    require(gemv_large_fits(rows, n, T), "large tiles", rows, n, T, cus);
                    require(left > 0 && (long) left * T <= 4l * 4 * cus, "four items a wave", rows, n, T, cus);
                    require(g == GemvRows::large_rest || (g == GemvRows::small_tiles && gemv_small_tiles(rows, T) > 2l * cus), "instead of a second launch or of more than two small tiles a CU", rows, n, T, cus);
                }
    if (!spread) return std::printf("FAILED: never spread\n"), 1;
    std::printf("ok %ld\n", checked);
    return 0;
}
