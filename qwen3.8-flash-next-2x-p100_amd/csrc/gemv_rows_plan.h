// Which kernel takes a product of f32 weight rows (a router's) over more rows of x than a window has. A plain function of the
// shape and the device's CUs, compiled (by the plan test) for the host too, so that the lines below can be looked at at every
// shape without running a kernel.
#pragma once

namespace fnx {

constexpr int RM_TILE = 32;                  // the large tiles (k_gemv_rows_mfma): rows of x and of W
constexpr int RS_TILE = 16, RS_COLS = 256;   // the small ones (k_gemv_rows_mfma16); the columns of a stage

enum class GemvRows {
    many,         // k_gemv_rows_many: no tiles
    small_tiles,
    large_tiles,
    large_rest,   // the large tiles, and a second launch (k_gemv_rows_many) for the weight rows past the last full tile
    large_spread  // the large tiles, those weight rows' items (such a row x a row of x) over the waves of all CUs
};
inline long gemv_small_tiles(int rows, int T) { return (long) ((T + RS_TILE - 1) / RS_TILE) * ((rows + RS_TILE - 1) / RS_TILE); }
// The weight rows past the last full large tile ride with the tiles' blocks, an item (such a row x a row of x) a wave of the four, as
// long as a row of tiles has a wave for each of its 32 items a left row.
inline bool gemv_rest_along(int rows) { return 8 * (rows % RM_TILE) <= rows / RM_TILE; }

// The small tiles where the larger ones would leave CUs idle, or cannot be had; the larger ones read each row from the L2 half as
// often, and that is the time of a long chunk. A CU takes its small tiles one after the other, 4.5 us each.
// Three take longer than its one large one: up to two a CU. 513 weight rows of 2,048, weights in turn, us (small / large): 64 rows of x 5.7 /
// 13.2, 128 10.0 / 13.4, 240 10.2 / 13.4, 280 14.3 / 13.7, 320 15.1 / 13.5; 257 weight rows, 482 rows of x 15.9 / 13.3.
// Where the left weight rows want a second launch (11 us and more, whatever it computes), four a CU. 2,048 columns (small / large and
// rest): 33 weight rows, 2,900 rows of x 18.1 / 34.9, 5,000 24.5 / 47.1, 6,000 29.8 / 48.1; 65, 1,633 17.4 / 24.2, 3,200 25.3 / 35.4; 129, 897
// 17.0 / 23.9, 1,300 19.1 / 24.4; 300, 512 16.7 / 25.0; 1,000, 140 14.2 / 24.7, 240 19.5 / 25.6. Between 7/2 and four a CU most shapes still gain, their
// large tiles being more than a round of the CUs: 97, 2,330 25.4 / 35.0; 161, 1,480 25.8 / 34.6; 193, 1,240 25.9 / 34.5; 300, 780 24.4 / 35.3; those whose large
// tiles are one round are a little behind: 129, 1,600 24.3 / 24.5, 1,728 25.0 / 24.6, 1,808 25.3 / 25.0, 225, 1,020 24.8 / 24.4, and at five 129, 1,820 29.2 / 25.1. Wider
// rows the same: of 4,096, 129, 1,500 39.4 / 40.9, 1,808 44.5 / 41.6, 161, 1,480 43.8 / 58.8; of 8,192, 129, 1,500 71.9 / 73.8, 1,808 81.0 / 75.4, 300, 800 76.7 / 109, 65,
// 3,200 79.4 / 108.
// Where the large ones cannot be had, k_gemv_rows_many is the other kernel: it reads a row of x once for four weight rows a
// wave, and fills the chip only with many rows. The narrower the rows, the more of a small tile's time is its start and its
// end, so it is the better one up to 5/2, 8 and 12 tiles a CU at widths of 512, 1024 and 1536, and always from 2048 on.
// 513 weight rows, us (small / many): 512 wide, 64 rows 4.5 / 6.9, 300 9.6 / 10.2, 450 11.9 / 10.7, 3000 66.6 / 44.1; 1024 wide, 64
// 5.1 / 9.7, 1000 30.4 / 31.8, 1500 48.6 / 41.6; 1536 wide, 64 5.7 / 12.4, 1000 42.8 / 43.5, 1500 60.9 / 57.5; 2560 wide, 64 7.3 / 17.8,
// 3000 163 / 185; 2048 weight rows of 1024, 300 32.5 / 32.6, 450 47.0 / 46.2; of 3072, 3000 647 / 750.
// T: more than a window's; cus: the device's. The pointers are 16-byte aligned (else: many).
inline bool gemv_large_fits(int rows, int n, int T) {   // the large tiles can be had
    return T >= 2 * RM_TILE && rows >= RM_TILE && n % 2048 == 0 && (unsigned long long) T * n * 4 < (1ull << 32) &&
           (unsigned long long) rows * n * 4 < (1ull << 32);
}
inline GemvRows gemv_rows_form(int rows, int n, int T, int cus) {   // where no items are spread (below)
    const bool large = gemv_large_fits(rows, n, T);
    const long tiles = gemv_small_tiles(rows, T), most = 1l << 24;
    const long upto = large ? (gemv_rest_along(rows) ? 2l : 4l) * cus : n == 512 ? 5l * cus / 2 : n == 1024 ? 8l * cus : n == 1536 ? 12l * cus : most;
    if (n % (2 * RS_COLS) == 0 && tiles < most && tiles <= upto) return GemvRows::small_tiles;
    if (!large) return GemvRows::many;
    return gemv_rest_along(rows) ? GemvRows::large_tiles : GemvRows::large_rest;
}
// Large tiles with the left weight rows' items spread over the waves of all CUs, up to four each, instead of the small tiles or the second
// launch that the form says: from where the small tiles are more than two a CU, the line of the rows that ride along. 2,048 columns, us (as the
// form says / so): 33 weight rows, 2,900 rows of x 18.0 / 16.8; 65, 1,633 17.4 / 14.9, 4,000 36.3 / 18.4; 97, 2,330 25.3 / 16.2; 129, 918 17.7 / 13.7, 1,820
// 25.0 / 15.4, 4,096 37.9 / 29.3; 161, 770 17.2 / 13.4; 258, 500 16.3 / 13.6, 1,500 35.5 / 26.1; 1,000, 500 36.9 / 27.5.
inline bool gemv_rest_spread(int rows, int n, int T, int cus) {
    return gemv_large_fits(rows, n, T) && rows % RM_TILE && !gemv_rest_along(rows) && gemv_small_tiles(rows, T) > 2l * cus && (long) (rows % RM_TILE) * T <= 16l * cus;
}
inline GemvRows gemv_rows_route(int rows, int n, int T, int cus) {   // the kernel that runs
    return gemv_rest_spread(rows, n, T, cus) ? GemvRows::large_spread : gemv_rows_form(rows, n, T, cus);
}

}  // namespace fnx
