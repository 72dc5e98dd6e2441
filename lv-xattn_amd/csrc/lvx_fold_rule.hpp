// Which launch folds the parts that a forward launch leaves (lvx_fwd.hip, lvx_rowwise.hip); host code alone, so that it can be tested
// as such.
#pragma once
#include <cstdint>

namespace lvx {

// Lanes (of merge_kernel; chains of fold_before) that share the parts of a row: as many as the parts need, four parts each,
// and the chip has room for.
inline int fold_chains(int nparts, int64_t rows) {
    return nparts > 8 && rows < 16384 ? 4 : nparts > 4 && rows < 32768 ? 2 : 1;
}

// 16-byte chunks that each of `wgs` work-groups of 256 threads folds of `rows` rows of so many, and those it folds at a time.  Whole
// rows, and no more than that: the rows of a head are then folded on the XCD that computed them, and by every work-group (in
// multiples of 256 chunks 200 rows x 32 heads of 64, 6 parts of 4 tiles, took half of 192 work-groups and 14.1 us a round instead of 12.3).
constexpr int64_t FOLD_PASS = 512;
inline int64_t fold_per_wg(int64_t rows, int row_chunks, int64_t wgs) { return (rows + wgs - 1) / wgs * row_chunks; }

// Whether the parts (nparts of `rows` rows of so many 16-byte chunks, over batch and heads) are folded by the next launch of
// a round loop, of `wgs` work-groups, instead of by one of their own.  A launch of its own costs 4 to 6 us; in the next one the fold
// stands in front of a work-group's first tile, 2 to 4 us for a pass.  So it rides where one pass is enough, or two on most
// of the chip, and all work-groups start at once.  us a round, its own launch -> riding:
//   one pass   256 rows x 32 heads, 8 parts of 13 tiles of 64 keys 35.0 -> 34.2; 4 x 16 heads, 102 rows, 8 of 4 19.6 -> 17.8; heads of
//              64, 2 x 16, 256 rows, 4 of 13 22.1 -> 21.0
//   two        441 rows x 32 heads, 4 parts of 16 tiles, 256 work-groups 38.9 -> 37.6; 158 rows x 32, 6 of 4, 144 16.4 -> 17.4
//   four       2 x 16 heads, 256 rows, 2 parts of 13, 64 work-groups 27.4 -> 30.3
//   480 work-groups (256 CUs), three passes: 2 x 64 heads, 280 rows, 3 parts of 39 145 -> 149
inline bool fold_rides(int nparts, int64_t rows, int row_chunks, int64_t wgs, int n_cu) {
    const int64_t passes = (fold_per_wg(rows, row_chunks, wgs) + FOLD_PASS - 1) / FOLD_PASS;
    return nparts > 1 && fold_chains(nparts, rows) <= 2 && wgs <= n_cu && (passes <= 1 || (passes == 2 && 4 * wgs > 3 * n_cu));
}

// Whether the launch of the form for few rows folds its own parts, of `cols` (row, head) columns per kv head.  The last work-group then has
// the fold to itself: a column a wave, and 1.0 us more for every further column of a wave, where a launch of its own spreads them
// over the chip.  us a pass, its own launch -> inside:
//   4 columns  8 kv heads x 6404 keys in 29 parts 12.2 -> 11.4, 4 x 8 x 1601 in 8 11.2 -> 10.6, heads of 64 6404 in 51 11.0 -> 9.3
//   8          8 x 6404 in 29 12.3 -> 13.4, 4 x 8 x 1601 in 8 11.2 -> 11.6, heads of 64 1601 in 26 9.0 -> 8.1, 6404 in 34 10.8 -> 11.8
//   16         8 x 6404 in 29 12.7 -> 17.3
inline bool fold_inside(int nparts, int64_t cols) { return nparts > 1 && cols <= 4; }

}  // namespace lvx
