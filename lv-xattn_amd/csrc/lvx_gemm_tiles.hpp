// Which of the hand-scheduled GEMM tiles a product takes (lvx_gemm.hip); host code alone, so that it can be tested as such.
#pragma once
#include <cstdint>

namespace lvx {

enum GemmTile { TILE_256_256, TILE_256_128, TILE_224_256 };     // rows x columns

// The tile whose rounds of work-groups on `n_cu` CUs cost least, for C [M, N] of `nprob` problems; `lower`: there is a 224-row
// tile for this layout.  Prices of a round against one of 256 x 256, in thousandths:
//   256 x 128: 0.615 (2046 x 4096 x 4096: one round of 256 wide 81 us, one of 128 60; 5000 x 4096 of 2 x 1024 three rounds
//     95 us, two of 224 rows 89; 12808 x 4096 x 1024 twice: two rounds 184, four of 128 214).
//   224 x 256: 0.915, of rounds that are full: an eighth less work, a quarter more LDS reads per MFMA, and the matrix pipe
//     under the same power.  In as many rounds as 256 rows need it always wins, 2 % where those are full and 10 where they are
//     not, because it leaves fewer CUs idle: 6404 x 4096 x 1024 twice 91.6 us -> 88.0, 12808 184 -> 174, 28000 382 -> 362, dX 6404
//     x 4096 of 2 x 1024 103 -> 96.4, 25000 372 -> 349.  In one round more it loses up to ten rounds of 256 rows (57000
//     in 8 instead of 7 744 -> 762, 66000 in 10 instead of 9 883 -> 899, 76848 in 11 instead of 10 1028 -> 1034, with the norm 1058
//     -> 1073) and wins from eleven (84000 1134 -> 1121, dX 42000 593 -> 582); two more are always too many (150000 in 21
//     instead of 19 1980 -> 1983, 108000 in 16 instead of 14 1419 -> 1455).
inline GemmTile gemm_tile(int64_t M, int64_t N, int nprob, int n_cu, bool lower) {
    auto rounds = [&](int tm, int tn) { return ((M + tm - 1) / tm * nprob * ((N + tn - 1) / tn) + n_cu - 1) / n_cu; };
    const int64_t wide = 1000 * rounds(256, 256), narrow = 615 * rounds(256, 128);
    const int64_t low = lower ? 915 * rounds(224, 256) : INT64_MAX;
    if (low < wide && low < narrow) return TILE_224_256;
    return narrow < wide ? TILE_256_128 : TILE_256_256;
}

}  // namespace lvx
