// How many rows the experts' large tiles have (sm_moe_tiles.hip): 256, or 128.
//
// 256 from 128 rows per expert on average, else 128 (moe_tiles_kernel, us with 128 / 256 rows, two sizes: 16 experts of 2048 x 1536, 32
// of 1024 x 768: 96 rows per expert 99 / 120, 53 / 75; 128 rows 142 / 120, 78 / 76; 384 rows 229 / 189, 126 / 124; 2048 rows 942 / 734,
// 634 / 514).
//
// Walked over by kWalkers workgroups, one per CU: with fewer than one and a half tiles of 256 rows each, those of 128 share the work out better
// (us with 128 / 256 rows: 4 experts of 2048 x 4096, 192 tiles 94 / 105, 320 131 / 130, 448 194 / 179; 8 of 1024 x 768, 216 77 / 81, 408
// 122 / 130; 16 of 2048 x 1536, 288 132 / 152, 384 174 / 176, 864 377 / 359; 8 of 4096 x 14336, 896 729 / 700, 1344 1139 / 979), but where
// those of 256 fill one round and those of 128 need two: a tile of 128 rows takes 0.5 of the time of one of 256, and 0.07 more for every
// 1024 k (8 experts of 3072 x 2048, 448 rows each 180 / 154, 2 of 4096 x 2048, 1960 rows 220 / 190).  1300 calls of 100 to 430 tiles, 140 of
// them on this line: 0.94 of the time of 128 rows; 7 of the 140 are slower by more than 3 %, up to 1.24 x, whose groups are of unlike size
// and take a tile or two more than the round has.  Below 2048 k it does not pay (76 further calls 1.04, 39 of them slower by more than 3 %).
#pragma once
#include <stdint.h>

constexpr int kWalkers = 256, kWalk256 = 384;

static inline int moe_tile_rows(int64_t pairs, int E) { return pairs >= (int64_t)128 * E ? 256 : 128; }

// Whether tiles that are walked over and could have 256 rows have 128.  `cols`: column tiles of the first product, over K
static inline bool moe_walk_low(int64_t pairs, int E, int cols, int K) {
    const int64_t about = (pairs / 256 + E / 2) * cols;                 // (half a tile of every group is empty)
    if (about >= kWalk256) return false;
    auto even = [&](int rows) { return (pairs + (int64_t)rows * E - 1) / ((int64_t)rows * E) * E * cols; };      // (groups of like size)
    return !(K >= 2048 && even(256) <= kWalkers && even(128) > kWalkers + kWalkers / 2);
}
