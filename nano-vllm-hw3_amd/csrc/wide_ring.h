// Whether groups' tiles of 96 rows (ql_gemm_wide.h) hold weights for 128 k instead of 64: at most one tile for every CU, which then has the registers.
//
// What it saves is a weight's way from memory for every 64 k, what it costs is a longer start.  Few row tiles have their weights from
// memory, more of them have them from L2; over long K the way counts in both.  500 calls of 100 to 256 tiles, weights not in a cache, times the
// figure with 64 k (up to 4 row tiles / 5 to 8 / more), groups of 128 and 256:
//   fp8:   to 512 k 1.04 / 1.04 / 1.05   to 1024 0.96 / 1.05 / 1.05   to 2048 0.93 / 0.95 / 1.02   to 4096 0.92 / 0.92 / 0.96   beyond 0.90 / 0.92 / 0.93
//   int8:  to 512 k 1.02 / 1.05 / 1.06   to 1024 0.97 / 1.04 / 1.05   to 2048 0.94 / 0.97 / 1.02   to 4096 0.94 / 0.93 / 0.94   beyond 0.89 / 0.92 / 0.91
// groups of 64 in fp8: to 512 k 1.00 to 1.02, to 1024 0.94 / 0.96 / 1.01, to 2048 0.90 / 0.90 / 0.98, beyond 0.90 to 0.92.  On these lines all of
// them 0.957, 2 of the 500 slower by more than 3 % (5 and 6 %).
#pragma once
#include <stdint.h>

static inline bool wide_alone(int64_t row_tiles, int64_t col_tiles, int64_t K) {
    if (row_tiles * col_tiles > 256) return false;
    return K > 2048 || (K > 1024 && row_tiles <= 8) || (K > 512 && row_tiles <= 4);
}
