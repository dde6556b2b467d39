// How the prompt attention kernels' workgroups are dealt to the eight dies, each with an L2 of its own.  A kernel's work is
// `tiles` row tiles (tile 0 the heaviest: the last rows, which see most keys) of each of B sequences by G groups of heads; a
// (sequence, group) pair's tiles read the same keys and values.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define ROW_DEAL_FN __host__ __device__ __forceinline__
#else
#define ROW_DEAL_FN inline
#endif

// Two grids; consecutive workgroups go to the dies in turn.
// Few pairs, which would leave dies idle, or more than the other grid holds: (tiles, G, B), every tile to the next die (run 0); tiles
// are counted from the end of the longest sequence.
// Else eight pairs after eight pairs, (8 tiles, ceil(B G / 8)), tiles counted from a sequence's own end: a run of kRowRun neighbouring
// tiles of a pair on one die, whose L2 then reads their keys once, and the next run of the pair as many dies further on as a
// sequence's heads take, so that one long prompt among short ones has the whole chip.  (All tiles of a pair on one die / runs / dealt one
// by one in an older kernel, us: 2000 tokens and 31 single ones in latent attention, 16 heads: 269 / 94 / 104; 8192 and 7 single ones 3292 /
// 508 / 850; 8 x 1000 90 / 82 / 164.  16 / 2 heads, paged, 8192 and 7 single ones 1266 / 363 / 792.  Runs of 4 and of 16 are within 3 %.)
// The number of a pair's places is odd: a die deals its workgroups to its shader engines in turn, too, and with an even one the
// single tiles of the short sequences all met on one of them (500 tokens and 127 single ones, 16 / 8 heads: 331 / 126 us).  Below
// eight tiles the empty place would cost more (8 x 100 tokens, 32 / 8 heads: 8.9 / 10.7 us).
constexpr int kRowRun = 8;

struct RowGrid { uint32_t x, y, z; int run; };

static inline RowGrid row_grid(int64_t tiles, int B, int G) {
    const int64_t pairs = (int64_t)B * G;
    if ((pairs >= 32 || pairs % 8 == 0) && pairs <= 8 * 65535 && tiles < 1 << 20)        // (2^32 threads in x, 65535 groups in y)
        return {(uint32_t)(8 * (tiles < 8 ? tiles : tiles | 1)), (uint32_t)((pairs + 7) / 8), 1u, kRowRun};
    return {(uint32_t)tiles, (uint32_t)G, (uint32_t)B, 0};
}

struct RowTile { int b, g, tile; };                  // b < 0: nothing to do

// the first row of tile `tile` of a sequence of `rows` rows, in tiles of `size`; negative or past the rows: nothing to do.  (Counted
// from a sequence's own end its heavy tiles come early also where it is short and continues a long cached prefix: eight prompts of
// 900 to 1100 tokens, two of them half cached, latent attention: 93 us counted from the longest one's end, 81 so.)
ROW_DEAL_FN int row_first(int run, int tile, int tiles, int rows, int size) {
    return ((run ? (rows + size - 1) / size : tiles) - 1 - tile) * size;
}

// the tile of workgroup (x, y, z)
ROW_DEAL_FN RowTile row_tile(uint32_t x, uint32_t y, uint32_t z, int run, int tiles, int B, int G) {
    if (run == 0) return {(int)z, (int)y, (int)x};
    const int tile = x >> 3, step = G & -G;          // step: a divisor of eight (or a multiple, which stays), 8 / step dies per pair
    const int pair = 8 * (int)y + (((int)(x & 7) - step * (tile / run)) & 7);
    if (pair >= B * G || tile >= tiles) return {-1, 0, 0};
    return {pair / G, pair % G, tile};
}
