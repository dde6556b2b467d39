// How the 32-row form's workgroups, one for each (row tile, block of 32 columns), are dealt to the eight dies, each with an L2 of its own:
// consecutive workgroups, x first, go to the dies in turn, and those of a die to its 32 CUs in turn.
//
// Tile after tile, a tile's column blocks (filled up to a multiple of eight) one behind the other.  A die so has every eighth block,
// and the tiles of one expert meet its weights in one L2.  Tiles that no expert uses, which come last, have no workgroups between those of
// used ones: an empty workgroup takes its turn, and where a column block's used tiles were followed by its empty ones a CU of a die
// had up to six waves of 54 and another none.  Whole calls, us, weights not in a cache, a block's tiles on neighbouring dies / a block's
// tiles on one die / here: 16 experts of 2048 x 1536, 4 for each of 4 tokens 56 / 56 / 48, of 64 73 / 74 / 67; 8 of 2048 x 1536, 4 for each of 33
// tokens 43.5 / 50.5 / 41.3; 32 of 2048 x 768, one for each of 9 tokens 26.5 / 32.9 / 25.7, of 32 50 / 49 / 47; 1574 calls of 1 to 512 tokens and 4
// to 256 experts: 0.94 of the first, at most 1.045, and 0.95 of the second.
#pragma once
#include <stdint.h>

#ifdef __HIPCC__
#include <hip/hip_runtime.h>
#define MOE_DEAL_FN __host__ __device__ __forceinline__
#else
#define MOE_DEAL_FN inline
#endif

struct MoeGrid { uint32_t x, y, z; };
struct MoePlace { int tile, block; };                // tile >= tiles or block * 32 >= columns: nothing to do

constexpr uint32_t kMoeDealRows = 32768;             // (at most 65535 groups in y)

static inline MoeGrid moe_grid(int tiles, int columns) {
    const uint32_t t = (uint32_t)tiles, z = (t + kMoeDealRows - 1) / kMoeDealRows;
    return {8u * (((uint32_t)columns + 255u) / 256u), z > 1 ? kMoeDealRows : t, z};
}

MOE_DEAL_FN MoePlace moe_place(uint32_t x, uint32_t y, uint32_t z) { return {(int)(z * kMoeDealRows + y), (int)x}; }
