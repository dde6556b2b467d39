// The grouping in front of the expert products: (token, choice) pairs sorted by expert into tiles of `unit` rows.
//
// One workgroup, because every row number depends on every count.  What it spends its time in are the LDS counters: with one
// counter per expert all waves meet on a few addresses, so every wave (or a few of them, for very many experts) counts on a
// copy of its own, and the position that its counter returned is kept, so that pairs are counted once and not twice; and the
// loads, which a thread therefore requests sixteen at a time (32768 pairs over 16 experts: 35 -> 25 us).
#include <algorithm>

#include "sm_common.h"

namespace sm {

constexpr int kAlignThreads = 1024, kAlignWaves = kAlignThreads / 64, kBatch = 16;
constexpr int64_t kMaxBlocks = 64, kManyPairs = 12288;         // (16 experts, us, one workgroup / two launches: 8192 pairs 9.2 / 9.4, 12000 11.0 / 9.3)

__global__ __launch_bounds__(kAlignThreads) void moe_align_kernel(const int32_t* __restrict__ idx, int P, int E, int copies, int unit,
                                                                  int max_tiles, int32_t* __restrict__ row_pair,
                                                                  int32_t* __restrict__ tile_expert, int32_t* __restrict__ pair_row) {
    extern __shared__ int cnt[];                // [copies][E]: counts, then the first row of the copy's pairs
    const int lane = threadIdx.x & 63;
    int* mine = cnt + (threadIdx.x >> 6) % copies * E;
    const int max_rows = max_tiles * unit;
    // Up to kHeld pairs per thread stay in registers, experts asked for in front of everything else (256 pairs over 16 experts: 3.4 us, with
    // both read again from memory behind the sums, and the copies of waves without pairs counted one by one, 5.2)
    constexpr int kHeld = 4;
    const bool held = P <= kHeld * kAlignThreads;
    int he[kHeld], hr[kHeld];
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
        const int p = (int)threadIdx.x + j * kAlignThreads;
        he[j] = held && p < P ? idx[p] : -1;
    }
    for (int i = threadIdx.x; i < copies * E; i += kAlignThreads) cnt[i] = 0;
    for (int i = threadIdx.x; i < max_tiles; i += kAlignThreads) tile_expert[i] = -1;
    for (int i = threadIdx.x; i < max_rows; i += kAlignThreads) row_pair[i] = -1;
    __syncthreads();
    if (held)
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            if ((unsigned)he[j] >= (unsigned)E) he[j] = -1;
            hr[j] = he[j] >= 0 ? atomicAdd(&mine[he[j]], 1) : 0;
        }
    for (int p0 = threadIdx.x; p0 < P && !held; p0 += kBatch * kAlignThreads) {
        int e[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int p = p0 + j * kAlignThreads;
            e[j] = p < P ? idx[p] : -1;
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) e[j] = e[j] >= 0 && e[j] < E ? atomicAdd(&mine[e[j]], 1) : 0;
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int p = p0 + j * kAlignThreads;
            if (p < P) pair_row[p] = e[j];
        }
    }
    __syncthreads();
    if (threadIdx.x < 64) {                     // a wave takes 64 experts at a time
        int tiles = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane;
            int total = 0, k[kAlignWaves];      // (all copies' counts at once)
#pragma unroll
            for (int c = 0; c < kAlignWaves; ++c) k[c] = c < copies && e < E ? cnt[c * E + e] : 0;
#pragma unroll
            for (int c = 0; c < kAlignWaves; ++c) total += k[c];
            const int n = (total + unit - 1) / unit;
            int upto = n;                       // tiles of the experts up to this one
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(upto, o);
                if (lane >= o) upto += v;
            }
            const int first = tiles + upto - n;
            if (e < E) {
                for (int i = 0; i < n && first + i < max_tiles; ++i) tile_expert[first + i] = e;
                int row = first * unit;
#pragma unroll
                for (int c = 0; c < kAlignWaves; ++c) {
                    if (c < copies) cnt[c * E + e] = row;
                    row += k[c];
                }
            }
            tiles += __shfl(upto, 63);
        }
    }
    __syncthreads();
    if (held) {
#pragma unroll
        for (int j = 0; j < kHeld; ++j) {
            const int p = (int)threadIdx.x + j * kAlignThreads;
            if (p >= P) continue;
            const int row = he[j] >= 0 ? mine[he[j]] + hr[j] : 0;
            if (he[j] >= 0 && row < max_rows) row_pair[row] = p;
            pair_row[p] = min(row, max_rows - 1);
        }
        return;
    }
    for (int p0 = threadIdx.x; p0 < P; p0 += kBatch * kAlignThreads) {
        int e[kBatch], r[kBatch];
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int p = p0 + j * kAlignThreads;
            e[j] = p < P ? idx[p] : -1;
            r[j] = p < P ? pair_row[p] : 0;
        }
#pragma unroll
        for (int j = 0; j < kBatch; ++j) {
            const int p = p0 + j * kAlignThreads;
            if (e[j] < 0 || e[j] >= E) continue;
            const int row = mine[e[j]] + r[j];
            if (row < max_rows) row_pair[row] = p;
            pair_row[p] = min(row, max_rows - 1);
        }
    }
}

// Many pairs: blocks of `chunk` of them count at the same time, then every block works out where its pairs of each expert begin.  Two
// launches instead of one, and the counts of all blocks go through memory: `counts`, [blocks][E].  (32768 pairs over 16 experts 25 -> 10 us.)
__global__ __launch_bounds__(kAlignThreads) void moe_align_count_kernel(const int32_t* __restrict__ idx, int P, int E, int copies, int chunk,
                                                                        int max_rows, int max_tiles, int32_t* __restrict__ row_pair,
                                                                        int32_t* __restrict__ tile_expert, int32_t* __restrict__ pair_row,
                                                                        int32_t* __restrict__ counts) {
    extern __shared__ int cnt[];                // [copies][E]: counts, then the copy's first position among the block's pairs
    int* mine = cnt + (threadIdx.x >> 6) % copies * E;
    const int begin = blockIdx.x * chunk, end = min(P, begin + chunk);
    for (int i = threadIdx.x; i < copies * E; i += kAlignThreads) cnt[i] = 0;
    for (int i = blockIdx.x * kAlignThreads + threadIdx.x; i < max_tiles; i += gridDim.x * kAlignThreads) tile_expert[i] = -1;
    for (int i = blockIdx.x * kAlignThreads + threadIdx.x; i < max_rows; i += gridDim.x * kAlignThreads) row_pair[i] = -1;
    __syncthreads();
    for (int p = begin + threadIdx.x; p < end; p += kAlignThreads) {
        const int e = idx[p];
        pair_row[p] = e >= 0 && e < E ? atomicAdd(&mine[e], 1) : 0;
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += kAlignThreads) {
        int at = 0;
        for (int c = 0; c < copies; ++c) {
            const int k = cnt[c * E + e];
            cnt[c * E + e] = at;
            at += k;
        }
        counts[(size_t)blockIdx.x * E + e] = at;
    }
    __syncthreads();
    for (int p = begin + threadIdx.x; p < end; p += kAlignThreads) {
        const int e = idx[p];
        if (e >= 0 && e < E) pair_row[p] += mine[e];
    }
}

__global__ __launch_bounds__(kAlignThreads) void moe_align_place_kernel(const int32_t* __restrict__ idx, int P, int E, int chunk, int unit,
                                                                        int max_tiles, int32_t* __restrict__ row_pair,
                                                                        int32_t* __restrict__ tile_expert, int32_t* __restrict__ pair_row,
                                                                        const int32_t* __restrict__ counts) {
    extern __shared__ int cnt[];                // [E] tiles, then first rows of this block's pairs; [E] pairs of the blocks before it
    int* before = cnt + E;
    const int begin = blockIdx.x * chunk, end = min(P, begin + chunk), max_rows = max_tiles * unit;
    for (int e = threadIdx.x; e < E; e += kAlignThreads) {
        int total = 0, mine = 0;
#pragma unroll 8
        for (int b = 0; b < (int)gridDim.x; ++b) {
            const int k = counts[(size_t)b * E + e];
            mine += b < (int)blockIdx.x ? k : 0;
            total += k;
        }
        cnt[e] = (total + unit - 1) / unit;
        before[e] = mine;
    }
    __syncthreads();
    if (threadIdx.x < 64) {                     // a wave takes 64 experts at a time
        const int lane = threadIdx.x;
        int tiles = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + lane, n = e < E ? cnt[e] : 0;
            int upto = n;                       // tiles of the experts up to this one
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const int v = __shfl_up(upto, o);
                if (lane >= o) upto += v;
            }
            const int first = tiles + upto - n;
            if (e < E) {
                if (blockIdx.x == 0)
                    for (int i = 0; i < n && first + i < max_tiles; ++i) tile_expert[first + i] = e;
                cnt[e] = first * unit + before[e];
            }
            tiles += __shfl(upto, 63);
        }
    }
    __syncthreads();
    for (int p = begin + threadIdx.x; p < end; p += kAlignThreads) {
        const int e = idx[p];
        if (e < 0 || e >= E) continue;
        const int row = cnt[e] + pair_row[p];
        if (row < max_rows) row_pair[row] = p;
        pair_row[p] = min(row, max_rows - 1);
    }
}

// tiles of `unit` rows: every pair of idx gets a row, a tile's rows belong to one expert; rows without a pair hold -1, tiles
// without rows expert -1.  `counts`, if given: room for kMaxBlocks x E numbers, which many pairs are grouped with
int launch_moe_align(const int32_t* idx, int64_t P, int E, int unit, int max_tiles, int32_t* row_pair, int32_t* tile_expert,
                     int32_t* pair_row, int32_t* counts, hipStream_t s) {
    int copies = kAlignWaves;
    while ((int64_t)copies * E * sizeof(int) > 64 * 1024) copies >>= 1;      // (E <= 4096: four copies at least)
    if (counts && P >= kManyPairs) {
        const int64_t per = (P + kMaxBlocks - 1) / kMaxBlocks;               // at most kMaxBlocks blocks, of 2 kAlignThreads pairs at least
        const int chunk = (int)std::max<int64_t>(2, (per + kAlignThreads - 1) / kAlignThreads) * kAlignThreads;
        const int blocks = (int)((P + chunk - 1) / chunk);
        hipLaunchKernelGGL(moe_align_count_kernel, dim3((unsigned)blocks), dim3(kAlignThreads), (size_t)copies * E * sizeof(int), s, idx,
                           (int)P, E, copies, chunk, max_tiles * unit, max_tiles, row_pair, tile_expert, pair_row, counts);
        SM_CHECK_LAUNCH("sm_moe_align (counts)");
        hipLaunchKernelGGL(moe_align_place_kernel, dim3((unsigned)blocks), dim3(kAlignThreads), (size_t)2 * E * sizeof(int), s, idx, (int)P,
                           E, chunk, unit, max_tiles, row_pair, tile_expert, pair_row, counts);
        SM_CHECK_LAUNCH("sm_moe_align");
        return SM_OK;
    }
    copies = (int)std::min<int64_t>(copies, (P + 63) / 64);                  // (waves without pairs need none)
    hipLaunchKernelGGL(moe_align_kernel, dim3(1), dim3(kAlignThreads), (size_t)copies * E * sizeof(int), s, idx, (int)P, E, copies, unit,
                       max_tiles, row_pair, tile_expert, pair_row);
    SM_CHECK_LAUNCH("sm_moe_align");
    return SM_OK;
}

}  // namespace sm
