// Expert products for many tokens on the matrix cores (bf16): the (token, expert) pairs are grouped by expert into
// tiles of 32 rows (sm_moe_align.hip), so that one wave multiplies 32 rows of one expert by 32 of its output
// columns; gate and up are produced together and leave as the clamped GLU, the down product leaves per pair and a
// last launch sums a token's pairs with their weights (and the shared expert) in a fixed order.
//
// A row of the result depends only on its own inputs: which other pairs share its tile does not change it, so the
// (arbitrary) order of pairs inside an expert's group leaves every value as it is.
//
// Both matrices are K-contiguous and a lane multiplies 32 consecutive k of one row in a 64-k step (four MFMA steps; the k order
// inside a step is free as long as both operands agree).  Weights go from global memory straight to the MFMA registers, in the
// order that their layout gives them; activations go through registers and LDS.
#include <algorithm>

#include "sm_common.h"
#include "sm_moe_deal.h"

namespace sm {

constexpr int kRowsPerTile = 32;

__device__ __forceinline__ float glu_bf16(float g, float u, float limit, float alpha, int act) {
    // the products leave the matrix unit in bf16, as a GEMM's output would
    return gated_act((float)(bf16_t)g, (float)(bf16_t)u, limit, alpha, act);
}

__device__ __forceinline__ bf16x8 load8(const unsigned short* p, int k, int K) {
    i32x4 v = {0, 0, 0, 0};
    if (k + 8 <= K) v = *(const i32x4*)(p + k);
    return __builtin_bit_cast(bf16x8, v);
}

// GATE_UP: A = h rows gathered by token, B = the expert's gate and up rows, out = act [rows, N] (N = F, K = W)
// else:    A = act rows,                 B = the expert's down rows,       out = per-row products [rows, N] (N = W, K = F)
// MODE 0: the down product; 1: gate and up with a gated activation (act_kind); 2: the up product alone with a plain one.
// in_wts != NULL (modes 1, 2): pair p's products are scaled by in_wts[p] before the activation (a weight on the expert's input)
//
// A wave is a workgroup: sixteen tiles by 48 column blocks are three waves for every CU, where workgroups of four waves left a
// quarter of the CUs without work.  Bound by the weights, read once, and by what a short kernel takes to begin and end (64 tokens,
// top 4 of 16 experts of 2048 x 1536: gate and up 44 us, 4.6 TB/s; down 23, 4.4).  Lanes that read their own rows of the activations from
// global memory touched 64 cache lines with every load, and rows without a pair as many as the others: 46 and 37 us.
// FEW: rows of a handful of tokens, of which a load touches only as many cache lines whichever lane asks for what; LDS would only stand between
// the load and the product, and a step's few waves cover nothing of it.  (The down product's rows are the pairs' own, and take the way through
// LDS.)  Whole calls, us, rows through LDS / to the lanes that multiply them: 1 token, top 1 of 4 plain experts of 4096 x 768 25.3 / 21.3, of 2048 x
// 1536 21.9 / 20.0; 8 tokens, top 2 of 16 experts of 2048 x 1536 62 / 62, 12 tokens 63 / 67, but with few waves on the chip, 12 tokens of 4 experts of 2048 x 256, 20.5 / 18.6.
template <int MODE, bool FEW>
__global__ __launch_bounds__(64) void moe_grouped_kernel(const unsigned short* __restrict__ a, const unsigned short* __restrict__ w,
                                                          const int32_t* __restrict__ row_pair, const int32_t* __restrict__ tile_expert,
                                                          unsigned short* __restrict__ out, int tiles, int top, unsigned top_inv, int N, int K, float limit,
                                                          float alpha, int act_kind, const float* __restrict__ in_wts) {
    constexpr bool GATE_UP = MODE == 1, FROM_TOKENS = MODE != 0;
    const MoePlace place = moe_place(blockIdx.x, blockIdx.y, blockIdx.z);
    const int tile = place.tile, n0 = place.block * 32;
    if (n0 >= N || tile >= tiles) return;
    const int lane = threadIdx.x, l31 = lane & 31, hi = lane >> 5;
    // The tile's rows come 128 bytes at a time, eight lanes to a row, and go through LDS to the lanes that multiply them (chunk c
    // of row r at place c ^ (r / 2 & 7)): a lane reading its own row would touch a cache line of its own with every load.  Rows
    // without a pair repeat one that has a place in memory; nobody reads their sums.
    __shared__ __attribute__((aligned(1024))) unsigned char rows[2][FEW ? 16 : kRowsPerTile * 128];
    __shared__ __attribute__((aligned(16))) int pairs[kRowsPerTile];
    const int sub = lane >> 3, chunk = lane & 7;
    const unsigned short* arow[4];
    // (the rows' pairs all at once, beside the expert and with no branch between them: one behind the other is four trips to memory)
    int pair[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) pair[j] = row_pair[tile * kRowsPerTile + (FEW ? l31 : 8 * j + sub)];
    const int e = tile_expert[tile];
    if (e < 0) return;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        pairs[FEW ? l31 : 8 * j + sub] = pair[j];             // (several lanes, one number)
        const unsigned p = (unsigned)max(pair[j], 0);
        if (FROM_TOKENS) {                                    // pair / top: the product with 1 / top is at most one too large
            const unsigned q = top > 1 ? __umulhi(p, top_inv) : p;
            arow[j] = a + (size_t)(q - (q * (unsigned)top > p ? 1u : 0u)) * K + (FEW ? 32 * hi + 8 * j : 8 * chunk);
        } else {
            arow[j] = a + (size_t)(tile * kRowsPerTile + (pair[j] < 0 ? 0 : 8 * j + sub)) * K + 8 * chunk;
        }
    }
    // weights in the tiled layout of sm_moe_tile_weights: block (expert, 32-row block, 64-k step) = 4 KB, chunk s of
    // lane L at 16 (64 s + L): a wave's load is one contiguous KB
    const int nb32 = (N + 31) / 32, ksteps = (K + 63) / 64;
    const unsigned short* bp = w + (((size_t)e * (GATE_UP ? 2 : 1) * nb32 + n0 / 32) * ksteps) * 2048 + 8 * lane;
    const unsigned short* bp2 = bp + (size_t)nb32 * ksteps * 2048;      // the up blocks follow the gate blocks
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    f32x16 acc = {0}, acc2 = {0};
    // A ring of 64-k steps in flight: with a handful of rows per expert (decode) a wave's few MFMAs per step hide nothing, so
    // the weight stream has to be kept busy by outstanding loads: three steps of gate and up (36 KB per wave), six of a single
    // product (24 KB of weights).  No condition stands around a load of the ring (one would make every load wait for the one
    // before it): past the last whole step it loads that step again, and a shorter last step comes by itself.
    constexpr int RING = GATE_UP ? 3 : 6;
    struct Stage { bf16x8 a[4], b[4], b2[4]; };
    auto request = [&](Stage& st, int step) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            st.a[s] = *(const bf16x8*)(arow[s] + (size_t)step * 64);
            st.b[s] = *(const bf16x8*)(bp + (size_t)step * 2048 + 512 * s);
            if (GATE_UP) st.b2[s] = *(const bf16x8*)(bp2 + (size_t)step * 2048 + 512 * s);
        }
    };
    const int put = sub * 128 + 16 * (chunk ^ (sub >> 1)), get = l31 * 128, swz = (l31 >> 1) & 7;
    auto consume = [&](const Stage& st, unsigned char* lds) {
        bf16x8 av[4];
        if constexpr (FEW) {
#pragma unroll
            for (int s = 0; s < 4; ++s) av[s] = st.a[s];
        } else {
            // (one wave, whose LDS accesses are carried out in their order: nothing to wait for but the order itself)
#pragma unroll
            for (int j = 0; j < 4; ++j) *(bf16x8*)(lds + 1024 * j + (put ^ (64 * (j & 1)))) = st.a[j];
            asm volatile("" ::: "memory");
            __builtin_amdgcn_wave_barrier();
#pragma unroll
            for (int s = 0; s < 4; ++s) av[s] = *(const bf16x8*)(lds + get + 16 * ((4 * hi + s) ^ swz));
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[s], st.b[s], acc, 0, 0, 0);
            if (GATE_UP) acc2 = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[s], st.b2[s], acc2, 0, 0, 0);
        }
        if constexpr (!FEW) asm volatile("" ::: "memory");
    };
    const int full = K / 64;
    if (full > 0) {
        Stage st[RING];
#pragma unroll
        for (int i = 0; i < RING; ++i) request(st[i], min(i, full - 1));
        int step = 0;
        for (; step + RING <= full; step += RING)
#pragma unroll
            for (int i = 0; i < RING; ++i) {
                consume(st[i], rows[i & 1]);
                request(st[i], min(step + RING + i, full - 1));
            }
#pragma unroll
        for (int i = 0; i < RING; ++i)
            if (step + i < full) consume(st[i], rows[i & 1]);
    }
    if (K % 64 != 0) {                                        // zeros past the end of a row (the weights end in zeros)
        Stage st;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            st.a[s] = FEW ? load8(arow[s] - 32 * hi - 8 * s, full * 64 + 32 * hi + 8 * s, K) : load8(arow[s] - 8 * chunk, full * 64 + 8 * chunk, K);
            st.b[s] = *(const bf16x8*)(bp + (size_t)full * 2048 + 512 * s);
            if (GATE_UP) st.b2[s] = *(const bf16x8*)(bp2 + (size_t)full * 2048 + 512 * s);
        }
        consume(st, rows[0]);
    }
    if (n0 + l31 >= N) return;
    int p[16];
    float iw[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        p[r] = pairs[(r & 3) + 8 * (r >> 2) + 4 * hi];
        iw[r] = FROM_TOKENS && in_wts && p[r] >= 0 ? in_wts[p[r]] : 1.f;
    }
    with_act<MODE>(act_kind, [&](auto kind) {
        constexpr int ACT = decltype(kind)::value;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            if (p[r] < 0) continue;
            const int orow = tile * kRowsPerTile + (r & 3) + 8 * (r >> 2) + 4 * hi;
            const float v = GATE_UP ? glu_bf16(acc[r] * iw[r], acc2[r] * iw[r], limit, alpha, ACT)
                                    : (MODE == 2 ? plain_act((float)(bf16_t)(acc[r] * iw[r]), ACT) : acc[r]);
            out[(size_t)orow * N + n0 + l31] = __builtin_bit_cast(unsigned short, (bf16_t)v);
        }
    });
}

// A token's pairs summed with their weights, in a fixed order, V channels per thread: 8 where rows and pointers allow 16-byte
// accesses (64 tokens of 2048 channels: 4 us, 8192 tokens: 29 us, 5.8 TB/s; two bytes per access and a workgroup per token took 12
// and 80).
template <int V>
__global__ __launch_bounds__(256) void moe_combine_kernel(const unsigned short* __restrict__ prod, const int32_t* __restrict__ pair_row,
                                                          const float* __restrict__ wts, const unsigned short* __restrict__ shared,
                                                          unsigned short* __restrict__ y, int64_t items, int top, int W,
                                                          const float* __restrict__ shared_scale) {
    struct alignas(2 * V) Pack { bf16_t v[V]; };
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= items) return;
    const int per = W / V;
    const int64_t t = i / per;
    const int c = (int)(i - t * per) * V;
    float tot[V];
#pragma unroll
    for (int v = 0; v < V; ++v) tot[v] = 0.f;
#pragma unroll 4
    for (int k = 0; k < top; ++k) {
        const size_t r = pair_row[t * top + k];
        const float w = wts ? wts[t * top + k] : 1.f;
        const Pack x = *(const Pack*)(prod + r * W + c);
#pragma unroll
        for (int v = 0; v < V; ++v) tot[v] += w * (float)x.v[v];
    }
    if (shared) {
        const float w = shared_scale ? shared_scale[t] : 1.f;
        const Pack x = *(const Pack*)(shared + t * W + c);
#pragma unroll
        for (int v = 0; v < V; ++v) tot[v] += w * (float)x.v[v];
    }
    Pack o;
#pragma unroll
    for (int v = 0; v < V; ++v) o.v[v] = (bf16_t)tot[v];
    *(Pack*)(y + t * W + c) = o;
}

}  // namespace sm

using namespace sm;

extern "C" int sm_moe_grouped_tiles(int64_t T, int top, int E) {
    if (T <= 0 || top <= 0 || E <= 0) return 0;
    return (int)((T * top + kRowsPerTile - 1) / kRowsPerTile + E);
}

extern "C" int sm_moe_grouped(const void* h, const int32_t* idx, const float* wts, const void* w_gu, const void* w_down,
                              const void* shared, const float* shared_scale, int weight_in, float limit, float alpha, int act_kind, void* y, int64_t T, int top, int E, int W, int F,
                              int32_t* row_pair, int32_t* tile_expert, int32_t* pair_row, void* act, void* prod, void* stream) {
    if (T < 0 || top < 1 || E < 1 || W < 1 || F < 1 || act_kind < 0 || act_kind > SM_ACT_LAST ||
        (T > 0 && (!h || !idx || !wts || !w_gu || !w_down || !row_pair || !tile_expert || !pair_row || !act || !prod))) {
        set_error("sm_moe_grouped: bad argument");
        return SM_EINVAL;
    }
    if (W % 8 || F % 8 || E > 4096 || T * top > (int64_t)1 << 30) {
        set_error("sm_moe_grouped: needs W %% 8 == 0, F %% 8 == 0, at most 4096 experts");
        return SM_ESHAPE;
    }
    if (T == 0) return SM_OK;
    const int tiles = sm_moe_grouped_tiles(T, top, E);
    const unsigned top_inv = top > 1 ? (unsigned)((((uint64_t)1 << 32) + top - 1) / top) : 0;
    hipStream_t s = as_stream(stream);
    if (int rc = launch_moe_align(idx, T * top, E, kRowsPerTile, tiles, row_pair, tile_expert, pair_row, nullptr, s)) return rc;
    const bool few = T <= 8 || (T <= 32 && std::min<int64_t>(T * top, E) * ((F + 31) / 32) <= 256);
    auto grid = [&](int n) {
        const MoeGrid g = moe_grid(tiles, n);
        return dim3(g.x, g.y, g.z);
    };
#define SM_GROUPED(MODE_, FEW_)                                                                                                          \
    hipLaunchKernelGGL((moe_grouped_kernel<MODE_, FEW_>), grid(F), dim3(64), 0, s,                                                     \
                       (const unsigned short*)h, (const unsigned short*)w_gu, row_pair, tile_expert, (unsigned short*)act, tiles, top, top_inv, \
                       F, W, limit, alpha, act_kind, weight_in ? wts : nullptr)
    if (act_is_gated(act_kind)) {
        if (few) SM_GROUPED(1, true); else SM_GROUPED(1, false);
    } else {
        if (few) SM_GROUPED(2, true); else SM_GROUPED(2, false);
    }
#undef SM_GROUPED
    SM_CHECK_LAUNCH("sm_moe_grouped (gate/up)");
    hipLaunchKernelGGL((moe_grouped_kernel<0, false>), grid(W), dim3(64), 0, s,
                       (const unsigned short*)act, (const unsigned short*)w_down, row_pair, tile_expert, (unsigned short*)prod, tiles, top, top_inv, W,
                       F, 0.f, 0.f, 0, (const float*)nullptr);
    SM_CHECK_LAUNCH("sm_moe_grouped (down)");
    if (y == nullptr) return SM_OK;               // the caller sums a token's pairs itself
    return sm_moe_combine(prod, pair_row, weight_in ? nullptr : wts, shared, shared_scale, y, T, top, W, stream);
}

// The grouping and the final sum on their own, for callers that run the expert products themselves (the engine gives
// large groups to the vendor GEMM, one call per expert on the rows sm_moe_align put together).
extern "C" int sm_moe_align(const int32_t* idx, int64_t T, int top, int E, int32_t* row_pair, int32_t* tile_expert,
                            int32_t* pair_row, void* stream) {
    if (T < 0 || top < 1 || E < 1 || E > 4096 || (T > 0 && (!idx || !row_pair || !tile_expert || !pair_row))) {
        set_error("sm_moe_align: bad argument");
        return SM_EINVAL;
    }
    if (T == 0) return SM_OK;
    return launch_moe_align(idx, T * top, E, kRowsPerTile, sm_moe_grouped_tiles(T, top, E), row_pair, tile_expert, pair_row,
                            nullptr, as_stream(stream));
}

extern "C" int sm_moe_combine(const void* prod, const int32_t* pair_row, const float* wts, const void* shared,
                              const float* shared_scale, void* y, int64_t T, int top, int W, void* stream) {
    if (T < 0 || top < 1 || W < 1 || (shared_scale && !shared) || (T > 0 && (!prod || !pair_row || !y))) {
        set_error("sm_moe_combine: bad argument");
        return SM_EINVAL;
    }
    if (T == 0) return SM_OK;
    const bool wide = W % 8 == 0 && ((uintptr_t)prod | (uintptr_t)shared | (uintptr_t)y) % 16 == 0;
    const int per = wide ? W / 8 : W;
    const int64_t most = (((int64_t)1 << 32) - 256) / per;     // tokens of one launch: a grid holds fewer than 2^32 threads
    for (int64_t t = 0; t < T; t += most) {
        const int64_t items = std::min(most, T - t) * per;
        const dim3 grid((unsigned)((items + 255) / 256));
        const unsigned short* sh = shared ? (const unsigned short*)shared + t * W : nullptr;
#define SM_COMBINE(V_)                                                                                                         \
    hipLaunchKernelGGL(moe_combine_kernel<V_>, grid, dim3(256), 0, as_stream(stream), (const unsigned short*)prod, pair_row + t * top,    \
                       wts ? wts + t * top : nullptr, sh, (unsigned short*)y + t * W, items, top, W,                              \
                       shared_scale ? shared_scale + t : nullptr)
        if (wide) SM_COMBINE(8); else SM_COMBINE(1);
#undef SM_COMBINE
        SM_CHECK_LAUNCH("sm_moe_combine");
    }
    return SM_OK;
}
