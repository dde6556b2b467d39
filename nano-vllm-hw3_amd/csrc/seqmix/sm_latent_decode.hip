// Latent attention for single-token queries (decode) on the matrix cores.  The H heads of a sequence's one token are
// the query rows (they all see the same keys); the keys are split over workgroups in whole tiles, every
// (sequence, split) leaves an unnormalised partial state {m * c, l, O} in the workspace, and a second launch merges
// the splits in order.  The split count is the caller's and does not depend on the sequences' lengths.
#include "sm_latent_tile.h"

namespace sm {

// floats per (sequence, split, head) in the workspace: scaled maximum, sum, RP outputs
__host__ __device__ constexpr int part_stride(int nb) { return 32 * nb + 2; }

// SLIM: rows of exactly 32 NB columns on 16 bytes, in the loop of 32-key tiles (latent_slim_loop), which goes straight to LDS.  A split is
// a few tiles behind the latency of its first loads, so what counts is how many workgroups run beside each other; the other loop, with a
// tile in registers on its way, spills in one wave of 256 columns.  Below 96 columns it has registers enough, and its tiles of 64 keys half
// the steps (us, 32 heads of 64 columns, other loop / this one: 64 sequences of 1000 keys 13.6 / 14.2, 600 46 / 49).  Microseconds with the merge, other loop / this one, rows of
// 192 + 64: 64 sequences of about 1000 keys 28 / 22 (16 heads), 42 / 35 (64 heads), 8 sequences 21 / 18, 256 of about 450 41 / 31, 16 of
// 3500 with 128 heads 49 / 40.  256 registers, so that two waves share a SIMD, where a workgroup has two or four waves:
// 35 against 42 at 64 heads; one wave alone holds more than that and would spill (30 against 22).
template <int NB, int NBV, int WAVES, bool SLIM>
__global__ __launch_bounds__(64 * WAVES, SLIM && WAVES > 1 ? 2 : 1) void latent_attn_decode_kernel(const unsigned short* __restrict__ q,
                                                                        const unsigned short* __restrict__ cache,
                                                                        const int32_t* __restrict__ block_tables,
                                                                        const int32_t* __restrict__ ctx, float* __restrict__ ws,
                                                                        float c_log2, int H, int R, int block_size,
                                                                        int max_blocks, int splits, int window) {
    // (the slim loop has two buffers of half a tile)
    __shared__ __attribute__((aligned(1024))) unsigned char lds[SLIM ? SlimGeom<NB>::BYTES : TileGeom<NB>::LDS_BYTES];
    __shared__ __attribute__((aligned(1024))) unsigned char lds2[SLIM ? SlimGeom<NB>::BYTES : 16];
    const int sp = blockIdx.x, b = blockIdx.y;
    const int n = ctx[b];
    // the visible keys start at the tile that holds key n - window; whole tiles per split
    const int first = window > 0 ? max(0, n - window) / kTileKeys * kTileKeys : 0;
    const int per = ((n - first + kTileKeys - 1) / kTileKeys + splits - 1) / splits * kTileKeys;
    const int k_lo = first + sp * per, k_hi = min(n, k_lo + per);
    const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = 32 * wave + l31;
    float* part = ws + (((size_t)b * splits + sp) * H + min(r, H - 1)) * part_stride(NBV);
    if (k_lo >= k_hi) {                                      // an empty split: the merge skips l == 0
        if (r < H && hi == 0) { part[0] = -INFINITY; part[1] = 0.f; }
        return;
    }
    const int rc = min(r, H - 1);
    f32x16 oacc[NBV];
    float m_run, l_tot;
    const unsigned short* qrow = q + ((size_t)b * H + rc) * R;
    const int32_t* table = block_tables + (size_t)b * max_blocks;
    if constexpr (SLIM)
        latent_slim_loop<NB, NBV, WAVES>(qrow, cache, table, block_size, k_lo, k_hi, n - 1, n - 1, n - 1, c_log2, window, lds, lds2, oacc,
                                         m_run, l_tot);
    else
        latent_tile_loop<NB, NBV, WAVES>(qrow, cache, table, R, block_size, k_lo, k_hi, n - 1, n - 1, c_log2, window, lds, oacc, m_run,
                                         l_tot);
    if (r >= H) return;
    if (hi == 0) { part[0] = l_tot > 0.f ? m_run * c_log2 : -INFINITY; part[1] = l_tot; }
#pragma unroll
    for (int d = 0; d < NBV; ++d)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq)
#pragma unroll
            for (int e = 0; e < 4; ++e) part[2 + 32 * d + 8 * rq + 4 * hi + e] = oacc[d][4 * rq + e];
}

// A workgroup per (sequence, head), one wave or four: of four each adds up every fourth split, two columns per lane, and the waves'
// sums meet in LDS.  The splits' maxima and sums are read a split per lane in front of the outputs.  (One wave walking the splits one
// after another, a column per lane, three dependent rounds of loads per split: 17 us for 64 sequences of 16 heads and up to
// 11 splits, against 21 of the attention itself.)
// One wave where four have nothing to share out, up to five splits, and where the rows fill the chip several times over, from 6400 (us of
// the whole step with four / one): 256 sequences of about 450 keys, 64 heads of 32 columns, 4 splits 33.5 / 22.6; 512 of 300, 64 heads of
// 192 + 64, 2 splits 82 / 52; 128 of 1000, 64 heads, 8 splits 14 % more with four; 16 heads of 100 sequences, 8 splits 13 % less.
template <int WAVES, int U>
__global__ __launch_bounds__(64 * WAVES) void latent_decode_merge_kernel(const float* __restrict__ ws, unsigned short* __restrict__ o, int H,
                                                                         int R, int splits, int stride, const float* __restrict__ sink) {
    __shared__ float2 part[WAVES][64];
    typedef unsigned short u16x2 __attribute__((ext_vector_type(2), aligned(2)));      // (workspace and output as the caller has them)
    typedef float f32x2 __attribute__((ext_vector_type(2), aligned(4)));
    const size_t row = blockIdx.x;                          // b * H + h
    const size_t b = row / H, h = row % H;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const float* first = ws + (b * splits * H + h) * stride;
    const size_t step = (size_t)H * stride;
    // (an empty split has sum 0 and outputs that nobody wrote: it counts for nothing)
    // A wave's first U splits of the first two column blocks are asked for in front of the maximum, which they do not wait for: with one
    // round of loads behind another the kernel took 6.9 us of 20.6 (64 sequences of 16 heads, 11 splits of 192 columns), so 4.5.  (With six asked for
    // where there is one, 400 sequences of 128 heads of 64 + 64 took 35.1 us, not 32.5.)
    const f32x2 ml = lane < splits ? *(const f32x2*)(first + lane * step) : f32x2{-INFINITY, 0.f};
    f32x2 ahead[2][U];
#pragma unroll
    for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int u = 0; u < U; ++u)
            ahead[k][u] = *(const f32x2*)(first + min(wave + u * WAVES, splits - 1) * step + 2 + min(128 * k + 2 * lane, R - 2));
    __builtin_amdgcn_sched_barrier(0);
    float M = ml.y > 0.f ? ml.x : -INFINITY;
    for (int s = lane + 64; s < splits; s += 64) {
        const f32x2 more = *(const f32x2*)(first + s * step);
        if (more.y > 0.f) M = fmaxf(M, more.x);
    }
    M = wave_max(M);
    const float fl = ml.y > 0.f ? __builtin_amdgcn_exp2f(ml.x - M) : 0.f;
    float L = ml.y > 0.f ? fl * ml.y : 0.f;
    for (int s = lane + 64; s < splits; s += 64) {
        const f32x2 more = *(const f32x2*)(first + s * step);
        if (more.y > 0.f) L += __builtin_amdgcn_exp2f(more.x - M) * more.y;
    }
    L = wave_sum(L);
    const float inv = sink ? sink_inv(M, L, sink[h]) : 1.f / L;
    const unsigned long long counts = __builtin_amdgcn_ballot_w64(ml.y > 0.f);
    auto block = [&](int c0, const f32x2* have) __attribute__((always_inline)) {      // (R % 4 == 0)
        const int c = c0 + 2 * lane;
        float2 acc = make_float2(0.f, 0.f);
        auto add = [&](int s, f32x2 x) __attribute__((always_inline)) {
            if (s < 64) {
                if (counts >> s & 1) {
                    const float f = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, fl), s));
                    acc.x += f * x.x;
                    acc.y += f * x.y;
                }
            } else {
                const f32x2 more = *(const f32x2*)(first + s * step);
                const float f = __builtin_amdgcn_exp2f(more.x - M);
                if (more.y > 0.f) { acc.x += f * x.x; acc.y += f * x.y; }
            }
        };
        int s = wave;
        if (have)
#pragma unroll
            for (int u = 0; u < U; ++u, s += WAVES)
                if (s < splits) add(s, have[u]);
        // (four at a time: a lane's number cannot be read by another while the compiler has loads to move over the condition)
        for (; s < splits; s += 4 * WAVES) {
            f32x2 x[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) x[u] = *(const f32x2*)(first + min(s + u * WAVES, splits - 1) * step + 2 + min(c, R - 2));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < 4; ++u)
                if (s + u * WAVES < splits) add(s + u * WAVES, x[u]);
        }
        if (WAVES > 1) {
            part[wave][lane] = acc;
            __syncthreads();
        }
        if (wave == 0 && c < R) {
#pragma unroll
            for (int v = 1; v < WAVES; ++v) { acc.x += part[v][lane].x; acc.y += part[v][lane].y; }
            const u16x2 o2 = {__builtin_bit_cast(unsigned short, (bf16_t)(acc.x * inv)), __builtin_bit_cast(unsigned short, (bf16_t)(acc.y * inv))};
            *(u16x2*)(o + row * R + c) = o2;
        }
        if (WAVES > 1) __syncthreads();
    };
    block(0, ahead[0]);
    if (R > 128) block(128, ahead[1]);
    for (int c0 = 256; c0 < R; c0 += 128) block(c0, nullptr);
}

// the padded value width the kernel SM_BY_LATENT_SIZE picks for (R, RV)
static int padded_nbv(int R, int RV) {
    const int nb = (R + 31) / 32, nbv = (RV + 31) / 32;
    int got = 0;
#define SM_PICK(NB_, NBV_) got = NBV_
    SM_BY_LATENT_SIZE(nb, nbv, SM_PICK);
#undef SM_PICK
    return got;
}

}  // namespace sm

using namespace sm;

extern "C" size_t sm_latent_decode_workspace_bytes(int64_t B, int H, int R, int splits) {
    if (B <= 0 || H <= 0 || R <= 0 || splits <= 0) return 0;
    return (size_t)B * splits * H * part_stride(padded_nbv(R, R)) * sizeof(float);       // (a narrower value part needs less)
}

extern "C" int sm_latent_attn_decode(const void* q, const void* cache, const int32_t* block_tables, const int32_t* ctx, void* o,
                                     float scale, int64_t B, int H, int R, int block_size, int max_blocks, int splits,
                                     void* workspace, size_t workspace_bytes, int RV, int window, const float* sink,
                                     void* stream) {
    if (RV <= 0) RV = R;
    if (B < 0 || H < 1 || R < 1 || RV > R || window < 0 || block_size < 1 || max_blocks < 1 || splits < 1 ||
        (B > 0 && (!q || !cache || !block_tables || !ctx || !o || !workspace))) {
        set_error("sm_latent_attn_decode: bad argument");
        return SM_EINVAL;
    }
    if (R % 8 || RV % 4 || R > 256 || block_size % 64 || H > 128 || B > 65535 || splits > 65535) {
        set_error("sm_latent_attn_decode: needs R %% 8 == 0, R <= 256, block_size %% 64 == 0, H <= 128");
        return SM_ESHAPE;
    }
    if (workspace_bytes < sm_latent_decode_workspace_bytes(B, H, R, splits)) {
        set_error("sm_latent_attn_decode: workspace too small");
        return SM_EWORKSPACE;
    }
    if (B == 0) return SM_OK;
    const int nb = (R + 31) / 32, nbv = (RV + 31) / 32, waves = H <= 32 ? 1 : (H <= 64 ? 2 : 4);
    dim3 grid((unsigned)splits, (unsigned)B);
    const float c = scale * 1.4426950408889634f;
    hipStream_t s = as_stream(stream);
#define SM_DEC(NB_, NBV_, W_) do { if (R == 32 * NB_ && (uintptr_t)cache % 16 == 0) SM_DEC_(NB_, NBV_, W_, (NB_ >= 3)); else SM_DEC_(NB_, NBV_, W_, false); } while (0)
#define SM_DEC_(NB_, NBV_, W_, SLIM_)                                                                                      \
    hipLaunchKernelGGL((latent_attn_decode_kernel<NB_, NBV_, W_, SLIM_>), grid, dim3(64 * W_), 0, s, (const unsigned short*)q, \
                       (const unsigned short*)cache, block_tables, ctx, (float*)workspace, c, H, R, block_size, max_blocks, \
                       splits, window)
#define SM_DEC_W(NB_, NBV_) do { if (waves == 1) SM_DEC(NB_, NBV_, 1); else if (waves == 2) SM_DEC(NB_, NBV_, 2); else SM_DEC(NB_, NBV_, 4); } while (0)
    SM_BY_LATENT_SIZE(nb, nbv, SM_DEC_W);
#undef SM_DEC_W
#undef SM_DEC_
#undef SM_DEC
    SM_CHECK_LAUNCH("sm_latent_attn_decode");
#define SM_MERGE(WAVES_, U_)                                                                                                   \
    hipLaunchKernelGGL((latent_decode_merge_kernel<WAVES_, U_>), dim3((unsigned)(B * H)), dim3(64 * WAVES_), 0, s, (const float*)workspace, \
                       (unsigned short*)o, H, RV, splits, part_stride(padded_nbv(R, RV)), sink)
    if (splits <= 5 || B * H >= 6400) {
        if (splits <= 2) SM_MERGE(1, 2); else SM_MERGE(1, 6);
    } else {
        SM_MERGE(4, 4);
    }
#undef SM_MERGE
    SM_CHECK_LAUNCH("sm_latent_attn_decode (merge)");
    return SM_OK;
}
