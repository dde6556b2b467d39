// Decode attention of few query heads per key/value head: the keys and values go through the vector unit as they arrive, nothing is
// staged.  With one, two or four query heads per group the matrix cores' tile of 32 rows is almost all padding, and its way through
// LDS takes the registers that loads in flight need: what bounds the step is the stream of the cache.
//
// A workgroup of four waves owns one (sequence, split, key/value head); a wave takes half a tile of the walk (32 keys) at a time.
// Eight lanes share a key, 16 bytes of every 128 each, so a key's lanes read whole 128-byte runs; four keys per lane are in flight
// (two with four heads, whose state takes the registers).  Scores are bf16 dot-product instructions (exact products, float32 sums), weights
// and outputs float32.  The 32 states of the workgroup's key slots (8 per wave) are merged pairwise by a lane exchange, then in LDS, in
// a fixed order; the split's state {maximum in log2 units, sum, outputs} is left in the workspace as attn_decode_kernel does.
//
// Microseconds with the merge, attn_decode_kernel / this one (caches not in L2; floor = the cache at 6.1 TB/s): 64 sequences of 700 to
// 1300 keys, heads 16 / 8 of 128: 71 / 52 (floor 43), 16 / 4 of 128: 48 / 38 (22), 16 / 8 of 64: 43 / 32 (22), window 256 with capped
// scores 34 / 22 (11); 64 of 1700 to 1800: 102 / 80 (75); 16 of 700 to 1300, 16 / 8 of 128: 36 / 22 (11); 4 of them 25 / 13; one of 100
// keys 15 / 7.4.  512 to 3072 workgroups measured within 5 % of each other, so the splits stay those of the other form.  Only waves with keys leave states:
// with all four's merged whatever their keys, 256 sequences of 32 keys, 16 / 4 heads of 128, took 17.7 us, not 16.4, where the other form takes 15.5
// (more than 768 workgroups of up to 64 keys and four heads of 128: the only ones that it is faster for, by up to 0.9 us).
#pragma once
#include "hm_attn_tile.h"

#include <type_traits>

namespace hm {

template <int D, int REP, int MODE>
__global__ __launch_bounds__(256) void attn_decode_stream_kernel(const unsigned short* __restrict__ q, const unsigned short* __restrict__ kc,
                                                                 const unsigned short* __restrict__ vc,
                                                                 const int32_t* __restrict__ block_tables, const int32_t* __restrict__ ctx,
                                                                 int window, int keep_first, float c_log2, float pre,
                                                                 float* __restrict__ ws, int H, int G, int block_size, int max_blocks,
                                                                 int splits, int chunk) {
    typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
    constexpr int NL = D / 64, U = REP == 4 ? 2 : 4, STRIDE = D + 2;       // 16-byte pieces of a key per lane; keys in flight per lane
    __shared__ float st_m[16][REP], st_l[16][REP];
    __shared__ __attribute__((aligned(16))) float st_acc[16][REP][D];
    const int sp = blockIdx.x, b = blockIdx.y, g = blockIdx.z;
    const int n = ctx[b];
    const auto walk = make_walk(n - 1, n - 1, window, keep_first, 0, chunk);
    // whole pairs of tiles per split: the four waves take half a tile each
    const int nt = walk.count(n), per = ((nt + splits - 1) / splits + 1) & ~1;
    const int vt_lo = sp * per, vt_hi = min(nt, vt_lo + per);
    float* part = ws + (((size_t)b * splits + sp) * H + g * REP) * STRIDE;
    if (vt_lo >= vt_hi) {                                    // an empty split: the merge skips sums of 0
        if (threadIdx.x < REP) { part[threadIdx.x * STRIDE] = -INFINITY; part[threadIdx.x * STRIDE + 1] = 0.f; }
        return;
    }
    const int lane = threadIdx.x & 63, slot = lane >> 3, seg = lane & 7;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    int qp[REP][4 * NL];                                     // pairs of q as they lie in memory
    float acc[REP][8 * NL], m[REP], l[REP];
#pragma unroll
    for (int h = 0; h < REP; ++h) {
#pragma unroll
        for (int p = 0; p < NL; ++p) {
            const i32x4 a = *(const i32x4*)(q + ((size_t)b * H + g * REP + h) * D + 64 * p + 8 * seg);
#pragma unroll
            for (int j = 0; j < 4; ++j) qp[h][4 * p + j] = a[j];
        }
#pragma unroll
        for (int j = 0; j < 8 * NL; ++j) acc[h][j] = 0.f;
        m[h] = -INFINITY;
        l[h] = 0.f;
    }
    const int32_t* table = block_tables + (size_t)b * max_blocks;
    const int chunk_lo = chunk > 0 ? (n - 1) / chunk * chunk : 0;
    const size_t head = (size_t)g * D + 8 * seg, pitch = (size_t)G * D;
    // half h of the walk: its first key, and the cache row of key 0 of its page (a tile lies in one cache block)
    auto first_key = [&](int half) { return walk.key0(half >> 1) + 32 * (half & 1); };
    auto page_row = [&](int key) {
        const int page = key / block_size;
        return ((int64_t)table[page] - page) * block_size;
    };
    // (32 U keys' worth of halves: with two keys per lane a half takes two steps)
    constexpr int STEPS = 4 / U;
    int half = 2 * vt_lo + wave;
    const int end = 2 * vt_hi - (first_key(2 * vt_hi - 1) >= n ? 1 : 0);    // (the last tile's second half may lie past the last key)
    const int used = min(4, end - 2 * vt_lo);                // waves that have keys: short sequences have no states of the others to merge
    int key0 = half < end ? first_key(half) : 0;
    int64_t row0 = half < end ? page_row(key0) : 0;
    for (; half < end; half += 4) {
        const int next = min(half + 4, end - 1), nkey0 = first_key(next);
        const int64_t nrow0 = page_row(nkey0);               // (asked for a step ahead)
#pragma unroll
        for (int st = 0; st < STEPS; ++st) {
            i32x4 kk[U][NL], vv[U][NL];
            size_t at[U];
            const int k0 = key0 + 8 * U * st + slot;
#pragma unroll
            for (int u = 0; u < U; ++u) {
                // (keys past the last one: that one's row, masked below; all read once, past the caches)
                at[u] = (size_t)(row0 + min(k0 + 8 * u, n - 1)) * pitch + head;
#pragma unroll
                for (int p = 0; p < NL; ++p) kk[u][p] = __builtin_nontemporal_load((const i32x4*)(kc + at[u] + 64 * p));
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int p = 0; p < NL; ++p) vv[u][p] = __builtin_nontemporal_load((const i32x4*)(vc + at[u] + 64 * p));
            // (All asked for first, keys in front of values, and a key's products behind its own loads: left alone the compiler moves half of the
            // loads to their use and takes the keys' products in turn, which waits for all of them.  64 sequences of 700 to 1300 keys, 16 / 8 heads
            // of 128: 54.1 us, so 52.9; 275 shapes 0.99.)
            __builtin_amdgcn_sched_barrier(0);
            float sc[U][REP];
#pragma unroll
            for (int u = 0; u < U; ++u) {
#pragma unroll
                for (int h = 0; h < REP; ++h) {
                    sc[u][h] = 0.f;
#pragma unroll
                    for (int j = 0; j < 4 * NL; ++j) {
                        const int kd = kk[u][j >> 2][j & 3];   // (a value: a bit cast of the element itself reads the vector's first one)
                        sc[u][h] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, qp[h][j]), __builtin_bit_cast(bf16x2, kd), sc[u][h], false);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            bool seen[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int key = k0 + 8 * u;
                seen[u] = key < n && key >= chunk_lo && (window <= 0 || n - 1 - key < window || key < keep_first);
            }
#pragma unroll
            for (int h = 0; h < REP; ++h) {
                float sv[U], mn = m[h];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    float s = group_sum<8>(sc[u][h]);
                    // tanh(z) = 1 - 2 / (1 + e^2z); both infinities come out right
                    if (MODE == kSoftcap) s = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s * pre));
                    sv[u] = seen[u] ? s * c_log2 : -INFINITY;
                    mn = fmaxf(mn, sv[u]);
                }
                const bool none = mn == -INFINITY;           // the slot has seen nothing yet
                const float mc = none ? 0.f : mn, alpha = none ? 1.f : __builtin_amdgcn_exp2f(m[h] - mn);
                float psum = 0.f;
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    sc[u][h] = __builtin_amdgcn_exp2f(sv[u] - mc);
                    psum += sc[u][h];
                }
                l[h] = l[h] * alpha + psum;
                m[h] = mn;
#pragma unroll
                for (int j = 0; j < 8 * NL; ++j) acc[h][j] *= alpha;
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int j = 0; j < 4 * NL; ++j) {           // a pair of values is widened once for all heads
                    const unsigned vd = (unsigned)vv[u][j >> 2][j & 3];
                    const float lo = __builtin_bit_cast(float, vd << 16), hi = __builtin_bit_cast(float, vd & 0xFFFF0000u);
#pragma unroll
                    for (int h = 0; h < REP; ++h) {
                        acc[h][2 * j] = __builtin_fmaf(sc[u][h], lo, acc[h][2 * j]);
                        acc[h][2 * j + 1] = __builtin_fmaf(sc[u][h], hi, acc[h][2 * j + 1]);
                    }
                }
        }
        key0 = nkey0;
        row0 = nrow0;
    }
    // two slots share 16 lanes: lane ^ 8 holds the other's state of the same channels
    auto other = [](float v) {
        return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x128, 0xF, 0xF, false));
    };
    const int state = 4 * wave + (lane >> 4);
    if (wave < used)
#pragma unroll
        for (int h = 0; h < REP; ++h) {
            const float mo = other(m[h]), lo = other(l[h]), mn = fmaxf(m[h], mo), mc = mn == -INFINITY ? 0.f : mn;
            const float wa = __builtin_amdgcn_exp2f(m[h] - mc), wb = __builtin_amdgcn_exp2f(mo - mc);
            if (lane % 16 == 0) { st_m[state][h] = mn; st_l[state][h] = l[h] * wa + lo * wb; }
#pragma unroll
            for (int j = 0; j < 8 * NL; ++j) {
                const float o = other(acc[h][j]);
                acc[h][j] = acc[h][j] * wa + o * wb;
            }
            if ((lane & 8) == 0) {
#pragma unroll
                for (int p = 0; p < NL; ++p)
#pragma unroll
                    for (int e = 0; e < 8; e += 4)
                        *(float4*)&st_acc[state][h][64 * p + 8 * seg + e] =
                            make_float4(acc[h][8 * p + e], acc[h][8 * p + e + 1], acc[h][8 * p + e + 2], acc[h][8 * p + e + 3]);
            }
        }
    __syncthreads();
    auto merge = [&](auto states) __attribute__((always_inline)) {
        constexpr int S = decltype(states)::value;
        for (int o = threadIdx.x; o < REP * D; o += 256) {
            const int h = o / D, d = o % D;
            float M = st_m[0][h];
#pragma unroll
            for (int s = 1; s < S; ++s) M = fmaxf(M, st_m[s][h]);
            const float mc = M == -INFINITY ? 0.f : M;
            float num = 0.f, den = 0.f;
#pragma unroll
            for (int s = 0; s < S; ++s) {
                const float w = __builtin_amdgcn_exp2f(st_m[s][h] - mc);
                num += w * st_acc[s][h][d];
                den += w * st_l[s][h];
            }
            float* p = part + h * STRIDE;
            p[2 + d] = num;
            if (d == 0) { p[0] = den > 0.f ? M : -INFINITY; p[1] = den; }
        }
    };
    using std::integral_constant;
    if (used == 4) merge(integral_constant<int, 16>{});
    else if (used == 3) merge(integral_constant<int, 12>{});
    else if (used == 2) merge(integral_constant<int, 8>{});
    else merge(integral_constant<int, 4>{});
}

}  // namespace hm
