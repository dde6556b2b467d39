// The outer-product recurrences of hm_outer.hip over prompts, 32 tokens at a time on the matrix cores.
//
// With G_t the product of a chunk's decays up to token t, D_ti that of the decays after i up to t, S the state in front of the
// chunk (f32 [D keys, V]) and r the lengths' reciprocals, the chunk's strengths W [32, V] solve a triangular system,
//   (I + A) W = R,  A_ti = beta_t rk_t rk_i (k_t . k_i) D_ti (i < t),  R_t = beta_t (v_t - G_t rk_t S^T k_t)
// (state-space form: W = beta v), and then
//   o_t = rq_t (G_t S^T q_t + sum_{i <= t} D_ti rk_i (q_t . k_i) w_i) + skip v_t,   S <- G_31 S + sum_i D_31,i rk_i k_i w_i^T.
// Everything that does not depend on the state is worked out for all chunks at once (prepare): P_ti = rq_t rk_i (q_t . k_i) D_ti,
// T = (I + A)^-1 by forward substitution, and four numbers per token.  The walk over a sequence's chunks is left with five
// products per chunk: K S, Q S, T R, P W and K^T W.
//
// Precision: the stored q, k are bf16 and enter the products exactly; every float32 operand (S, T, R, P, W) enters as the sum of
// three bf16 numbers, which is the number itself, and of the nine products of two such sums the six above 2^-24 of the result
// are kept, the leading one in a sum of its own; sums are float32, products of decays double.  Against float64 the results are as near
// as the token-by-token walk's: 8 prompts of 900 to 1100 tokens, 16 heads: gated delta 128 x 128 o 2.7e-7 of its norm (walk 2.95e-7),
// state 4.4e-7 (4.8e-7); state space 128 x 64 o 1.68e-7 (1.68e-7), state 3.19e-7 (3.25e-7).  A token that is not finite spoils
// its own and later tokens, as in the walk, and none in front of it.
//
// The walk is one workgroup of two waves per (sequence, head, 32 value channels), half of the keys each, the state in the
// accumulators of the products: lane l holds column l & 31 and the keys 32 blk + 16 (r >> 3) + 8 (l >> 5) + (r & 7) of its wave's,
// register r.  That is the order in which a lane's eight numbers of a B operand come (8 keys in a row: a row of K or Q is read from
// LDS in 16-byte pieces as the A operand), so the state never moves; strengths and results keep tokens (r & 3) + 8 (r >> 2) +
// 4 (l >> 5) per lane, and the prepared A operands are stored in that order.  The waves add up their parts of K S in LDS, work out the
// same strengths, and give each other half of the results' rows at the next meeting, so that both have the same work.
//
// Against the walk that takes token after token, bound by the float32 vector unit and its chain of lane sums at two waves per
// SIMD: 8 prompts of 900 to 1100 tokens, 16 heads of 128 x 128: 418 us there, here 29 (prepare) + 117 (walk), 3.1 us per chunk at one wave
// per SIMD: 800 vector instructions, five cycles each (a third of them the splits), 0.8 us of matrix work, the rest their chain K S -> R -> W -> S
// and its waits.  The walk took 143 with numbers split one at a time (each rounded once more to be packed), the waves' halves of the results chosen
// element by element (through indexed moves) and the products' results in the accumulation registers (a copy for every number read).
// Four waves of 32 keys: 195 us (the strengths worked out four times); results all in one wave, v read from global memory: 175 us.
#include "hm_attn_tile.h"
#include "hm_outer.h"

#include <type_traits>

namespace hm {

constexpr int kChunk = 32;
typedef float f32x4 __attribute__((ext_vector_type(4)));
// bytes of a prepared (chunk, head): P as three terms of an A operand, the tokens' coefficients, T as P
constexpr int kTermBytes = 2 * 64 * 16, kOperand = 3 * kTermBytes, kCoefAt = kOperand, kEndAt = kCoefAt + kChunk * 16, kTAt = kOperand + 1024,
              kPrepared = kTAt + kOperand;

// chunks are numbered q0 / 32 + b + chunk: numbers of different sequences never meet
__device__ __forceinline__ size_t prepared_at(int q0, int b, int chunk, int h, int H) {
    return ((size_t)(q0 / kChunk + b + chunk) * H + h) * kPrepared;
}

struct Terms { bf16x8 v[3]; };              // x = v[0] + v[1] + v[2], exactly

__device__ __forceinline__ Terms split8(const float* x) {
    // (two at a time: one conversion rounds and packs both; element by element the compiler rounds every number once more to pack it)
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
    typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
    u32x4 t[3];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        float a = x[2 * e], b = x[2 * e + 1];
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const unsigned u = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a, b}), bf16x2));
            t[j][e] = u;
            a -= __builtin_bit_cast(float, u << 16);
            b -= __builtin_bit_cast(float, u & 0xFFFF0000u);
        }
    }
    return {__builtin_bit_cast(bf16x8, t[0]), __builtin_bit_cast(bf16x8, t[1]), __builtin_bit_cast(bf16x8, t[2])};
}

// big += a b of the leading terms, small += the five products down to 2^-24 of it: the large sums take few roundings
__device__ __forceinline__ void mul_terms(const bf16x8* a, const Terms& b, f32x16& big, f32x16& small) {
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[2], b.v[0], small, 0, 0, 0);
    big = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b.v[0], big, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b.v[2], small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b.v[1], small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[0], b.v[1], small, 0, 0, 0);
    small = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[1], b.v[0], small, 0, 0, 0);
}

__device__ __forceinline__ f32x16 zeros() {
    f32x16 z;
#pragma unroll
    for (int r = 0; r < 16; ++r) z[r] = 0.f;
    return z;
}

__device__ __forceinline__ float lane_value(float v, int lane) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// One wave per (chunk, sequence, head).  Lane l stands for token l & 31.
template <int DK, bool DELTA>
__global__ __launch_bounds__(64) void outer_chunk_prepare_kernel(const bf16_t* __restrict__ rows, int64_t stride, int q_off, int k_off,
                                                                 const float* __restrict__ gates, const int32_t* __restrict__ qstart,
                                                                 unsigned char* __restrict__ work, int H, int G) {
    constexpr int PITCH = 36;
    __shared__ __attribute__((aligned(16))) float at[kChunk * PITCH];          // column j of A, row by row
    const int b = blockIdx.y, h = blockIdx.z, gr = h / (H / G);
    const int q0 = qstart[b], n = qstart[b + 1] - q0;
    const int c = blockIdx.x, t0 = c * kChunk;
    if (t0 >= n) return;
    const int lane = threadIdx.x, l31 = lane & 31, hi = lane >> 5;
    const bool valid = t0 + l31 < n;                          // past the portion's end: the identity step
    const size_t tok = q0 + min(t0 + l31, n - 1);
    const bf16_t *q = rows + tok * stride + q_off + (size_t)gr * DK + 8 * hi, *k = rows + tok * stride + k_off + (size_t)gr * DK + 8 * hi;
    const float4 *gp = (const float4*)(gates + (tok * H + h) * 8);
    const float4 ga = gp[0], gb = gp[1];
    const float g = valid ? ga.x : 1.f, beta = valid ? ga.y : 0.f, rk = valid ? ga.w : 0.f, rq = valid ? gb.w : 0.f;
    f32x16 kk, qk;                                            // [i, t]: lane: token t, register r: i = (r & 3) + 8 (r >> 2) + 4 hi
#pragma unroll
    for (int r = 0; r < 16; ++r) kk[r] = qk[r] = 0.f;
#pragma unroll
    for (int ks = 0; ks < DK / 16; ++ks) {
        i32x4 kv = *(const i32x4*)(k + 16 * ks), qv = *(const i32x4*)(q + 16 * ks);
        if (!valid) { kv = i32x4{0, 0, 0, 0}; qv = kv; }
        const bf16x8 kf = __builtin_bit_cast(bf16x8, kv), qf = __builtin_bit_cast(bf16x8, qv);
        if (DELTA) kk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, kf, kk, 0, 0, 0);
        qk = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf, qk, 0, 0, 0);
    }
    // D_ti rk_i, from i = t down (zero for i > t); and the products over the whole chunk.  In double: a product of up to 32 decays
    // is the one place where the chunk would round more often than the token-by-token walk does.
    float m0[16], m1[16];
    double cur = 0., end = 1., dend = 0.;
#pragma unroll
    for (int i = kChunk - 1; i >= 0; --i) {
        if (i < kChunk - 1) cur *= (double)lane_value(g, i + 1);
        if (l31 == i) { cur = 1.; dend = end; }
        end *= (double)lane_value(g, i);
        const float m = (float)(cur * (double)lane_value(rk, i));
        if (i & 4) m1[(i & 3) + 4 * (i >> 3)] = m; else m0[(i & 3) + 4 * (i >> 3)] = m;
    }
    const double Gt = cur * (double)lane_value(g, 0);         // (cur is D_t0 now)
    unsigned char* out = work + prepared_at(q0, b, c, h, H);
    float p[16], a[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const float m = hi ? m1[r] : m0[r];
        const int i = (r & 3) + 8 * (r >> 2) + 4 * hi;
        p[r] = i <= l31 ? rq * (qk[r] * m) : 0.f;             // (chosen, not multiplied: a later token's NaN stays out)
        if (DELTA) a[r] = i < l31 ? beta * rk * (kk[r] * m) : 0.f;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        const Terms t = split8(p + 8 * ks);
#pragma unroll
        for (int j = 0; j < 3; ++j) *(bf16x8*)(out + j * kTermBytes + ks * 1024 + 16 * lane) = t.v[j];
    }
    if (hi == 0)
        *(float4*)(out + kCoefAt + 16 * l31) =
            make_float4(beta, (float)(Gt * (double)(beta * rk)), (float)(Gt * (double)rq), (float)(dend * (double)rk));
    if (lane == 0) *(float*)(out + kEndAt) = (float)end;
    if constexpr (DELTA) {
        // a token's row that is not finite is left out here (the rows of earlier tokens would multiply it by zero) and put in below
        float z = 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) z = __builtin_fmaf(a[r], 0.f, z);
        z += __shfl_xor(z, 32);
#pragma unroll
        for (int r = 0; r < 16; ++r) a[r] = z == 0.f ? a[r] : 0.f;
#pragma unroll
        for (int r = 0; r < 16; ++r) at[((r & 3) + 8 * (r >> 2) + 4 * hi) * PITCH + l31] = a[r];
        __syncthreads();
        // row t of (I + A)^-1, from its diagonal down: x (I + A) = e_t
        float x[kChunk];
#pragma unroll
        for (int j = kChunk - 1; j >= 0; --j) {
            float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i4 = (j + 1) / 4; i4 < kChunk / 4; ++i4) {
                const float4 v = *(const float4*)(at + j * PITCH + 4 * i4);
                const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (4 * i4 + u > j) s[u] += x[4 * i4 + u] * e[u];
            }
            x[j] = j == l31 ? 1.f : j < l31 ? -((s[0] + s[1]) + (s[2] + s[3])) : 0.f;
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            float y[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int i = 16 * ks + (e & 3) + 8 * (e >> 2);
                y[e] = (hi ? x[i + 4] : x[i]) + z;
            }
            const Terms t = split8(y);
#pragma unroll
            for (int j = 0; j < 3; ++j) *(bf16x8*)(out + kTAt + j * kTermBytes + ks * 1024 + 16 * lane) = t.v[j];
        }
    }
}

// The first of a column's 32 tokens (16 in this lane, 16 in the one 32 further) whose x is not finite, its non-finite x made zero; 32
// where there is none.  The triangular products multiply a token by zeros above the diagonal, and zero times infinity is not zero.
__device__ __forceinline__ int first_spoiled(float* x, int hi) {
    float z = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) z = __builtin_fmaf(x[r], 0.f, z);
    if (!__any(!(z == 0.f))) return kChunk;
    int first = kChunk;
#pragma unroll
    for (int r = 0; r < 16; ++r) asm volatile("" : "+v"(x[r]));      // (or the comparisons are made in front of the branch)
#pragma unroll
    for (int r = 15; r >= 0; --r)
        if (!(fabsf(x[r]) <= 3.402823466e38f)) {
            x[r] = 0.f;
            first = (r & 3) + 8 * (r >> 2) + 4 * hi;
        }
    return min(first, __shfl_xor(first, 32));
}

template <int DK, bool DELTA>
__global__ __launch_bounds__(128, 1) void outer_chunk_walk_kernel(const bf16_t* __restrict__ rows, int64_t stride, int q_off, int k_off,
                                                                  int v_off, const unsigned char* __restrict__ work,
                                                                  const float* __restrict__ skip_w, float* __restrict__ state,
                                                                  const int32_t* __restrict__ qstart, const int32_t* __restrict__ seq_pos0,
                                                                  const int32_t* __restrict__ seq_slot, float* __restrict__ o, int H, int G,
                                                                  int V) {
    constexpr int NB = DK / 64;                               // blocks of 32 keys of a wave
    typedef SlimGeom<DK / 32> GM;
    typedef __attribute__((address_space(1))) const void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;
    constexpr int ROWS = kChunk * GM::RB, PREP = 2 * ROWS;    // bytes of a chunk's K (and Q); where its prepared part lies
    constexpr int KQ = ROWS / 2048, NP = (DELTA ? kPrepared : kTAt) / 1024, VAT = PREP + 1024 * NP;
    __shared__ __attribute__((aligned(1024))) unsigned char buf0[VAT + kChunk * 64];
    __shared__ __attribute__((aligned(1024))) unsigned char buf1[VAT + kChunk * 64];
    // Either wave's part of K S, and of the other's rows of results.  swap_k: written between a chunk's first and second meeting, read
    // behind the second one.  swap_o: wave w reads swap_o[.][w] of chunk c behind the first meeting of chunk c + 1, and the other wave
    // writes the place again at the end of a chunk.  The delta form's second meeting lies between the two; the state-space form
    // has one meeting per chunk, so its chunks take two places in turn, and the first meeting of chunk c + 2 lies between.
    __shared__ __attribute__((aligned(16))) f32x4 swap_k[2][4][64], swap_o[DELTA ? 1 : 2][2][2][64];
    const int b = blockIdx.x, h = blockIdx.y, gr = h / (H / G), lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int col = blockIdx.z * 32 + l31;
    const int q0 = qstart[b], n = qstart[b + 1] - q0;
    if (n <= 0) return;
    float* st = state + ((size_t)seq_slot[b] * H + h) * (size_t)DK * V + (size_t)(32 * NB * wave + 8 * hi) * V + col;
    const bool fresh = seq_pos0[b] == 0;
    const float skip = DELTA ? 0.f : skip_w[h];
    f32x16 S[NB];
#pragma unroll
    for (int blk = 0; blk < NB; ++blk)
#pragma unroll
        for (int r = 0; r < 16; ++r) S[blk][r] = fresh ? 0.f : st[(size_t)(32 * blk + 16 * (r >> 3) + (r & 7)) * V];

    const bf16_t *ks0 = rows + (size_t)q0 * stride + k_off + (size_t)gr * DK, *qs0 = rows + (size_t)q0 * stride + q_off + (size_t)gr * DK;
    const bf16_t* vs0 = rows + (size_t)q0 * stride + v_off + (size_t)h * V + blockIdx.z * 32;
    // a chunk's K, Q, V (rows past the end: the last one, cleared before use) and prepared part: 1 KB pieces to the two waves in turn
    int row_of[KQ], ch_of[KQ];
    size_t off_of[KQ];
#pragma unroll
    for (int j = 0; j < KQ; ++j) {
        const int c = 64 * (2 * j + wave) + lane;
        row_of[j] = c / GM::CH;
        ch_of[j] = 8 * ((c % GM::CH) ^ GM::swz(row_of[j]));
        off_of[j] = (size_t)row_of[j] * stride + ch_of[j];
    }
    const int v_row = 16 * wave + (lane >> 2);
    auto load_chunk = [&](unsigned char* buf, int t0) {
        const unsigned char* prep = work + prepared_at(q0, b, t0 / kChunk, h, H) + 1024 * wave + 16 * lane;
        const bool whole = t0 + kChunk <= n;
        __builtin_amdgcn_global_load_lds((gvoid*)(vs0 + (size_t)min(t0 + v_row, n - 1) * stride + 8 * (lane & 3)),
                                         (lvoid*)(buf + VAT + 1024 * wave), 16, 0, 0);
#pragma unroll
        for (int j = 0; j < KQ; ++j) {
            const size_t off = whole ? (size_t)t0 * stride + off_of[j] : (size_t)min(t0 + row_of[j], n - 1) * stride + ch_of[j];
            const int at = 1024 * (2 * j + wave);
            __builtin_amdgcn_global_load_lds((gvoid*)(ks0 + off), (lvoid*)(buf + at), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gvoid*)(qs0 + off), (lvoid*)(buf + ROWS + at), 16, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < NP / 2; ++j)
            __builtin_amdgcn_global_load_lds((gvoid*)(prep + 2048 * j), (lvoid*)(buf + PREP + 1024 * (2 * j + wave)), 16, 0, 0);
        if (NP % 2 && wave == 0)
            __builtin_amdgcn_global_load_lds((gvoid*)(prep + 1024 * (NP - 1)), (lvoid*)(buf + PREP + 1024 * (NP - 1)), 16, 0, 0);
    };
    // row l31, chunk 2 (16 keys) + hi, as the A operand of K S and Q S; columns of K for K^T W by the transposing read, the two
    // middle quads of 16 keys exchanged (the state's order of keys)
    const int gq = (lane >> 4) & 1, ti = lane & 15, tq = ti >> 2, pq = ((ti & 1) << 1) | ((ti >> 1) & 1);
    const int r_at = GM::at(l31, hi) ^ (64 * NB * wave), c_at = (GM::at(4 * hi + tq, 2 * gq + (pq >> 1)) + 8 * (pq & 1)) ^ (64 * NB * wave),
              v_at = 64 * (4 * hi + tq) + 32 * gq + 8 * (ti & 3),
              c_at8 = (GM::at(4 * hi + tq + 8, 2 * gq + (pq >> 1)) + 8 * (pq & 1)) ^ (64 * NB * wave);

    // LDS accesses of both waves in front of it are done; loads from global memory go on (__syncthreads would wait for them)
    auto meet = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    double part[8];                                          // the last chunk's results of tokens 16 wave..: this wave's part
    // (in double: in float32 the state-space form's error was 1 to 5 % above the token-by-token walk's; 1 us, measured when the walk took 142)
    // their sum with the other wave's part, written before the last meeting (turn: 0 for an even chunk of the portion, 1 for an odd one)
    auto store_rows = [&](int t0, bool whole, int turn) {
        float* orow = o + ((size_t)(q0 + t0 + 16 * wave + 4 * hi) * H + h) * V + col;
#pragma unroll
        for (int r4 = 0; r4 < 2; ++r4) {
            const f32x4 y = swap_o[DELTA ? 0 : turn][wave][r4][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int t = e + 8 * r4;
                if (whole || t0 + 16 * wave + 4 * hi + t < n) orow[(size_t)t * H * V] = (float)(part[4 * r4 + e] + (double)y[e]);
            }
        }
    };
    auto chunk = [&](unsigned char* buf, unsigned char* nxt, int t0, int turn) {
        const int left = n - t0;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // the chunk has landed (and rows of results a whole chunk old)
        meet();
        if (t0 > 0) store_rows(t0 - kChunk, true, turn ^ 1);
        if (left < kChunk) {                                  // an absent token's row: zeros, whatever the one in its place holds
            for (int i = left * GM::RB + 16 * (int)threadIdx.x; i < ROWS; i += 2048) {
                *(i32x4*)(buf + i) = i32x4{0, 0, 0, 0};
                *(i32x4*)(buf + ROWS + i) = i32x4{0, 0, 0, 0};
            }
            for (int i = left * 64 + 16 * (int)threadIdx.x; i < kChunk * 64; i += 2048) *(i32x4*)(buf + VAT + i) = i32x4{0, 0, 0, 0};
            meet();
        }
        const unsigned char* prep = buf + PREP;
        Terms s[2 * NB];                                      // the wave's part of the state, 16 keys at a time
#pragma unroll
        for (int ks = 0; ks < 2 * NB; ++ks) {
            float x[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) x[e] = S[ks >> 1][8 * (ks & 1) + e];
            s[ks] = split8(x);
        }
        f32x16 ksb = zeros(), kss = zeros(), qsb = zeros(), qss = zeros();
        if (DELTA) {                                          // each wave has its keys' part of K S
#pragma unroll
            for (int ks = 0; ks < 2 * NB; ++ks) {
                const bf16x8 kf = *(const bf16x8*)(buf + (r_at ^ (32 * ks)));
                kss = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, s[ks].v[2], kss, 0, 0, 0);
                ksb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, s[ks].v[0], ksb, 0, 0, 0);
                kss = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, s[ks].v[1], kss, 0, 0, 0);
            }
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4) {
                f32x4 x;
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = ksb[4 * r4 + e] += kss[4 * r4 + e];
                swap_k[wave][r4][lane] = x;
            }
            meet();
        }
        if (t0 + kChunk < n) load_chunk(nxt, t0 + kChunk);    // (the other buffer was last read in front of the first meeting)
        __builtin_amdgcn_sched_barrier(0);
        float v[16];                                          // column l31 of V, by the transposing read
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                (s16x4 __attribute__((address_space(3)))*)(buf + VAT + v_at + 512 * r4));
#pragma unroll
            for (int e = 0; e < 4; ++e) v[4 * r4 + e] = to_f(__builtin_bit_cast(bf16_t, (short)x[e]));
        }
        float w[16], wd[16], cq[16];
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4) {
            f32x4 x = {0.f, 0.f, 0.f, 0.f};
            if (DELTA) x = swap_k[wave ^ 1][r4][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int r = 4 * r4 + e;
                const float4 cf = *(const float4*)(prep + kCoefAt + 16 * ((r & 3) + 8 * (r >> 2) + 4 * hi));      // beta, beta G rk, G rq, D_31 rk
                w[r] = cf.x * v[r];
                if (DELTA) w[r] -= cf.y * (ksb[r] + x[e]);
                cq[r] = cf.z;
                wd[r] = cf.w;
            }
        }
#pragma unroll
        for (int ks = 0; ks < 2 * NB; ++ks) {                 // and of Q S (independent of what surrounds it)
            const bf16x8 qf = *(const bf16x8*)(buf + ROWS + (r_at ^ (32 * ks)));
            qss = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, s[ks].v[2], qss, 0, 0, 0);
            qsb = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, s[ks].v[0], qsb, 0, 0, 0);
            qss = __builtin_amdgcn_mfma_f32_32x32x16_bf16(qf, s[ks].v[1], qss, 0, 0, 0);
        }
        if (DELTA) {
            f32x16 big = zeros(), small = zeros();
            const int first = first_spoiled(w, hi);
#pragma unroll
            for (int ks = 0; ks < 2; ++ks) {
                bf16x8 m[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) m[j] = *(const bf16x8*)(prep + kTAt + j * kTermBytes + ks * 1024 + 16 * lane);
                mul_terms(m, split8(w + 8 * ks), big, small);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) w[r] = big[r] + small[r];
            if (__any(first < kChunk))
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    asm volatile("" : "+v"(w[r]));
                    if ((r & 3) + 8 * (r >> 2) + 4 * hi >= first) w[r] = __builtin_nanf("");
                }
        }
        const float end = *(const float*)(prep + kEndAt);
#pragma unroll
        for (int r = 0; r < 16; ++r) wd[r] *= w[r];
        f32x16 ib[NB], is[NB];
#pragma unroll
        for (int blk = 0; blk < NB; ++blk) ib[blk] = is[blk] = zeros();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const Terms d = split8(wd + 8 * ks);
#pragma unroll
            for (int blk = 0; blk < NB; ++blk) {
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4 __attribute__((address_space(3)))*)(buf + (c_at ^ (64 * blk)) + 16 * GM::RB * ks));
                const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4 __attribute__((address_space(3)))*)(buf + (c_at8 ^ (64 * blk)) + 16 * GM::RB * ks));
                const s16x8 kt8 = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                const bf16x8 kt = __builtin_bit_cast(bf16x8, kt8);
                is[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kt, d.v[2], is[blk], 0, 0, 0);
                ib[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kt, d.v[0], ib[blk], 0, 0, 0);
                is[blk] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kt, d.v[1], is[blk], 0, 0, 0);
            }
        }
        {                                                     // P W of the wave's half of the strengths, and the parts of the results
            const int first = first_spoiled(w, hi);
            if (__any(first < kChunk))
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    asm volatile("" : "+v"(cq[r]));
                    if ((r & 3) + 8 * (r >> 2) + 4 * hi >= first) cq[r] = __builtin_nanf("");
                }
            // (one form per wave: chosen element by element, the halves go through indexed register moves)
            auto results = [&](auto second) __attribute__((always_inline)) {
                constexpr int KEPT = second ? 8 : 0, GIVEN = 8 - KEPT;
                f32x16 big = zeros(), small = zeros();
                bf16x8 m[3];
#pragma unroll
                for (int j = 0; j < 3; ++j) m[j] = *(const bf16x8*)(prep + j * kTermBytes + (KEPT / 8) * 1024 + 16 * lane);
                mul_terms(m, split8(w + KEPT), big, small);
#pragma unroll
                for (int r4 = 0; r4 < 2; ++r4) {
                    f32x4 y;
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const int r = 4 * r4 + e, g = GIVEN + r, k = KEPT + r;
                        y[e] = cq[g] * (qsb[g] + qss[g]) + (big[g] + small[g]);
                        const double c = cq[k], qb = qsb[k], qs = qss[k], pb = big[k], ps = small[k];
                        part[r] = c * (qb + qs) + (pb + ps);
                        if (!DELTA) part[r] += (double)skip * (double)v[k];
                    }
                    swap_o[DELTA ? 0 : turn][wave ^ 1][r4][lane] = y;
                }
            };
            if (wave) results(std::true_type{});
            else results(std::false_type{});
        }
#pragma unroll
        for (int blk = 0; blk < NB; ++blk)
#pragma unroll
            for (int r = 0; r < 16; ++r) S[blk][r] = end * S[blk][r] + (ib[blk][r] + is[blk][r]);
    };
    load_chunk(buf0, 0);
    for (int t0 = 0; t0 < n; t0 += 2 * kChunk) {
        chunk(buf0, buf1, t0, 0);
        if (t0 + kChunk < n) chunk(buf1, buf0, t0 + kChunk, 1);
    }
    meet();
    store_rows((n - 1) / kChunk * kChunk, false, (n - 1) / kChunk & 1);
#pragma unroll
    for (int blk = 0; blk < NB; ++blk)
#pragma unroll
        for (int r = 0; r < 16; ++r) st[(size_t)(32 * blk + 16 * (r >> 3) + (r & 7)) * V] = S[blk][r];
}

template <bool DELTA>
static void launch_chunks(const void* rows_, int64_t stride, int q_off, int k_off, int v_off, const GateArgs<bf16_t>& ga, float* gates,
                          void* work, float* state, const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, float* o,
                          int B, int64_t T, int H, int G, int D, int V, int max_q, hipStream_t s) {
    const bf16_t* rows = (const bf16_t*)rows_;
    const int64_t items = T * G;
    hipLaunchKernelGGL((outer_gates_kernel<bf16_t, 8, DELTA>), dim3((unsigned)((items + 15) / 16)), dim3(256), 0, s, rows, stride, q_off,
                       k_off, ga, gates, items, H, G, D);
    const dim3 pg((unsigned)((max_q + kChunk - 1) / kChunk), (unsigned)B, (unsigned)H), wg((unsigned)B, (unsigned)H, (unsigned)(V / 32));
#define HM_CHUNKS(DK)                                                                                                              \
    do {                                                                                                                           \
        hipLaunchKernelGGL((outer_chunk_prepare_kernel<DK, DELTA>), pg, dim3(64), 0, s, rows, stride, q_off, k_off, gates, qstart,   \
                           (unsigned char*)work, H, G);                                                                            \
        hipLaunchKernelGGL((outer_chunk_walk_kernel<DK, DELTA>), wg, dim3(128), 0, s, rows, stride, q_off, k_off, v_off,             \
                           (const unsigned char*)work, ga.skip, state, qstart, seq_pos0, seq_slot, o, H, G, V);                    \
    } while (0)
    if (D == 64) HM_CHUNKS(64); else HM_CHUNKS(128);
#undef HM_CHUNKS
}

static int chunk_args_bad(const char* name, int64_t stride, int q_off, int k_off, int v_off, const void* rows, const void* work, int B,
                          int64_t T, int D, int V) {
    if (B > 0 && T > 0 && !work) { set_error("%s: bad argument", name); return HM_EINVAL; }
    if ((D != 64 && D != 128) || V % 32 != 0 || B > 65535) {
        set_error("%s: 64 or 128 key channels, value channels a multiple of 32, at most 65535 sequences", name);
        return HM_ESHAPE;
    }
    if ((stride | q_off | k_off | v_off) % 8 != 0 || (uintptr_t)rows % 16 != 0 || (uintptr_t)work % 16 != 0) {
        set_error("%s: rows and their parts must start on 16 bytes", name);
        return HM_EINVAL;
    }
    return 0;
}

}  // namespace hm

using namespace hm;

extern "C" size_t hm_outer_chunk_work_bytes(int64_t T, int B, int H) {
    if (T <= 0 || B <= 0 || H <= 0) return 0;
    return (size_t)(T / kChunk + B + 1) * H * kPrepared;
}

extern "C" int hm_gated_delta_chunks(const void* rows, int64_t stride, int q_off, int k_off, int v_off, const void* pre,
                                     int64_t pre_stride, int b_off, int a_off, const float* A, const float* dt_bias, float unit_eps,
                                     float q_scale, float* gates, void* work, float* state, const int32_t* qstart,
                                     const int32_t* seq_pos0, const int32_t* seq_slot, float* o, int B, int64_t T, int H, int G, int D,
                                     int V, int max_q, void* stream) {
    int rc = outer_args_bad("hm_gated_delta_chunks", stride, q_off, k_off, v_off, pre_stride, b_off, a_off, rows, pre, A, dt_bias, gates,
                            state, qstart, seq_pos0, seq_slot, o, B, T, H, G, D, V, max_q < 2 ? 2 : max_q);
    if (!rc) rc = chunk_args_bad("hm_gated_delta_chunks", stride, q_off, k_off, v_off, rows, work, B, T, D, V);
    if (rc) return rc;
    if (B == 0 || T == 0 || max_q == 0) return HM_OK;
    GateArgs<bf16_t> ga = {(const bf16_t*)pre, pre_stride, b_off, a_off, A, dt_bias, nullptr, unit_eps, q_scale};
    launch_chunks<true>(rows, stride, q_off, k_off, v_off, ga, gates, work, state, qstart, seq_pos0, seq_slot, o, B, T, H, G, D, V, max_q,
                        as_stream(stream));
    HM_CHECK_LAUNCH("hm_gated_delta_chunks");
    return HM_OK;
}

extern "C" int hm_state_space_chunks(const void* rows, int64_t stride, int x_off, int b_off, int c_off, const void* pre, int64_t pre_stride,
                                     int dt_off, const float* A, const float* dt_bias, const float* D, float* gates, void* work,
                                     float* state, const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, float* y, int B,
                                     int64_t T, int H, int G, int N, int V, int max_q, void* stream) {
    int rc = outer_args_bad("hm_state_space_chunks", stride, c_off, b_off, x_off, pre_stride, 0, dt_off, rows, pre, A, dt_bias, gates,
                            state, qstart, seq_pos0, seq_slot, y, B, T, H, G, N, V, max_q < 2 ? 2 : max_q);
    if (!rc) rc = chunk_args_bad("hm_state_space_chunks", stride, c_off, b_off, x_off, rows, work, B, T, N, V);
    if (rc) return rc;
    if (B > 0 && T > 0 && !D) { set_error("hm_state_space_chunks: bad argument"); return HM_EINVAL; }
    if (B == 0 || T == 0 || max_q == 0) return HM_OK;
    GateArgs<bf16_t> ga = {(const bf16_t*)pre, pre_stride, 0, dt_off, A, dt_bias, D, 0.f, 1.f};
    launch_chunks<false>(rows, stride, c_off, b_off, x_off, ga, gates, work, state, qstart, seq_pos0, seq_slot, y, B, T, H, G, N, V, max_q,
                         as_stream(stream));
    HM_CHECK_LAUNCH("hm_state_space_chunks");
    return HM_OK;
}
