// The outer-product recurrences of hm_outer.hip over prompts, 32 tokens at a time on the matrix cores.
//
// With G_t the product of a chunk's decays up to token t, D_ti that of the decays after i up to t, S the state in front of the
// chunk (f32 [D keys, V]) and r the lengths' reciprocals, the chunk's strengths W [32, V] solve a triangular system,
//   (I + A) W = R,  A_ti = beta_t rk_t rk_i (k_t . k_i) D_ti (i < t),  R_t = beta_t (v_t - G_t rk_t S^T k_t)
// (state-space form: W = beta v), and then
//   o_t = rq_t (G_t S^T q_t + sum_{i <= t} D_ti rk_i (q_t . k_i) w_i) + skip v_t,   S <- G_31 S + sum_i D_31,i rk_i k_i w_i^T.
// Everything that does not depend on the state is worked out for all chunks at once (prepare): P_ti = rq_t rk_i (q_t . k_i) D_ti,
// N = (I + A)^-1 - I by forward substitution, and four numbers per token.  The walk over a sequence's chunks is left with five
// products per chunk: K S, Q S, N R (W = R + N R), P W and K^T W.
//
// Precision: the stored q, k are bf16 and enter the products exactly; every float32 operand (S, N, R, P, W) enters as the sum of
// three bf16 numbers, which is the number itself, and of the nine products of two such sums the six above 2^-24 of the result
// are kept, the leading one in a sum of its own (but for K^T W); sums are float32, products of decays double.  Against float64 the results are
// nearer than the token-by-token walk's: 8 prompts of 900 to 1100 tokens, 8 heads, in norm: gated delta 128 x 128 o 1.30e-7 (walk 1.50e-7), state
// 1.04e-7 (1.18e-7); state space 128 x 64 o 1.53e-7 (1.91e-7), state 1.41e-7 (1.86e-7).  A token that is not finite spoils
// its own and later tokens, as in the walk, and none in front of it.
//
// The walk is one workgroup of 2 NW waves per (sequence, head, 16 NW value channels).  Wave w < NW keeps 16 columns of the state in the
// accumulators of its products: lane l holds column l & 15 and of every 32 keys 8 (l >> 4) + 0..7.  That is the order in which a lane's
// eight numbers of a B operand come (a row of K or Q is read from LDS in 16-byte pieces as the A operand), so the state never moves; the
// 32 tokens' strengths lie in the lanes as 4 (l >> 4) + 0..3 and 16 further, and the prepared A operands are stored in that order.
// Its partner w + NW, on the same SIMD with four columns' waves, asks for the chunks two ahead and makes the results of the chunk before
// from the strengths that it is handed through LDS.  One meeting per chunk.
//
// Against the walk that takes token after token, bound by the float32 vector unit and its chain of lane sums at two waves per
// SIMD: 8 prompts of 900 to 1100 tokens, 16 heads of 128 x 128: 418 us there, here 22 (prepare) + 68 (walk); one such prompt 9 + 46 us.
// What is left of a chunk's 3800 cycles: the chain S -> K S -> R -> W -> S of one wave, 380 vector instructions of 4.5 cycles (8 for a
// conversion to bf16) and 85 matrix ones of 16, next to 3300 cycles of its partner, and LDS (58 KB per chunk and 16 columns).
// With two waves of half the keys each on 32 columns, which both work out the strengths and give each other parts of the results in
// LDS, the walk took 118 (one prompt: 90).  Against 72 (49), with the state's sums apart: one wave per SIMD with all of a chunk's work 99 (75);
// the state's terms handed on through LDS so that the partner makes Q S too 85 (63: LDS is then the bound); results in double here as
// well 78 (57).
#include "hm_attn_tile.h"
#include "hm_outer.h"

namespace hm {

constexpr int kChunk = 32;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef bf16_t bf16x2 __attribute__((ext_vector_type(2)));
typedef bf16_t bf16x4 __attribute__((ext_vector_type(4)));

// A prepared (chunk, head): P, and T with the delta form, as A operands of 16 rows (tokens): three terms each, of rows 0..15 the
// columns 0..15 (the others are zero), of rows 16..31 all; four coefficients per token; the whole chunk's decay.  Column 8 g + e of a
// lane's eight stands for token 4 g + e, or 16 + 4 g + e - 4 from e = 4 on: the order in which a lane holds strengths.
constexpr int kTermLow = 64 * 8, kTermBytes = kTermLow + 64 * 16, kOperand = 3 * kTermBytes, kPrepared = 10240;
constexpr int kBeta = 0, kOldKey = kChunk, kOldQuery = 2 * kChunk, kLeft = 3 * kChunk;       // beta, beta G rk, G rq, D_31 rk (state space: D_31 beta)
template <bool DELTA>
struct Prepared {
    static constexpr int kTAt = kOperand, kCoefAt = DELTA ? 2 * kOperand : kOperand, kEndAt = kCoefAt + kChunk * 16,
                         kPieces = (kEndAt + 4 + 1023) / 1024;
    static_assert(1024 * kPieces <= kPrepared, "whole pieces are read");
};

// chunks are numbered q0 / 32 + b + chunk: numbers of different sequences never meet
__device__ __forceinline__ size_t prepared_at(int q0, int b, int chunk, int h, int H) {
    return ((size_t)(q0 / kChunk + b + chunk) * H + h) * kPrepared;
}

struct Terms { bf16x8 v[3]; };              // x = v[0] + v[1] + v[2], exactly

// a - u[0], b - u[1] (exact): a product with (-1, 0) and (0, -1) added up.  The factors are kept from the compiler, which would take
// them for the inline constant -1.0 and that for both halves.
struct Minus {
    bf16x2 lo, hi;
    __device__ __forceinline__ Minus() {
        unsigned l = 0x0000BF80u, h = 0xBF800000u;
        asm volatile("" : "+s"(l), "+s"(h));
        lo = __builtin_bit_cast(bf16x2, l);
        hi = __builtin_bit_cast(bf16x2, h);
    }
};

// each term the nearest bf16 to what the terms in front of it leave: products of two such sums may drop what is below 2^-24 of them
// (here and below all numbers term by term: a dot product's result may be read three instructions later)
template <int N>
__device__ __forceinline__ void split(const float* x, const Minus& minus, unsigned (&t)[3][N / 2]) {
    float a[N];
#pragma unroll
    for (int e = 0; e < N; ++e) a[e] = x[e];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int e = 0; e < N / 2; ++e) t[j][e] = __builtin_bit_cast(unsigned, __builtin_convertvector((f32x2{a[2 * e], a[2 * e + 1]}), bf16x2));
        if (j < 2)
#pragma unroll
            for (int e = 0; e < N; ++e)
                a[e] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, t[j][e / 2]), e & 1 ? minus.hi : minus.lo, a[e], false);
    }
}

__device__ __forceinline__ Terms split8(const float* x, const Minus& minus) {
    unsigned t[3][4];
    split<8>(x, minus, t);
    Terms r;
#pragma unroll
    for (int j = 0; j < 3; ++j) r.v[j] = __builtin_bit_cast(bf16x8, (u32x4{t[j][0], t[j][1], t[j][2], t[j][3]}));
    return r;
}

// each term the upper 16 bits of what the terms in front of it leave (the conversion takes twice as long): for products with numbers
// that are bf16 themselves, of which none is dropped
__device__ __forceinline__ Terms cut8(const float* x, const Minus& minus) {
    u32x4 t[3];
    float a[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) a[e] = x[e];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
            t[j][e] = __builtin_amdgcn_perm(__builtin_bit_cast(unsigned, a[2 * e + 1]), __builtin_bit_cast(unsigned, a[2 * e]), 0x07060302u);
        if (j < 2)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const unsigned u = t[j][e / 2];
                a[e] = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, u), e & 1 ? minus.hi : minus.lo, a[e], false);
            }
    }
    return {__builtin_bit_cast(bf16x8, t[0]), __builtin_bit_cast(bf16x8, t[1]), __builtin_bit_cast(bf16x8, t[2])};
}

__device__ __forceinline__ f32x4 zeros4() { return f32x4{0.f, 0.f, 0.f, 0.f}; }

// A lower triangular prepared operand (32 x 32), a lane's part
struct Lower {
    s16x4 a0[3];
    bf16x8 a1[3];
    __device__ __forceinline__ void read(const unsigned char* op, int lane) {
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            a0[j] = *(const s16x4*)(op + j * kTermBytes + 8 * lane);
            a1[j] = *(const bf16x8*)(op + j * kTermBytes + kTermLow + 16 * lane);
        }
    }
    // times 16 columns of strengths: rows 0..15 in [0], 16..31 in [1].  big has the products of the leading terms (of rows 16..31 and columns
    // 16..31: more), small the five down to 2^-24 of them: the large sums take few roundings.
    __device__ __forceinline__ void times(const Terms& b, f32x4 (&big)[2], f32x4& more, f32x4 (&small)[2]) const {
        s16x4 b0[3], b1;
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            const s16x8 x = __builtin_bit_cast(s16x8, b.v[j]);
            b0[j] = s16x4{x[0], x[1], x[2], x[3]};
            if (j == 0) b1 = s16x4{x[4], x[5], x[6], x[7]};
        }
        const s16x8 a = __builtin_bit_cast(s16x8, a1[0]);
        constexpr int A[5] = {2, 0, 1, 0, 1}, B[5] = {0, 2, 1, 1, 0};
        big[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0[0], b0[0], zeros4(), 0, 0, 0);
        big[1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(s16x4{a[0], a[1], a[2], a[3]}, b0[0], zeros4(), 0, 0, 0);
        more = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(s16x4{a[4], a[5], a[6], a[7]}, b1, zeros4(), 0, 0, 0);
        small[0] = small[1] = zeros4();
#pragma unroll
        for (int i = 0; i < 5; ++i) {
            small[0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a0[A[i]], b0[B[i]], small[0], 0, 0, 0);
            small[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a1[A[i]], b.v[B[i]], small[1], 0, 0, 0);
        }
    }
};

template <int CTRL>
__device__ __forceinline__ float of_quad(float v) {            // the value of lane CTRL / 0x55 of each four
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}

// One wave per (chunk, sequence, head), from the rows and the gates' pre-activations.  Lane (l15, g4) has the products of tokens t = l15
// and 16 + l15 with the tokens i = 4 g4 + 0..3 and 16 + 4 g4 + 0..3: as the 16-row products leave them and as the walk reads them, so
// they are stored as they lie.
//
// The decays D_ti are products in double, put together from quads of tokens: t's part of its quad, the quads between, the rest of
// i's quad; a product of up to 32 decays is the one place where the chunk would round more often than the token-by-token walk does.
// (I + A)^-1 by blocks of 16: T11 and T22 by forward substitution, a column per lane, T21 = -T22 A21 T11 by the float32 matrix products.
//
// 8 prompts of 900 to 1100 tokens, 16 heads of 128 x 128: 22 us (state space, 32 heads of 128 x 64: 26) of which the stores are 5, 4096 waves of
// 990 vector instructions and a way of 6 us each (one prompt: 9 us).  With a kernel of its own for the gates in front, products of
// decays token by token and the whole of (I + A)^-1 by substitution in 32 lanes of 64 it was 32 + 11 (27 + 12; 11 + 5).  Four chunks
// per workgroup, or a group's heads side by side on one die: no difference.
template <int DK, bool DELTA>
__global__ __launch_bounds__(64) void outer_chunk_prepare_kernel(const bf16_t* __restrict__ rows, int64_t stride, int q_off, int k_off,
                                                                 GateArgs<bf16_t> ga, const int32_t* __restrict__ qstart,
                                                                 unsigned char* __restrict__ work, int H, int G) {
    constexpr int AP = 36, TP = 20;                           // floats between rows of A, columns of T: whole 16 bytes, every bank once
    typedef Prepared<DELTA> PR;
    __shared__ double own[kChunk], rest[kChunk], quad[8], between[8][8];
    __shared__ f32x4 inside[kChunk], token[kChunk];
    __shared__ __attribute__((aligned(16))) float row_a[DELTA ? kChunk * AP : 4], col_t[DELTA ? 2 : 1][DELTA ? 16 * TP : 4];
    const int b = blockIdx.y, h = blockIdx.z, gr = h / (H / G);
    const int q0 = qstart[b], n = qstart[b + 1] - q0;
    const int c = blockIdx.x, t0 = c * kChunk;
    if (t0 >= n) return;
    const int lane = threadIdx.x, l31 = lane & 31, l15 = lane & 15, g4 = lane >> 4;
    const Minus minus;
    f32x4 kk00 = zeros4(), kk10 = zeros4(), kk11 = zeros4(), qk00 = zeros4(), qk10 = zeros4(), qk11 = zeros4();
    float qq = 0.f, ksq = 0.f;                                // of token l31
    {
        bf16x8 k[2][DK / 32], q[2][DK / 32];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const int t = t0 + 16 * tb + l15;
            const bf16_t* row = rows + (size_t)(q0 + min(t, n - 1)) * stride + (size_t)gr * DK + 8 * g4;
#pragma unroll
            for (int ks = 0; ks < DK / 32; ++ks) {
                k[tb][ks] = *(const bf16x8*)(row + k_off + 32 * ks);
                q[tb][ks] = *(const bf16x8*)(row + q_off + 32 * ks);
            }
        }
        if (t0 + kChunk > n)                                  // past the portion's end: the identity step
#pragma unroll
            for (int tb = 0; tb < 2; ++tb)
#pragma unroll
                for (int ks = 0; ks < DK / 32; ++ks)
                    if (t0 + 16 * tb + l15 >= n) {
                        asm volatile("" : "+v"(k[tb][ks]), "+v"(q[tb][ks]));      // (or every chunk makes the choice)
                        k[tb][ks] = q[tb][ks] = __builtin_bit_cast(bf16x8, (i32x4{0, 0, 0, 0}));
                    }
#pragma unroll
        for (int ks = 0; ks < DK / 32; ++ks) {
            if (DELTA) {
                kk00 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[0][ks], k[0][ks], kk00, 0, 0, 0);
                kk11 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[1][ks], k[1][ks], kk11, 0, 0, 0);
                kk10 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[0][ks], k[1][ks], kk10, 0, 0, 0);
            }
            qk00 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[0][ks], q[0][ks], qk00, 0, 0, 0);
            qk11 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[1][ks], q[1][ks], qk11, 0, 0, 0);
            qk10 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(k[0][ks], q[1][ks], qk10, 0, 0, 0);
        }
        if (DELTA) {                                          // the squared lengths (on the products' diagonals they have larger errors)
            auto square = [&](const bf16x8 (&x)[2][DK / 32]) {
                float sum[2];
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) {
                    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
                    for (int ks = 0; ks < DK / 32; ++ks)
#pragma unroll
                        for (int e = 0; e < 4; ++e) {
                            const bf16x2 u = {x[tb][ks][2 * e], x[tb][ks][2 * e + 1]};
                            s[e] = __builtin_amdgcn_fdot2_f32_bf16(u, u, s[e], false);
                        }
                    sum[tb] = (s[0] + s[1]) + (s[2] + s[3]);
                    sum[tb] += __shfl_xor(sum[tb], 16);
                    sum[tb] += __shfl_xor(sum[tb], 32);
                }
                return lane & 16 ? sum[1] : sum[0];
            };
            qq = square(q);
            ksq = square(k);
        }
    }
    // ---- lane l31 (either half): the gates of that token, and its quad's decays
    Gates gt = make_gates<bf16_t, DELTA>(ga, q0 + min(t0 + l31, n - 1), h, qq, ksq, 0.f);
    if (t0 + l31 >= n) {
        gt.g = 1.f;
        gt.a1 = gt.rk = gt.rq = 0.f;
    }
    const int e4 = lane & 3;
    {
        const double g0 = of_quad<0x00>(gt.g), g1 = of_quad<0x55>(gt.g), g2 = of_quad<0xAA>(gt.g), g3 = of_quad<0xFF>(gt.g);
        const double r0 = of_quad<0x00>(gt.rk), r1 = of_quad<0x55>(gt.rk), r2 = of_quad<0xAA>(gt.rk), r3 = of_quad<0xFF>(gt.rk);
        const double g12 = g1 * g2, g23 = g2 * g3, g123 = g1 * g23;
        const double x0 = e4 == 0 ? 1. : e4 == 1 ? g1 : e4 == 2 ? g12 : g123, x1 = e4 == 1 ? 1. : e4 == 2 ? g2 : g23, x2 = e4 == 2 ? 1. : g3;
        own[l31] = g0 * x0;
        rest[l31] = (e4 == 0 ? g123 : e4 == 1 ? g23 : e4 == 2 ? g3 : 1.) * (double)gt.rk;
        inside[l31] = f32x4{(float)(x0 * r0), (float)(x1 * r1), (float)(x2 * r2), (float)r3};       // (of tokens behind t: not used)
        token[l31] = f32x4{gt.a1, gt.rk, gt.rq, 0.f};
        if (e4 == 3) quad[l31 >> 2] = g0 * x0;
    }
    __syncthreads();
    {
        double r = 1.;                                        // the quads between q = lane & 7 and lane >> 3
#pragma unroll
        for (int s = 1; s < 7; ++s)
            if (s > (lane & 7) && s < lane >> 3) r *= quad[s];
        between[lane >> 3][lane & 7] = r;
    }
    __syncthreads();
    unsigned char* out = work + prepared_at(q0, b, c, h, H);
    if (lane < kChunk) {
        const int q = lane >> 2;
        const double first = quad[0], last = quad[7], in_front = q > 0 ? first * between[q][0] : 1., behind = q < 7 ? between[7][q] * last : 1.;
        const double Gt = own[lane] * in_front;
        float* coef = (float*)(out + PR::kCoefAt);
        coef[kBeta + lane] = gt.a1;
        coef[kOldKey + lane] = (float)(Gt * (double)(gt.a1 * gt.rk));
        coef[kOldQuery + lane] = (float)(Gt * (double)gt.rq);
        coef[kLeft + lane] = (float)(rest[lane] * behind * (DELTA ? 1. : (double)gt.a1));
        if (lane == 0) *(float*)(out + PR::kEndAt) = (float)(first * between[7][0] * last);
    }
    // D_ti rk_i for t and the quad q of i; of later tokens anything
    auto decay = [&](int t, int q) {
        const double d = own[t] * between[t >> 2][q];
        const f32x4 in = inside[t];
        f32x4 m;
#pragma unroll
        for (int e = 0; e < 4; ++e) m[e] = (t >> 2) == q ? in[e] : (float)(d * rest[4 * q + e]);
        return m;
    };
    const f32x4 m00 = decay(l15, g4), m10 = decay(16 + l15, g4), m11 = decay(16 + l15, 4 + g4), tk0 = token[l15], tk1 = token[16 + l15];
    // three terms of rows 0..15 (columns 4 g4..) and of rows 16..31 (columns 4 g4.. and 16 + 4 g4..)
    auto put = [&](unsigned char* op, const f32x4& x00, const f32x4& x10, const f32x4& x11) {
        typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
        const float low[4] = {x00[0], x00[1], x00[2], x00[3]}, up[8] = {x10[0], x10[1], x10[2], x10[3], x11[0], x11[1], x11[2], x11[3]};
        unsigned tl[3][2], tu[3][4];
        split<4>(low, minus, tl);
        split<8>(up, minus, tu);
#pragma unroll
        for (int j = 0; j < 3; ++j) {
            *(u32x2*)(op + j * kTermBytes + 8 * lane) = u32x2{tl[j][0], tl[j][1]};
            *(u32x4*)(op + j * kTermBytes + kTermLow + 16 * lane) = u32x4{tu[j][0], tu[j][1], tu[j][2], tu[j][3]};
        }
    };
    {
        f32x4 p00, p10, p11;
#pragma unroll
        for (int e = 0; e < 4; ++e) {                         // (chosen, not multiplied: a later token's NaN stays out)
            const bool seen = 4 * g4 + e <= l15;
            p00[e] = seen ? tk0[2] * (qk00[e] * m00[e]) : 0.f;
            p10[e] = tk1[2] * (qk10[e] * m10[e]);
            p11[e] = seen ? tk1[2] * (qk11[e] * m11[e]) : 0.f;
        }
        put(out, p00, p10, p11);
    }
    if constexpr (DELTA) {
        const float s0 = tk0[0] * tk0[1], s1 = tk1[0] * tk1[1];
        f32x4 a00, a10, a11;
        float z0 = 0.f, z1 = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const bool seen = 4 * g4 + e < l15;
            a00[e] = seen ? s0 * (kk00[e] * m00[e]) : 0.f;
            a10[e] = s1 * (kk10[e] * m10[e]);
            a11[e] = seen ? s1 * (kk11[e] * m11[e]) : 0.f;
            z0 = __builtin_fmaf(a00[e], 0.f, z0);
            z1 = __builtin_fmaf(a10[e], 0.f, __builtin_fmaf(a11[e], 0.f, z1));
        }
        // a token's row that is not finite is left out here (the rows of earlier tokens would multiply it by zero) and put in below
        z0 += __shfl_xor(z0, 16);
        z1 += __shfl_xor(z1, 16);
        z0 += __shfl_xor(z0, 32);
        z1 += __shfl_xor(z1, 32);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            a00[e] = z0 == 0.f ? a00[e] : 0.f;
            a10[e] = z1 == 0.f ? a10[e] : 0.f;
            a11[e] = z1 == 0.f ? a11[e] : 0.f;
        }
        *(f32x4*)(row_a + l15 * AP + 4 * g4) = a00;
        *(f32x4*)(row_a + (16 + l15) * AP + 16 + 4 * g4) = a11;
        __syncthreads();
        // column l15 of the block's inverse: (I + A) x = e
        const int tb = l31 >> 4;
        const float* rows_a = row_a + 16 * tb * (AP + 1);
        float x[16];
#pragma unroll
        for (int t = 0; t < 16; ++t) {
            float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i4 = 0; i4 < (t + 3) / 4; ++i4) {
                const f32x4 v = *(const f32x4*)(rows_a + t * AP + 4 * i4);
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (4 * i4 + u < t) s[u] += v[u] * x[4 * i4 + u];
            }
            x[t] = t == l15 ? 1.f : t > l15 ? -((s[0] + s[1]) + (s[2] + s[3])) : 0.f;
        }
        if (lane < kChunk)
#pragma unroll
            for (int i = 0; i < 4; ++i) *(f32x4*)(col_t[tb] + l15 * TP + 4 * i) = f32x4{x[4 * i], x[4 * i + 1], x[4 * i + 2], x[4 * i + 3]};
        __syncthreads();
        // T21: the order of the sums is the lanes', k = 4 g4 + s in step s
        const f32x4 t11 = *(const f32x4*)(col_t[0] + l15 * TP + 4 * g4);
        f32x4 t22, u = zeros4(), t21 = zeros4(), n00, n10, n11;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            t22[s] = col_t[1][(4 * g4 + s) * TP + l15];
            u = __builtin_amdgcn_mfma_f32_16x16x4f32(a10[s], t11[s], u, 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) t21 = __builtin_amdgcn_mfma_f32_16x16x4f32(t22[s], u[s], t21, 0, 0, 0);
        *(f32x4*)(row_a + l15 * TP + 4 * g4) = t21;            // (A's rows are done with)
        __syncthreads();
#pragma unroll
        for (int e = 0; e < 4; ++e) {                         // (the diagonal's ones stay out: W = R + N R)
            const bool one = 4 * g4 + e == l15;
            n00[e] = (one ? 0.f : col_t[0][(4 * g4 + e) * TP + l15]) + z0;
            n10[e] = z1 - row_a[(4 * g4 + e) * TP + l15];
            n11[e] = (one ? 0.f : t22[e]) + z1;
        }
        put(out + PR::kTAt, n00, n10, n11);
    }
}

__device__ __forceinline__ bool spoiled(const float* x) {
    float z0 = 0.f, z1 = 0.f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        z0 = __builtin_fmaf(x[r], 0.f, z0);
        z1 = __builtin_fmaf(x[4 + r], 0.f, z1);
    }
    const float z = z0 + z1;
    return __builtin_expect(__any(!(z == 0.f)), 0);
}

// The first of a column's 32 tokens (8 in this lane, the others in those 16, 32 and 48 further) whose x is not finite, its non-finite x
// made zero; 32 where there is none.  The triangular products multiply a token by zeros above the diagonal, and zero times infinity is not zero.
__device__ __forceinline__ int first_spoiled(float* x, int g) {
    int first = kChunk;
#pragma unroll
    for (int r = 0; r < 8; ++r) asm volatile("" : "+v"(x[r]));       // (or the comparisons are made in front of the caller's branch)
#pragma unroll
    for (int r = 7; r >= 0; --r)
        if (!(fabsf(x[r]) <= 3.402823466e38f)) {
            x[r] = 0.f;
            first = (r & 3) + 16 * (r >> 2) + 4 * g;
        }
    first = min(first, __shfl_xor(first, 16));
    return min(first, __shfl_xor(first, 32));
}

template <int DK, int NW, bool DELTA>
__global__ __launch_bounds__(128 * NW) void outer_chunk_walk_kernel(const bf16_t* __restrict__ rows, int64_t stride, int q_off, int k_off,
                                                                    int v_off, const unsigned char* __restrict__ work,
                                                                    const float* __restrict__ skip_w, float* __restrict__ state,
                                                                    const int32_t* __restrict__ qstart, const int32_t* __restrict__ seq_pos0,
                                                                    const int32_t* __restrict__ seq_slot, float* __restrict__ o, int H, int G,
                                                                    int V) {
    constexpr int KS = DK / 32;                               // steps of 32 keys
    typedef SlimGeom<DK / 32> GM;
    typedef Prepared<DELTA> PR;
    typedef __attribute__((address_space(1))) const void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;
    constexpr int ROWS = kChunk * GM::RB, PREP = 2 * ROWS;    // bytes of a chunk's K (and Q); where its prepared part lies
    constexpr int KQ = ROWS / (1024 * NW), VAT = PREP + 1024 * PR::kPieces, VP = 32 * NW;         // (VP: bytes of a row of V)
    constexpr int LOADS = 2 * KQ + 1 + PR::kPieces / NW;      // a wave's per chunk, at least
    __shared__ __attribute__((aligned(1024))) unsigned char buf0[VAT + kChunk * VP];
    __shared__ __attribute__((aligned(1024))) unsigned char buf1[VAT + kChunk * VP];
    __shared__ __attribute__((aligned(1024))) unsigned char buf2[VAT + kChunk * VP];
    // what a chunk's results are made of: the strengths and the state's part (state space: a double in two numbers), read behind the next
    // meeting while the next chunk's are written to the other half
    constexpr int GIVEN = DELTA ? 4 : 6;
    __shared__ __attribute__((aligned(16))) f32x4 given[2][NW][GIVEN][64];
    const int b = blockIdx.x, h = blockIdx.y, gr = h / (H / G), lane = threadIdx.x & 63, l15 = lane & 15, g = lane >> 4;
    const int warp = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = warp % NW;
    const int col = (blockIdx.z * NW + wave) * 16 + l15;
    const int q0 = qstart[b], n = qstart[b + 1] - q0;
    if (n <= 0) return;
    const int r_at = GM::at(l15, g);                          // row l15, chunk g (8 keys), as the A operand of K S and Q S
    const int v_at = VP * (4 * g + (l15 >> 2)) + 32 * wave + 8 * (l15 & 3);        // the wave's columns of V, by the transposing read
    const Minus minus;

    // LDS accesses of all waves in front of it are done; loads from global memory go on (__syncthreads would wait for them)
    auto meet = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };
    auto clear_absent = [&](unsigned char* buf, int left) {   // an absent token's row: zeros, whatever the one in its place holds
        for (int i = left * GM::RB + 16 * (int)threadIdx.x; i < ROWS; i += 2048 * NW) {
            *(i32x4*)(buf + i) = i32x4{0, 0, 0, 0};
            *(i32x4*)(buf + ROWS + i) = i32x4{0, 0, 0, 0};
        }
        for (int i = left * VP + 16 * (int)threadIdx.x; i < kChunk * VP; i += 2048 * NW) *(i32x4*)(buf + VAT + i) = i32x4{0, 0, 0, 0};
        meet();
    };
    auto transposed = [&](const unsigned char* at) {
        return __builtin_bit_cast(bf16x4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((s16x4 __attribute__((address_space(3)))*)at));
    };
    auto in_turn = [&](auto&& chunk) {
        for (int t0 = 0, turn = 0; t0 < n; t0 += 3 * kChunk, turn ^= 1) {
            chunk(buf0, buf2, t0, turn);
            if (t0 + kChunk < n) chunk(buf1, buf0, t0 + kChunk, turn ^ 1);
            if (t0 + 2 * kChunk < n) chunk(buf2, buf1, t0 + 2 * kChunk, turn);
        }
    };

    if (warp < NW) {                                          // the state and the strengths
        float* st = state + ((size_t)seq_slot[b] * H + h) * (size_t)DK * V + (size_t)(8 * g) * V + col;
        const bool fresh = seq_pos0[b] == 0;
        const float skip = DELTA ? 0.f : skip_w[h];
        f32x4 S[KS][2];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) S[ks][e >> 2][e & 3] = fresh ? 0.f : st[(size_t)(32 * ks + e) * V];
        // columns of K for K^T W by the transposing read: rows 4 g.., of 32 keys those 8 i + 0..3, i = 0..3
        const int c_at = GM::at(4 * g + (l15 >> 2), l15 & 3);
        in_turn([&](unsigned char* buf, unsigned char*, int t0, int turn) __attribute__((always_inline)) {
            meet();
            if (n - t0 < kChunk) clear_absent(buf, n - t0);
            const unsigned char* prep = buf + PREP;
            // everything that the chunk brings is asked for before the first product
            bf16x8 kf[KS][2], qf[KS][2];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) {
                    if (DELTA) kf[ks][tb] = *(const bf16x8*)(buf + (r_at ^ (64 * ks)) + 16 * GM::RB * tb);
                    else qf[ks][tb] = *(const bf16x8*)(buf + ROWS + (r_at ^ (64 * ks)) + 16 * GM::RB * tb);
                }
            const f32x4* coef = (const f32x4*)(prep + PR::kCoefAt) + g;
            f32x4 beta[2], ck[2], cq[2], left[2];
            bf16x4 vx[2];
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                vx[tb] = transposed(buf + VAT + v_at + 16 * VP * tb);
                beta[tb] = coef[kBeta / 4 + 4 * tb];
                if (DELTA) ck[tb] = coef[kOldKey / 4 + 4 * tb];
                cq[tb] = coef[kOldQuery / 4 + 4 * tb];
                left[tb] = coef[kLeft / 4 + 4 * tb];
            }
            const float end = *(const float*)(prep + PR::kEndAt);
            Lower N;
            if (DELTA) N.read(prep + PR::kTAt, lane);
            float w[8], wd[8];
            f32x4 kb[2] = {zeros4(), zeros4()}, kl[2] = {zeros4(), zeros4()}, qb[2] = {zeros4(), zeros4()}, qc[2] = {zeros4(), zeros4()},
                  ql[2] = {zeros4(), zeros4()};
            Terms s[KS];                                      // the wave's columns of the state, 32 keys at a time
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
                float x[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) x[e] = S[ks][e >> 2][e & 3];
                s[ks] = cut8(x, minus);
                if (DELTA) {
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb) kl[tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks][tb], s[ks].v[2], kl[tb], 0, 0, 0);
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb) kb[tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks][tb], s[ks].v[0], kb[tb], 0, 0, 0);
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb) kl[tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kf[ks][tb], s[ks].v[1], kl[tb], 0, 0, 0);
                }
            }
            if (DELTA)
#pragma unroll
                for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                    for (int tb = 0; tb < 2; ++tb) qf[ks][tb] = *(const bf16x8*)(buf + ROWS + (r_at ^ (64 * ks)) + 16 * GM::RB * tb);
#pragma unroll
            for (int r = 0; r < 8; ++r) {
                const float v = to_f(vx[r >> 2][r & 3]);
                w[r] = beta[r >> 2][r & 3] * v;
                if (!DELTA) wd[r] = left[r >> 2][r & 3] * v;
            }
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) ql[tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[ks][tb], s[ks].v[2], ql[tb], 0, 0, 0);
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) {
                    f32x4& q = ks < KS / 2 ? qb[tb] : qc[tb];
                    q = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[ks][tb], s[ks].v[0], q, 0, 0, 0);
                }
#pragma unroll
                for (int tb = 0; tb < 2; ++tb) ql[tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[ks][tb], s[ks].v[1], ql[tb], 0, 0, 0);
            }
            bf16x8 kt[KS][2];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int half = 0; half < 2; ++half)
                    kt[ks][half] = __builtin_shufflevector(transposed(buf + (c_at ^ (64 * ks)) + 8 * half),
                                                           transposed(buf + (c_at ^ (64 * ks)) + 8 * half + 16 * GM::RB), 0, 1, 2, 3, 4, 5, 6, 7);
            if (DELTA) {
#pragma unroll
                for (int r = 0; r < 8; ++r) w[r] -= ck[r >> 2][r & 3] * (kb[r >> 2][r & 3] + kl[r >> 2][r & 3]);
                auto solve = [&](float* x) {
                    f32x4 big[2], more, small[2];
                    N.times(split8(x, minus), big, more, small);
#pragma unroll
                    for (int r = 0; r < 8; ++r) x[r] += (r < 4 ? big[0][r & 3] : big[1][r & 3] + more[r & 3]) + small[r >> 2][r & 3];
                };
                float r0[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) r0[r] = w[r];
                solve(w);
                if (spoiled(w)) {                             // (a row that is not finite leaves none of its column finite)
                    const int first = first_spoiled(r0, g);
                    solve(r0);
#pragma unroll
                    for (int r = 0; r < 8; ++r) w[r] = (r & 3) + 16 * (r >> 2) + 4 * g >= first ? __builtin_nanf("") : r0[r];
                }
            }
#pragma unroll
            for (int tb = 0; tb < 2; ++tb) {
                f32x4* to = &given[turn][wave][tb][lane];
                to[0] = f32x4{w[4 * tb], w[4 * tb + 1], w[4 * tb + 2], w[4 * tb + 3]};
                if (DELTA) {
                    to[128] = cq[tb] * (qb[tb] + (qc[tb] + ql[tb]));
                } else {
                    // (in double, here and where P W is added: in float32 the error was 1 to 5 % above the token-by-token walk's)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const double z = (double)cq[tb][e] * ((double)qb[tb][e] + (double)qc[tb][e] + (double)ql[tb][e]) +
                                         (double)skip * (double)to_f(vx[tb][e]);
                        to[128][e] = (float)z;
                        to[256][e] = (float)(z - (double)(float)z);
                    }
                }
            }
#pragma unroll
            for (int r = 0; r < 8; ++r)
                if (DELTA) wd[r] = left[r >> 2][r & 3] * w[r];
            const Terms d = cut8(wd, minus);
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    // (one sum from the smallest terms up: with the leading ones in a sum of their own, as above, the state was up to 2 % further
                    // from float64, and the walk 2 to 5 % slower)
                    f32x4 sum = zeros4();
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt[ks][half], d.v[2], sum, 0, 0, 0);
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt[ks][half], d.v[1], sum, 0, 0, 0);
                    sum = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kt[ks][half], d.v[0], sum, 0, 0, 0);
#pragma unroll
                    for (int e = 0; e < 4; ++e) S[ks][half][e] = end * S[ks][half][e] + sum[e];
                }
        });
        meet();
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int e = 0; e < 8; ++e) st[(size_t)(32 * ks + e) * V] = S[ks][e >> 2][e & 3];
        return;
    }

    // the loads and the results
    const bf16_t *ks0 = rows + (size_t)q0 * stride + k_off + (size_t)gr * DK, *qs0 = rows + (size_t)q0 * stride + q_off + (size_t)gr * DK;
    const bf16_t* vs0 = rows + (size_t)q0 * stride + v_off + (size_t)h * V + blockIdx.z * 16 * NW;
    // a chunk's K, Q, V (rows past the end: the last one, cleared before use) and prepared part: 1 KB pieces to the waves in turn
    int row_of[KQ], ch_of[KQ];
    size_t off_of[KQ];
#pragma unroll
    for (int j = 0; j < KQ; ++j) {
        const int c = 64 * (NW * j + wave) + lane;
        row_of[j] = c / GM::CH;
        ch_of[j] = 8 * ((c % GM::CH) ^ GM::swz(row_of[j]));
        off_of[j] = (size_t)row_of[j] * stride + ch_of[j];
    }
    const int v_row = (64 * wave + lane) / (2 * NW), v_ch = 8 * (lane % (2 * NW));
    auto load_chunk = [&](unsigned char* buf, int t0) {
        const unsigned char* prep = work + prepared_at(q0, b, t0 / kChunk, h, H) + 1024 * wave + 16 * lane;
        const bool whole = t0 + kChunk <= n;
        __builtin_amdgcn_global_load_lds((gvoid*)(vs0 + (size_t)min(t0 + v_row, n - 1) * stride + v_ch),
                                         (lvoid*)(buf + VAT + 1024 * wave), 16, 0, 0);
#pragma unroll
        for (int j = 0; j < KQ; ++j) {
            const size_t off = whole ? (size_t)t0 * stride + off_of[j] : (size_t)min(t0 + row_of[j], n - 1) * stride + ch_of[j];
            const int at = 1024 * (NW * j + wave);
            __builtin_amdgcn_global_load_lds((gvoid*)(ks0 + off), (lvoid*)(buf + at), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((gvoid*)(qs0 + off), (lvoid*)(buf + ROWS + at), 16, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < PR::kPieces / NW; ++j)
            __builtin_amdgcn_global_load_lds((gvoid*)(prep + 1024 * NW * j), (lvoid*)(buf + PREP + 1024 * (NW * j + wave)), 16, 0, 0);
        if (PR::kPieces % NW != 0 && wave < PR::kPieces % NW) {
            constexpr int J = PR::kPieces / NW;
            __builtin_amdgcn_global_load_lds((gvoid*)(prep + 1024 * NW * J), (lvoid*)(buf + PREP + 1024 * (NW * J + wave)), 16, 0, 0);
        }
    };
    // what the chunk leaves in registers for its results, which are worked out behind the next meeting
    Lower P;
    auto results = [&](int t0, bool whole, int turn) {
        float w[8];
        f32x4 q[2][2];
#pragma unroll
        for (int tb = 0; tb < 2; ++tb) {
            const f32x4* from = &given[turn][wave][tb][lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) w[4 * tb + e] = from[0][e];
#pragma unroll
            for (int i = 0; i < (DELTA ? 1 : 2); ++i) q[i][tb] = from[128 * (i + 1)];
        }
        int first = kChunk;
        if (spoiled(w)) first = first_spoiled(w, g);
        f32x4 pb[2], pm, pl[2];
        P.times(split8(w, minus), pb, pm, pl);
        float* orow = o + ((size_t)(q0 + t0 + 4 * g) * H + h) * V + col;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            const int i = r & 3, tb = r >> 2, t = i + 16 * tb;
            float y;
            if (DELTA) {
                y = q[0][tb][i] + (r < 4 ? pb[0][i] + pl[0][i] : pb[1][i] + (pm[i] + pl[1][i]));
            } else {
                double z = ((double)q[0][tb][i] + (double)q[1][tb][i]) + ((double)pb[tb][i] + (double)pl[tb][i]);
                if (r >= 4) z += (double)pm[i];
                y = (float)z;
            }
            if (t + 4 * g >= first) y = __builtin_nanf("");
            if (whole || t0 + 4 * g + t < n) orow[(size_t)t * H * V] = y;
        }
    };
    load_chunk(buf0, 0);
    if (n > kChunk) load_chunk(buf1, kChunk);
    in_turn([&](unsigned char* buf, unsigned char* nxt, int t0, int turn) __attribute__((always_inline)) {
        const int left = n - t0;
        // the chunk has landed: what was asked for behind it are the next chunk's loads and, from the third chunk on, eight rows of results
        if (t0 > kChunk && left > kChunk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS + 8) : "memory");
        else if (t0 > kChunk) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        else if (left > kChunk) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(LOADS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        meet();
        if (left < kChunk) clear_absent(buf, left);
        if (left > 2 * kChunk) load_chunk(nxt, t0 + 2 * kChunk);      // (its buffer was last read in front of this meeting)
        if (t0 > 0) results(t0 - kChunk, true, turn ^ 1);
        const unsigned char* prep = buf + PREP;
        P.read(prep, lane);
    });
    meet();
    const int last = (n - 1) / kChunk;
    results(last * kChunk, false, last & 1);
}

template <bool DELTA>
static void launch_chunks(const void* rows_, int64_t stride, int q_off, int k_off, int v_off, const GateArgs<bf16_t>& ga, void* work, float* state, const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, float* o,
                          int B, int H, int G, int D, int V, int max_q, hipStream_t s) {
    const bf16_t* rows = (const bf16_t*)rows_;
    // Four waves of columns share a chunk's K, Q and prepared part, two have a SIMD each and LDS to themselves: where every CU has at most one
    // workgroup of two, those (us of a call, 16 heads, portions of 1000 tokens, two / four: 128 x 128 delta 1 portion 59 / 62, state space 47 / 57).
    // Beyond: with 128 keys a CU has LDS for one workgroup of either, and four take half the rounds (128 x 64, 12 portions, delta 124 / 88, state
    // space 103 / 78).  With 64 keys two workgroups of two waves fit and take turns on its SIMDs, each loading its own K, Q and prepared part, where
    // four waves have those once (64 x 64: 8 portions 59 / 65 and 46 / 58, 12 portions 83 / 73 and 65 / 61, 16 portions 90 / 80 and 70 / 67); from
    // 513 to 768 workgroups of two, one round and a half of the four's, those are ahead once more (20 portions 121 / 123 and 96 / 106), beyond
    // that behind (32 portions 171 / 152 and 132 / 129).
    const int nw = V % 64 == 0 && (int64_t)B * H * (V / 32) > 256 ? 4 : 2;
    const dim3 pg((unsigned)((max_q + kChunk - 1) / kChunk), (unsigned)B, (unsigned)H), wg((unsigned)B, (unsigned)H, (unsigned)(V / (16 * nw)));
#define HM_CHUNKS(DK, NW)                                                                                                              \
    do {                                                                                                                           \
        hipLaunchKernelGGL((outer_chunk_prepare_kernel<DK, DELTA>), pg, dim3(64), 0, s, rows, stride, q_off, k_off, ga, qstart,      \
                           (unsigned char*)work, H, G);                                                                            \
        hipLaunchKernelGGL((outer_chunk_walk_kernel<DK, NW, DELTA>), wg, dim3(128 * NW), 0, s, rows, stride, q_off, k_off, v_off,             \
                           (const unsigned char*)work, ga.skip, state, qstart, seq_pos0, seq_slot, o, H, G, V);                    \
    } while (0)
    if (nw == 4) { if (D == 64) HM_CHUNKS(64, 4); else HM_CHUNKS(128, 4); }
    else { if (D == 64) HM_CHUNKS(64, 2); else HM_CHUNKS(128, 2); }
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
                            state, qstart, seq_pos0, seq_slot, o, B, T, H, G, D, V, max_q < 1 ? max_q : 1);
    if (!rc) rc = chunk_args_bad("hm_gated_delta_chunks", stride, q_off, k_off, v_off, rows, work, B, T, D, V);
    if (rc) return rc;
    if (B == 0 || T == 0 || max_q == 0) return HM_OK;
    GateArgs<bf16_t> ga = {(const bf16_t*)pre, pre_stride, b_off, a_off, A, dt_bias, nullptr, unit_eps, q_scale};
    launch_chunks<true>(rows, stride, q_off, k_off, v_off, ga, work, state, qstart, seq_pos0, seq_slot, o, B, H, G, D, V, max_q, as_stream(stream));
    HM_CHECK_LAUNCH("hm_gated_delta_chunks");
    return HM_OK;
}

extern "C" int hm_state_space_chunks(const void* rows, int64_t stride, int x_off, int b_off, int c_off, const void* pre, int64_t pre_stride,
                                     int dt_off, const float* A, const float* dt_bias, const float* D, float* gates, void* work,
                                     float* state, const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, float* y, int B,
                                     int64_t T, int H, int G, int N, int V, int max_q, void* stream) {
    int rc = outer_args_bad("hm_state_space_chunks", stride, c_off, b_off, x_off, pre_stride, 0, dt_off, rows, pre, A, dt_bias, gates,
                            state, qstart, seq_pos0, seq_slot, y, B, T, H, G, N, V, max_q < 1 ? max_q : 1);
    if (!rc) rc = chunk_args_bad("hm_state_space_chunks", stride, c_off, b_off, x_off, rows, work, B, T, N, V);
    if (rc) return rc;
    if (B > 0 && T > 0 && !D) { set_error("hm_state_space_chunks: bad argument"); return HM_EINVAL; }
    if (B == 0 || T == 0 || max_q == 0) return HM_OK;
    GateArgs<bf16_t> ga = {(const bf16_t*)pre, pre_stride, 0, dt_off, A, dt_bias, D, 0.f, 1.f};
    launch_chunks<false>(rows, stride, c_off, b_off, x_off, ga, work, state, qstart, seq_pos0, seq_slot, y, B, H, G, N, V, max_q, as_stream(stream));
    HM_CHECK_LAUNCH("hm_state_space_chunks");
    return HM_OK;
}
