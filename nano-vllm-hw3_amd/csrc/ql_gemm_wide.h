// Prefill-sized fused dequant GEMM for gfx950:  y[M,N] = x[M,K] . dequant(qw[N,K])^T  on tiles of 32 MT x 256   (kernel template)
//
// Four waves side by side: a wave owns all 32 MT rows and 64 weight columns (two strips of 32), so that an activation fragment read
// from LDS serves two matrix products.  (One strip per wave, as in the tiles of ql_gemm_kernel.h, needs 16 bytes per lane from LDS
// for every 32 cycles of the matrix unit, which is all that LDS delivers to four SIMDs.)  Two workgroups share a CU, and one's
// barriers, first loads and epilogue run under the other's products: up to 256 registers per lane, 128 of them sums.
//   * Activations go from global memory straight to LDS (16 bytes per lane, no registers in between), 256 bytes of a row per step
//     (128 k in 16 bits, 256 k in 8), two buffers: the loads of step t + 1 are issued behind the one barrier of step t.  16-byte
//     chunk c of row r lies at place c ^ (r & 15): a lane reads its row's chunk, and 16 rows hit 16 places of the 256-byte bank row.
//   * Weights go from global memory to the registers of the wave that multiplies them (16 bytes per lane and 32-k product), RW
//     products ahead: a register is loaded again as soon as its weights are widened.  They are widened once for 32 MT rows.
//   * Per-group sums take a second set of accumulators, so 96 rows are the most there, and weights are loaded 64 k ahead.
//   * Tiles are dealt to the eight dies in contiguous runs of an order that goes through panels of eight row tiles, so that the
//     tiles a die has at hand form a square and its L2 sees activations and weights several times.
// The k order of a sum is that of the other tiles: results agree with theirs bit for bit (per-group scales: fused multiply-adds of
// the same group sums in the same order).
//
// Bound by the matrix cores in 16 bits (1.15 to 1.2 PFLOP/s, what a library product of 8192 reaches too), by the vector unit beside
// them with int8 groups (widening 50 %, folds 25 % of the time), by both and LDS in 8 bits.  4099 rows, Qwen3-4B shapes,
// microseconds of the 128 x 256 tile with one strip per wave / here (without the waits by position, see load_a): weight-only int8 qkv 158 / 134, o 113 / 84, gate_up 398 / 349,
// down 223 / 191; groups of 128 178 / 154, 136 / 97, 500 / 405, 269 / 218; fp8 x fp8 106 / 71, 82 / 44, 311 / 180, 158 / 93.
#pragma once
#include "ql_gemm_kernel.h"

namespace ql {

constexpr int kWidePanel = 8;                 // row tiles of a panel

// FG: 32-k products behind which a group's sum is folded into the total with its scale (0: no groups)
template <int ACT, bool FP8W, int FG, int MT, bool ROPE>
__global__ __launch_bounds__(256, 2) void qgemm_wide_kernel(const GemmParams p) {
    constexpr bool INT = ACT == ACT_I8, GROUP = FG > 0;
    constexpr int AB = ACT == ACT_BF16 ? 2 : 1, KS = 256 / AB, SUB = KS / 32, BM = 32 * MT, BUF = BM * 256;
    constexpr int NA = 2 * MT;                                // 1 KB pieces of activations a wave loads per step
    constexpr int FS = GROUP ? SUB / (FG + !FG) : 0;                  // folds per step
    using acc_t = typename std::conditional<INT, i32x16, f32x16>::type;
    typedef __attribute__((address_space(3))) void lvoid;
    typedef __attribute__((address_space(1))) const unsigned char* gbytes;    // (global from the start: uniform base + 32-bit offset)
    __shared__ __attribute__((aligned(1024))) unsigned char buf0[BUF];
    __shared__ __attribute__((aligned(1024))) unsigned char buf1[BUF];
    __shared__ float sxs[ACT == ACT_BF16 ? 1 : BM];

    const unsigned C = (unsigned)p.ntile_n, R = ((unsigned)p.M + BM - 1) / BM, total = C * R;
    const unsigned per = (total + 7) >> 3, lin = (blockIdx.x & 7u) * per + (blockIdx.x >> 3);
    if ((blockIdx.x >> 3) >= per || lin >= total) return;
    const unsigned panel = lin / (kWidePanel * C), in = lin - panel * kWidePanel * C;
    const unsigned h = min((unsigned)kWidePanel, R - panel * kWidePanel);
    const unsigned bx = in / h, by = panel * kWidePanel + (in - bx * h);

    const int lane = threadIdx.x & 63, l31 = lane & 31, lh = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int m0 = (int)by * BM, n0 = (int)bx * 256 + wave * 64;
    const int steps = p.K / KS;                               // (host: K % KS == 0)

    // activations: piece i = rows 8 MT wave + 4 i .. + 3 of the tile (rows past M: the last one, never stored)
    unsigned aoff[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int row = 8 * MT * wave + 4 * i + (lane >> 4);
        aoff[i] = (unsigned)min(m0 + row, p.M - 1) * (unsigned)p.K * AB + 16u * (unsigned)((lane & 15) ^ (row & 15));
    }
    // (as buffer loads: behind a global load to LDS the compiler lets no load's registers be read before every load has arrived, so the
    // first weights of a step, or the third with groups, waited for activations just asked for.  With waits by position 4099 rows of
    // the Qwen3-4B projections take 857 us with groups of 128, not 914)
    // (the host's pass over a kernel knows no buffer resources)
#ifdef __HIP_DEVICE_COMPILE__
    const auto xrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, (unsigned)p.M * (unsigned)p.K * AB, 0x00020000);
#endif
    auto load_a = [&](unsigned char* buf, int t) {
#ifdef __HIP_DEVICE_COMPILE__
#pragma unroll
        for (int i = 0; i < NA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xrsrc, (lvoid*)(buf + (8 * MT * wave + 4 * i) * 256), 16, aoff[i], t * 256, 0, 0);
#endif
    };
    // weights: as in the other tiles (columns past N: the last strip or row, never stored)
    const unsigned kmul = p.wtiled ? 32u : 1u;
    unsigned woff[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = n0 + 32 * j;
        woff[j] = p.wtiled ? min((unsigned)(n >> 5), (unsigned)((p.N + 31) / 32 - 1)) * (unsigned)p.K * 32u + (unsigned)lane * 16u
                           : (unsigned)min(n + l31, p.N - 1) * (unsigned)p.K + (unsigned)(16 * lh);
    }
    auto load_w = [&](int k, int j) -> i32x4 {
        asm volatile("" : "+v"(woff[j]));
        return *(const __attribute__((address_space(1))) i32x4*)((gbytes)p.w + (unsigned)k * kmul + woff[j]);
    };
    // a group's scale (group k / group of the lane's columns; 4 N K / group bytes of them, so 32 bits hold an offset)
    unsigned swoff[2];
    if constexpr (GROUP) {
#pragma unroll
        for (int j = 0; j < 2; ++j) swoff[j] = (unsigned)min(n0 + 32 * j + l31, p.N - 1) * (unsigned)(p.K / p.group) * 4u;
    }
    auto load_s = [&](int k, int j) -> float {
        asm volatile("" : "+v"(swoff[j]));
        const unsigned g = __umulhi((unsigned)k >> 5, p.gmagic);   // (groups of 64 and more: never 0)
        return *(const __attribute__((address_space(1))) float*)((gbytes)p.sw + 4u * g + swoff[j]);
    };

    acc_t acc[MT][2], accg[GROUP ? MT : 1][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

    constexpr int RW = GROUP ? 2 : 4;                         // 32-k products that weights are loaded ahead
    i32x4 raw[RW][2];
    float sc[GROUP ? FS : 1][2];
    load_a(buf0, 0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < RW; ++s)
#pragma unroll
        for (int j = 0; j < 2; ++j) raw[s][j] = load_w(32 * s, j);
    if constexpr (GROUP) {
#pragma unroll
        for (int f = 0; f < FS; ++f)
#pragma unroll
            for (int j = 0; j < 2; ++j) sc[f][j] = load_s(32 * FG * f, j);
    }
    if constexpr (ACT != ACT_BF16) {
        if ((int)threadIdx.x < BM) sxs[threadIdx.x] = p.sx[min(m0 + (int)threadIdx.x, p.M - 1)];
    }

    // the lane's places: chunk 4 s + 2 lh + q (16 bits) or 2 s + lh (8 bits) of its row in a fragment
    unsigned place[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        const int chunk = ACT == ACT_BF16 ? 4 * (c >> 1) + 2 * lh + (c & 1) : 2 * c + lh;
        place[c] = (unsigned)(l31 * 256 + 16 * (chunk ^ (l31 & 15)));
        asm volatile("" : "+v"(place[c]));                    // (one register each, whatever the buffer and the fragment)
    }
    // One step.  The wait counter is positional: behind a step's activation loads come its 2 SUB weight loads and 2 FS scales, so
    // at most that many outstanding means that the activations are in LDS (the weights of the step behind go on); behind the barrier
    // everybody's are, and nobody reads the other buffer any more.
    constexpr int AFTER = 2 * SUB + 2 * FS;
    static_assert(AFTER < 64, "the wait counter's range");
    auto step = [&](unsigned char* cur, unsigned char* nxt, int t) __attribute__((always_inline)) {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0070 | (AFTER & 15) | (AFTER >> 4) << 14);      // vmcnt(AFTER) lgkmcnt(0)
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int tn = min(t + 1, steps - 1);                 // (past the end: the last step again, which nobody reads)
        load_a(nxt, tn);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        const int kn = tn * KS;
        // the weights of the product RW behind product s of this step
        auto next_w = [&](int s, int j) -> i32x4 { return load_w(s + RW < SUB ? t * KS + 32 * (s + RW) : kn + 32 * (s + RW - SUB), j); };
        if constexpr (ACT == ACT_BF16) {
            if constexpr (GROUP) {
#pragma unroll
                for (int s = 0; s < SUB; ++s) {
                    const int f = s / FG;
#pragma unroll
                    for (int q = 0; q < 2; ++q) {
                        bf16x8 b[2];
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            b[j] = widen8<FP8W>(raw[s % RW][j][2 * q], raw[s % RW][j][2 * q + 1]);
                            if (q == 1) raw[s % RW][j] = next_w(s, j);
                        }
#pragma unroll
                        for (int i = 0; i < MT; ++i) {
                            const bf16x8 a = *(const bf16x8*)(cur + i * 8192 + place[2 * s + q]);
#pragma unroll
                            for (int j = 0; j < 2; ++j) {
                                if (s % FG == 0 && q == 0) accg[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[j], f32x16{}, 0, 0, 0);
                                else accg[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[j], accg[i][j], 0, 0, 0);
                            }
                        }
                        __builtin_amdgcn_sched_barrier(0);
                    }
                    if (s % FG == FG - 1) {
#pragma unroll
                        for (int j = 0; j < 2; ++j) {
                            const float g = sc[f][j];
                            sc[f][j] = load_s(kn + 32 * FG * f, j);
#pragma unroll
                            for (int i = 0; i < MT; ++i)
#pragma unroll
                                for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(accg[i][j][r], g, acc[i][j][r]);
#pragma unroll
                            for (int i = 0; i < MT; ++i) asm volatile("" : "+v"(acc[i][j]));
                        }
                    }
                }
            } else {
                bf16x8 b[2][2][2];
                auto widen = [&](bf16x8 (&o)[2][2], int s) __attribute__((always_inline)) {
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const i32x4 w = raw[s][j];
                        raw[s][j] = next_w(s, j);
                        o[j][0] = widen8<FP8W>(w[0], w[1]);
                        o[j][1] = widen8<FP8W>(w[2], w[3]);
                    }
                };
                widen(b[0], 0);
#pragma unroll
                for (int s = 0; s < SUB; ++s) {
                    if (s + 1 < SUB) widen(b[(s + 1) & 1], s + 1);
#pragma unroll
                    for (int i = 0; i < MT; ++i)
#pragma unroll
                        for (int q = 0; q < 2; ++q) {
                            const bf16x8 a = *(const bf16x8*)(cur + i * 8192 + place[2 * s + q]);
#pragma unroll
                            for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b[s & 1][j][q], acc[i][j], 0, 0, 0);
                        }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        } else if constexpr (INT) {
#pragma unroll
            for (int s = 0; s < SUB; ++s) {
                i32x4 w[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    w[j] = raw[s % RW][j];
                    raw[s % RW][j] = next_w(s, j);
                }
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const i32x4 a = *(const i32x4*)(cur + i * 8192 + place[s]);
#pragma unroll
                    for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, w[j], acc[i][j], 0, 0, 0);
                }
                if (s & 1) __builtin_amdgcn_sched_barrier(0);
            }
        } else {
            typedef int i32x8 __attribute__((ext_vector_type(8)));
#pragma unroll
            for (int s = 0; s < SUB; s += 2) {                // two 32-k products in one of 64 k (unit scales), as the other tiles
                i32x8 w[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const i32x4 e = raw[s % RW][j], o = raw[(s + 1) % RW][j];
                    w[j] = i32x8{e[0], e[1], e[2], e[3], o[0], o[1], o[2], o[3]};
                    raw[s % RW][j] = next_w(s, j);
                    raw[(s + 1) % RW][j] = next_w(s + 1, j);
                }
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const i32x4 e = *(const i32x4*)(cur + i * 8192 + place[s]);
                    const i32x4 o = *(const i32x4*)(cur + i * 8192 + place[s + 1]);
                    const i32x8 a = {e[0], e[1], e[2], e[3], o[0], o[1], o[2], o[3]};
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a, w[j], acc[i][j], 0, 0, 0, 0x7F7F7F7F, 0, 0x7F7F7F7F);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_s_waitcnt(0x0F70);                       // vmcnt(0): fewer loads than AFTER follow the first activations
    {
        int t = 0;
        for (; t + 1 < steps; t += 2) {
            step(buf0, buf1, t);
            step(buf1, buf0, t + 1);
        }
        if (t < steps) step(buf0, buf1, t);
    }

    // ---- epilogue: scales, bias, one rounding; the tile as bf16 through LDS (rows of the first half in buf0, the others in buf1; a
    // half-wave's 32 columns and those of the other half, four rows below, on different banks), then 16 bytes per lane to memory
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    float sw[2] = {1.f, 1.f}, bias[2] = {0.f, 0.f};
    const bool has_bias = p.bias != nullptr;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int n = min(n0 + 32 * j + l31, p.N - 1);
        if constexpr (!GROUP) sw[j] = p.sw[(size_t)n * p.sw_stride];
        if (has_bias) bias[j] = bf16_bits_to_f32(p.bias[n]);
    }
    auto outv = [&](int i, int j, int r) -> bf16_t {
        float v = (float)acc[i][j][r];
        if constexpr (ACT != ACT_BF16) v = __fmul_rn(v, sxs[32 * i + (r & 3) + 8 * (r >> 2) + 4 * lh]);
        if constexpr (!GROUP) v = __fmul_rn(v, sw[j]);
        if (has_bias) {
            if (p.bias_after_round) v = __fadd_rn((float)(bf16_t)v, bias[j]);
            else v = __fadd_rn(v, bias[j]);
        }
        return (bf16_t)v;
    };
    // byte offset of 16-byte chunk c of a row of the image (RS bytes per row), and the half it lies in
    auto half = [&](int row) -> unsigned char* { return row >= BM / 2 ? buf1 : buf0; };
    auto put = [&](int RS, int i, int r, int chunk, unsigned short v) {
        const int rowc = 32 * i + (r & 3) + 8 * (r >> 2);    // (+ 4 lh: the swizzle's bit)
        unsigned char* base = (rowc >= BM / 2 ? buf1 : buf0) + (rowc >= BM / 2 ? rowc - BM / 2 : rowc) * RS;
        *(unsigned short*)(base + 4 * lh * RS + 16 * (chunk ^ (4 * (((rowc >> 2) & 1) ^ lh))) + 2 * (l31 & 7)) = v;
    };
    auto piece = [&](int RS, int row, int chunk) -> u16x8 {
        const unsigned char* base = half(row) + (row >= BM / 2 ? row - BM / 2 : row) * RS;
        return *(const u16x8*)(base + 16 * (chunk ^ (4 * ((row >> 2) & 1))));
    };
    if (!ROPE && p.silu) {
        // strip 0 of a wave is gate, strip 1 up of the same 32 outputs
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                put(256, i, r, 4 * wave + (l31 >> 3), silu_mul_bf16((float)outv(i, 0, r), (float)outv(i, 1, r)));
        __syncthreads();
        const int I = p.N >> 1;
#pragma unroll 4
        for (int e = threadIdx.x; e < BM * 16; e += 256) {
            const int row = e >> 4, c = e & 15, col = (int)bx * 128 + 8 * c;
            if (m0 + row < p.M && col < I) *(u16x8*)(p.y + (size_t)(m0 + row) * I + col) = piece(256, row, c);
        }
        return;
    }
    // (ROPE: the tile's columns are two whole 128-wide heads, eight lanes per (row, head), as in the other tiles.  A thread has one head
    // and 2 MT rows; their cache slots and positions are requested in front of the image, their cosines and sines behind it, all at
    // once: one row behind the other, each a chain of two trips to memory, took 6076 x 4096 outputs of 1024 k 85 us instead of 70)
    constexpr int NR = ROPE ? 2 * MT : 1;
    const int rc = threadIdx.x & 7, rhead = (int)bx * 2 + (((int)threadIdx.x >> 3) & 1), rrow = (int)threadIdx.x >> 4;
    int64_t rpos[NR];
    RopePre pre[NR];
    if constexpr (ROPE) {
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int t = min(m0 + rrow + 16 * i, p.M - 1);
            pre[i].slot = p.rope.slot_mapping ? p.rope.slot_mapping[t] : -1;
            rpos[i] = p.rope.positions ? p.rope.positions[t] : (int64_t)t;
        }
    }
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                put(512, i, r, 8 * wave + 4 * j + (l31 >> 3), __builtin_bit_cast(unsigned short, outv(i, j, r)));
    if constexpr (ROPE) {
        const unsigned short* nw = rhead < p.rope.Hq ? p.rope.qw : p.rope.kw;
        u16x8 w1 = {0, 0, 0, 0, 0, 0, 0, 0}, w2 = w1;
        if (nw) { w1 = *(const u16x8*)(nw + 8 * rc); w2 = *(const u16x8*)(nw + 64 + 8 * rc); }
#pragma unroll
        for (int i = 0; i < NR; ++i) {                        // (value heads too, which leave them unused)
            const float* cs = p.rope.cos_sin + rpos[i] * 128 + 8 * rc;
            pre[i].w1 = w1;
            pre[i].w2 = w2;
#pragma unroll
            for (int e = 0; e < 8; ++e) { pre[i].c[e] = cs[e]; pre[i].sn[e] = cs[64 + e]; }
        }
    }
    __syncthreads();
    if constexpr (ROPE) {
        if (rhead >= p.rope.Hq + 2 * p.rope.Hkv) return;
#pragma unroll
        for (int i = 0; i < NR; ++i) {
            const int row = rrow + 16 * i;
            if (m0 + row >= p.M) break;                       // (whole 8-lane groups leave together)
            rope_store_piece(piece(512, row, 16 * (rhead & 1) + rc), piece(512, row, 16 * (rhead & 1) + 8 + rc), m0 + row, rhead, 8 * rc, p.rope, pre[i]);
        }
    } else {
#pragma unroll 4
        for (int e = threadIdx.x; e < BM * 32; e += 256) {
            const int row = e >> 5, c = e & 31, col = (int)bx * 256 + 8 * c;
            if (m0 + row < p.M && col < p.N) *(u16x8*)(p.y + (size_t)(m0 + row) * p.N + col) = piece(512, row, c);
        }
    }
}

template <int ACT, bool FP8W, int FG, bool ROPE>
kern_t pick_wide_impl(int mt) {
    switch (mt) {
        case 2: return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 2, ROPE>;
        case 3: return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 3, ROPE>;
        case 4: if constexpr (FG == 0) return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 4, ROPE>; break;
    }
    return nullptr;
}

template <bool FP8W, bool ROPE>
kern_t pick_wide_w16(int mt, int group) {
    if (group == 0) return pick_wide_impl<ACT_BF16, FP8W, 0, ROPE>(mt);
    return group == 64 ? pick_wide_impl<ACT_BF16, FP8W, 2, ROPE>(mt) : pick_wide_impl<ACT_BF16, FP8W, 4, ROPE>(mt);
}

}  // namespace ql
