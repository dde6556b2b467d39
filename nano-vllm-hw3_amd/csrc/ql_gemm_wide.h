// Prefill-sized fused dequant GEMM for gfx950:  y[M,N] = x[M,K] . dequant(qw[N,K])^T  on tiles of 32 MT x 256   (kernel template)
//
// Four waves side by side: a wave owns all 32 MT rows and 64 weight columns (two strips of 32), so that an activation fragment read
// from LDS serves two matrix products.  (One strip per wave, as in the tiles of ql_gemm_kernel.h, needs 16 bytes per lane from LDS
// for every 32 cycles of the matrix unit, which is all that LDS delivers to four SIMDs.)  Two workgroups share a CU, and one's
// barriers, first loads and epilogue run under the other's products: up to 256 registers per lane, 128 of them sums.
//   * Activations go from global memory straight to LDS (16 bytes per lane, no registers in between), 256 bytes of a row per step
//     (128 k in 16 bits, 256 k in 8), two buffers.  8 bits: the loads of step t + 1 are issued behind the one barrier of step t.  16 bits:
//     those of step t + 2 behind the barrier in front of step t's last product, which is held in registers by then (step16).  16-byte
//     chunk c of row r lies at place c ^ (r & 15): a lane reads its row's chunk, and 16 rows hit 16 places of the 256-byte bank row.
//   * Weights go from global memory to the registers of the wave that multiplies them (16 bytes per lane and 32-k product), RW
//     products ahead: a register is loaded again as soon as its weights are widened.  They are widened once for 32 MT rows.
//   * Per-group sums take a second set of accumulators, so 96 rows are the most there, and there weights are loaded 64 k ahead (64 rows
//     have registers for 128 k: groups of 128, one tile per CU, 0.84 x the time of 64 k).  With nothing beside it on its CU a workgroup
//     takes a weight's way from memory for every 64 k, and has twice the registers: 96 rows of at most one tile per CU have weights 128 k
//     ahead too where that pays (wide_ring.h; not groups of 64 in int8: the compiler moves a fold's sums through accumulation registers, 1.07).
//   * Tiles are dealt to the eight dies in contiguous runs of an order that goes through panels of eight row tiles, so that the
//     tiles a die has at hand form a square and its L2 sees activations and weights several times.
// The k order of a sum is that of the other tiles: results agree with theirs bit for bit (per-group scales: fused multiply-adds of
// the same group sums in the same order).
//
// Bound by the matrix cores in 16 bits and by the power they take (random operands run at 1.7 to 2.0 GHz of 2.4; 1.15 to 1.25 PFLOP/s, where a
// library product in bf16, which widens nothing, reaches 1.2 at these shapes and 1.5 to 1.6 at 8192 x 8192 of 8192 k), by the vector unit beside them
// with int8 groups, by both and LDS in 8 bits.  4099 rows, Qwen3-4B shapes,
// microseconds of the 128 x 256 tile with one strip per wave / of this one with every product's weights widened in front of its matrix
// instructions: weight-only int8 qkv 158 / 134, o 113 / 84, gate_up 398 / 349, down 223 / 191; groups of 128 178 / 154, 136 / 97, 500 / 405,
// 269 / 218; fp8 x fp8 106 / 71, 82 / 44, 311 / 180, 158 / 93.  With step16, all four and groups of 128: 811, not 859.  256 to 8192 rows of
// the Qwen3 shapes and others, times the figure before: 96 rows of a tile 0.90 in int8, 0.89 in fp8, 128 rows 0.95 and 0.94, groups of
// 128 on 64 rows 0.87 (0.64 at best), on 96 rows 0.94.
#pragma once
#include "ql_gemm_kernel.h"
#include "step_window.h"

namespace ql {

constexpr int kWidePanel = 8;                 // row tiles of a panel

// FG: 32-k products behind which a group's sum is folded into the total with its scale (0: no groups).  ALONE: at most one workgroup for every CU
template <int ACT, bool FP8W, int FG, int MT, bool ROPE, bool ALONE = false>
__global__ __launch_bounds__(256, ALONE ? 1 : 2) void qgemm_wide_kernel(const GemmParams p) {
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

    // activations: piece i = rows 8 MT wave + 4 i .. + 3 of the tile (rows past M lie behind the resource's end: zeros, never stored)
    const int arow = 8 * MT * wave + (lane >> 4);
    // (a row is a multiple of 256 bytes; 8 MT wave is one of 8 rows, so that 4 i only changes bits 2 and 3 of a row's number)
    unsigned abase = (unsigned)(m0 + arow) * (unsigned)p.K * AB + 16u * (unsigned)((lane & 15) ^ (arow & 15));
    auto aoff = [&](int i) -> unsigned {
        return (abase ^ (16u * ((unsigned)((8 * MT * wave + 4 * i) ^ (8 * MT * wave)) & 12u))) + (unsigned)(4 * i) * (unsigned)p.K * AB;
    };
    // (8 bits have registers for the places, and are up to 6 % faster with them: 6000 x 4096 of 2048 k in fp8 66 us, not 70)
    constexpr bool KEPT = ACT != ACT_BF16;
    unsigned akept[KEPT ? NA : 1];
#pragma unroll
    for (int i = 0; i < (KEPT ? NA : 0); ++i) akept[i] = aoff(i);
    // (as buffer loads: behind a global load to LDS the compiler lets no load's registers be read before every load has arrived, so the
    // first weights of a step, or the third with groups, waited for activations just asked for.  With waits by position 4099 rows of
    // the Qwen3-4B projections take 857 us with groups of 128, not 914)
    // (the host's pass over a kernel knows no buffer resources)
#ifdef __HIP_DEVICE_COMPILE__
    const unsigned xbytes = (unsigned)p.M * (unsigned)p.K * AB;
#endif
    auto load_a = [&](unsigned char* buf, int t) {
        if constexpr (!KEPT) asm volatile("" : "+v"(abase));  // (worked out anew at every step, or each would keep its register)
#ifdef __HIP_DEVICE_COMPILE__
        // (a step past the last one finds an empty resource, at its start: nothing is read; 8 bits have none)
        const StepWindow win = KEPT ? StepWindow{xbytes, t * 256u} : step_window(t, steps, 256u, xbytes);
        const auto xrsrc = __builtin_amdgcn_make_buffer_rsrc((void*)p.x, 0, win.bytes, 0x00020000);
#pragma unroll
        for (int i = 0; i < NA; ++i)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xrsrc, (lvoid*)(buf + (8 * MT * wave + 4 * i) * 256), 16, KEPT ? akept[i] : aoff(i), win.at, 0, 0);
#endif
    };
    // weights: as in the other tiles (strips past N: the last one, never stored; N is a multiple of 32).  A lane's place in a strip in a
    // register, whatever the strip; what is uniform goes into the address
    const unsigned kmul = p.wtiled ? 32u : 1u;
    unsigned wplace = p.wtiled ? (unsigned)lane * 16u : (unsigned)l31 * (unsigned)p.K + (unsigned)(16 * lh);
    unsigned col[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) col[j] = (unsigned)min(n0 + 32 * j, p.N - 32);
    unsigned wkept[2] = {col[0] * (unsigned)p.K + wplace, col[1] * (unsigned)p.K + wplace};
    auto load_w = [&](int k, int j) -> i32x4 {
        if constexpr (KEPT) {
            asm volatile("" : "+v"(wkept[j]));
            return *(const __attribute__((address_space(1))) i32x4*)((gbytes)p.w + (unsigned)k * kmul + wkept[j]);
        }
        asm volatile("" : "+v"(wplace));
        return *(const __attribute__((address_space(1))) i32x4*)((gbytes)p.w + (col[j] * (unsigned)p.K + (unsigned)k * kmul) + wplace);
    };
    // a group's scale (group k / group of the lane's columns; 4 N K / group bytes of them, so 32 bits hold an offset)
    unsigned splace = GROUP ? (unsigned)l31 * (unsigned)(p.K / p.group) * 4u : 0u;
    auto load_s = [&](int k, int j) -> float {
        asm volatile("" : "+v"(splace));
        const unsigned g = __umulhi((unsigned)k >> 5, p.gmagic);   // (groups of 64 and more: never 0)
        return *(const __attribute__((address_space(1))) float*)((gbytes)p.sw + 4u * (g + col[j] * (unsigned)(p.K / p.group)) + splace);
    };

    acc_t acc[MT][2], accg[GROUP ? MT : 1][2];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0;

    constexpr int RW = GROUP && MT > 2 && !ALONE ? 2 : 4;     // 32-k products that weights are loaded ahead
    i32x4 raw[RW][2];
    // a group's scales; groups of 64 on 64 rows are over before one group's way from memory: theirs are asked for a step ahead
    constexpr int SD = GROUP && FG == 2 && MT == 2 ? 2 : 1;
    float sc[SD][2] = {};
    load_a(buf0, 0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < RW; ++s)
#pragma unroll
        for (int j = 0; j < 2; ++j) raw[s][j] = load_w(32 * s, j);
    if constexpr (ACT != ACT_BF16) {
        if ((int)threadIdx.x < BM) sxs[threadIdx.x] = p.sx[min(m0 + (int)threadIdx.x, p.M - 1)];
    }

    // the lane's places, 8 bits: chunk 2 s + lh of its row in a fragment
    unsigned place[8];
#pragma unroll
    for (int c = 0; c < (ACT == ACT_BF16 ? 0 : 8); ++c) {
        const int chunk = 2 * c + lh;
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
        if constexpr (INT) {
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
    // 16 bits: a step is 2 SUB products of 16 k, 2 MT matrix instructions each; between them the widening of the next product's weights and
    // the reads of its activations, each into the registers that the last of them has left, so that one wave of a SIMD keeps the matrix unit
    // as busy as two (a wave issues up to five vector instructions in the 32 cycles of a matrix one; with all of a product's in front of its
    // matrix instructions, two waves took the time of both units added up).  In front of a step's last product its activations are all
    // read: the barrier stands there, behind it the next step's are in LDS and read, and those of the step after next take their place.
    bf16x8 ga[MT], gb[2][2];
    auto step16 = [&](unsigned char* cur, unsigned char* nxt, int t) __attribute__((always_inline)) {
        const int kn = min(t + 1, steps - 1) * KS;
        auto next_w = [&](int s, int j) -> i32x4 { return load_w(s + RW < SUB ? t * KS + 32 * (s + RW) : kn + 32 * (s + RW - SUB), j); };
        int tid = threadIdx.x;                                // (worked out anew, as the activations' places: registers are short)
        asm volatile("" : "+v"(tid));
        // (chunk 4 s + 2 lh + q of the row lies at `at` ^ 16 (4 s + q))
        const unsigned at = (unsigned)((tid & 31) * 256 + 16 * ((tid >> 4 & 2) ^ (tid & 15)));
#pragma unroll
        for (int p = 0; p < 2 * SUB; ++p) {
            const int s = p >> 1, q = p & 1, pn = (p + 1) % (2 * SUB), sn = pn >> 1;
            const bool last = p == 2 * SUB - 1, fold = GROUP && p % (2 * (FG + !FG)) == 0;
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            if (last) {                                       // vmcnt(AFTER) lgkmcnt(0), as below
                __builtin_amdgcn_s_waitcnt(0x0070 | (AFTER & 15) | (AFTER >> 4) << 14);
                __builtin_amdgcn_s_barrier();
                asm volatile("" ::: "memory");
                __builtin_amdgcn_sched_barrier(0);
                load_a(cur, t + 2);
            }
            const unsigned char* from = last ? nxt : cur;
            const unsigned next = at ^ (64u * (pn >> 1) + 16u * (pn & 1));
            float g[2] = {0.f, 0.f};
            if constexpr (GROUP) {
                if (fold) {                                   // the group in front of this one
                    const int slot = SD == 2 && p == 0 ? 1 : 0;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        g[j] = p > 0 || t > 0 ? sc[slot][j] : 0.f;
                        sc[slot][j] = load_s(SD == 1 ? t * KS + 32 * s : p == 0 ? t * KS + 32 * FG : kn, j);   // (this one's, for the next fold)
                        if (MT == 2) continue;                // (its folds stand between the products)
#pragma unroll
                        for (int i = 0; i < MT; ++i)
#pragma unroll
                            for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(accg[i][j][r], g[j], acc[i][j][r]);
#pragma unroll
                        for (int i = 0; i < MT; ++i) asm volatile("" : "+v"(acc[i][j]));
                    }
                    if (MT != 2) __builtin_amdgcn_sched_barrier(0);
                }
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) {
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if constexpr (GROUP) {
                        if (fold && MT == 2) {
#pragma unroll
                            for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(accg[i][j][r], g[j], acc[i][j][r]);
                            asm volatile("" : "+v"(acc[i][j]));
                        }
                        if (fold) accg[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ga[i], gb[q][j], f32x16{}, 0, 0, 0);
                        else accg[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ga[i], gb[q][j], accg[i][j], 0, 0, 0);
                    } else {
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ga[i], gb[q][j], acc[i][j], 0, 0, 0);
                    }
                }
                ga[i] = *(const bf16x8*)(from + i * 8192 + next);
            }
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                gb[q ^ 1][j] = widen8<FP8W>(raw[sn % RW][j][2 * (q ^ 1)], raw[sn % RW][j][2 * (q ^ 1) + 1]);
                if (q == 0) raw[s % RW][j] = next_w(s, j);
            }
            constexpr int V = ((FP8W ? 8 : 24) + 2 * MT) / (2 * MT);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    if (fold && MT == 2) __builtin_amdgcn_sched_group_barrier(0x002, 16, 0);
                    __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                    __builtin_amdgcn_sched_group_barrier(0x002, V, 0);
                    if (j == 1) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                    if (last) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
                }
        }
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (ACT == ACT_BF16) {
        if constexpr (SD == 2)
#pragma unroll
            for (int j = 0; j < 2; ++j) sc[0][j] = load_s(0, j);
        load_a(buf1, 1);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_waitcnt(0x0F70 | NA);              // vmcnt(NA): the first step's activations, and the weights
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if constexpr (GROUP) {
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r) accg[i][j][r] = 0;
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) gb[0][j] = widen8<FP8W>(raw[0][j][0], raw[0][j][1]);
#pragma unroll
        for (int i = 0; i < MT; ++i) ga[i] = *(const bf16x8*)(buf0 + i * 8192 + l31 * 256 + 16 * ((2 * lh) ^ (l31 & 15)));
    } else {
        __builtin_amdgcn_s_waitcnt(0x0F70);                   // vmcnt(0): fewer loads than AFTER follow the first activations
    }
    {
        auto one = [&](unsigned char* cur, unsigned char* nxt, int t) __attribute__((always_inline)) {
            if constexpr (ACT == ACT_BF16) step16(cur, nxt, t);
            else step(cur, nxt, t);
        };
        int t = 0;
        for (; t + 1 < steps; t += 2) {
            one(buf0, buf1, t);
            one(buf1, buf0, t + 1);
        }
        if (t < steps) one(buf0, buf1, t);
    }
    if constexpr (GROUP) {                                    // the last group
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[i][j][r] = __builtin_fmaf(accg[i][j][r], sc[SD - 1][j], acc[i][j][r]);
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
kern_t pick_wide_impl(int mt, bool alone = false) {
    switch (mt) {
        case 2: return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 2, ROPE>;
        case 3:
            if constexpr (FG > 2 || (FG == 2 && FP8W))
                if (alone) return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 3, ROPE, true>;
            return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 3, ROPE>;
        case 4: if constexpr (FG == 0) return (kern_t)qgemm_wide_kernel<ACT, FP8W, FG, 4, ROPE>; break;
    }
    return nullptr;
}

template <bool FP8W, bool ROPE>
kern_t pick_wide_w16(int mt, int group, bool alone) {
    if (group == 0) return pick_wide_impl<ACT_BF16, FP8W, 0, ROPE>(mt);
    return group == 64 ? pick_wide_impl<ACT_BF16, FP8W, 2, ROPE>(mt, alone) : pick_wide_impl<ACT_BF16, FP8W, 4, ROPE>(mt, alone);
}

}  // namespace ql
