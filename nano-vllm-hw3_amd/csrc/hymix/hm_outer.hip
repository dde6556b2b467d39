// Recurrences whose per-head float32 state S [D, V] takes one gated outer product per token and is read in the same step:
//   S <- g S + k w^T,   o = S^T q + skip v,
// with g, the strength of w and the lengths of k and q given by the token:
//   gated delta rule      w = beta (v - (g S)^T k^),  k^ = k / sqrt(sum k^2 + eps), q^ = scale q / sqrt(sum q^2 + eps)
//   state-space dual      w = dt v                   (k = B, q = C, v = x)
// Both are walked in one form.  With the sums over the OLD state d1 = S^T k, d2 = S^T q of the vectors as they are stored,
//   w = a1 v - b2 d1,   o = gq d2 + kq w + skip v,   S <- g S + k (rk w),
// so the two sums of a token wait for nothing of that token, and everything that is not a sum over the state is a number per
// (token, head): gates [T, H, 8] f32 = {g, a1, b2, rk, gq, kq, skip, rq}.  A head reads the q and k of group h / (H / G).
// The state f32 [slots, H, D, V] is read at a portion's start (zero at position 0, whatever the slot holds) and left at its
// end.  Three kernels: the gates (parallel over tokens), the walk over portions, and a step of single tokens that works out
// its gates itself.
#include <algorithm>

#include "hm_outer.h"

namespace hm {

// The walk.  One workgroup of 256 threads per (sequence, head, 32 CV value channels).  A thread keeps CV neighbouring columns
// of S over DK / 8 key channels in registers (DK >= D): a column is spread over 8 neighbouring lanes, four channels each of
// every 32, and the sums over the state are a butterfly over those lanes, so their order is fixed by DK alone.  CH tokens'
// q, k, v and gates are staged in LDS at a time; the next chunk is requested from global memory before the current chunk's
// tokens run and written to the other buffer after them (one barrier per chunk).  Beyond the portion's end a chunk is padded
// with the identity step (g = 1, everything else 0).  A column's outputs are kept by its lanes in turn and leave CH tokens at
// a time.
template <typename T, int DK, int CV, int VEC, bool DELTA>
__global__ __launch_bounds__(256) void outer_walk_kernel(const T* __restrict__ rows, int64_t stride, int q_off, int k_off, int v_off,
                                                         const float* __restrict__ gates, float* __restrict__ state,
                                                         const int32_t* __restrict__ qstart, const int32_t* __restrict__ seq_pos0,
                                                         const int32_t* __restrict__ seq_slot, float* __restrict__ o, int H, int G,
                                                         int D, int V) {
    constexpr int SL = 8, CH = 8, KS = DK / SL, COLS = 256 / SL * CV, TOK = 2 * DK + COLS, PT = TOK / VEC, NR = (CH * PT + 255) / 256;
    static_assert(CH == SL, "a chunk's tokens are kept by a column's lanes");
    struct alignas(sizeof(T) * VEC) Pack { T v[VEC]; };
    __shared__ __attribute__((aligned(16))) float buf[2][CH * TOK];
    __shared__ __attribute__((aligned(16))) float gbuf[2][CH * 8];
    const int b = blockIdx.x, hd = blockIdx.y, gr = hd / (H / G);
    const int q0 = qstart[b], n = qstart[b + 1] - q0;
    if (n <= 0) return;
    const int tid = threadIdx.x, slice = tid % SL, col = tid / SL;
    const int j0 = blockIdx.z * COLS + col * CV;           // the thread's first value channel
    float* st = state + ((size_t)seq_slot[b] * H + hd) * (size_t)D * V;
    const bool fresh = seq_pos0[b] == 0;
    float s[KS][CV];                                       // key channel 32 m + 4 slice + e at index 4 m + e
#pragma unroll
    for (int ii = 0; ii < KS; ++ii) {
        const int i = 32 * (ii / 4) + 4 * slice + ii % 4;
#pragma unroll
        for (int c = 0; c < CV; ++c) s[ii][c] = (!fresh && j0 + c < V && i < D) ? st[(size_t)i * V + j0 + c] : 0.f;
    }
    // what a thread fetches does not change from chunk to chunk (column -1: padding)
    int col_of[NR], tok_of[NR];
#pragma unroll
    for (int k = 0; k < NR; ++k) {
        const int e = tid + 256 * k;
        const int tc = e / PT, rem = (e - tc * PT) * VEC;
        int c = -1;
        if (e < CH * PT) {
            if (rem < 2 * DK) {
                const int part = rem / DK, i = rem - part * DK;
                if (i < D) c = (part ? k_off : q_off) + gr * D + i;
            } else {
                const int jj = blockIdx.z * COLS + (rem - 2 * DK);
                if (jj < V) c = v_off + hd * V + jj;
            }
        }
        col_of[k] = c;
        tok_of[k] = tc;
    }
    Pack regs[NR];
    float greg = 0.f;
    auto request = [&](int tok0) {
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const int tok = tok0 + tok_of[k];
            Pack val;
#pragma unroll
            for (int e = 0; e < VEC; ++e) val.v[e] = from_f<T>(0.f);
            if (col_of[k] >= 0 && tok < n) val = *(const Pack*)(rows + (size_t)(q0 + tok) * stride + col_of[k]);
            regs[k] = val;
        }
        if (tid < CH * 8) {
            const int tok = tok0 + tid / 8;
            greg = tok < n ? gates[((size_t)(q0 + tok) * H + hd) * 8 + tid % 8] : (tid % 8 == 0 ? 1.f : 0.f);
        }
    };
    auto deposit = [&](int which) {
#pragma unroll
        for (int k = 0; k < NR; ++k) {
            const int e = tid + 256 * k;
            if (e < CH * PT) {
                float* p = buf[which] + e * VEC;
                if (VEC == 8) {
                    *(float4*)p = make_float4(to_f(regs[k].v[0]), to_f(regs[k].v[1 % VEC]), to_f(regs[k].v[2 % VEC]), to_f(regs[k].v[3 % VEC]));
                    *(float4*)(p + 4) = make_float4(to_f(regs[k].v[4 % VEC]), to_f(regs[k].v[5 % VEC]), to_f(regs[k].v[6 % VEC]), to_f(regs[k].v[7 % VEC]));
                } else {
#pragma unroll
                    for (int v = 0; v < VEC; ++v) p[v] = to_f(regs[k].v[v]);
                }
            }
        }
        if (tid < CH * 8) gbuf[which][tid] = greg;
    };
    request(0);
    deposit(0);
    __syncthreads();
    int which = 0;
    for (int tok0 = 0; tok0 < n; tok0 += CH) {
        const bool more = tok0 + CH < n;
        if (more) request(tok0 + CH);
        float keep[CV];
#pragma unroll
        for (int c = 0; c < CV; ++c) keep[c] = 0.f;
#pragma unroll
        for (int tc = 0; tc < CH; ++tc) {
            const float* p = buf[which] + tc * TOK;
            const float4 ga = *(const float4*)(gbuf[which] + tc * 8), gb = *(const float4*)(gbuf[which] + tc * 8 + 4);
            float d1[CV], d2[CV], kk[KS];
#pragma unroll
            for (int c = 0; c < CV; ++c) { d1[c] = 0.f; d2[c] = 0.f; }
#pragma unroll
            for (int m = 0; m < KS / 4; ++m) {             // 16-byte LDS reads: 8 lanes read 32 neighbouring channels
                const float4 q4 = *(const float4*)(p + 32 * m + 4 * slice), k4 = *(const float4*)(p + DK + 32 * m + 4 * slice);
                const float qe[4] = {q4.x, q4.y, q4.z, q4.w};
                kk[4 * m] = k4.x; kk[4 * m + 1] = k4.y; kk[4 * m + 2] = k4.z; kk[4 * m + 3] = k4.w;
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int c = 0; c < CV; ++c) {
                        if (DELTA) d1[c] += s[4 * m + e][c] * kk[4 * m + e];
                        d2[c] += s[4 * m + e][c] * qe[e];
                    }
            }
            float w[CV];
#pragma unroll
            for (int c = 0; c < CV; ++c) {
                const float vj = p[2 * DK + col * CV + c];
                w[c] = ga.y * vj;
                if (DELTA) w[c] -= ga.z * group_sum<SL>(d1[c]);
                d2[c] = group_sum<SL>(d2[c]);
                const float out = gb.x * d2[c] + gb.y * w[c] + gb.z * vj;
                keep[c] = slice == tc ? out : keep[c];
                w[c] *= ga.w;
            }
#pragma unroll
            for (int ii = 0; ii < KS; ++ii)
#pragma unroll
                for (int c = 0; c < CV; ++c) s[ii][c] = ga.x * s[ii][c] + kk[ii] * w[c];
        }
        if (tok0 + slice < n) {
            float* orow = o + ((size_t)(q0 + tok0 + slice) * H + hd) * V;
#pragma unroll
            for (int c = 0; c < CV; ++c)
                if (j0 + c < V) orow[j0 + c] = keep[c];
        }
        if (more) {
            deposit(which ^ 1);                // the other buffer was last read one chunk ago, before that chunk's barrier
            __syncthreads();
            which ^= 1;
        }
    }
#pragma unroll
    for (int ii = 0; ii < KS; ++ii) {
        const int i = 32 * (ii / 4) + 4 * slice + ii % 4;
#pragma unroll
        for (int c = 0; c < CV; ++c)
            if (j0 + c < V && i < D) st[(size_t)i * V + j0 + c] = s[ii][c];
    }
}

// Single tokens.  One workgroup of 256 threads per (sequence, head, 4 CT columns): a thread owns four neighbouring columns of
// every (256 / CT)-th key channel, RPT of them at most, all requested at once; the gates are worked out while they arrive.
// The sums over the key channels run over the wave, then over the four waves through LDS.
template <typename T, int RPT, bool WIDE, bool DELTA>
__global__ __launch_bounds__(256) void outer_step_kernel(const T* __restrict__ rows, int64_t stride, int q_off, int k_off, int v_off,
                                                         GateArgs<T> ga, float* __restrict__ state, const int32_t* __restrict__ qstart,
                                                         const int32_t* __restrict__ seq_pos0, const int32_t* __restrict__ seq_slot,
                                                         float* __restrict__ o, int H, int G, int D, int V, int CT) {
    __shared__ float qs[256], ks[256];
    __shared__ __attribute__((aligned(16))) float part[4][2][128];        // per wave: d1, d2 of up to 4 CT columns
    const int b = blockIdx.x, hd = blockIdx.y, gr = hd / (H / G);
    const int t = qstart[b];
    if (qstart[b + 1] - t <= 0) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int rg = tid / CT, RG = 256 / CT, cl = tid % CT * 4, j0 = blockIdx.z * CT * 4 + cl;
    float* st = state + ((size_t)seq_slot[b] * H + hd) * (size_t)D * V + j0;
    const bool fresh = seq_pos0[b] == 0;
    float4 s[RPT];
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int i = rg + r * RG;
        s[r] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (!fresh && i < D) {
            if (WIDE) {
                if (j0 < V) s[r] = *(const float4*)(st + (size_t)i * V);
            } else {
                if (j0 < V) s[r].x = st[(size_t)i * V];
                if (j0 + 1 < V) s[r].y = st[(size_t)i * V + 1];
                if (j0 + 2 < V) s[r].z = st[(size_t)i * V + 2];
                if (j0 + 3 < V) s[r].w = st[(size_t)i * V + 3];
            }
        }
    }
    const T* row = rows + (size_t)t * stride;
    const T *q = row + q_off + (size_t)gr * D, *k = row + k_off + (size_t)gr * D, *v = row + v_off + (size_t)hd * V + j0;
    float qq = 0.f, kk = 0.f, kq = 0.f;
    for (int i = lane; i < D; i += 64) {       // (every wave has the sums)
        const float a = to_f(q[i]), c = to_f(k[i]);
        if (wave == 0) { qs[i] = a; ks[i] = c; }
        qq += a * a;
        kk += c * c;
        kq += a * c;
    }
    if (DELTA) { qq = group_sum<64>(qq); kk = group_sum<64>(kk); }
    kq = group_sum<64>(kq);
    const Gates gt = make_gates<T, DELTA>(ga, t, hd, qq, kk, kq);
    float vv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) vv[c] = j0 + c < V ? to_f(v[c]) : 0.f;
    __syncthreads();
    float d1[4] = {0.f, 0.f, 0.f, 0.f}, d2[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int i = rg + r * RG;
        if (i < D) {
            const float a = ks[i], c = qs[i];
            if (DELTA) { d1[0] += s[r].x * a; d1[1] += s[r].y * a; d1[2] += s[r].z * a; d1[3] += s[r].w * a; }
            d2[0] += s[r].x * c; d2[1] += s[r].y * c; d2[2] += s[r].z * c; d2[3] += s[r].w * c;
        }
    }
    for (int m = CT; m < 64; m <<= 1) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (DELTA) d1[c] += __shfl_xor(d1[c], m);
            d2[c] += __shfl_xor(d2[c], m);
        }
    }
    if (lane < CT) {
        *(float4*)&part[wave][0][cl] = make_float4(d1[0], d1[1], d1[2], d1[3]);
        *(float4*)&part[wave][1][cl] = make_float4(d2[0], d2[1], d2[2], d2[3]);
    }
    __syncthreads();
    float w[4], out[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
        float e1 = 0.f, e2 = 0.f;
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            if (DELTA) e1 += part[u][0][cl + c];
            e2 += part[u][1][cl + c];
        }
        w[c] = gt.a1 * vv[c];
        if (DELTA) w[c] -= gt.b2 * e1;
        out[c] = gt.gq * e2 + gt.kq * w[c] + gt.skip * vv[c];
        w[c] *= gt.rk;
    }
    if (rg == 0) {
        float* orow = o + ((size_t)t * H + hd) * V + j0;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (j0 + c < V) orow[c] = out[c];
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
        const int i = rg + r * RG;
        if (i < D) {
            const float a = ks[i];
            const float4 n4 = make_float4(gt.g * s[r].x + a * w[0], gt.g * s[r].y + a * w[1], gt.g * s[r].z + a * w[2], gt.g * s[r].w + a * w[3]);
            if (WIDE) {
                if (j0 < V) *(float4*)(st + (size_t)i * V) = n4;
            } else {
                if (j0 < V) st[(size_t)i * V] = n4.x;
                if (j0 + 1 < V) st[(size_t)i * V + 1] = n4.y;
                if (j0 + 2 < V) st[(size_t)i * V + 2] = n4.z;
                if (j0 + 3 < V) st[(size_t)i * V + 3] = n4.w;
            }
        }
    }
}

template <typename DT, bool DELTA>
static void launch_outer(const void* rows_, int64_t stride, int q_off, int k_off, int v_off, const GateArgs<DT>& ga, float* gates,
                         float* state, const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, float* o, int B,
                         int64_t T, int H, int G, int D, int V, int max_q, hipStream_t s) {
    const DT* rows = (const DT*)rows_;
    if (max_q <= 1) {
        int ct = 8;                            // threads across the columns: up to 32, four columns each
        while (ct < 32 && ct * 4 < V) ct <<= 1;
        const int rpt = (D * ct + 255) / 256;
        const bool wide = V % 4 == 0 && (uintptr_t)state % 16 == 0;
        dim3 grid((unsigned)B, (unsigned)H, (unsigned)((V + 4 * ct - 1) / (4 * ct)));
#define HM_STEP(R, W)                                                                                                        \
    hipLaunchKernelGGL((outer_step_kernel<DT, R, W, DELTA>), grid, dim3(256), 0, s, rows, stride, q_off, k_off, v_off, ga, state, \
                       qstart, seq_pos0, seq_slot, o, H, G, D, V, ct)
#define HM_STEP_W(R) do { if (wide) HM_STEP(R, true); else HM_STEP(R, false); } while (0)
        if (rpt <= 4) HM_STEP_W(4); else if (rpt <= 8) HM_STEP_W(8); else if (rpt <= 16) HM_STEP_W(16); else HM_STEP_W(32);
#undef HM_STEP_W
#undef HM_STEP
        return;
    }
    const uintptr_t bits = (uintptr_t)rows;
    const bool packs = (stride | q_off | k_off | v_off | D | V) % 8 == 0 && bits % (8 * sizeof(DT)) == 0;
    const int64_t items = T * G;
    dim3 ggrid((unsigned)((items + 15) / 16));
    if (packs)
        hipLaunchKernelGGL((outer_gates_kernel<DT, 8, DELTA>), ggrid, dim3(256), 0, s, rows, stride, q_off, k_off, ga, gates, items, H, G, D);
    else
        hipLaunchKernelGGL((outer_gates_kernel<DT, 1, DELTA>), ggrid, dim3(256), 0, s, rows, stride, q_off, k_off, ga, gates, items, H, G, D);
    // columns per thread: two of them let every q and k value read from LDS meet two columns, one gives more workgroups
    const int cv = V >= 64 && (int64_t)B * H * ((V + 63) / 64) >= 512 ? 2 : 1;
#define HM_WALK(DK, CV, P)                                                                                                    \
    hipLaunchKernelGGL((outer_walk_kernel<DT, DK, CV, P, DELTA>), dim3((unsigned)B, (unsigned)H, (unsigned)((V + 32 * CV - 1) / (32 * CV))), \
                       dim3(256), 0, s, rows, stride, q_off, k_off, v_off, gates, state, qstart, seq_pos0, seq_slot, o, H, G, D, V)
#define HM_WALK_C(DK)                                                                                \
    do {                                                                                             \
        if (!packs) HM_WALK(DK, 1, 1);                                                               \
        else if (cv == 2) HM_WALK(DK, 2, 8);                                                         \
        else HM_WALK(DK, 1, 8);                                                                      \
    } while (0)
    if (D <= 32) HM_WALK_C(32); else if (D <= 64) HM_WALK_C(64); else if (D <= 128) HM_WALK_C(128); else HM_WALK_C(256);
#undef HM_WALK_C
#undef HM_WALK
}

}  // namespace hm

using namespace hm;

extern "C" int hm_gated_delta(int dtype, const void* rows, int64_t stride, int q_off, int k_off, int v_off, const void* pre,
                              int64_t pre_stride, int b_off, int a_off, const float* A, const float* dt_bias, float unit_eps,
                              float q_scale, float* gates, float* state, const int32_t* qstart, const int32_t* seq_pos0,
                              const int32_t* seq_slot, float* o, int B, int64_t T, int H, int G, int D, int V, int max_q, void* stream) {
    const int rc = outer_args_bad("hm_gated_delta", stride, q_off, k_off, v_off, pre_stride, b_off, a_off, rows, pre, A, dt_bias, gates,
                                  state, qstart, seq_pos0, seq_slot, o, B, T, H, G, D, V, max_q);
    if (rc) return rc;
    if (B == 0 || T == 0 || max_q == 0) return HM_OK;
    HM_DISPATCH(dtype, "hm_gated_delta",
                GateArgs<DT> ga = {(const DT*)pre, pre_stride, b_off, a_off, A, dt_bias, nullptr, unit_eps, q_scale};
                launch_outer<DT, true>(rows, stride, q_off, k_off, v_off, ga, gates, state, qstart, seq_pos0, seq_slot, o, B, T, H, G,
                                       D, V, max_q, as_stream(stream)));
    HM_CHECK_LAUNCH("hm_gated_delta");
    return HM_OK;
}

extern "C" int hm_state_space(int dtype, const void* rows, int64_t stride, int x_off, int b_off, int c_off, const void* pre,
                              int64_t pre_stride, int dt_off, const float* A, const float* dt_bias, const float* D, float* gates,
                              float* state, const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, float* y, int B,
                              int64_t T, int H, int G, int N, int V, int max_q, void* stream) {
    const int rc = outer_args_bad("hm_state_space", stride, c_off, b_off, x_off, pre_stride, 0, dt_off, rows, pre, A, dt_bias, gates,
                                  state, qstart, seq_pos0, seq_slot, y, B, T, H, G, N, V, max_q);
    if (rc) return rc;
    if (B > 0 && T > 0 && !D) { set_error("hm_state_space: bad argument"); return HM_EINVAL; }
    if (B == 0 || T == 0 || max_q == 0) return HM_OK;
    HM_DISPATCH(dtype, "hm_state_space",
                GateArgs<DT> ga = {(const DT*)pre, pre_stride, 0, dt_off, A, dt_bias, D, 0.f, 1.f};
                launch_outer<DT, false>(rows, stride, c_off, b_off, x_off, ga, gates, state, qstart, seq_pos0, seq_slot, y, B, T, H, G,
                                        N, V, max_q, as_stream(stream)));
    HM_CHECK_LAUNCH("hm_state_space");
    return HM_OK;
}
