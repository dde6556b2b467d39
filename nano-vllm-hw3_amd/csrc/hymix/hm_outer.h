// What the forms of the outer-product recurrences (hm_outer.hip, hm_outer_chunk.hip) share: the gates of a token, and the
// checks of the entry points.
#pragma once
#include "hm_common.h"

namespace hm {

// what turns a token's projections into its gates
template <typename T>
struct GateArgs {
    const T* pre;              // delta: the pre-activations of beta and of the decay's step; state space: of the step size dt
    int64_t pre_stride;
    int b_off, a_off;          // their columns, one per head (state space: a_off only)
    const float* A;            // f32 [H], the decay's rate (negative)
    const float* dt_bias;      // f32 [H]
    const float* skip;         // f32 [H], state space only
    float unit_eps, q_scale;   // delta only
};

struct Gates { float g, a1, b2, rk, gq, kq, skip, rq; };

// qq, kk, kq = the sums of q^2, k^2 and q k over the head's D channels (state space: kq alone)
template <typename T, bool DELTA>
__device__ __forceinline__ Gates make_gates(const GateArgs<T>& a, int64_t t, int h, float qq, float kk, float kq) {
    const T* row = a.pre + (size_t)t * a.pre_stride;
    const float dt = softplus_f(to_f(row[a.a_off + h]) + a.dt_bias[h]);
    Gates r;
    r.g = expf(a.A[h] * dt);
    if (DELTA) {
        const float rq = a.q_scale / sqrtf(qq + a.unit_eps);
        r.rq = rq;
        r.rk = 1.f / sqrtf(kk + a.unit_eps);
        r.a1 = sigmoid_f(to_f(row[a.b_off + h]));
        r.b2 = r.a1 * r.g * r.rk;
        r.gq = r.g * rq;
        r.kq = r.rk * rq * kq;
        r.skip = 0.f;
    } else {
        r.rq = r.rk = 1.f;
        r.a1 = dt;
        r.b2 = 0.f;
        r.gq = r.g;
        r.kq = kq;
        r.skip = a.skip[h];
    }
    return r;
}

// 16 lanes per (token, group of heads), VEC channels per access
template <typename T, int VEC, bool DELTA>
__global__ __launch_bounds__(256) void outer_gates_kernel(const T* __restrict__ rows, int64_t stride, int q_off, int k_off,
                                                          GateArgs<T> ga, float* __restrict__ gates, int64_t items, int H, int G,
                                                          int D) {
    struct alignas(sizeof(T) * VEC) Pack { T v[VEC]; };
    const int64_t item = (int64_t)blockIdx.x * 16 + (threadIdx.x >> 4);
    if (item >= items) return;                 // (whole groups of 16 lanes)
    const int li = threadIdx.x & 15;
    const int64_t t = item / G;
    const int gr = (int)(item - t * G), rep = H / G;
    const T* q = rows + (size_t)t * stride + q_off + (size_t)gr * D;
    const T* k = rows + (size_t)t * stride + k_off + (size_t)gr * D;
    float qq = 0.f, kk = 0.f, kq = 0.f;
    for (int i = li * VEC; i < D; i += 16 * VEC) {
        const Pack pq = *(const Pack*)(q + i), pk = *(const Pack*)(k + i);
#pragma unroll
        for (int e = 0; e < VEC; ++e) {
            const float a = to_f(pq.v[e]), b = to_f(pk.v[e]);
            qq += a * a;
            kk += b * b;
            kq += a * b;
        }
    }
    if (DELTA) { qq = group_sum<16>(qq); kk = group_sum<16>(kk); }
    kq = group_sum<16>(kq);
    for (int j = li; j < rep; j += 16) {
        const int h = gr * rep + j;
        const Gates r = make_gates<T, DELTA>(ga, t, h, qq, kk, kq);
        float4* out = (float4*)(gates + ((size_t)t * H + h) * 8);
        out[0] = make_float4(r.g, r.a1, r.b2, r.rk);
        out[1] = make_float4(r.gq, r.kq, r.skip, r.rq);
    }
}

static int outer_args_bad(const char* name, int64_t stride, int q_off, int k_off, int v_off, int64_t pre_stride, int b_off, int a_off,
                          const void* rows, const void* pre, const float* A, const float* dt_bias, const float* gates, const float* state,
                          const int32_t* qstart, const int32_t* seq_pos0, const int32_t* seq_slot, const float* o, int B, int64_t T, int H,
                          int G, int D, int V, int max_q) {
    if (B < 0 || T < 0 || H < 1 || G < 1 || H % G != 0 || D < 1 || V < 1 || q_off < 0 || k_off < 0 || v_off < 0 || b_off < 0 || a_off < 0 ||
        max_q < 0 || stride < (int64_t)q_off + (int64_t)G * D || stride < (int64_t)k_off + (int64_t)G * D ||
        stride < (int64_t)v_off + (int64_t)H * V || pre_stride < (int64_t)a_off + H || pre_stride < (int64_t)b_off + H ||
        (B > 0 && T > 0 && (!rows || !pre || !A || !dt_bias || !state || !qstart || !seq_pos0 || !seq_slot || !o || (max_q > 1 && !gates)))) {
        set_error("%s: bad argument", name);
        return HM_EINVAL;
    }
    if (D > 256 || H > 65535 || V > 32 * 65535) { set_error("%s: at most 256 key channels and 65535 heads", name); return HM_ESHAPE; }
    if ((uintptr_t)gates % 16 != 0) { set_error("%s: gates must be 16-byte aligned", name); return HM_EINVAL; }
    return 0;
}

}  // namespace hm
