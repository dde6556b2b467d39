// Mixture of experts: the router (softmax or sigmoid scores, an optional correction that only steers the choice,
// group-limited top-k, weights renormalised or not) and the expert products
// in their memory-bound form, one (token, chosen expert) pair at a time.
#include "sm_common.h"

namespace sm {

constexpr int kMaxExperts = 1024, kMaxTop = 32;

// The wave's sums of d[0 .. N - 1]: halving the values with every step, lane l ends with value l / (64 / N) in d[0].
template <int N, int O, int M>
__device__ __forceinline__ void fold_wave(float (&d)[M], int lane) {
    if constexpr (O == 0) {
        return;
    } else if constexpr (N > 1) {
        const bool up = (lane & O) != 0;
#pragma unroll
        for (int i = 0; i < N / 2; ++i) d[i] = (up ? d[i + N / 2] : d[i]) + __shfl_xor(up ? d[i] : d[i + N / 2], O);
        fold_wave<N / 2, O / 2>(d, lane);
    } else {
        d[0] += __shfl_xor(d[0], O);
        fold_wave<1, O / 2>(d, lane);
    }
}

// From the logits to the choice: tokens t0 .. t0 + nt - 1, token i's E logits at z_all + i RS, then room for its group scores, then (with
// gate_w) the gate's logit.  Called by all `waves` waves of a workgroup behind a barrier.
__device__ __forceinline__ void finish_routes(float* z_all, int RS, int64_t t0, int nt, int wave, int waves, int32_t* __restrict__ idx,
                                              float* __restrict__ wts, int E, int top, int groups, int keep, int score,
                                              const float* __restrict__ correction, int group_top, int renorm,
                                              const float* __restrict__ bias, const float* __restrict__ gate_w, float* __restrict__ gate_out) {
    const int lane = threadIdx.x & 63;
    if (groups <= 1 && E <= 256) {
        // no groups: a wave finishes a token, lane l holding the scores of the experts l, l + 64, ...
        for (int i = wave; i < nt; i += waves) {
            const int64_t t = t0 + i;
            const float* z = z_all + i * RS;
            if (gate_w != nullptr && lane == 0) gate_out[t] = 1.f / (1.f + expf(-z[RS - 1]));
            float s[4], c[4], mx = -INFINITY, sum = 0.f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = lane + 64 * j;
                s[j] = e < E ? z[e] + (bias ? bias[e] : 0.f) : -INFINITY;
                mx = fmaxf(mx, s[j]);
            }
            if (score == SM_ROUTE_SIGMOID) {
#pragma unroll
                for (int j = 0; j < 4; ++j) s[j] = 1.f / (1.f + expf(-s[j]));
            } else {
                mx = wave_max(mx);
#pragma unroll
                for (int j = 0; j < 4; ++j) { s[j] = expf(s[j] - mx); sum += s[j]; }
                const float inv = 1.f / wave_sum(sum);
#pragma unroll
                for (int j = 0; j < 4; ++j) s[j] *= inv;
            }
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = lane + 64 * j;
                c[j] = e < E ? s[j] + (correction ? correction[e] : 0.f) : -INFINITY;
            }
            float tot = 0.f, my_w = 0.f;
            int my_e = 0;
            const int span = E <= 16 ? 16 : E <= 32 ? 32 : 64;
            for (int k = 0; k < top; ++k) {
                float bv = -INFINITY;
                int be = E;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (c[j] > bv) { bv = c[j]; be = lane + 64 * j; }
                for (int o = span >> 1; o > 0; o >>= 1) {        // (the lanes past the experts hold -inf)
                    const float ov = __shfl_xor(bv, o);
                    const int oe = __shfl_xor(be, o);
                    if (ov > bv || (ov == bv && oe < be)) { bv = ov; be = oe; }
                }
                be = min(__builtin_amdgcn_readfirstlane(be), E - 1);
                float w = 0.f;
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    if (be == lane + 64 * j) { w = s[j]; c[j] = -INFINITY; }
                w = __shfl(w, be & 63);
                tot += w;
                if (lane == k) { my_w = w; my_e = be; }
            }
            if (lane < top) {                    // top <= 32
                idx[(size_t)t * top + lane] = my_e;
                wts[(size_t)t * top + lane] = my_w * (renorm ? 1.f / (tot + 1e-20f) : 1.f);
            }
        }
        return;
    }
    if (threadIdx.x >= nt) return;
    // groups (or very many experts): one thread finishes a token, the selections one after another
    const int64_t t = t0 + threadIdx.x;
    float* z = z_all + threadIdx.x * RS;
    if (gate_w != nullptr) gate_out[t] = 1.f / (1.f + expf(-z[RS - 1]));
    if (bias != nullptr)
        for (int e = 0; e < E; ++e) z[e] += bias[e];
    if (score == SM_ROUTE_SIGMOID) {
        for (int e = 0; e < E; ++e) z[e] = 1.f / (1.f + expf(-z[e]));
    } else {
        float mx = -INFINITY;
        for (int e = 0; e < E; ++e) mx = fmaxf(mx, z[e]);
        float sum = 0.f;
        for (int e = 0; e < E; ++e) { z[e] = expf(z[e] - mx); sum += z[e]; }
        const float inv = 1.f / sum;
        for (int e = 0; e < E; ++e) z[e] *= inv;
    }
    float* gs = z + E;
    // a chosen expert's score becomes -inf (no score is); the weights wait in wts for their sum.  (No array per thread: those
    // cost every token of this kernel its registers.)
    auto take = [&](int k, int best, float& tot) {
        const float w = best < 0 ? 0.f : z[best];
        idx[(size_t)t * top + k] = best < 0 ? 0 : best;
        wts[(size_t)t * top + k] = w;
        tot += w;
        if (best >= 0) z[best] = -INFINITY;
    };
    auto leave = [&](float tot) {
        const float rn = renorm ? 1.f / (tot + 1e-20f) : 1.f;
        for (int k = 0; k < top; ++k) wts[(size_t)t * top + k] *= rn;
    };
    if (correction != nullptr || group_top > 1) {
        // The general form: choice scores c = s + correction (they may be negative) decide, the weights are s.  A group
        // scores the sum of its `group_top` largest c; experts outside the best `keep` groups count as -inf.
        const int per = E / groups;
        bool ok_all = groups <= 1;
        if (!ok_all) {
            for (int g = 0; g < groups; ++g) {
                float tot = 0.f;
                int used[4] = {-1, -1, -1, -1};                 // group_top <= 4
                for (int k = 0; k < group_top && k < per; ++k) {
                    int best = -1;
                    float bv = -INFINITY;
                    for (int e = 0; e < per; ++e) {
                        bool taken = false;
                        for (int j = 0; j < k; ++j) taken |= used[j] == e;
                        const float c = z[g * per + e] + (correction ? correction[g * per + e] : 0.f);
                        if (!taken && (best < 0 || c > bv)) { bv = c; best = e; }
                    }
                    used[k] = best;
                    tot += bv;
                }
                gs[g] = tot;
            }
            // keep the best groups: a kept group's score becomes +inf, the others' -inf afterwards
            for (int k = 0; k < keep; ++k) {
                int best = -1;
                float bv = -INFINITY;
                for (int g = 0; g < groups; ++g)
                    if (gs[g] != INFINITY && (best < 0 || gs[g] > bv)) { bv = gs[g]; best = g; }
                if (best >= 0) gs[best] = INFINITY;
            }
        }
        float tot = 0.f;
        for (int k = 0; k < top; ++k) {
            int best = -1;
            float bv = -INFINITY;
            for (int e = 0; e < E; ++e) {
                if (!ok_all && gs[e / per] != INFINITY) continue;
                const float c = z[e] + (correction ? correction[e] : 0.f);
                if (z[e] != -INFINITY && (best < 0 || c > bv)) { bv = c; best = e; }
            }
            take(k, best, tot);
        }
        leave(tot);
        return;
    }
    if (groups > 1) {
        const int per = E / groups;
        for (int g = 0; g < groups; ++g) {
            float m = -1.f;
            for (int e = 0; e < per; ++e) m = fmaxf(m, z[g * per + e]);
            gs[g] = m;
        }
        // mark the best `keep` groups by negating the others' score; a dropped group's experts become ineligible
        for (int k = 0; k < keep; ++k) {
            int best = -1;
            float bv = -1.f;
            for (int g = 0; g < groups; ++g)
                if (gs[g] >= 0.f && gs[g] > bv) { bv = gs[g]; best = g; }
            if (best >= 0) gs[best] = -2.f;                     // -2 = kept
        }
    }
    float tot = 0.f;
    for (int k = 0; k < top; ++k) {
        int best = -1;
        float bv = -1.f;
        for (int e = 0; e < E; ++e) {
            if (groups > 1 && gs[e / (E / groups)] != -2.f) continue;
            if (z[e] != -INFINITY && z[e] > bv) { bv = z[e]; best = e; }
        }
        take(k, best, tot);
    }
    leave(tot);
}

// kRouteTokens = tokens per workgroup: every router row read serves all of them
template <typename T, int kRouteTokens>
__global__ __launch_bounds__(256, kRouteTokens == 8 ? 3 : 4) void moe_route_kernel(const T* __restrict__ h, const float* __restrict__ router_w,
                                                        int32_t* __restrict__ idx, float* __restrict__ wts, int64_t T_all, int W,
                                                        int E, int top, int groups, int keep, int score,
                                                        const float* __restrict__ correction, int group_top, int renorm,
                                                        int staged, const float* __restrict__ bias,
                                                        const float* __restrict__ gate_w, float* __restrict__ gate_out) {
    // per token: E scores, `groups` group scores and, with gate_w, the gate's logit; then the staged rows
    extern __shared__ float z_all[];
    const int RS = E + groups + (gate_w ? 1 : 0), rows = E + (gate_w ? 1 : 0);     // the gate's row follows the experts'
    const int64_t t0 = (int64_t)blockIdx.x * kRouteTokens;
    const int nt = (int)min((int64_t)kRouteTokens, T_all - t0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (staged && kRouteTokens == 1) {
        // one token: its row and four router rows, 1024 channels of them at once, go to registers side by side (through LDS and 256
        // channels at a time, 64 tokens of 2048 channels and 16 experts took 9.6 us, not 8.2)
        constexpr int U = 4;
        struct alignas(sizeof(T) * 4) Pack4 { T v[4]; };
        const T* src = h + (size_t)t0 * W;
        for (int e0 = 4 * wave; e0 < rows; e0 += 16) {
            const float* wr[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = min(e0 + j, rows - 1);
                wr[j] = e < E ? router_w + (size_t)e * W : gate_w;
            }
            float d[4] = {0.f, 0.f, 0.f, 0.f};
            for (int c0 = lane * 4; c0 < W; c0 += 256 * U) {
                Pack4 hv[U];
                float4 wv[U][4];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int c = min(c0 + 256 * u, W - 4);
                    hv[u] = *(const Pack4*)(src + c);
#pragma unroll
                    for (int j = 0; j < 4; ++j) wv[u][j] = *(const float4*)(wr[j] + c);
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (c0 + 256 * u < W) {
                        const float x0 = to_f(hv[u].v[0]), x1 = to_f(hv[u].v[1]), x2 = to_f(hv[u].v[2]), x3 = to_f(hv[u].v[3]);
#pragma unroll
                        for (int j = 0; j < 4; ++j) d[j] += x0 * wv[u][j].x + x1 * wv[u][j].y + x2 * wv[u][j].z + x3 * wv[u][j].w;
                    }
            }
            fold_wave<4, 32>(d, lane);
            const int e = e0 + lane / 16;
            if (lane % 16 == 0 && e < rows) z_all[e < E ? e : RS - 1] = d[0];
        }
    } else if (staged) {
        // the workgroup's token rows (one contiguous piece of h) go to LDS once; every expert's row is then read once per
        // workgroup in 16-byte pieces and meets all the tokens there
        T* h_lds = (T*)(z_all + (kRouteTokens * RS + 3) / 4 * 4);
        const T* src = h + (size_t)t0 * W;
        struct alignas(sizeof(T) * 4) Pack4 { T v[4]; };
        for (int i0 = threadIdx.x * 4; i0 < nt * W; i0 += 8 * 1024) {     // W % 4 == 0; eight pieces of a thread in flight
            Pack4 piece[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) piece[j] = *(const Pack4*)(src + min(i0 + 1024 * j, nt * W - 4));
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (i0 + 1024 * j < nt * W) *(Pack4*)(h_lds + i0 + 1024 * j) = piece[j];
        }
        __syncthreads();
        // four experts at a time: a token's piece read from LDS and widened meets four router rows (one row at a time, the
        // LDS reads and the 6 lane moves of every single sum were most of the kernel: 8192 tokens of 2048 channels, 16
        // experts: 53 -> 29 us; 64 tokens 16 -> 9)
        for (int e0 = 4 * wave; e0 < rows; e0 += 16) {
            const float* wr[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int e = min(e0 + j, rows - 1);
                wr[j] = e < E ? router_w + (size_t)e * W : gate_w;
            }
            constexpr int N = 4 * kRouteTokens;
            float d[N];
#pragma unroll
            for (int i = 0; i < N; ++i) d[i] = 0.f;
            float4 nxt[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) nxt[j] = *(const float4*)(wr[j] + min(lane * 4, W - 4));
#pragma unroll 1
            for (int c = lane * 4; c < W; c += 256) {
                float4 wv[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    wv[j] = nxt[j];
                    nxt[j] = *(const float4*)(wr[j] + min(c + 256, W - 4));
                }
#pragma unroll
                for (int i = 0; i < kRouteTokens; ++i) {           // (rows past nt: whatever LDS holds, nobody reads their sums)
                    const Pack4 hv = *(const Pack4*)(h_lds + (size_t)i * W + c);
                    const float x0 = to_f(hv.v[0]), x1 = to_f(hv.v[1]), x2 = to_f(hv.v[2]), x3 = to_f(hv.v[3]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) d[4 * i + j] += x0 * wv[j].x + x1 * wv[j].y + x2 * wv[j].z + x3 * wv[j].w;
                }
            }
            fold_wave<N, 32>(d, lane);
            const int v = lane / (64 / N), e = e0 + v % 4;
            if (lane % (64 / N) == 0 && e < rows) z_all[v / 4 * RS + (e < E ? e : RS - 1)] = d[0];
        }
    } else {
        for (int e = wave; e < rows; e += 4) {
            const float* wr = e < E ? router_w + (size_t)e * W : gate_w;
            float d[kRouteTokens];
            for (int i = 0; i < kRouteTokens; ++i) d[i] = 0.f;
            for (int c = lane; c < W; c += 64) {
                const float wv = wr[c];
                for (int i = 0; i < kRouteTokens; ++i)
                    if (i < nt) d[i] += to_f(h[(size_t)(t0 + i) * W + c]) * wv;
            }
            for (int i = 0; i < kRouteTokens; ++i) {
                const float sum = wave_sum(d[i]);
                if (lane == 0) z_all[i * RS + (e < E ? e : RS - 1)] = sum;
            }
        }
    }
    __syncthreads();
    finish_routes(z_all, RS, t0, nt, wave, 4, idx, wts, E, top, groups, keep, score, correction, group_top, renorm, bias, gate_w, gate_out);
}

// The logits on the matrix cores, in float32: sixteen tokens by 16 NT rows of the router (the gate's row follows the experts') per
// workgroup, whose waves share the width among them, 32 channels a wave in turn; their sums meet in LDS and are added in wave order.  A lane
// holds eight consecutive channels of one token and of one router row per 32 channels (the instruction's four k are channels 8 apart,
// which both operands agree on), so everything comes in 16-byte loads, U steps of them at once, and a router row is read once
// for sixteen tokens.  For many tokens: it is then bound by the reads of h, where staging the tokens in LDS and multiplying on the vector
// unit spent its time in LDS reads and widening (16 experts, us: 8192 tokens of 2048 channels 28 -> 19, 4096 21 -> 13; 64 experts,
// 8192 tokens of 4096 channels, which did not fit LDS, 2255 -> 88).  Below 2048 tokens a workgroup per token is as fast or faster (64
// tokens 8.2 and 12.5: sixteen waves in few workgroups begin and end later), from 65 rows on the products of sixteen tokens are.
template <typename T, int NT>
__global__ __launch_bounds__(1024, NT == 1 && sizeof(T) == 2 ? 8 : 4) void moe_route_mfma_kernel(const T* __restrict__ h, const float* __restrict__ router_w,
                                                              int32_t* __restrict__ idx, float* __restrict__ wts, int64_t T_all, int W,
                                                              int E, int top, int groups, int keep, int score,
                                                              const float* __restrict__ correction, int group_top, int renorm,
                                                              const float* __restrict__ bias, const float* __restrict__ gate_w,
                                                              float* __restrict__ gate_out) {
    constexpr int WAVES = 16, U = NT <= 2 ? 4 : 2;
    __shared__ float part[WAVES][NT][4][64];
    __shared__ float z_all[16 * (32 * NT + 1)];                 // (as many groups as experts at most)
    const int RS = E + groups + (gate_w ? 1 : 0), rows = E + (gate_w ? 1 : 0);
    const int64_t t0 = (int64_t)blockIdx.x * 16;
    const int nt = (int)min((int64_t)16, T_all - t0);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, l15 = lane & 15, c0 = 8 * (lane >> 4);
    struct alignas(16) Eight { T v[8]; };
    struct alignas(16) Eight32 { float v[8]; };
    const T* src = h + (size_t)(t0 + min(l15, nt - 1)) * W + c0;
    const float* wr[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        const int e = min(16 * n + l15, rows - 1);
        wr[n] = (e < E ? router_w + (size_t)e * W : gate_w) + c0;
    }
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    f32x4 acc[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    int left = (W / 32 - wave + WAVES - 1) / WAVES, k = 32 * wave;
    auto some = [&](auto count) {                              // the next steps of this wave, all their loads in front
        constexpr int C = decltype(count)::value;
        Eight x[C];
        Eight32 w[C][NT];
#pragma unroll
        for (int u = 0; u < C; ++u) {
            x[u] = *(const Eight*)(src + k + 32 * WAVES * u);
#pragma unroll
            for (int n = 0; n < NT; ++n) w[u][n] = *(const Eight32*)(wr[n] + k + 32 * WAVES * u);
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int u = 0; u < C; ++u)
#pragma unroll
            for (int j = 0; j < 8; ++j)
#pragma unroll
                for (int n = 0; n < NT; ++n) acc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(to_f(x[u].v[j]), w[u][n].v[j], acc[n], 0, 0, 0);
        left -= C;
        k += 32 * WAVES * C;
    };
    while (left >= U) some(std::integral_constant<int, U>{});
    if (left >= 2) some(std::integral_constant<int, 2>{});
    if (left >= 1) some(std::integral_constant<int, 1>{});
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) part[wave][n][r][lane] = acc[n][r];
    __syncthreads();
    for (int i = threadIdx.x; i < NT * 256; i += 1024) {        // token 4 (l / 16) + r, row 16 n + l % 16
        const int n = i >> 8, r = (i >> 6) & 3, l = i & 63, token = 4 * (l >> 4) + r, e = 16 * n + (l & 15);
        float sum = 0.f;
#pragma unroll
        for (int v = 0; v < WAVES; ++v) sum += part[v][n][r][l];
        if (e < rows) z_all[token * RS + (e < E ? e : RS - 1)] = sum;
    }
    __syncthreads();
    finish_routes(z_all, RS, t0, nt, wave, WAVES, idx, wts, E, top, groups, keep, score, correction, group_top, renorm, bias, gate_w, gate_out);
}

// workgroup = one (token, expert) pair; every wave produces outputs f = wave, wave + 4, ...
template <typename T>
__global__ __launch_bounds__(256) void moe_pairs_gate_up_kernel(const T* __restrict__ h, const int32_t* __restrict__ idx,
                                                                const T* __restrict__ w_gu, float limit, float alpha,
                                                                T* __restrict__ act, int top, int W, int F, int act_kind,
                                                                const float* __restrict__ in_wts) {
    extern __shared__ float h_lds[];
    const int64_t p = blockIdx.x, t = p / top;
    const int e = idx[p];
    const float iw = in_wts ? in_wts[p] : 1.f;       // a weight on the expert's input: the products are linear in it
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int c = threadIdx.x; c < W; c += 256) h_lds[c] = to_f(h[(size_t)t * W + c]);
    __syncthreads();
    if (!act_is_gated(act_kind)) {                   // one product per expert: w_gu is [E, F, W]
        const T* wu = w_gu + (size_t)e * F * W;
        for (int f = wave; f < F; f += 4) {
            const T* u_row = wu + (size_t)f * W;
            float u = 0.f;
            for (int c = lane; c < W; c += 64) u += h_lds[c] * to_f(u_row[c]);
            u = wave_sum(u);
            if (lane == 0) act[(size_t)p * F + f] = from_f<T>(plain_act(to_f(from_f<T>(u * iw)), act_kind));
        }
        return;
    }
    const T* wg = w_gu + (size_t)e * 2 * F * W;
    for (int f = wave; f < F; f += 4) {
        const T* g_row = wg + (size_t)f * W;
        const T* u_row = wg + (size_t)(F + f) * W;
        float g = 0.f, u = 0.f;
        for (int c = lane; c < W; c += 64) {
            const float x = h_lds[c];
            g += x * to_f(g_row[c]);
            u += x * to_f(u_row[c]);
        }
        g = wave_sum(g);
        u = wave_sum(u);
        // the products leave the matrix unit in the storage type, as a GEMM's output would
        if (lane == 0) act[(size_t)p * F + f] = from_f<T>(gated_act(to_f(from_f<T>(g * iw)), to_f(from_f<T>(u * iw)), limit, alpha, act_kind));
    }
}

// workgroup = one token; every wave produces output columns w = wave, wave + 4, ...
template <typename T>
__global__ __launch_bounds__(256) void moe_pairs_down_kernel(const T* __restrict__ act, const int32_t* __restrict__ idx,
                                                             const float* __restrict__ wts, const T* __restrict__ w_down,
                                                             const T* __restrict__ shared, T* __restrict__ y, int top, int W, int F,
                                                             int staged, const float* __restrict__ shared_scale) {
    extern __shared__ float a_lds[];             // top * F activations of the token's pairs (staged: they fit)
    const int64_t t = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (staged) {
        for (int c = threadIdx.x; c < top * F; c += 256) a_lds[c] = to_f(act[(size_t)t * top * F + c]);
        __syncthreads();
    }
    const T* a_row = act + (size_t)t * top * F;
    for (int w = wave; w < W; w += 4) {
        float tot = 0.f;
        for (int k = 0; k < top; ++k) {
            const int e = idx[(size_t)t * top + k];
            const T* row = w_down + ((size_t)e * W + w) * F;
            float d = 0.f;
            if (staged) {
                for (int c = lane; c < F; c += 64) d += a_lds[k * F + c] * to_f(row[c]);
            } else {                                 // the same sum from global memory
                for (int c = lane; c < F; c += 64) d += to_f(a_row[k * F + c]) * to_f(row[c]);
            }
            d = wave_sum(d);
            tot += (wts ? wts[(size_t)t * top + k] : 1.f) * to_f(from_f<T>(d));
        }
        if (lane == 0) {
            if (shared) tot += (shared_scale ? shared_scale[t] : 1.f) * to_f(shared[(size_t)t * W + w]);
            y[(size_t)t * W + w] = from_f<T>(tot);
        }
    }
}

}  // namespace sm

using namespace sm;

extern "C" int sm_moe_route(int dtype, const void* h, const float* router_w, int32_t* idx, float* wts, int64_t T, int W, int E,
                            int top, int groups, int keep, int score, const float* correction, int group_top, int renorm,
                            const float* bias, const float* gate_w, float* gate_out, void* stream) {
    if ((gate_w != nullptr) != (gate_out != nullptr) || T < 0 || W < 1 || E < 1 || top < 1 || (score != SM_ROUTE_SOFTMAX && score != SM_ROUTE_SIGMOID) || group_top < 1 ||
        group_top > 4 || (T > 0 && (!h || !router_w || !idx || !wts))) {
        set_error("sm_moe_route: bad argument");
        return SM_EINVAL;
    }
    if (groups < 1) groups = 1;
    if (E > kMaxExperts || top > kMaxTop || top > E || E % groups || keep < 1 || keep > groups || top > keep * (E / groups)) {
        set_error("sm_moe_route: unsupported routing shape (E=%d top=%d groups=%d keep=%d)", E, top, groups, keep);
        return SM_ESHAPE;
    }
    if (T == 0) return SM_OK;
    const int router_rows = E + (gate_w ? 1 : 0);
    const bool wide = ((uintptr_t)h | (uintptr_t)router_w | (uintptr_t)gate_w) % 16 == 0;
    if (wide && W % 32 == 0 && router_rows <= 64 && T >= 2048) {
#define SM_ROUTE(NT_)                                                                                                           \
    hipLaunchKernelGGL((moe_route_mfma_kernel<DT, NT_>), dim3((unsigned)((T + 15) / 16)), dim3(1024), 0, as_stream(stream), (const DT*)h, \
                       router_w, idx, wts, T, W, E, top, groups, keep, score, correction, group_top, renorm, bias, gate_w, gate_out)
        SM_DISPATCH(dtype, "sm_moe_route", if (router_rows <= 16) SM_ROUTE(1); else if (router_rows <= 32) SM_ROUTE(2); else SM_ROUTE(4));
#undef SM_ROUTE
        SM_CHECK_LAUNCH("sm_moe_route");
        return SM_OK;
    }
    // the token rows of a workgroup are staged in LDS when they fit and the rows can be moved in pieces of four channels
    const int tok = T >= 4096 ? 8 : (T >= 1024 ? 4 : 1);       // enough workgroups for a small step
    const size_t scores = ((size_t)tok * (E + groups + (gate_w ? 1 : 0)) * 4 + 15) / 16 * 16;
    const size_t rows = (size_t)tok * W * (dtype == SM_F32 ? 4 : 2);
    const int staged = W % 4 == 0 && scores + rows <= 60 * 1024 && wide;
#define SM_ROUTE(TOK_)                                                                                                          \
    hipLaunchKernelGGL((moe_route_kernel<DT, TOK_>), dim3((unsigned)((T + TOK_ - 1) / TOK_)), dim3(256), scores + (staged ? rows : 0), \
                       as_stream(stream), (const DT*)h, router_w, idx, wts, T, W, E, top, groups, keep, score, correction, group_top, \
                       renorm, staged, bias, gate_w, gate_out)
    SM_DISPATCH(dtype, "sm_moe_route", if (tok == 8) SM_ROUTE(8); else if (tok == 4) SM_ROUTE(4); else SM_ROUTE(1));
#undef SM_ROUTE
    SM_CHECK_LAUNCH("sm_moe_route");
    return SM_OK;
}

extern "C" int sm_moe_pairs_gate_up(int dtype, const void* h, const int32_t* idx, const void* w_gu, float limit, float alpha,
                                    int act_kind, const float* in_wts, void* act, int64_t T, int top, int W, int F, void* stream) {
    if (T < 0 || top < 1 || W < 1 || F < 1 || act_kind < 0 || act_kind > SM_ACT_LAST || (T > 0 && (!h || !idx || !w_gu || !act))) {
        set_error("sm_moe_pairs_gate_up: bad argument");
        return SM_EINVAL;
    }
    if ((size_t)W * 4 > 60000) { set_error("sm_moe_pairs_gate_up: width too large"); return SM_ESHAPE; }
    if (T == 0) return SM_OK;
    SM_DISPATCH(dtype, "sm_moe_pairs_gate_up",
                hipLaunchKernelGGL(moe_pairs_gate_up_kernel<DT>, dim3((unsigned)(T * top)), dim3(256), (size_t)W * 4,
                                   as_stream(stream), (const DT*)h, idx, (const DT*)w_gu, limit, alpha, (DT*)act, top, W, F, act_kind,
                                   in_wts));
    SM_CHECK_LAUNCH("sm_moe_pairs_gate_up");
    return SM_OK;
}

extern "C" int sm_moe_pairs_down(int dtype, const void* act, const int32_t* idx, const float* wts, const void* w_down,
                                 const void* shared, const float* shared_scale, void* y, int64_t T, int top, int W, int F,
                                 void* stream) {
    if (T < 0 || top < 1 || W < 1 || F < 1 || (shared_scale && !shared) || (T > 0 && (!act || !idx || !w_down || !y))) {
        set_error("sm_moe_pairs_down: bad argument");
        return SM_EINVAL;
    }
    if (T == 0) return SM_OK;
    const int staged = (size_t)top * F * 4 <= 60000;            // a token's activations in LDS when they fit
    SM_DISPATCH(dtype, "sm_moe_pairs_down",
                hipLaunchKernelGGL(moe_pairs_down_kernel<DT>, dim3((unsigned)T), dim3(256), staged ? (size_t)top * F * 4 : 0,
                                   as_stream(stream), (const DT*)act, idx, wts, (const DT*)w_down, (const DT*)shared, (DT*)y, top, W,
                                   F, staged, shared_scale));
    SM_CHECK_LAUNCH("sm_moe_pairs_down");
    return SM_OK;
}
