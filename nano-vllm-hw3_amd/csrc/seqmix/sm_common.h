// Shared helpers of libseqmix (gfx950 only).
#pragma once
#include <hip/hip_runtime.h>
#include <stdarg.h>
#include <stdint.h>
#include <stdio.h>

#include <type_traits>

#include "../../../include/seqmix.h"

namespace sm {

typedef __bf16 bf16_t;
typedef bf16_t bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));

void set_error(const char* fmt, ...);

template <typename T> __device__ __forceinline__ float to_f(T v) { return (float)v; }
template <typename T> __device__ __forceinline__ T from_f(float v) { return (T)v; }   // bf16: round to nearest even

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
    return v;
}
__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
    return v;
}

// sum over a workgroup of up to 16 waves; `red` = 16 floats of LDS; every thread gets the total
__device__ __forceinline__ float block_sum(float v, float* red) {
    v = wave_sum(v);
    const int wave = threadIdx.x >> 6, nw = (blockDim.x + 63) >> 6;
    __syncthreads();                      // red may still be read from a previous call
    if ((threadIdx.x & 63) == 0) red[wave] = v;
    __syncthreads();
    float t = 0.f;
    for (int i = 0; i < nw; ++i) t += red[i];
    return t;
}

// what a feed-forward applies between its two products (SM_ACT_*): a gated form of a gate and an up product (clamped GLU,
// SiLU or tanh-GELU gate), or a function of the up product alone (exact or tanh GELU, squared ReLU)
__device__ __forceinline__ float gelu_erf(float z) { return 0.5f * z * (1.f + erff(z * 0.70710678118654752f)); }
__device__ __forceinline__ float gelu_tanh(float z) {
    return 0.5f * z * (1.f + tanhf(0.7978845608028654f * (z + 0.044715f * z * z * z)));
}
// n / d for d >= 1: a division's remainder step without its scaling (d 2^-32 and its reciprocal are never subnormal), the special cases
// by the division's own last instruction.  7 instructions for 11: a gate's outputs are a sixth of the expert tiles' cycles.
// Not correctly rounded in every case, but nearly: the first quotient is off by 1.5 units at most (the reciprocal's one, the product's half), its
// remainder is exact, and the reciprocal scales that with a relative error of 2^-21 (2^-20 where it is subnormal): 0.5 units + 2^-19.
// Gates of 2^22 numbers each (normal ones, +-90, +-e^85, -86 to -89; alpha 1 and 8) have the errors of the division, largest and mean, to
// every digit shown: the exponential's are 4 to 64 units.
__device__ __forceinline__ float quotient(float n, float d) {
    const float r = __builtin_amdgcn_rcpf(d * 0x1p-32f) * 0x1p-32f, q = n * r;
    return __builtin_amdgcn_div_fixupf(__builtin_fmaf(__builtin_fmaf(-q, d, n), r, q), d, n);
}
// the gated forms: g' = min(g, limit), u' = clamp(u, +-limit), g' sigmoid(alpha g') (u' + 1) (SM_ACT_CLAMPED_GLU), or with
// SM_ACT_SILU_GLU the same without the one: silu(g) u for limit = +inf and alpha = 1; SM_ACT_GELU_TANH_GLU: gelu_tanh(g) u
__device__ __forceinline__ float gated_act(float g, float u, float limit, float alpha, int act) {
    if (act == SM_ACT_GELU_TANH_GLU) return gelu_tanh(g) * u;
    // (minnum and maxnum as the hardware has them: the library's put a canonicalization in front of every operand, and a caller that has
    // numbers from memory does so itself, since a signalling NaN would come through)
    asm("v_min_f32 %0, %1, %2" : "=v"(g) : "s"(limit), "v"(g));
    u = __builtin_amdgcn_fmed3f(u, -fabsf(limit), limit);     // (min(max(u, -limit), limit), which is the limit for negative ones)
    const float y = quotient(g, 1.f + __builtin_amdgcn_exp2f(g * (-1.4426950408889634f * alpha)));
    return y * (act == SM_ACT_SILU_GLU ? u : u + 1.f);
}
__host__ __device__ __forceinline__ bool act_is_gated(int act) {
    return act == SM_ACT_CLAMPED_GLU || act == SM_ACT_SILU_GLU || act == SM_ACT_GELU_TANH_GLU;
}
__device__ __forceinline__ float plain_act(float z, int act) {
    if (act == SM_ACT_RELU_SQ) { z = fmaxf(z, 0.f); return z * z; }
    return act == SM_ACT_GELU_TANH ? gelu_tanh(z) : gelu_erf(z);
}

// f(kind as a constant) for the kinds that a kernel's mode can meet (0: none, 1: the gated forms, 2: the plain ones), so that a loop over
// outputs holds the code of one kind and no branches around it
template <int MODE, typename F>
__device__ __forceinline__ void with_act(int act, F f) {
    auto is = [&](auto kind) {
        if (act == decltype(kind)::value) f(kind);
    };
    if constexpr (MODE == 0) {
        f(std::integral_constant<int, 0>{});
    } else if constexpr (MODE == 1) {
        is(std::integral_constant<int, SM_ACT_CLAMPED_GLU>{});
        is(std::integral_constant<int, SM_ACT_SILU_GLU>{});
        is(std::integral_constant<int, SM_ACT_GELU_TANH_GLU>{});
    } else {
        is(std::integral_constant<int, SM_ACT_GELU>{});
        is(std::integral_constant<int, SM_ACT_GELU_TANH>{});
        is(std::integral_constant<int, SM_ACT_RELU_SQ>{});
    }
}

// the grouping of (token, choice) pairs by expert into tiles of `unit` rows (sm_moe_align.hip); SM_OK or an error code
int launch_moe_align(const int32_t* idx, int64_t P, int E, int unit, int max_tiles, int32_t* row_pair, int32_t* tile_expert,
                     int32_t* pair_row, int32_t* counts, hipStream_t s);

static inline hipStream_t as_stream(void* s) { return (hipStream_t)s; }

#define SM_CHECK_LAUNCH(name)                                                    \
    do {                                                                         \
        hipError_t e_ = hipGetLastError();                                       \
        if (e_ != hipSuccess) {                                                  \
            sm::set_error("%s: launch failed: %s", name, hipGetErrorString(e_)); \
            return SM_ELAUNCH;                                                   \
        }                                                                        \
    } while (0)

// run `call<T>` for the storage type named by a dtype code
#define SM_DISPATCH(dtype, name, ...)                                        \
    do {                                                                     \
        if ((dtype) == SM_F32) { typedef float DT; __VA_ARGS__; }             \
        else if ((dtype) == SM_BF16) { typedef sm::bf16_t DT; __VA_ARGS__; }  \
        else { sm::set_error("%s: unknown dtype %d", name, (int)(dtype)); return SM_EINVAL; } \
    } while (0)

}  // namespace sm
