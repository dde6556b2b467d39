// Output projection of up to 32 rows:  y[M, V] = x[M, K] . w[V, K]^T in bf16, one read of the vocabulary table.
//
// A wave is a workgroup and owns 32 columns and all of K.  Rows of the table come 128 bytes at a time, eight lanes to a row, and go
// through LDS to the lanes that multiply them (16-byte chunk c of row r at place c ^ (r / 2 & 7)); so do the activations, MR groups of
// eight rows of them.  RING steps of 64 k are in flight per wave, without a barrier anywhere.  The k order of a sum is that of the tiles
// in ql_gemm_kernel.h: the same bits.
//
// Bound by the table's bytes.  In those tiles a lane loads its own row, so that each load touches 64 cache lines, which are fetched
// again when the 32 KB next to the CU has dropped them: 12 rows, 151936 x 1024, 80 us there (3.9 TB/s), 53 here (5.8).
#include "ql_common.h"

namespace ql {

template <int MR, int RING>
__global__ __launch_bounds__(64) void head_rows_kernel(const unsigned short* __restrict__ x, const unsigned short* __restrict__ w,
                                                       unsigned short* __restrict__ y, int M, int V, int K) {
    __shared__ __attribute__((aligned(1024))) unsigned char lds_a[32 * 128];
    __shared__ __attribute__((aligned(1024))) unsigned char lds_b[32 * 128];
    const int lane = threadIdx.x, l31 = lane & 31, hi = lane >> 5, sub = lane >> 3, chunk = lane & 7;
    const int n0 = blockIdx.x * 32;
    const unsigned short *arow[MR], *brow[4];
#pragma unroll
    for (int j = 0; j < MR; ++j) arow[j] = x + (size_t)min(8 * j + sub, M - 1) * K + 8 * chunk;
#pragma unroll
    for (int j = 0; j < 4; ++j) brow[j] = w + (size_t)min(n0 + 8 * j + sub, V - 1) * K + 8 * chunk;
    struct Stage { i32x4 a[MR], b[4]; };
    typedef const __attribute__((address_space(1))) i32x4* gptr;
    auto request = [&](Stage& st, int step) {
#pragma unroll
        for (int j = 0; j < MR; ++j) st.a[j] = *(gptr)(arow[j] + (size_t)step * 64);
#pragma unroll
        for (int j = 0; j < 4; ++j) st.b[j] = __builtin_nontemporal_load((gptr)(brow[j] + (size_t)step * 64));
    };
    f32x16 acc = {0};
    const int put = sub * 128 + 16 * (chunk ^ (sub >> 1)), get = l31 * 128, swz = (l31 >> 1) & 7;
    auto consume = [&](const Stage& st) {
        // (one wave, whose LDS accesses are carried out in their order: nothing to wait for but the order itself)
#pragma unroll
        for (int j = 0; j < MR; ++j) *(i32x4*)(lds_a + 1024 * j + (put ^ (64 * (j & 1)))) = st.a[j];
#pragma unroll
        for (int j = 0; j < 4; ++j) *(i32x4*)(lds_b + 1024 * j + (put ^ (64 * (j & 1)))) = st.b[j];
        asm volatile("" ::: "memory");
        __builtin_amdgcn_wave_barrier();
        bf16x8 a[4], b[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {                          // k = 32 (s / 2) + 16 hi + 8 (s % 2) .. + 8 of the step
            const int place = 16 * ((4 * (s >> 1) + 2 * hi + (s & 1)) ^ swz);
            a[s] = *(const bf16x8*)(lds_a + get + place);
            b[s] = *(const bf16x8*)(lds_b + get + place);
        }
#pragma unroll
        for (int s = 0; s < 4; ++s) acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[s], b[s], acc, 0, 0, 0);
        asm volatile("" ::: "memory");
    };
    const int steps = K / 64;                                  // (no condition stands around a load: past the end the last step again)
    Stage st[RING];
#pragma unroll
    for (int i = 0; i < RING; ++i) request(st[i], min(i, steps - 1));
    int step = 0;
    for (; step + RING <= steps; step += RING)
#pragma unroll
        for (int i = 0; i < RING; ++i) {
            consume(st[i]);
            request(st[i], min(step + RING + i, steps - 1));
        }
#pragma unroll
    for (int i = 0; i < RING; ++i)
        if (step + i < steps) consume(st[i]);
    if (n0 + l31 >= V) return;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        const int row = (r & 3) + 8 * (r >> 2) + 4 * hi;
        if (row < M) y[(size_t)row * V + n0 + l31] = __builtin_bit_cast(unsigned short, (bf16_t)acc[r]);
    }
}

// up to 32 rows, K a multiple of 64, x and w on 16 bytes (the caller checks)
int launch_head_rows(const void* x, const void* w, void* y, int64_t M, int64_t V, int64_t K, hipStream_t s) {
    const dim3 grid((unsigned)((V + 31) / 32));
#define QL_HEAD(MR_)                                                                                                         \
    hipLaunchKernelGGL((head_rows_kernel<MR_, 4>), grid, dim3(64), 0, s, (const unsigned short*)x, (const unsigned short*)w, \
                       (unsigned short*)y, (int)M, (int)V, (int)K)
    if (M <= 8) QL_HEAD(1); else if (M <= 16) QL_HEAD(2); else QL_HEAD(4);
#undef QL_HEAD
    QL_CHECK_LAUNCH("ql_lmhead_logits");
    return QL_OK;
}

}  // namespace ql
