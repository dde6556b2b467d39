// Causal self-attention over packed variable-length sequences (prefill) for gfx950, flash style:
// scores are never materialised; each workgroup walks the K/V tiles of its query block with an
// online softmax.  head_dim = 128, bf16 in / bf16 out, f32 accumulation, grouped-query heads.
//
// Workgroup = 4 waves = the G = Hq/Hkv query heads of ONE kv head x (128/G) consecutive query rows,
// so each K/V tile staged in LDS serves all query heads that share it.  Each wave owns 32 query rows
// of one head.  Both products are computed transposed so that everything a softmax row needs sits
// in one lane (pair):
//   S^T = K . Q^T   (A = K rows from LDS with 16-byte reads, B = Q^T kept in registers):
//                   lane l holds query (l & 31) and the keys (r&3) + 8*(r>>2) + 4*(l>>5) of a tile
//   O^T += V^T . P^T (A = V^T through the transposing LDS read, B = P^T = the lane's own probabilities):
//                   the accumulator keeps query (l & 31) per lane, so the online rescale is lane-local.
// The k index of the second product is the KEY; its order inside a 16-key MFMA step is free as long
// as both operands agree, and it is chosen to be exactly the order in which the S^T accumulator
// registers already hold the keys - P never moves between lanes.
// K/V tiles (64 keys) go from global memory straight to LDS, 256-byte rows with an XOR swizzle of the 16-byte chunk
// index that keeps both the row reads (K) and the transposed reads (V) conflict-free: two buffers, one barrier per
// tile, the next tile's loads issued before the current tile's math.  Held in registers on its way a tile made it 294
// per wave, one wave per SIMD, and nothing filled its waits; at 191 two waves run one's exponentials beside the
// other's products: 8 prompts of 1024 tokens, 16 / 8 heads, 133 -> 74 us, one of 4096 tokens 222 -> 110, two of 1024 34 -> 30.
// (Tiles of 32 keys fit three waves and are no faster with full CUs, 76 and 128 us, and slower where a CU has one
// workgroup and a tile's chain of dependent steps is what counts: 128 us and 38.)
#include "ql_common.h"
#include "row_deal.h"

namespace ql {

typedef short s16x4 __attribute__((ext_vector_type(4)));


constexpr int kTileKeys = 64, NH = kTileKeys / 32;

__device__ __forceinline__ int kv_off(int row, int ch) {
    return 256 * row + 16 * (ch ^ (((row & 3) << 2) | ((row >> 2) & 3)));
}

// DMA: keys and values on 16 bytes, loaded straight to LDS; rows off 16 bytes go through registers
template <int G, bool DMA>
__global__ __launch_bounds__(256, 2) void attn_prefill_kernel(const unsigned short* __restrict__ q,
                                                              const unsigned short* __restrict__ k,
                                                              const unsigned short* __restrict__ v,
                                                              const int* __restrict__ cu_seqlens,
                                                              unsigned short* __restrict__ out, float c_log2, int Hq,
                                                              int Hkv, int kv_group, int blocks, int num_seqs, int run) {
    constexpr int SUBS = 4 / G;            // 32-row query blocks per head in this workgroup
    constexpr int QROWS = 32 * SUBS;
    constexpr int V_AT = kTileKeys * 256;  // the value tile behind the key tile
    __shared__ __attribute__((aligned(1024))) unsigned char buf0[2 * kTileKeys * 256];
    __shared__ __attribute__((aligned(1024))) unsigned char buf1[2 * kTileKeys * 256];

    const RowTile rt = row_tile(blockIdx.x, blockIdx.y, blockIdx.z, run, blocks, num_seqs, Hq / G);
    if (rt.b < 0) return;
    // a group of G query heads reads the K/V of kv head (group * G) / kv_group, which is the group itself when a kv
    // head's query heads form one group (kv_group == G: ratios 1, 2, 4); other ratios are dealt to several groups per
    // kv head
    const int seq = rt.b, hgrp = rt.g, hk = (hgrp * G) / kv_group;
    const int s0 = cu_seqlens[seq];
    const int L = cu_seqlens[seq + 1] - s0;
    const int q0 = row_first(run, rt.tile, blocks, L, QROWS);           // heaviest query blocks first
    if (q0 < 0 || q0 >= L) return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = wave % G, sub = wave / G;
    const int hq = hgrp * G + g;
    const int l31 = lane & 31, hi = lane >> 5;
    const int qw0 = q0 + sub * 32;
    const int qrow = qw0 + l31;                                      // this lane's query (within the sequence)
    const int kend = min(L, q0 + QROWS);
    const int ntiles = (kend + kTileKeys - 1) / kTileKeys;

    // Q^T as the B operand: 8 k-steps of 16 dims, lane holds dims 16*ks + 8*hi .. +8 of its query
    bf16x8 qf[8];
    {
        const unsigned short* qp = q + ((size_t)(s0 + min(qrow, L - 1)) * Hq + hq) * 128 + 8 * hi;
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qf[ks] = *(const bf16x8*)(qp + 16 * ks);
    }

    // a tile: eight pieces of 1 KB (four rows) per tensor, two per wave; lane l brings the chunk that belongs at 16 l
    typedef i32x4 anywhere __attribute__((aligned(2)));
    typedef __attribute__((address_space(1))) const void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;
    const unsigned short *ks0 = k + ((size_t)s0 * Hkv + hk) * 128, *vs0 = v + ((size_t)s0 * Hkv + hk) * 128;
    auto load_tile = [&](unsigned char* buf, int kt0) {
#pragma unroll
        for (int j = 0; j < 2 * NH; ++j) {
            const int i = wave + 4 * j, row = 4 * i + (lane >> 4);
            const int ch = (lane & 15) ^ (((row & 3) << 2) | ((row >> 2) & 3));
            const size_t off = (size_t)min(kt0 + row, L - 1) * Hkv * 128 + 8 * ch;
            if constexpr (DMA) {
                __builtin_amdgcn_global_load_lds((gvoid*)(ks0 + off), (lvoid*)(buf + 1024 * i), 16, 0, 0);
                __builtin_amdgcn_global_load_lds((gvoid*)(vs0 + off), (lvoid*)(buf + V_AT + 1024 * i), 16, 0, 0);
            } else {
                *(i32x4*)(buf + 1024 * i + 16 * lane) = *(const anywhere*)(ks0 + off);
                *(i32x4*)(buf + V_AT + 1024 * i + 16 * lane) = *(const anywhere*)(vs0 + off);
            }
        }
    };
    auto landed = [&]() {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
    };

    f32x16 oacc[4];
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[d][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    // Transposed-read address pieces of this lane: 16-lane group gq picks dims 16*gq .. +16 of a 32-dim block.  A chunk's
    // number enters its place by exclusive or, so the reads' addresses are one base each, changed in the chunk's bits.
    const int gq = (lane >> 4) & 1, ti = lane & 15, tq = ti >> 2, tp = ti & 3;
    const int k_at = kv_off(l31, hi), v_at = kv_off(4 * hi + tq, 2 * gq + (tp >> 1)) + 8 * (tp & 1),
              v_at8 = kv_off(4 * hi + tq + 8, 2 * gq + (tp >> 1)) + 8 * (tp & 1);

    auto work = [&](const unsigned char* buf, int kt0) {
        if (kt0 > qw0 + 31) return;                                  // no row of this wave sees the tile
        // ---- S^T = K . Q^T
        f32x16 s[NH];
#pragma unroll
        for (int j = 0; j < NH; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[j][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 8; ++ks) {
                const bf16x8 kf = *(const bf16x8*)(buf + (k_at ^ (32 * ks)) + 8192 * j);
                s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[j], 0, 0, 0);
            }
        }
        // ---- causal mask (only tiles that reach past this wave's first query) and online softmax
        if (kt0 + kTileKeys - 1 > qw0) {
#pragma unroll
            for (int j = 0; j < NH; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int key = kt0 + 32 * j + (r & 3) + 8 * (r >> 2) + 4 * hi;
                    if (key > qrow) s[j][r] = -INFINITY;
                }
        }
        float mx = s[0][0];
#pragma unroll
        for (int j = 0; j < NH; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[j][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 32));                          // the other half of this query's keys
        const float m_new = fmaxf(m_run, mx);                        // finite: key 0 is visible to every query
        const float alpha = __builtin_amdgcn_exp2f((m_run - m_new) * c_log2);
        const float mc = m_new * c_log2;
        float psum = 0.f;
        bf16x8 pf[2 * NH];                                           // P^T fragments, 16 keys each
#pragma unroll
        for (int t = 0; t < 2 * NH; ++t)
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t >> 1][8 * (t & 1) + e], c_log2, -mc));
                psum += p;
                pf[t][e] = (bf16_t)p;
            }
        l_run = l_run * alpha + psum;
        m_run = m_new;
        if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {        // skip the rescale while no maximum moved
#pragma unroll
            for (int d = 0; d < 4; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) oacc[d][r] *= alpha;
        }
        // ---- O^T += V^T . P^T: rows 16 t + 4 hi + tq and 8 further on, chunk 4 d + 2 gq + tp / 2
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int t = 0; t < 2 * NH; ++t) {
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4 __attribute__((address_space(3)))*)(buf + V_AT + (v_at ^ (64 * d)) + 4096 * t));
                const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4 __attribute__((address_space(3)))*)(buf + V_AT + (v_at8 ^ (64 * d)) + 4096 * t));
                typedef short s16x8 __attribute__((ext_vector_type(8)));
                const s16x8 vv = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vv), pf[t], oacc[d], 0, 0, 0);
            }
    };
    load_tile(buf0, 0);
    landed();
    for (int it = 0; it < ntiles; it += 2) {
        if (it + 1 < ntiles) load_tile(buf1, (it + 1) * kTileKeys);
        work(buf0, it * kTileKeys);
        landed();
        if (it + 1 >= ntiles) break;
        if (it + 2 < ntiles) load_tile(buf0, (it + 2) * kTileKeys);
        work(buf1, (it + 1) * kTileKeys);
        landed();
    }

    // ---- normalise and store: lane holds dims 32*d + 8*(r>>2) + 4*hi + (r&3) of its query
    const float l_tot = l_run + __shfl_xor(l_run, 32);
    if (qrow >= L) return;
    const float inv = 1.f / l_tot;
    unsigned short* op = out + ((size_t)(s0 + qrow) * Hq + hq) * 128 + 4 * hi;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            u16x4 o4;
#pragma unroll
            for (int e = 0; e < 4; ++e) o4[e] = __builtin_bit_cast(unsigned short, (bf16_t)(oacc[d][4 * rq + e] * inv));
            *(u16x4*)(op + 32 * d + 8 * rq) = o4;
        }
}

}  // namespace ql

using namespace ql;

extern "C" int ql_attn_prefill(const void* q, const void* k, const void* v, const int* cu_seqlens, void* out, float scale,
                               int num_seqs, int max_seqlen, int Hq, int Hkv, int head_dim, void* stream) {
    if (num_seqs < 0 || max_seqlen < 0 || Hq <= 0 || Hkv <= 0 ||
        (num_seqs > 0 && max_seqlen > 0 && (!q || !k || !v || !cu_seqlens || !out))) {
        set_error("ql_attn_prefill: bad argument");
        return QL_EINVAL;
    }
    if (head_dim != 128 || Hq % Hkv) { set_error("ql_attn_prefill: head_dim must be 128 and Hq %% Hkv == 0"); return QL_ESHAPE; }
    const int kv_group = Hq / Hkv;
    const int G = (kv_group % 4 == 0) ? 4 : (kv_group % 2 == 0) ? 2 : 1;     // query heads per workgroup
    if (num_seqs == 0 || max_seqlen == 0) return QL_OK;
    if (num_seqs > 65535 || Hq / G > 65535) { set_error("ql_attn_prefill: too many sequences or heads"); return QL_ESHAPE; }
    const int qrows = 128 / G, blocks = (max_seqlen + qrows - 1) / qrows;
    const RowGrid rg = row_grid(blocks, num_seqs, Hq / G);
    dim3 grid(rg.x, rg.y, rg.z), block(256);
    const float c = scale * 1.4426950408889634f;
    hipStream_t s = as_stream(stream);
    const bool dma = ((uintptr_t)k | (uintptr_t)v) % 16 == 0;
#define QL_PF(G_) do { if (dma) QL_PF_(G_, true); else QL_PF_(G_, false); } while (0)
#define QL_PF_(G_, DMA_)                                                                                       \
    hipLaunchKernelGGL((attn_prefill_kernel<G_, DMA_>), grid, block, 0, s, (const unsigned short*)q, (const unsigned short*)k, \
                       (const unsigned short*)v, cu_seqlens, (unsigned short*)out, c, Hq, Hkv, kv_group, blocks, num_seqs, rg.run)
    if (G == 1) QL_PF(1); else if (G == 2) QL_PF(2); else QL_PF(4);
#undef QL_PF
#undef QL_PF_
    QL_CHECK_LAUNCH("ql_attn_prefill");
    return QL_OK;
}
