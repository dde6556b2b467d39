// Latent attention on the matrix cores, portions of any length: a workgroup of four waves owns 128 consecutive
// query rows of ONE sequence's portion (rows run token by token, head by head, so a row's last visible key is the
// position of its token) and walks the cache tiles up to the last row's position.
#include "../row_deal.h"
#include "sm_latent_tile.h"

namespace sm {

// SLIM: rows of exactly 32 NB columns on 16 bytes, in the loop of 32-key tiles (latent_slim_loop)
template <int NB, int NBV, bool SLIM>
__global__ __launch_bounds__(256, SLIM ? 2 : 1) void latent_attn_tiles_kernel(const unsigned short* __restrict__ q,
                                                                const unsigned short* __restrict__ cache,
                                                                const int32_t* __restrict__ block_tables,
                                                                const int32_t* __restrict__ qstart,
                                                                const int32_t* __restrict__ seq_pos0,
                                                                unsigned short* __restrict__ o, float c_log2, int H, int R,
                                                                int block_size, int max_blocks, int RV, int window,
                                                                const float* __restrict__ sink, int B, int tiles, int run) {
    // (the slim loop has two buffers of half a tile)
    __shared__ __attribute__((aligned(1024))) unsigned char lds[SLIM ? SlimGeom<NB>::BYTES : TileGeom<NB>::LDS_BYTES];
    __shared__ __attribute__((aligned(1024))) unsigned char lds2[SLIM ? SlimGeom<NB>::BYTES : 16];
    const RowTile rt = row_tile(blockIdx.x, blockIdx.y, blockIdx.z, run, tiles, B, 1);
    if (rt.b < 0) return;
    const int b = rt.b;
    const int q0 = qstart[b], rows = (qstart[b + 1] - q0) * H;
    const int tile0 = row_first(run, rt.tile, tiles, rows, 128);               // heaviest tiles first
    if (tile0 < 0 || tile0 >= rows) return;
    const int pos0 = seq_pos0[b];
    const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = tile0 + 32 * wave + l31;
    const int rc = min(r, rows - 1);
    const int row_pos = pos0 + rc / H;
    const int wave_min_pos = pos0 + min(tile0 + 32 * wave, rows - 1) / H;
    const int k_hi = pos0 + min(tile0 + 127, rows - 1) / H + 1;
    // with a window the walk starts at the tile that holds the first key the workgroup's first row sees
    constexpr int TK = SLIM ? kSlimKeys : kTileKeys;
    const int k_lo = window > 0 ? max(0, pos0 + tile0 / H - window + 1) / TK * TK : 0;
    f32x16 oacc[NBV];
    float m_run, l_tot;
    const unsigned short* qrow = q + ((size_t)q0 * H + rc) * R;
    const int32_t* table = block_tables + (size_t)b * max_blocks;
    if constexpr (SLIM) {
        const int wave_max_pos = pos0 + min(tile0 + 32 * wave + 31, rows - 1) / H;
        latent_slim_loop<NB, NBV, 4>(qrow, cache, table, block_size, k_lo, k_hi, row_pos, wave_min_pos, wave_max_pos, c_log2, window, lds, lds2,
                                  oacc, m_run, l_tot);
    } else {
        latent_tile_loop<NB, NBV, 4>(qrow, cache, table, R, block_size, k_lo, k_hi, row_pos, wave_min_pos, c_log2, window, lds, oacc, m_run,
                                     l_tot);
    }
    if (r >= rows) return;
    const float inv = sink ? sink_inv(m_run * c_log2, l_tot, sink[r % H]) : 1.f / l_tot;
    unsigned short* op = o + ((size_t)q0 * H + r) * RV + 4 * hi;
#pragma unroll
    for (int d = 0; d < NBV; ++d)
#pragma unroll
        for (int rq = 0; rq < 4; ++rq) {
            if (32 * d + 8 * rq + 4 * hi >= RV) continue;
            u16x4 o4;
#pragma unroll
            for (int e = 0; e < 4; ++e) o4[e] = __builtin_bit_cast(unsigned short, (bf16_t)(oacc[d][4 * rq + e] * inv));
            *(u16x4*)(op + 32 * d + 8 * rq) = o4;
        }
}

}  // namespace sm

using namespace sm;

extern "C" int sm_latent_attn_tiles(const void* q, const void* cache, const int32_t* block_tables, const int32_t* qstart,
                                    const int32_t* seq_pos0, void* o, float scale, int B, int max_q, int H, int R, int block_size,
                                    int max_blocks, int RV, int window, const float* sink, void* stream) {
    if (RV <= 0) RV = R;
    if (B < 0 || max_q < 0 || H < 1 || R < 1 || RV > R || window < 0 || block_size < 1 || max_blocks < 1 ||
        (B > 0 && max_q > 0 && (!q || !cache || !block_tables || !qstart || !seq_pos0 || !o))) {
        set_error("sm_latent_attn_tiles: bad argument");
        return SM_EINVAL;
    }
    if (R % 8 || RV % 4 || R > 256 || block_size % 64 || B > 65535) {
        set_error("sm_latent_attn_tiles: needs R %% 8 == 0, R <= 256, block_size %% 64 == 0, at most 65535 sequences");
        return SM_ESHAPE;
    }
    if (B == 0 || max_q == 0) return SM_OK;
    const int64_t tiles = ((int64_t)max_q * H + 127) / 128;
    const RowGrid rg = row_grid(tiles, B, 1);
    dim3 grid(rg.x, rg.y, rg.z), block(256);
    const float c = scale * 1.4426950408889634f;
    hipStream_t s = as_stream(stream);
    const int nb = (R + 31) / 32, nbv = (RV + 31) / 32;
    // Rows whose 256 columns are all values need more than the 256 registers of two waves per SIMD and spill: that pays only where two
    // workgroups share a CU.  Where a CU has one, the other loop's steps of 64 keys are half as many (us, other loop / this one, 16
    // heads: 6 prompts of 195 to 411 tokens 34 / 42, 1 x 2000 115 / 151, 8 x 300 30 / 38, 1 x 4096 (512 tiles) 243 / 304; 16 x 300
    // (608 tiles) 56 / 45, 8 x 1000 150 / 126; 8 heads, 8 x 1000 (504 tiles) 82 / 95).
    const bool shared_cus = tiles * B > 512;
    // Rows of 32 to 96 columns with up to 64 values: the other loop has registers enough for the tile on its way, and without a window a
    // row tile's chain of steps is what counts as long as all of them run beside each other (us, other / this one: 8 heads, rows of 32
    // columns, 1 x 6000 97 / 106, 40 x 70 8.7 / 9.7; of 64, 1 x 2000 44 / 47, 2 x 1500 34 / 36; 16 heads, 8 x 300 12.0 / 11.9; of 64 + 32,
    // 32 heads, 1 x 2000 54 / 58).  Up to 512 row tiles, 768 where a sequence has half as many as fit (of 64, 16 heads, 1 x 6000 135 /
    // 141; of 64 + 32 152 / 164; short ones, 32 heads, 40 x 70 14.0 / 10.4); above, throughput counts (16 heads, 8 x 1100 42 / 36; 64
    // heads, 1 x 2000 70 / 60), and with a window, whose few steps do not lie in the loads' way (1 x 2000, window 256 17 / 13).
    const bool chain = window <= 0 && tiles * B <= (tiles >= 256 ? 768 : 512);
    const bool aligned = (uintptr_t)cache % 16 == 0;
#define SM_TILES(NB_, NBV_)                                                                                             \
    do {                                                                                                                \
        if (R == 32 * NB_ && aligned && (NBV_ < 8 || shared_cus) && !(NB_ <= 3 && NBV_ <= 2 && chain)) SM_TILES_(NB_, NBV_, true); \
        else SM_TILES_(NB_, NBV_, false);                                                                               \
    } while (0)
#define SM_TILES_(NB_, NBV_, SLIM_)                                                                                       \
    hipLaunchKernelGGL((latent_attn_tiles_kernel<NB_, NBV_, SLIM_>), grid, block, 0, s, (const unsigned short*)q,                 \
                       (const unsigned short*)cache, block_tables, qstart, seq_pos0, (unsigned short*)o, c, H, R, block_size, \
                       max_blocks, RV, window, sink, B, (int)tiles, rg.run)
    SM_BY_LATENT_SIZE(nb, nbv, SM_TILES);
#undef SM_TILES
#undef SM_TILES_
    SM_CHECK_LAUNCH("sm_latent_attn_tiles");
    return SM_OK;
}
