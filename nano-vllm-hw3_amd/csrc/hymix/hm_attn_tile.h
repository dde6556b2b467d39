// The tile loop of paged key/value attention on the matrix cores (bf16 operands, f32 accumulation).
//
// A wave owns 32 query rows that read the same key/value head (the query heads of one group, token after token).  Both
// products are computed transposed, so that everything a softmax row needs sits in one lane pair:
//   S^T = K . Q^T    (A = key rows of a 64-key tile from LDS, B = Q^T kept in registers): lane l holds query (l & 31)
//                    and the keys (r & 3) + 8 (r >> 2) + 4 (l >> 5) of a 32-key half;
//   O^T += V^T . P^T (A = the value tile through the transposing LDS read, B = the lane's own probabilities): the
//                    accumulator keeps query (l & 31) per lane, so the online rescale is lane-local.
// Head sizes are padded to 32 NBK / 32 NBV columns of zeros; LDS rows are an odd number of 16-byte chunks apart.  The
// next tile's global loads are issued before the current tile's math and land in LDS after it.  A tile never straddles
// a cache block (block_size % 64 == 0); rows past the last needed key are read from that key's row and masked.
//
// Tiles are 64 keys from key 0, whatever the step brings, so the order of every sum depends on positions alone.  With a
// window the walk is over a list: the tiles that hold kept first tokens, then the tiles from the window's start; tiles
// between are skipped (every score in them is masked, and a masked score adds an exact zero).  With pooled blocks the
// list starts with tiles of 64 pooled entries (block means, read from the pooled caches row by row through the block
// table); an entry is masked for the rows whose window has not yet passed its block.
#pragma once
#include "hm_common.h"

namespace hm {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef unsigned short u16x4 __attribute__((ext_vector_type(4)));
typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef short s16x8 __attribute__((ext_vector_type(8)));

constexpr int kTileKeys = 64;

template <int NB>
struct TileGeom {
    static constexpr int P = 32 * NB, CH = P / 8, RS = P * 2 + 16, LDS_BYTES = kTileKeys * RS;
};

// The list of tiles of TK keys a group of rows walks.  keep_tiles tiles from key 0, then tiles from key win_lo (a multiple of
// TK, >= TK keep_tiles) up to the causal end.
template <int TK = kTileKeys>
struct TileWalk {
    int pool_tiles, n_pool, keep_tiles, win_lo;
    // first key of token tile vt (vt >= pool_tiles); a pooled tile vt < pool_tiles starts at entry TK vt
    __device__ __forceinline__ int key0(int vt) const {
        const int u = vt - pool_tiles;
        return u < keep_tiles ? u * TK : win_lo + (u - keep_tiles) * TK;
    }
    __device__ __forceinline__ int count(int n_keys) const {
        return pool_tiles + keep_tiles + (n_keys - win_lo + TK - 1) / TK;
    }
};

// min_pos / max_pos = the smallest / largest position among the rows that walk together
// chunk > 0: a row also sees nothing before the start of its own chunk of `chunk` positions
template <int TK = kTileKeys>
__device__ __forceinline__ TileWalk<TK> make_walk(int min_pos, int max_pos, int window, int keep_first, int pool, int chunk = 0) {
    TileWalk<TK> w;
    w.n_pool = pooled_seen(max_pos, window, pool);
    w.pool_tiles = (w.n_pool + TK - 1) / TK;
    int lo = window > 0 ? max(0, min_pos - window + 1) : 0;
    if (chunk > 0) lo = max(lo, min_pos / chunk * chunk);
    w.win_lo = lo / TK * TK;
    w.keep_tiles = window > 0 ? min((keep_first + TK - 1) / TK, w.win_lo / TK) : 0;
    return w;
}

// The mask of a tile of 32 PARTS keys, counted from a lane's first: a row sees the last `near` keys up to its own, key `ahead`, and those up to
// `kept`.  LATER / EARLIER: whether the tile has keys behind some row's own, and keys in front of some row's window (or chunk); both are
// uniform over a wave, and most masked tiles have one kind.  Without && and ||: with them the compiler branches lane by lane, 626 instructions
// per tile of 64 (162 with both kinds in one comparison, 64 and 96 in two).
template <bool LATER, bool EARLIER, int PARTS>
__device__ __forceinline__ void mask_side(f32x16 (&s)[PARTS], int ahead, int near, int kept) {
    asm volatile("");                                      // (a branch around it, not selects that every tile runs)
    const int first = ahead - near;
#pragma unroll
    for (int j = 0; j < PARTS; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int c = 32 * j + (r & 3) + 8 * (r >> 2);
            if (LATER) s[j][r] = c <= ahead ? s[j][r] : -INFINITY;
            if (EARLIER) s[j][r] = ((c > first) | (c <= kept)) ? s[j][r] : -INFINITY;
        }
}

template <int PARTS>
__device__ __forceinline__ void mask_tile(f32x16 (&s)[PARTS], bool later, bool earlier, int ahead, int near, int kept) {
    if (later) mask_side<true, false>(s, ahead, near, kept);
    if (earlier) mask_side<false, true>(s, ahead, near, kept);
}

// Walks tiles [vt_lo, vt_hi) of `walk` for the calling lane's query row at position row_pos; wave_min_pos / wave_max_pos = the
// smallest / largest position of the wave's rows.  Every wave of the workgroup must call this with the same tiles.  On return oacc holds the
// unnormalised output (lane: query l & 31, columns 32 d + 8 (r >> 2) + 4 (l >> 5) + (r & 3)), m_run the row maximum of
// the raw scores (-inf if the row saw no key) and l_tot the sum of exp2((s - m_run) * c_log2) over the row.
// MODE kSigmoid: the weight of a visible key is sigmoid(score * scale + bias), pre = the row's bias times log2(e); the weights
// are not normalised, oacc is the output itself, m_run = 0 and l_tot = 1.  MODE kSoftcap: scores are bent to
// cap tanh(score * scale / cap) before the mask; pre = 2 log2(e) scale / cap, c_log2 = cap log2(e), and "raw scores" are the tanh.
constexpr int kSoftmax = 0, kSigmoid = 1, kSoftcap = 2;

template <int NBK, int NBV, int WAVES, int MODE = kSoftmax>
__device__ __forceinline__ void kv_tile_loop(const unsigned short* __restrict__ qrow, const unsigned short* __restrict__ kc,
                                             const unsigned short* __restrict__ vc, const int32_t* __restrict__ table, int D, int V,
                                             int G, int g, int block_size, TileWalk<> walk, int vt_lo, int vt_hi, int n_keys,
                                             int row_pos, int wave_min_pos, int wave_max_pos, int window, int keep_first, float c_log2,
                                             const unsigned short* __restrict__ kp, const unsigned short* __restrict__ vp,
                                             int pool, int pool_rows, unsigned char* lds_k, unsigned char* lds_v, f32x16 (&oacc)[NBV], float& m_run,
                                             float& l_tot, int chunk = 0, float pre = 0.f) {
    constexpr bool SIG = MODE == kSigmoid;
    typedef TileGeom<NBK> GK;
    typedef TileGeom<NBV> GV;
    constexpr int NLK = GK::CH / WAVES, NLV = GV::CH / WAVES;      // 16-byte chunks a thread stages per tile
    const int tid = threadIdx.x, lane = tid & 63, l31 = lane & 31, hi = lane >> 5;

    bf16x8 qf[2 * NBK];                                    // Q^T as the B operand: k-step ks = columns 16 ks + 8 hi .. +8
#pragma unroll
    for (int ks = 0; ks < 2 * NBK; ++ks) {
        const int c0 = 16 * ks + 8 * hi;
        i32x4 v = {0, 0, 0, 0};
        if (c0 < D) v = *(const i32x4*)(qrow + c0);
        qf[ks] = __builtin_bit_cast(bf16x8, v);
    }

    i32x4 kreg[NLK], vreg[NLV];
    auto load_tile = [&](int vt) {
        if (vt < walk.pool_tiles) {                        // 64 pooled entries, each found through the block table
#pragma unroll
            for (int j = 0; j < NLK; ++j) {
                const int c = tid + 64 * WAVES * j;
                const int row = c / GK::CH, ch = c % GK::CH;
                const int e = min(vt * kTileKeys + row, walk.n_pool - 1);
                const size_t prow = (size_t)table[e / pool_rows] * pool_rows + e % pool_rows;
                i32x4 v = {0, 0, 0, 0};
                if (ch * 8 < D) v = *(const i32x4*)(kp + (prow * G + g) * D + ch * 8);
                kreg[j] = v;
            }
#pragma unroll
            for (int j = 0; j < NLV; ++j) {
                const int c = tid + 64 * WAVES * j;
                const int row = c / GV::CH, ch = c % GV::CH;
                const int e = min(vt * kTileKeys + row, walk.n_pool - 1);
                const size_t prow = (size_t)table[e / pool_rows] * pool_rows + e % pool_rows;
                i32x4 v = {0, 0, 0, 0};
                if (ch * 8 < V) v = *(const i32x4*)(vp + (prow * G + g) * V + ch * 8);
                vreg[j] = v;
            }
            return;
        }
        const int kt0 = walk.key0(vt);
        const size_t row0 = (size_t)table[kt0 / block_size] * block_size + (kt0 % block_size);
#pragma unroll
        for (int j = 0; j < NLK; ++j) {
            const int c = tid + 64 * WAVES * j;
            const int row = c / GK::CH, ch = c % GK::CH;
            const int key = min(kt0 + row, n_keys - 1) - kt0;
            i32x4 v = {0, 0, 0, 0};
            if (ch * 8 < D) v = *(const i32x4*)(kc + ((row0 + key) * G + g) * D + ch * 8);
            kreg[j] = v;
        }
#pragma unroll
        for (int j = 0; j < NLV; ++j) {
            const int c = tid + 64 * WAVES * j;
            const int row = c / GV::CH, ch = c % GV::CH;
            const int key = min(kt0 + row, n_keys - 1) - kt0;
            i32x4 v = {0, 0, 0, 0};
            if (ch * 8 < V) v = *(const i32x4*)(vc + ((row0 + key) * G + g) * V + ch * 8);
            vreg[j] = v;
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (int j = 0; j < NLK; ++j) {
            const int c = tid + 64 * WAVES * j;
            *(i32x4*)(lds_k + (c / GK::CH) * GK::RS + (c % GK::CH) * 16) = kreg[j];
        }
#pragma unroll
        for (int j = 0; j < NLV; ++j) {
            const int c = tid + 64 * WAVES * j;
            *(i32x4*)(lds_v + (c / GV::CH) * GV::RS + (c % GV::CH) * 16) = vreg[j];
        }
    };

#pragma unroll
    for (int d = 0; d < NBV; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[d][r] = 0.f;
    m_run = -INFINITY;
    float l_run = 0.f;
    const int gq = (lane >> 4) & 1, ti = lane & 15, tq = ti >> 2, tp = ti & 3;      // transposed-read address pieces

    const int my_pool = pooled_seen(row_pos, window, pool);   // pooled entries this row sees
    const int chunk_lo = chunk > 0 ? row_pos / chunk * chunk : 0;
    const int near = window > 0 ? min(window, row_pos + 1 - chunk_lo) : row_pos + 1 - chunk_lo,
              kept = window > 0 ? min(keep_first - 1, row_pos) : -1;    // (the last of the kept ones that the row sees)
    const int wave_chunk_lo = chunk > 0 ? wave_max_pos / chunk * chunk : 0;
    load_tile(vt_lo);
    store_tile();
    __syncthreads();
#pragma unroll
    for (int ks = 0; ks < 2 * NBK; ++ks) asm volatile("" ::"v"(__builtin_bit_cast(i32x4, qf[ks])));   // loaded before the loop
    for (int vt = vt_lo; vt < vt_hi; ++vt) {
        const bool pooled = vt < walk.pool_tiles;
        const int kt0 = pooled ? vt * kTileKeys : walk.key0(vt);
        const bool more = vt + 1 < vt_hi;
        if (more) load_tile(vt + 1);

        f32x16 s[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[j][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 2 * NBK; ++ks) {
                const bf16x8 kf = *(const bf16x8*)(lds_k + (32 * j + l31) * GK::RS + (2 * ks + hi) * 16);
                s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[j], 0, 0, 0);
            }
        }
        if (SIG) {                                           // the logit in log2 units, before the mask
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[j][r] = __builtin_fmaf(s[j][r], c_log2, pre);
        }
        if (MODE == kSoftcap) {                              // tanh(z) = 1 - 2 / (1 + e^2z); both infinities come out right
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    s[j][r] = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[j][r] * pre));
        }
        // (a tile that every row of the wave sees whole needs no mask; a pooled one hides what the row's window has not passed yet)
        mask_tile(s, pooled | (kt0 + kTileKeys - 1 > wave_min_pos), !pooled & ((window > 0 & wave_max_pos - kt0 >= window) | (kt0 < wave_chunk_lo)),
                  (pooled ? my_pool - 1 : row_pos) - kt0 - 4 * hi, near, kept - kt0 - 4 * hi);
        bf16x8 pf[2][2];
        if (SIG) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 8; ++e)          // a masked logit is -inf: exp2(+inf) = inf and the weight is 0
                        pf[j][t][e] = (bf16_t)__builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-s[j][8 * t + e]));
        } else {
            float mx = s[0][0];
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[j][r]);
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float m_new = fmaxf(m_run, mx);
            // a row may have seen nothing yet (its window starts in a later tile): no rescale, and every weight is zero
            const bool none = m_new == -INFINITY;
            const float alpha = none ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * c_log2);
            const float mc = none ? 0.f : m_new * c_log2;
            float psum = 0.f;
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int e = 0; e < 8; ++e) {
                        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[j][8 * t + e], c_log2, -mc));
                        psum += p;
                        pf[j][t][e] = (bf16_t)p;
                    }
            l_run = l_run * alpha + psum;
            m_run = m_new;
            if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
                for (int d = 0; d < NBV; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[d][r] *= alpha;
            }
        }
#pragma unroll
        for (int d = 0; d < NBV; ++d)
#pragma unroll
            for (int j = 0; j < 2; ++j)
#pragma unroll
                for (int t = 0; t < 2; ++t) {
                    const int r0 = 32 * j + 16 * t + 4 * hi;
                    const int c0 = 4 * d + 2 * gq;
                    const int off = (c0 + (tp >> 1)) * 16 + 8 * (tp & 1);
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (s16x4 __attribute__((address_space(3)))*)(lds_v + (r0 + tq) * GV::RS + off));
                    const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                        (s16x4 __attribute__((address_space(3)))*)(lds_v + (r0 + 8 + tq) * GV::RS + off));
                    const s16x8 vv = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                    oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vv), pf[j][t], oacc[d], 0, 0, 0);
                }
        __syncthreads();
        if (more) {
            store_tile();
            __syncthreads();
        }
    }
    l_tot = l_run + __shfl_xor(l_run, 32);
    if (SIG) { m_run = 0.f; l_tot = 1.f; }
}

// The same walk for head sizes of exactly 32 NBK and 32 NBV channels, whose tiles go from global memory straight to LDS: two
// buffers, one barrier per tile.  The loop above holds a tile in registers on its way (a wave then has 350 of them and its SIMD
// to itself, with nothing to fill its waits; held to 256 it takes 110 us where this one took 73 and the first 174: eight
// prompts of about 1000 tokens, 16 / 8 heads of 128, a window of 512, capped scores).  What is left is the vector unit's: three
// exponentials or reciprocals per capped score; 55 % of a SIMD's cycles are vector instructions, 20 % products, and a fifth of the time is
// the last workgroups' (two rounds of unequal ones).  Masks of one side, and pooled blocks in the same form, took 32 such prompts from 224 to
// 213 us, two of 3000 to 4000 tokens from 71 to 66.5, heads of 64 without a cap from 50 to 44.  Scores are what the loop above makes of
// them, bit for bit: with the cap's last multiply-add folded into what a score is worth, 1 to 4 % faster, the maximum that is taken off was
// rounded to 2^-24 of the cap and not of itself, and with a cap of 50 one result in 650 differed by a bf16
// rounding.  Tiles of 32 keys, which fit three waves, and cache blocks looked up a tile ahead measured the same.
// A row of 2 P bytes is kept in 16-byte chunks, chunk c of row r at place c ^ swz(r): the 16 lanes of a 16-byte read (rows
// that differ mod 16, one chunk) and the 32 of a transposed read (four rows, four chunks) then touch every bank once.  A
// wave none of whose rows sees a tile leaves it out: a masked score would add an exact zero.
constexpr int kSlimKeys = 64, kSlimParts = kSlimKeys / 32;

template <int NB>
struct SlimGeom {
    static constexpr int P = 32 * NB, CH = P / 8, RB = 2 * P, BYTES = kSlimKeys * RB, PIECES = BYTES / 1024;
    __device__ static __forceinline__ int swz(int r) {
        return CH % 16 == 0 ? ((r & 3) << 2 | (r >> 2 & 3)) : CH % 8 == 0 ? ((r >> 1 & 1) << 2 | (r >> 2 & 3)) : (r >> 2 & 3);
    }
    __device__ static __forceinline__ int at(int r, int ch) { return RB * r + 16 * (ch ^ swz(r)); }
};

template <int NBK, int NBV, int MODE>
__device__ __forceinline__ void kv_slim_loop(const unsigned short* __restrict__ qrow, const unsigned short* __restrict__ kc,
                                             const unsigned short* __restrict__ vc, const int32_t* __restrict__ table, int G, int g,
                                             int block_size, TileWalk<kSlimKeys> walk, int nt, int n_keys, int row_pos, int wave_min_pos,
                                             int wave_max_pos, int window, int keep_first, float c_log2,
                                             const unsigned short* __restrict__ kp, const unsigned short* __restrict__ vp, int pool,
                                             int pool_rows, unsigned char* buf0, unsigned char* buf1, f32x16 (&oacc)[NBV], float& m_run,
                                             float& l_tot, int chunk, float pre) {
    constexpr bool SIG = MODE == kSigmoid;
    typedef SlimGeom<NBK> GK;
    typedef SlimGeom<NBV> GV;
    typedef __attribute__((address_space(1))) const void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;
    const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    bf16x8 qf[2 * NBK];                                    // Q^T as the B operand: k-step ks = columns 16 ks + 8 hi .. +8
#pragma unroll
    for (int ks = 0; ks < 2 * NBK; ++ks) qf[ks] = *(const bf16x8*)(qrow + 16 * ks + 8 * hi);

    // one tile: pieces of 1 KB, dealt to the four waves; lane l of a piece brings the chunk that belongs at 16 l.  A lane's pieces are a
    // whole number of 16 rows apart, so its chunk is the same in all of them, and its place in a whole tile is one number.
    auto lane_row = [&](auto geom) { return wave * (64 / decltype(geom)::CH) + lane / decltype(geom)::CH; };
    auto lane_chunk = [&](auto geom) { return (lane % decltype(geom)::CH) ^ decltype(geom)::swz(lane_row(geom)); };
    const unsigned k_place = 2u * ((unsigned)lane_row(GK()) * (unsigned)(G * GK::P) + 8u * (unsigned)lane_chunk(GK())),
                   v_place = 2u * ((unsigned)lane_row(GV()) * (unsigned)(G * GV::P) + 8u * (unsigned)lane_chunk(GV()));
    auto load_part = [&](auto geom, unsigned char* to, const unsigned short* src, const unsigned short* psrc, int vt, int kt0, size_t row0,
                         unsigned place) {
        typedef decltype(geom) GG;
        constexpr int RP = 64 / GG::CH;                    // rows of a piece
        static_assert(64 % GG::CH == 0 && 4 * RP % 16 == 0 && GG::PIECES % 4 == 0, "pieces of whole rows");
        typedef __attribute__((address_space(1))) const unsigned char* gbytes;
        if (vt >= walk.pool_tiles && kt0 + kSlimKeys <= n_keys) {
            const gbytes from = (gbytes)(src + (row0 * G + g) * GG::P);
#pragma unroll
            for (int i0 = 0; i0 < GG::PIECES; i0 += 4)
                __builtin_amdgcn_global_load_lds((gvoid*)(from + (size_t)(i0 * RP) * (size_t)(2 * G * GG::P) + place),
                                                 (lvoid*)(to + 1024 * (i0 + wave)), 16, 0, 0);
            return;
        }
        const int ch = lane_chunk(geom);
#pragma unroll
        for (int i0 = 0; i0 < GG::PIECES; i0 += 4) {
            const int row = lane_row(geom) + i0 * RP;
            const unsigned short* from;
            if (vt < walk.pool_tiles) {                    // pooled entries, each found through the block table
                const int e = min(vt * kSlimKeys + row, walk.n_pool - 1);
                from = psrc + (((size_t)table[e / pool_rows] * pool_rows + e % pool_rows) * G + g) * GG::P;
            } else {
                from = src + ((row0 + min(row, n_keys - 1 - kt0)) * G + g) * GG::P;
            }
            __builtin_amdgcn_global_load_lds((gvoid*)(from + 8 * ch), (lvoid*)(to + 1024 * (i0 + wave)), 16, 0, 0);
        }
    };
    auto load_tile = [&](unsigned char* buf, int vt) {
        int kt0 = 0;
        size_t row0 = 0;
        if (vt >= walk.pool_tiles) {                       // (a tile lies in one cache block)
            kt0 = __builtin_amdgcn_readfirstlane(walk.key0(vt));
            const int page = kt0 / block_size;
            row0 = (size_t)table[page] * block_size + (kt0 - page * block_size);
        }
        load_part(GK(), buf, kc, kp, vt, kt0, row0, k_place);
        load_part(GV(), buf + GK::BYTES, vc, vp, vt, kt0, row0, v_place);
    };
    auto landed = [&]() {
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
    };

#pragma unroll
    for (int d = 0; d < NBV; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) oacc[d][r] = 0.f;
    m_run = -INFINITY;
    float l_run = 0.f;
    const int gq = (lane >> 4) & 1, ti = lane & 15, tq = ti >> 2, tp = ti & 3;      // transposed-read address pieces
    // a chunk's number enters its place by exclusive or: the reads' addresses are one base each, changed in the chunk's bits
    const int k_at = GK::at(l31, hi), v_at = GV::at(4 * hi + tq, 2 * gq + (tp >> 1)) + 8 * (tp & 1),
              v_at8 = GV::at(4 * hi + tq + 8, 2 * gq + (tp >> 1)) + 8 * (tp & 1);
    const int my_pool = pooled_seen(row_pos, window, pool);
    const int chunk_lo = chunk > 0 ? row_pos / chunk * chunk : 0;
    const int near = window > 0 ? min(window, row_pos + 1 - chunk_lo) : row_pos + 1 - chunk_lo,
              kept = window > 0 ? min(keep_first - 1, row_pos) : -1;    // (the last of the kept ones that the row sees)
    const int wave_chunk_lo = chunk > 0 ? wave_max_pos / chunk * chunk : 0, wave_chunk_first = chunk > 0 ? wave_min_pos / chunk * chunk : 0;

    auto work = [&](const unsigned char* buf, int vt) {
        const bool pooled = vt < walk.pool_tiles;
        const int kt0 = pooled ? vt * kSlimKeys : walk.key0(vt), kt1 = kt0 + kSlimKeys - 1;
        if (!pooled && (kt0 > wave_max_pos || kt1 < wave_chunk_first || (window > 0 && wave_min_pos - kt1 >= window && kt0 >= keep_first)))
            return;
        f32x16 s[kSlimParts];
#pragma unroll
        for (int j = 0; j < kSlimParts; ++j) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[j][r] = 0.f;
#pragma unroll
            for (int ks = 0; ks < 2 * NBK; ++ks) {
                const bf16x8 kf = *(const bf16x8*)(buf + (k_at ^ (32 * ks)) + 32 * GK::RB * j);        // row 32 j + l31, chunk 2 ks + hi
                s[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[ks], s[j], 0, 0, 0);
            }
        }
#pragma unroll
        for (int j = 0; j < kSlimParts; ++j) {
            if (SIG) {                                       // the logit in log2 units, before the mask
#pragma unroll
                for (int r = 0; r < 16; ++r) s[j][r] = __builtin_fmaf(s[j][r], c_log2, pre);
            }
            if (MODE == kSoftcap) {                          // tanh(z) = 1 - 2 / (1 + e^2z); both infinities come out right
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    s[j][r] = 1.f - 2.f * __builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(s[j][r] * pre));
            }
        }
        // (a tile that every row of the wave sees whole needs no mask; a pooled one hides what the row's window has not passed yet.  One form for
        // both takes 40 registers less: 64 channels 47.8 -> 45.2 us, 128 under a cap 70.5 -> 69.3; but 128 without a cap 56.9 -> 58.0)
        const bool later = kt1 > wave_min_pos, earlier = (window > 0 && wave_max_pos - kt0 >= window) || kt0 < wave_chunk_lo;
        if constexpr (MODE == kSoftmax && NBK == 4 && NBV == 4) {
            if (pooled) {
#pragma unroll
                for (int j = 0; j < kSlimParts; ++j)
#pragma unroll
                    for (int r = 0; r < 16; ++r)
                        if (kt0 + 32 * j + (r & 3) + 8 * (r >> 2) + 4 * hi >= my_pool) s[j][r] = -INFINITY;
            } else {
                mask_tile(s, later, earlier, row_pos - kt0 - 4 * hi, near, kept - kt0 - 4 * hi);
            }
        } else {
            mask_tile(s, pooled | later, !pooled & earlier, (pooled ? my_pool - 1 : row_pos) - kt0 - 4 * hi, near, kept - kt0 - 4 * hi);
        }
        bf16x8 pf[2 * kSlimParts];
        if (SIG) {
#pragma unroll
            for (int t = 0; t < 2 * kSlimParts; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e)              // a masked logit is -inf: exp2(+inf) = inf and the weight is 0
                    pf[t][e] = (bf16_t)__builtin_amdgcn_rcpf(1.f + __builtin_amdgcn_exp2f(-s[t >> 1][8 * (t & 1) + e]));
        } else {
            float mx = s[0][0];
#pragma unroll
            for (int j = 0; j < kSlimParts; ++j)
#pragma unroll
                for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[j][r]);
            mx = fmaxf(mx, __shfl_xor(mx, 32));
            const float m_new = fmaxf(m_run, mx);
            const bool none = m_new == -INFINITY;            // the row has seen nothing yet: no rescale, and every weight is zero
            const float alpha = none ? 1.f : __builtin_amdgcn_exp2f((m_run - m_new) * c_log2);
            const float mc = none ? 0.f : m_new * c_log2;
            float psum = 0.f;
#pragma unroll
            for (int t = 0; t < 2 * kSlimParts; ++t)
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t >> 1][8 * (t & 1) + e], c_log2, -mc));
                    psum += p;
                    pf[t][e] = (bf16_t)p;
                }
            l_run = l_run * alpha + psum;
            m_run = m_new;
            if (__builtin_amdgcn_ballot_w64(alpha != 1.f) != 0) {
#pragma unroll
                for (int d = 0; d < NBV; ++d)
#pragma unroll
                    for (int r = 0; r < 16; ++r) oacc[d][r] *= alpha;
            }
        }
#pragma unroll
        for (int d = 0; d < NBV; ++d)
#pragma unroll
            for (int t = 0; t < 2 * kSlimParts; ++t) {
                // rows 16 t + 4 hi + tq and 8 further on, chunk 4 d + 2 gq + tp / 2
                const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4 __attribute__((address_space(3)))*)(buf + GK::BYTES + (v_at ^ (64 * d)) + 16 * GV::RB * t));
                const s16x4 hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (s16x4 __attribute__((address_space(3)))*)(buf + GK::BYTES + (v_at8 ^ (64 * d)) + 16 * GV::RB * t));
                const s16x8 vv = {lo[0], lo[1], lo[2], lo[3], hi4[0], hi4[1], hi4[2], hi4[3]};
                oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, vv), pf[t], oacc[d], 0, 0, 0);
            }
    };
    load_tile(buf0, 0);
    landed();
    for (int vt = 0; vt < nt; vt += 2) {
        if (vt + 1 < nt) load_tile(buf1, vt + 1);
        work(buf0, vt);
        landed();
        if (vt + 1 >= nt) break;
        if (vt + 2 < nt) load_tile(buf0, vt + 2);
        work(buf1, vt + 1);
        landed();
    }
    l_tot = l_run + __shfl_xor(l_run, 32);
    if (SIG) { m_run = 0.f; l_tot = 1.f; }
}

}  // namespace hm
