// Expert products for large groups (prefill) on the matrix cores, bf16: tiles of 64 MB rows of one expert (MB = 4 or 2 by the
// size of the groups) by 256 rows of its weights (128 gate and the 128 up rows of the same outputs, or 256 plain ones).
//
// Row r of a group is the same sum whatever else shares its tile, so every form agrees bit for bit on a row's products
// (same k order inside a 64-k step, same accumulation).
#include "sm_common.h"
#include "sm_moe_rows.h"

namespace sm {

constexpr int kBigRows = 128;                 // tiles are one or two times as many rows

// MODE 0: the down product, A = act rows;  1: gate and up with a gated activation (act_kind), 2: the up product alone with a
// plain one, both with A = h rows gathered by token.  B = the expert's weight rows in the tiled layout (4 KB blocks of 32 rows
// x 64 k in lane order, see seq_ops.tile_expert_weights).  in_wts != NULL (modes 1, 2): pair p's products are scaled by
// in_wts[p] before the activation (a weight on the expert's input).
//
// Four waves, two by two: a wave owns 32 MB rows by 128 weight rows.  Both operands of a 64-k step go from global memory
// straight to LDS (16 bytes per lane, no registers in between): the weights as they lie, a token row as eight 16-byte chunks,
// chunk c of row r at place c ^ (r / 2 & 7), which spreads the 16-byte reads of 16 lanes over the 64 banks.  Two LDS buffers: the
// loads of step k + 2 are issued as soon as every wave has read step k, one whole step ahead of their use, and a wave's
// fragments are read from LDS one 16-k product ahead, across the barrier too.  (The buffers are two arrays and the loop is
// unrolled by two, so that the compiler sees that a read of one does not wait for the loads into the other.)
//
// Bound by the matrix cores and the power they may draw (with weights of zeros the same products take 10 % less): 128 x 128 per wave
// needs half of what LDS delivers (smaller wave tiles need all of it).  32768 rows over 16 experts: gate and up of 2 x 1536 x 2048
// in 435 us (0.95 PFLOP/s), down in 252 us (0.82).  A tile takes about 8 us beside its products: nothing covers its first loads and its
// last stores.  Of 20 us that it was in gate and up, 4 were the pairs of its rows, fetched and divided one behind the other, and
// 9 the activation's kind, asked for at every output.
template <int MODE, int MB, bool DMA>
__global__ __launch_bounds__(256, 1) void moe_tiles_kernel(const unsigned short* __restrict__ a, const unsigned short* __restrict__ w,
                                                           const int32_t* __restrict__ row_pair, const int32_t* __restrict__ tile_expert,
                                                           unsigned short* __restrict__ out, int top, unsigned top_inv, int N, int K, int tiles, int nct, int cols, int segs,
                                                           float limit, float alpha, int act_kind, const float* __restrict__ in_wts) {
    constexpr bool GATE_UP = MODE == 1, FROM_TOKENS = MODE != 0;
    constexpr int ROWS = 64 * MB, A_BYTES = ROWS * 128, BUF = A_BYTES + 8 * 4096;
    constexpr int NA = 2 * MB;                                // 1 KB pieces of A a wave loads per step (and 8 of B)
    __shared__ __attribute__((aligned(1024))) unsigned char buf0[BUF];
    __shared__ __attribute__((aligned(1024))) unsigned char buf1[BUF];
    // Workgroups go to the eight dies in turn; a die takes two neighbouring row tiles and one of `segs` parts of their column tiles
    // before its next such unit, so that its L2 sees a row tile's activations several times and a column tile's weights twice.
    const int id = blockIdx.x >> 3, turn = id / (2 * cols), in_unit = id - turn * 2 * cols;
    const int unit = turn * 8 + (blockIdx.x & 7), rows2 = unit / segs;
    const int tile = rows2 * 2 + (in_unit & 1), ct = (unit - rows2 * segs) * cols + (in_unit >> 1);
    if (tile >= tiles || ct >= nct) return;
    const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // (the pairs of a lane's rows all at once, beside the expert: one behind the other they took longer than a tile's 12 first steps)
    int pair[NA];
    if (FROM_TOKENS) {
#pragma unroll
        for (int i = 0; i < NA; ++i) pair[i] = row_pair[tile * ROWS + 8 * (wave * NA + i) + (lane >> 3)];
    }
    const int e = tile_expert[tile];
    if (e < 0) return;                                        // (uniform over the workgroup)
    const int wr = wave >> 1, wc = wave & 1;
    const int nb32 = (N + 31) / 32, ksteps = (K + 63) / 64;

    // what this lane loads: rows 8 (wave NA + i) + lane / 8 of the tile, the chunk that belongs at place lane % 8
    const int chunk = (lane & 7) ^ (lane >> 4);               // (i even; i odd: chunk ^ 4)
    const unsigned short* arow[NA];
#pragma unroll
    for (int i = 0; i < NA; ++i) {
        const int row = tile * ROWS + 8 * (wave * NA + i) + (lane >> 3), ch = chunk ^ (4 * (i & 1));
        if (FROM_TOKENS) {                                    // pair / top: the product with 1 / top is at most one too large
            const unsigned p = (unsigned)max(pair[i], 0), q = top > 1 ? __umulhi(p, top_inv) : p;
            arow[i] = a + (size_t)(q - (q * (unsigned)top > p ? 1u : 0u)) * K + 8 * ch;
        } else {
            arow[i] = a + (size_t)row * K + 8 * ch;
        }
    }
    // weight blocks 2 wave and 2 wave + 1 of the tile's eight: gate blocks first, then up blocks (blocks past N: the last one)
    const unsigned short* bblk[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int blk = 2 * wave + j;
        const int nb = GATE_UP ? min(4 * ct + (blk & 3), nb32 - 1) + (blk >= 4 ? nb32 : 0) : min(8 * ct + blk, nb32 - 1);
        bblk[j] = w + (((size_t)e * (GATE_UP ? 2 : 1) * nb32 + nb) * ksteps) * 2048 + 8 * lane;
    }
    typedef i32x4 anywhere __attribute__((aligned(2)));
    typedef __attribute__((address_space(1))) const void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;
    auto bring = [&](const unsigned short* from, unsigned char* to) {
        if constexpr (DMA) __builtin_amdgcn_global_load_lds((gvoid*)from, (lvoid*)to, 16, 0, 0);
        else *(i32x4*)(to + 16 * lane) = *(const anywhere*)from;
    };
    auto load_a = [&](unsigned char* buf, int ks, int i) { bring(arow[i] + (size_t)ks * 64, buf + 1024 * (wave * NA + i)); };
    auto load_b = [&](unsigned char* buf, int ks, int i) {
        bring(bblk[i >> 2] + (size_t)ks * 2048 + 512 * (i & 3), buf + A_BYTES + 4096 * (2 * wave + (i >> 2)) + 1024 * (i & 3));
    };
    auto load_step = [&](unsigned char* buf, int ks) {
#pragma unroll
        for (int i = 0; i < NA; ++i) load_a(buf, ks, i);
#pragma unroll
        for (int i = 0; i < 8; ++i) load_b(buf, ks, i);
    };
    auto landed = [&]() {                                     // this wave's loads are in LDS, then everybody's
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
    };

    f32x16 acc[MB][4];
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[m][n][r] = 0.f;

    struct Frags { bf16x8 a[MB], b[4]; };
    const int a_base = (32 * MB * wr + l31) * 128, a_x = (l31 >> 1) & 7;
    auto read = [&](Frags& f, const unsigned char* buf, int s) {       // k = 32 hi + 8 s .. + 8 of the step
        const int place = 16 * ((4 * hi + s) ^ a_x);
#pragma unroll
        for (int m = 0; m < MB; ++m) f.a[m] = *(const bf16x8*)(buf + a_base + 4096 * m + place);
#pragma unroll
        for (int n = 0; n < 4; ++n) {
            const int blk = GATE_UP ? 2 * wc + (n & 1) + 4 * (n >> 1) : 4 * wc + n;
            f.b[n] = *(const bf16x8*)(buf + A_BYTES + 4096 * blk + 1024 * s + 16 * lane);
        }
    };
    auto multiply = [&](const Frags& f) {
#pragma unroll
        for (int m = 0; m < MB; ++m)
#pragma unroll
            for (int n = 0; n < 4; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[n], f.a[m], acc[m][n], 0, 0, 0);
    };

    // The order of a product's instructions: the next product's LDS reads one by one between the first MFMAs, then the loads of
    // the step after next.  Left alone the compiler puts the reads in front of their use, and every product waits for LDS.
    auto interleave = [&](int loads) {
#pragma unroll
        for (int i = 0; i < MB + 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);          // an MFMA
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);          // an LDS read
        }
#pragma unroll
        for (int i = 0; i < 3 * MB - 4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            if (loads) __builtin_amdgcn_sched_group_barrier(0x020, (NA + 8 + 3 * MB - 5) / (3 * MB - 4), 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    Frags f0, f1;
    const int full = K / 64, last = full - 1;                 // whole steps; a shorter one follows them
    auto step = [&](unsigned char* cur, unsigned char* nxt, int ks) {
        read(f1, cur, 1);
        multiply(f0);
        interleave(0);
        read(f0, cur, 2);
        multiply(f1);
        interleave(0);
        read(f1, cur, 3);
        multiply(f0);
        interleave(0);
        landed();                                             // the next step is there, and nobody reads this one any more
        read(f0, nxt, 0);
        load_step(cur, min(ks + 2, last));                    // (past the end: the last step again, which nobody reads)
        multiply(f1);
        interleave(NA + 8);
    };
    if (full > 0) {
        load_step(buf0, 0);
        landed();
        load_step(buf1, min(1, last));
        read(f0, buf0, 0);
        int ks = 0;
        for (; ks + 1 < full; ks += 2) {
            step(buf0, buf1, ks);
            step(buf1, buf0, ks + 1);
        }
        if (ks < full) step(buf0, buf1, ks);
        landed();
    }
    if (K % 64 != 0) {                                        // zeros past the end of a token's row (the weights end in zeros)
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            i32x4 v = {0, 0, 0, 0};
            if (full * 64 + 8 * (chunk ^ (4 * (i & 1))) + 8 <= K) v = *(const anywhere*)(arow[i] + (size_t)full * 64);
            *(i32x4*)(buf0 + 1024 * (wave * NA + i) + 16 * lane) = v;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) load_b(buf0, full, i);
        landed();
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            read(f0, buf0, s);
            multiply(f0);
        }
        __syncthreads();
    }

    // The products leave the matrix unit in bf16, as a GEMM's output would, and go through LDS (rows 0 .. 32 MB - 1 in buf0, the
    // others in buf1; 16-byte chunk c of row r at place c ^ (r & 31)), so that a thread finishes eight neighbouring outputs.
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        float iw = 1.f;
        if (FROM_TOKENS && in_wts) {
            const int p = row_pair[tile * ROWS + 32 * (MB * wr + m) + l31];
            if (p >= 0) iw = in_wts[p];
        }
#pragma unroll
        for (int n = 0; n < 4; ++n)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const int blk = GATE_UP ? 2 * wc + (n & 1) + 4 * (n >> 1) : 4 * wc + n;
                u16x4 o4;
#pragma unroll
                for (int r = 0; r < 4; ++r) o4[r] = __builtin_bit_cast(unsigned short, (bf16_t)(acc[m][n][4 * q + r] * iw));
                *(u16x4*)((wr ? buf1 : buf0) + (32 * m + l31) * 512 + 16 * ((4 * blk + q) ^ l31) + 8 * hi) = o4;
            }
    }
    __syncthreads();
    constexpr int CH = GATE_UP ? 16 : 32;                     // finished chunks per row
    // (the activation's kind is chosen once, not at every output)
    auto finish = [&](auto kind) {
        constexpr int ACT = decltype(kind)::value;
#pragma unroll 4
        for (int i = threadIdx.x; i < ROWS * CH; i += 256) {      // (rows without a pair too: nobody reads what they leave)
            const int row = i / CH, c = i % CH, lrow = row & (32 * MB - 1);
            const int col = (GATE_UP ? 128 : 256) * ct + 8 * c;
            const unsigned char* src = (row >= 32 * MB ? buf1 : buf0) + lrow * 512;
            bf16x8 x = *(const bf16x8*)(src + 16 * (c ^ (row & 31)));
            if (GATE_UP) {
                const bf16x8 u = *(const bf16x8*)(src + 16 * ((c + 16) ^ (row & 31)));
#pragma unroll
                for (int r = 0; r < 8; ++r) x[r] = (bf16_t)gated_act((float)x[r], (float)u[r], limit, alpha, ACT);
            } else if (MODE == 2) {
#pragma unroll
                for (int r = 0; r < 8; ++r) x[r] = (bf16_t)plain_act((float)x[r], ACT);
            }
            if (col < N) *(bf16x8*)(out + ((size_t)tile * ROWS + row) * N + col) = x;      // (N % 8 == 0)
        }
    };
    with_act<MODE>(act_kind, finish);
}

// The same tiles walked by as many workgroups as there are CUs (K a multiple of 128, operands on 16 bytes): the loads of a tile's last two
// steps are the first two of the next tile, so neither the first loads nor the stores of a tile find the matrix cores idle for longer than
// the epilogue's own arithmetic.  The products leave by 8 KB of LDS per wave, 32 rows at a time, beside the two buffers that are
// being filled.
//
// What a step's 2048 cycles of products per SIMD leave room for decides: 128 KB of LDS reads (1024 cycles), and 64 one-KB loads that take the
// CU's way to L2 for 16 cycles each.  All behind one barrier at three quarters of the step, as in moe_tiles_kernel, those stood in the
// way of the products for half a step; over half of it, and with nothing but a place and a uniform offset per load, gate and up of the
// figures above took 464 us for 500 (under the profiler), behind a barrier each for weights and activations 438.  Now 768 to 620
// thousand cycles for 421 of products; the clock falls with the idle cycles (2.2 GHz with weights of zeros, 1.9 with random ones), so that
// time is won more slowly than cycles.  Whole calls (us, moe_tiles_kernel / here, weights not in a cache): 8192 tokens, top 4 of 16 experts
// of 2048 x 1536 725 / 630; 96 tokens top 4 of those 96 / 70; 512 rows for each of 4 of 2048 x 4096 217 / 131, 64 rows for each of 8 of 4096
// x 14336 795 / 539, 1500 rows 4812 / 3691; 24 rows for each of 128 of 2048 x 768 314 / 248.
//
// The used tiles, row tile pairs in turn, column tile by column tile within a pair, are cut into eight equal runs, one per die
// (workgroups go to the eight dies in turn), so that a die's L2 sees a row tile's activations several times and a column tile's weights
// twice; a run is dealt to its die's workgroups round by round.  What is left for a last round goes by halves (every other weight
// block, all rows) if there are twice as many workgroups.
template <int MODE, int MB>
__global__ __launch_bounds__(256, 1) void moe_tiles_walk_kernel(const unsigned short* __restrict__ a, const unsigned short* __restrict__ w,
                                                                const int32_t* __restrict__ row_pair, const int32_t* __restrict__ tile_expert,
                                                                unsigned short* __restrict__ out, int top, unsigned top_inv, int N, int K,
                                                                int tiles, int nct, float limit, float alpha, int act_kind,
                                                                const float* __restrict__ in_wts) {
    constexpr bool GATE_UP = MODE == 1, FROM_TOKENS = MODE != 0;
    constexpr int ROWS = 64 * MB, A_BYTES = ROWS * 128, BUF = A_BYTES + 8 * 4096, NA = 2 * MB;
    typedef __attribute__((address_space(1))) const void gvoid;
    typedef __attribute__((address_space(3))) void lvoid;
    __shared__ __attribute__((aligned(1024))) unsigned char buf0[BUF];
    __shared__ __attribute__((aligned(1024))) unsigned char buf1[BUF];
    __shared__ __attribute__((aligned(1024))) unsigned char image[4][8192];
    const int lane = threadIdx.x & 63, l31 = lane & 31, hi = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wr = wave >> 1, wc = wave & 1;
    const int nb32 = (N + 31) / 32, ksteps = K / 64;

    // the used tiles come first: 64 places of the rest are looked at per turn
    int used = 0;
    for (int most = tiles; used < most;) {
        const int stride = (most - used + 63) / 64, at = used + lane * stride;
        const int in = __popcll(__builtin_amdgcn_ballot_w64(at < most && tile_expert[min(at, tiles - 1)] >= 0));
        if (in == 0) break;
        most = min(most, used + in * stride);
        used += (in - 1) * stride + 1;
    }
    const int die = blockIdx.x & 7, slot = blockIdx.x >> 3, slots = gridDim.x >> 3;
    const int64_t total = (int64_t)used * nct;
    const int begin = (int)(total * die / 8), count = (int)(total * (die + 1) / 8) - begin, left = count % slots;
    const bool halves = left > 0 && 2 * left <= slots;
    const int whole = count / slots + (!halves && slot < left ? 1 : 0);        // whole tiles of this workgroup
    const bool half = halves && slot < 2 * left;                               // and one half
    if (whole == 0 && !half) return;
    const int hb = slot & 1;                                                   // its blocks: this one of every two
    struct Item { int tile, ct; };
    auto item = [&](int i) {                                                   // (i = whole: the half)
        const int pos = begin + (i < whole ? i * slots + slot : count - left + (slot >> 1));
        const int pair = pos / (2 * nct), in = pos - pair * 2 * nct;
        if (2 * pair + 1 < used) return Item{2 * pair + (in & 1), in >> 1};
        return Item{2 * pair, in};                                             // (the last of an odd number)
    };

    // What this lane loads: rows 8 (wave NA + i) + lane / 8 of the tile, the chunk that belongs at place lane % 8 (i even; i odd: chunk ^ 4);
    // and weight blocks 2 wave and 2 wave + 1 of the tile's eight: gate blocks first, then up blocks (blocks past N: the last one).  A
    // lane's place in a buffer resource and a uniform offset: no address is worked out per load.
    const int chunk = (lane & 7) ^ (lane >> 4);
    unsigned arow[NA], bblk[2];
    int pair[NA], e;
#ifdef __HIP_DEVICE_COMPILE__                                 // (the host's pass over a kernel knows no buffer resources)
    const auto arsrc = __builtin_amdgcn_make_buffer_rsrc((void*)a, 0, 0xFFFFFFFFu, 0x00020000);
    auto brsrc = arsrc;
#endif
    auto ask = [&](const Item& t) {                           // the pairs of the lane's rows all at once, beside the expert
        if (FROM_TOKENS) {
#pragma unroll
            for (int i = 0; i < NA; ++i) pair[i] = row_pair[t.tile * ROWS + 8 * (wave * NA + i) + (lane >> 3)];
        }
        e = tile_expert[t.tile];
    };
    auto point = [&](const Item& t) {
#pragma unroll
        for (int i = 0; i < NA; ++i) {
            unsigned row = (unsigned)(t.tile * ROWS + 8 * (wave * NA + i) + (lane >> 3));
            if (FROM_TOKENS) {                                // pair / top: the product with 1 / top is at most one too large
                const unsigned p = (unsigned)max(pair[i], 0), q = top > 1 ? __umulhi(p, top_inv) : p;
                row = q - (q * (unsigned)top > p ? 1u : 0u);
            }
            arow[i] = row * (unsigned)K * 2u + 16u * (unsigned)(chunk ^ (4 * (i & 1)));
        }
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int blk = 2 * wave + j;
            bblk[j] = (unsigned)(GATE_UP ? min(4 * t.ct + (blk & 3), nb32 - 1) + (blk >= 4 ? nb32 : 0) : min(8 * t.ct + blk, nb32 - 1)) * (unsigned)ksteps * 4096u;
        }
#ifdef __HIP_DEVICE_COMPILE__
        brsrc = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)e * (GATE_UP ? 2 : 1) * nb32 * ksteps * 2048), 0, 0xFFFFFFFFu, 0x00020000);
#endif
    };
    auto load_a = [&](unsigned char* buf, int ks, int i) {
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_raw_ptr_buffer_load_lds(arsrc, (lvoid*)(buf + 1024 * (wave * NA + i)), 16, arow[i], ks * 128, 0, 0);
#endif
    };
    auto load_b = [&](unsigned char* buf, int ks, int j, int place, int i) {
#ifdef __HIP_DEVICE_COMPILE__
        __builtin_amdgcn_raw_ptr_buffer_load_lds(brsrc, (lvoid*)(buf + A_BYTES + 4096 * (2 * wave + place) + 1024 * i), 16, 16 * lane,
                                                 bblk[j] + ks * 4096 + 1024 * i, 0, 0);
#endif
    };
    auto load_step = [&](unsigned char* buf, int ks) {
#pragma unroll
        for (int i = 0; i < NA; ++i) load_a(buf, ks, i);
#pragma unroll
        for (int i = 0; i < 8; ++i) load_b(buf, ks, i >> 2, i >> 2, i & 3);
    };
    auto landed = [&]() {                                     // this wave's loads are in LDS, then everybody's
        asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
        __syncthreads();
    };

    // a wave's blocks: two of gate and the two of up of the same outputs, or four plain ones; NB of them from block `from` on
    const int a_base = (32 * MB * wr + l31) * 128, a_x = (l31 >> 1) & 7;
    auto block = [&](int n) { return GATE_UP ? 2 * wc + (n & 1) + 4 * (n >> 1) : 4 * wc + n; };
    auto read_a = [&](auto& f, const unsigned char* buf, int s, int m) {       // k = 32 hi + 8 s .. + 8 of the step
        f.a[m] = *(const bf16x8*)(buf + a_base + 4096 * m + 16 * ((4 * hi + s) ^ a_x));
    };
    auto read_b = [&](auto& f, const unsigned char* buf, int s, int from) {
        constexpr int NB = sizeof(f.b) / sizeof(f.b[0]);
#pragma unroll
        for (int n = 0; n < NB; ++n)
            f.b[n] = *(const bf16x8*)(buf + A_BYTES + 4096 * (block(4 / NB * n) + from) + 1024 * s + 16 * lane);
    };
    auto read = [&](auto& f, const unsigned char* buf, int s, int from) {      // (in the order of their use)
        read_a(f, buf, s, 0);
        read_b(f, buf, s, from);
#pragma unroll
        for (int m = 1; m < MB; ++m) read_a(f, buf, s, m);
    };
    auto multiply = [&](auto& acc, const auto& f, auto first, int lo, int hi) __attribute__((always_inline)) {   // (a tile's first product has nothing to add to)
        constexpr int NB = sizeof(f.b) / sizeof(f.b[0]);
#pragma unroll
        for (int i = 0; i < MB * NB; ++i) {
            const int m = i / NB, n = i % NB;
            if (i >= lo && i < hi)
                acc[m][n] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(f.b[n], f.a[m], decltype(first)::value ? f32x16{} : acc[m][n], 0, 0, 0);
        }
    };
    // The order of a product's instructions: `reads` LDS reads one by one behind its first MFMAs, `loads` global loads among all of
    // them.  Left alone the compiler puts the reads in front of their use, and every product waits for LDS.
    auto interleave = [&](auto mfmas_, auto reads_, auto loads_) {
        constexpr int MFMAS = decltype(mfmas_)::value, READS = decltype(reads_)::value, LOADS = decltype(loads_)::value;
#pragma unroll
        for (int i = 0; i < MFMAS; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);          // an MFMA
#pragma unroll
            for (int j = READS * i / MFMAS; j < READS * (i + 1) / MFMAS; ++j) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
#pragma unroll
            for (int j = LOADS * i / MFMAS; j < LOADS * (i + 1) / MFMAS; ++j) __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // One step of 64 k, four products.  The loads of step `next` of the tile that the pointers name go to its buffer: the weights' as soon
    // as every wave has read its weights, behind the first product, the activations' behind the second, so that they spread over three
    // of the four: a load takes 16 cycles of the CU's way to L2, and a wave whose load finds the way taken issues no product either.
    // The wait counter is positional: at most this step's loads outstanding means that the next step is in LDS.
    auto step = [&](auto first, auto& acc, auto& f, unsigned char* cur, unsigned char* nxt, int next, int from) __attribute__((always_inline)) {
        constexpr int NB = sizeof(f[0].b) / sizeof(f[0].b[0]), P = MB * NB, CUT = P * 3 / 8, LB = 2 * NB;
        constexpr int L1 = (LB * 5 + 7) / 8, L3 = LB + NA * 3 / 8, L = LB + NA;
        using std::integral_constant;
        auto load = [&](int lo, int hi) {
#pragma unroll
            for (int i = 0; i < L; ++i) {
                if (i < lo || i >= hi) continue;
                if (i >= LB) load_a(cur, next, i - LB);
                else if (NB == 4) load_b(cur, next, i >> 2, i >> 2, i & 3);
                else load_b(cur, next, 0, from, i);           // (the half's block)
            }
        };
        auto meet = [&](auto count) {
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(decltype(count)::value);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        constexpr std::false_type more{};
        constexpr integral_constant<int, 0> none{};
        read(f[1], cur, 1, from);
        read_b(f[2], cur, 2, from);
        read_b(f[3], cur, 3, from);
        multiply(acc, f[0], first, 0, P);
        interleave(integral_constant<int, P>{}, integral_constant<int, MB + 3 * NB>{}, none);
#pragma unroll
        for (int m = 0; m < MB; ++m) read_a(f[2], cur, 2, m);
        multiply(acc, f[1], more, 0, CUT);
        interleave(integral_constant<int, CUT>{}, integral_constant<int, MB>{}, none);
        meet(integral_constant<int, 0xC07F | MB << 8>{});     // lgkmcnt(MB)
#pragma unroll
        for (int m = 0; m < MB; ++m) read_a(f[3], cur, 3, m);
        load(0, L1);
        multiply(acc, f[1], more, CUT, P);
        interleave(integral_constant<int, P - CUT>{}, integral_constant<int, MB>{}, integral_constant<int, L1>{});
        load(L1, LB);
        multiply(acc, f[2], more, 0, CUT);
        interleave(integral_constant<int, CUT>{}, none, integral_constant<int, LB - L1>{});
        meet(integral_constant<int, 0xC07F>{});               // lgkmcnt(0)
        load(LB, L3);
        multiply(acc, f[2], more, CUT, P);
        interleave(integral_constant<int, P - CUT>{}, none, integral_constant<int, L3 - LB>{});
        meet(integral_constant<int, 0x0F70 | L3>{});          // vmcnt(L3)
        read(f[0], nxt, 0, from);
        load(L3, L);
        multiply(acc, f[3], more, 0, P);
        interleave(integral_constant<int, P>{}, integral_constant<int, MB + NB>{}, integral_constant<int, L - L3>{});
    };

    // The products leave the matrix unit in bf16, as a GEMM's output would.  Through the wave's own LDS: 16-byte chunk c of row r at place
    // c ^ (r & 15), chunks of gate in front of those of up.
    auto leave = [&](auto& acc, const Item& t, int from) __attribute__((always_inline)) {
        constexpr int NB = sizeof(acc[0]) / sizeof(acc[0][0]), CH = 4 * NB / (GATE_UP ? 2 : 1);      // finished chunks per row
        unsigned char* img = image[wave];
        int ln = lane;                                        // (hidden, or its addresses would be kept in registers through the products)
        asm volatile("" : "+v"(ln));
        const int l31 = ln & 31, hi = ln >> 5;
        int first[MB];                                        // a group's rows without a pair are its last ones: 32 of them are left out
#pragma unroll
        for (int m = 0; m < MB; ++m) first[m] = row_pair[t.tile * ROWS + 32 * (MB * wr + m)];
        with_act<MODE>(act_kind, [&](auto kind) {             // (the activation's kind is chosen once, not at every output)
            constexpr int ACT = decltype(kind)::value;
#pragma unroll
            for (int m = 0; m < MB; ++m) {
                const int row0 = t.tile * ROWS + 32 * (MB * wr + m);
                if (first[m] < 0) continue;
                auto put = [&](auto weigh) {
#pragma unroll
                    for (int n = 0; n < NB; ++n) {
                        f32x16 x = acc[m][n];
                        asm volatile("" : "+v"(x));           // (taken here: all at once they are more than the registers beside them)
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            u16x4 o4;
#pragma unroll
                            for (int r = 0; r < 4; ++r) o4[r] = __builtin_bit_cast(unsigned short, (bf16_t)weigh(x[4 * q + r]));
                            *(u16x4*)(img + l31 * 256 + 16 * ((4 * n + q) ^ (l31 & 15)) + 8 * hi) = o4;
                        }
                    }
                };
                asm volatile("" ::: "memory");                // (one wave, whose LDS accesses are carried out in their order)
                __builtin_amdgcn_wave_barrier();
                if (FROM_TOKENS && in_wts) {
                    const int p = row_pair[row0 + l31];
                    const float iw = p >= 0 ? in_wts[p] : 1.f;
                    put([&](float v) { return v * iw; });
                } else {
                    put([](float v) { return v; });
                }
                asm volatile("" ::: "memory");
                __builtin_amdgcn_wave_barrier();
#pragma unroll 2
                for (int i = ln; i < 32 * CH; i += 64) {      // (single rows without a pair too: nobody reads what they leave)
                    const int row = i / CH, c = i % CH;
                    bf16x8 x = *(const bf16x8*)(img + row * 256 + 16 * (c ^ (row & 15)));
                    if (GATE_UP) {
                        const bf16x8 u = *(const bf16x8*)(img + row * 256 + 16 * ((c + CH) ^ (row & 15)));
#pragma unroll
                        for (int r = 0; r < 8; ++r) x[r] = (bf16_t)gated_act((float)x[r], (float)u[r], limit, alpha, ACT);
                    } else if (MODE == 2) {
#pragma unroll
                        for (int r = 0; r < 8; ++r) x[r] = (bf16_t)plain_act((float)x[r], ACT);
                    }
                    const int blk = (GATE_UP ? 2 * wc : 4 * wc) + 4 / NB * (c >> 2) + from;
                    const int col = (GATE_UP ? 128 : 256) * t.ct + 32 * blk + 8 * (c & 3);
                    if (col < N) *(bf16x8*)(out + (size_t)(row0 + row) * N + col) = x;      // (N % 8 == 0)
                }
            }
        });
    };

    struct Frags { bf16x8 a[MB], b[4]; };
    struct HalfFrags { bf16x8 a[MB], b[2]; };
    Item now = item(0);
    ask(now);
    point(now);
    load_step(buf0, 0);
    landed();
    load_step(buf1, 1);
    if (whole > 0) {
        Frags f[4];
        f32x16 acc[MB][4];
        read(f[0], buf0, 0, 0);
        for (int i = 0; i < whole; ++i) {
            const Item next = i + 1 < whole || half ? item(i + 1) : now;       // (none: this one's first steps again, which nobody reads)
            ask(next);
            auto two = [&](auto first, int ks) __attribute__((always_inline)) {              // (ks: the steps behind these two, which are loaded beside them)
                if (ks == ksteps) point(next);
                const int to = ks == ksteps ? 0 : ks;
                step(first, acc, f, buf0, buf1, to, 0);
                step(std::false_type{}, acc, f, buf1, buf0, to + 1, 0);
            };
            two(std::true_type{}, 2);
            for (int ks = 4; ks <= ksteps; ks += 2) two(std::false_type{}, ks);
            leave(acc, now, 0);
            now = next;
        }
    }
    if (half) {
        HalfFrags f[4];
        f32x16 acc[MB][2];
        if (hb) bblk[0] = bblk[1];
        read(f[0], buf0, 0, hb);
        auto two = [&](auto first, int ks) __attribute__((always_inline)) {
            const int to = min(ks, ksteps - 2);               // (past the end: the last steps again, which nobody reads)
            step(first, acc, f, buf0, buf1, to, hb);
            step(std::false_type{}, acc, f, buf1, buf0, to + 1, hb);
        };
        two(std::true_type{}, 2);
        for (int ks = 4; ks <= ksteps; ks += 2) two(std::false_type{}, ks);
        leave(acc, now, hb);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");          // (nothing may land in LDS that is no longer this workgroup's)
}

static int tile_count(int64_t T, int top, int E, int rows) { return (int)((T * top + rows - 1) / rows + E); }

// Units of work that a launch makes at least, by cutting the column tiles of its pairs of row tiles into parts: a pair of row tiles is
// one die's, so few of them left dies without any (us, 128-row tiles, weights not in a cache, whole pairs / parts: one expert of 4096 x
// 11008 687 / 295, two of 4096 x 4096 257 / 172, four of 2048 x 4096 184 / 138, eight of 4096 x 14336 970 / 807; 16 experts of
// 1024 x 768 58 / 59).  Two units per die: with one the largest of these is 30 % slower at 512 rows, with four the small ones lose up
// to 3 % to activations read by more dies.
constexpr int kUnits = 16;
// (an even number of whole steps; 32 bits hold the offsets into the rows and into an expert's weights, and a tile's number)
static bool walks(bool dma, int64_t a_rows, int K, int parts, int N, int64_t tiles) {
    return dma && K % 128 == 0 && a_rows * K * 2 < (int64_t)1 << 32 && (int64_t)parts * (N + 31) * K * 2 < (int64_t)1 << 32 &&
           tiles * (N / 128 + 1) < (int64_t)1 << 28;
}

template <int MODE>
static void launch_tiles(int rows, bool dma, int64_t a_rows, const void* a, const void* w, const int32_t* row_pair, const int32_t* tile_expert, void* out, int top,
                         int tiles, int N, int K, float limit, float alpha, int act_kind, const float* in_wts, hipStream_t s) {
    const int nct = MODE == 1 ? (N + 127) / 128 : (N + 255) / 256, pairs = (tiles + 1) / 2;
    const int want = (kUnits + pairs - 1) / pairs, cols = (nct + want - 1) / want, segs = (nct + cols - 1) / cols;
    const unsigned top_inv = top > 1 ? (unsigned)((((uint64_t)1 << 32) + top - 1) / top) : 0;
    dim3 grid((unsigned)((pairs * segs + 7) / 8 * 8 * 2 * cols));
#define SM_TILES(MB_, DMA_)                                                                                                             \
    hipLaunchKernelGGL((moe_tiles_kernel<MODE, MB_, DMA_>), grid, dim3(256), 0, s, (const unsigned short*)a, (const unsigned short*)w, \
                       row_pair, tile_expert, (unsigned short*)out, top, top_inv, N, K, tiles, nct, cols, segs, limit, alpha, act_kind, in_wts)
#define SM_WALK(MB_)                                                                                                                    \
    hipLaunchKernelGGL((moe_tiles_walk_kernel<MODE, MB_>), dim3(kWalkers), dim3(256), 0, s, (const unsigned short*)a, (const unsigned short*)w, \
                       row_pair, tile_expert, (unsigned short*)out, top, top_inv, N, K, tiles, nct, limit, alpha, act_kind, in_wts)
    if (walks(dma, a_rows, K, MODE == 1 ? 2 : 1, N, tiles)) {
        if (rows == 256) SM_WALK(4); else SM_WALK(2);
        return;
    }
#undef SM_WALK
    if (!dma) SM_TILES(2, false); else if (rows == 256) SM_TILES(4, true); else SM_TILES(2, true);
#undef SM_TILES
}

}  // namespace sm

using namespace sm;

// room for a call's rows, in units of 128 rows
extern "C" int sm_moe_tiles128_count(int64_t T, int top, int E) {
    if (T <= 0 || top <= 0 || E <= 0) return 0;
    const int rows = moe_tile_rows(T * top, E);
    return tile_count(T, top, E, rows) * (rows / kBigRows);
}

extern "C" int sm_moe_tiles128(const void* h, const int32_t* idx, const float* wts, const void* w_gu, const void* w_down,
                               const void* shared, const float* shared_scale, int weight_in, float limit, float alpha, int act_kind, void* y, int64_t T, int top, int E, int W, int F,
                               int32_t* row_pair, int32_t* tile_expert, int32_t* pair_row, void* act, void* prod, void* stream) {
    if (T < 0 || top < 1 || E < 1 || W < 1 || F < 1 || act_kind < 0 || act_kind > SM_ACT_LAST ||
        (T > 0 && (!h || !idx || !wts || !w_gu || !w_down || !row_pair || !tile_expert || !pair_row || !act || !prod))) {
        set_error("sm_moe_tiles128: bad argument");
        return SM_EINVAL;
    }
    if (W % 8 || F % 8 || E > 4096 || T * top > (int64_t)1 << 28) {
        set_error("sm_moe_tiles128: needs W %% 8 == 0, F %% 8 == 0, at most 4096 experts");
        return SM_ESHAPE;
    }
    if (T == 0) return SM_OK;
    // (operands off 16 bytes go through registers, in tiles of 128 rows, which need no more room)
    const bool dma = ((uintptr_t)h | (uintptr_t)act | (uintptr_t)w_gu | (uintptr_t)w_down) % 16 == 0;
    int rows = dma ? moe_tile_rows(T * top, E) : kBigRows, tiles = tile_count(T, top, E, rows);
    const bool gated = act_is_gated(act_kind);
    if (rows == 256 && moe_walk_low(T * top, E, gated ? (F + 127) / 128 : (F + 255) / 256, W)) {
        const int tiles128 = tile_count(T, top, E, kBigRows);  // (no more room than twice as many of 256 rows)
        if (walks(dma, T, W, gated ? 2 : 1, F, tiles128) && walks(dma, (int64_t)tiles128 * kBigRows, F, 1, W, tiles128)) {
            rows = kBigRows;
            tiles = tiles128;
        }
    }
    hipStream_t s = as_stream(stream);
    // (the counts of the grouping lie where the down product's results come later: 64 E numbers of 4 bytes, if that many fit)
    int32_t* counts = (int64_t)tiles * rows * W * 2 >= (int64_t)64 * E * 4 && (uintptr_t)prod % 4 == 0 ? (int32_t*)prod : nullptr;
    if (int rc = launch_moe_align(idx, T * top, E, rows, tiles, row_pair, tile_expert, pair_row, counts, s)) return rc;
    const float* in_wts = weight_in ? wts : nullptr;
    if (gated)
        launch_tiles<1>(rows, dma, T, h, w_gu, row_pair, tile_expert, act, top, tiles, F, W, limit, alpha, act_kind, in_wts, s);
    else
        launch_tiles<2>(rows, dma, T, h, w_gu, row_pair, tile_expert, act, top, tiles, F, W, limit, alpha, act_kind, in_wts, s);
    SM_CHECK_LAUNCH("sm_moe_tiles128 (gate/up)");
    launch_tiles<0>(rows, dma, (int64_t)tiles * rows, act, w_down, row_pair, tile_expert, prod, top, tiles, W, F, 0.f, 0.f, 0, nullptr, s);
    SM_CHECK_LAUNCH("sm_moe_tiles128 (down)");
    if (y == nullptr) return SM_OK;               // the caller sums a token's pairs itself
    return sm_moe_combine(prod, pair_row, weight_in ? nullptr : wts, shared, shared_scale, y, T, top, W, stream);
}
