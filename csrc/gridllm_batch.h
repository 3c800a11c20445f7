// Batch GEMM: out[M,N] = x[M,K] @ W[N,K]^T (bf16 I/O, f32 sums), for more rows
// than k_gemm_rows takes: k_gemm_tile up to 64 rows a block, k_gemm_fed above, and
// k_gemm_cols in 256 columns.
//
// A block has RT * 16 rows by CT * 16 columns of one of `splitk` parts of K. Pieces
// of 64 k of x and W come into rings in LDS by direct loads, 8 rows of 128 bytes
// each, their 16-byte pieces XOR-swizzled by the row through the addresses (no bank
// conflicts). Blocks of the same K part and neighbouring columns share an XCD, hence
// x's lines in its L2; those of other rows and the same columns follow each other.
//   EPI 1: W rows in groups of 64 gate | 64 up; a block takes CT * 8 of each and
//   stores the gated unit [M, N / 2].
//   splitk > 1: f32 partials [splitk][M][N] in ws. out == null otherwise: the
//   result, rounded to bf16, as f32 in ws (a vocabulary's scores: 256 rows of
//   128256 took 30 us to be widened behind it).
// Constraints: N % (16 CT) == 0 (128 for EPI 1), K % 64 == 0, kslice % 64 == 0; for
// k_gemm_tile and k_gemm_cols K <= BATCH_K, by which a tile's offsets fit into 32 bits
// (longer rows go to k_gemm_fed, whose loads have 64-bit addresses).
//
// Bound by a CU's loads: it has some 128 lines of 128 bytes on their way (counted:
// TCP_TCC_READ_REQ_LATENCY over time, with rings of 2 stages as of 6), for 500 cycles
// where x hits in L2 and 950 where W comes from memory, hence 51 KB a us (12288 x 3072,
// 192 rows, loads alone in tiles of 96 x 96: x 7.4 us, W 16.4, both 25.7; with W in the
// Infinity Cache both 16.2). So the tile is as large as the accumulators allow and all
// of the chip has one. ONCE: W is read past the Infinity Cache (see load_lds16_once), as one
// block of rows does. Several blocks of rows do not quite read it at one time, and what
// is past that cache has left L2, too (200 rows of 5120 x 3072, 96 by 64, 21.2 us past it,
// 17.1; but 48 of 2048 x 2048, 32 by 64, in 4 parts, 7.5 and 8.1). In all layers, prompts
// of 300, 400 and 700 tokens by 0.5b, 1.5b and 3b 1443 -> 1405, 2915 -> 2824, 5640 ->
// 5590; 400 by 4 layers of 1.5b, of which what is past the cache leaves much there, 427
// -> 441.
//
// Where W's rows are a multiple of 4096 bytes long, what all blocks read at a time, a
// piece of 128 bytes at the same place of each row, is in few of the memory's
// channels (800 MB in rows of 16384 bytes 4.0 TB/s, of 6144 5.7). Blocks of
// neighbouring columns then start some pieces of K further on and wrap (6.05): 45 rows
// of 128256 x 2048 134.7 -> 121.2 us, of 16384 x 2048 gated 20.1 -> 18.3. One piece, and
// ten for odd multiples of 2048 (in order: one row of 16384 x 2048 gated 14.0, 12.4, of
// 16384 x 6144 34.4, 33.5, of 11008 x 4096 18.1, 18.7; 45 rows of 128256 x 4096 187,
// 190). Parts of K are at different places anyway (24 rows of 3072 x 8192 in 5 parts
// 16.2 either way, 64 of 3072 x 12288 24.2, 23.1), and other rows are read as fast in
// order (24 rows of 5120 x 3072 12.8 us, 13.1; 16384 x 3072 22.8, 23.0).
#pragma once

#include <type_traits>

#include "gridllm_tiles.h"

#define BATCH_K (1 << 20)

struct BatchArgs {
    bf16_t* out;
    float* ws;
    const bf16_t *x, *w;
    int M, N, K, splitk, kslice, rblocks;
    GluParams glu;
};

// A block's place: its first row and column, column block, part and stages of K.
struct BatchTile {
    int m0, n0, col, ks, k0, stages;
};

template <int R, int C>
DEV_INLINE BatchTile batch_place(const BatchArgs& p, int item) {
    BatchTile t;
    const int cols = p.N / C;
    t.m0 = item % p.rblocks * R;
    t.col = item / p.rblocks % cols;
    t.n0 = t.col * C;
    t.ks = item / p.rblocks / cols;
    t.k0 = t.ks * p.kslice;
    t.stages = (min(p.K, t.k0 + p.kslice) - t.k0) >> 6;
    return t;
}

template <int R, int C>
DEV_INLINE bool batch_tile(const BatchArgs& p, BatchTile* t) {
    const int total = p.N / C * p.splitk * p.rblocks;
    const int each = (total + 7) >> 3;         // blocks of an XCD
    const int at = (int)(blockIdx.x >> 3);
    const int item = (int)(blockIdx.x & 7) * each + at;
    if (at >= each || item >= total) return false;
    *t = batch_place<R, C>(p, item);
    return true;
}

// The stage that a block starts at.
DEV_INLINE int batch_turn(const BatchArgs& p, const BatchTile& t) {
    if (p.K % 2048 || p.splitk > 1) return 0;
    return t.col * (p.K % 4096 ? 10 : 1) % t.stages;
}

// The row of W that is row r of a tile of C columns.
template <int C, int EPI>
DEV_INLINE int batch_row(int n0, int r) {
    if (EPI == 0) return n0 + r;
    const int c = (n0 >> 1) + r % (C / 2);
    return (c >> 6) * 128 + (c & 63) + (r >= C / 2 ? 64 : 0);
}

// A row of results, of which a lane has 4 columns in each of B tiles (the first of
// which is W's row n(b)); with gates the tiles' second half are the ups, and g(b) is
// where a unit goes.
template <int B, int EPI, class Col, class Unit>
DEV_INLINE void batch_store(const BatchArgs& p, int ks, int m, const f32x4* acc,
                            Col n, Unit g) {
    const int gq = (threadIdx.x & 63) >> 4;
    if (EPI && p.splitk == 1) {
#pragma unroll
        for (int b = 0; b < B / 2; ++b) {
            float f[4], u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                f[r] = acc[b][r];
                u[r] = acc[b + B / 2][r];
            }
            glu_units(f, f, u, p.glu);
            st4(p.out + (long)m * (p.N >> 1) + g(b) + gq * 4, f);
        }
        return;
    }
#pragma unroll
    for (int b = 0; b < B; ++b) {
        float f[4];
#pragma unroll
        for (int r = 0; r < 4; ++r)
            f[r] = p.splitk == 1 ? bf2f(f2bf(acc[b][r])) : acc[b][r];
        const int at = n(b) + gq * 4;
        if (p.splitk == 1 && p.out) st4(p.out + (long)m * p.N + at, f);
        else st4(p.ws + ((long)ks * p.M + m) * p.N + at, f);
    }
}

// Two waves have the same A rows of tiles, of two halves of K: they add them up
// through LDS (red: the pair's), one the first rows, the other the rest.
template <int A, int B, int C, int EPI>
DEV_INLINE void batch_join(const BatchArgs& p, const BatchTile& t, int m0, int kw,
                           f32x4 (&acc)[A][B], f32x4* red) {
    constexpr int FIRST = (A + 1) / 2;
    const int fr = threadIdx.x & 15;
    lds_barrier();                             // the tiles have been read
#pragma unroll
    for (int a = 0; a < A; ++a)
        if (kw == (a < FIRST))
#pragma unroll
            for (int b = 0; b < B; ++b) red[(a * B + b) * 64] = acc[a][b];
    lds_barrier();
#pragma unroll
    for (int a = 0; a < A; ++a) {
        if (kw == (a < FIRST)) continue;
        const int m = m0 + a * 16 + fr;
#pragma unroll
        for (int b = 0; b < B; ++b) acc[a][b] += red[(a * B + b) * 64];
        if (m < p.M)
            batch_store<B, EPI>(
                p, t.ks, m, acc[a],
                [&](int b) { return batch_row<C, EPI>(t.n0, b * 16); },
                [&](int b) { return (t.n0 >> 1) + b * 16; });
    }
}

// ===========================================================================
// Up to 64 rows a block (more in several). Bound by W's way from memory.
//
// 4 waves; a wave has half of the rows by half of the columns, so that it reads each
// operand piece from LDS for several products. Stages of x and W go into a ring of NB
// buffers, NB - 1 ahead. In the middle of a stage the waves meet: the next one is
// there, and this one's buffer is free, its second half being in registers; so the
// products of one half run while the other half is read.
// W through and past that cache (us, 2 GB of weights in turn, parts of K without what
// adds them up):
//   rows        1                24               64
//   5120x3072    7.5 ->  7.0      8.0 ->  7.6      9.7 ->  9.5
//   3072x8192   11.2 -> 10.4     11.5 -> 10.7     13.1 -> 12.4
//   16384x3072  20.7 -> 18.6     20.8 -> 19.4     22.8 -> 21.4 (gated)
//   128256x3072  141 ->  132      150 ->  138      166 ->  162
// Waves that load alone, as below, take .3 to .5 us more here: a block starts later.
// Loads by buffer descriptors, behind which waits for LDS are for what is needed (see
// tiles.h), without 64-bit addresses for each (x not in L2 either): 45 rows of 2048 x
// 2048 in 4 parts 4.7 -> 4.5, 3072 x 2048 7.9 -> 7.6, 64 of 3072 x 3072 in 5 7.3 -> 7.0,
// 128 of 128256 x 3072 173.5 -> 170, what W's way from memory bounds 0 to 2 %. The
// waves below, which only load, gain nothing by it.
// ===========================================================================
template <int RT, int CT>
struct GemmTile {
    static constexpr int R = RT * 16, C = CT * 16, THREADS = 256;
    static constexpr int STAGE = (R + C) * 128;         // bytes
    static constexpr int FIT = 160 * 1024 / STAGE;
    static constexpr int NB = FIT > 8 ? 8 : FIT;
    static constexpr int BYTES = NB * STAGE;
};

template <int RT, int CT, int EPI, bool ONCE>
__global__ void __launch_bounds__(256, 2)
k_gemm_tile(const BatchArgs p) {
    typedef GemmTile<RT, CT> Sh;
    constexpr int R = Sh::R, C = Sh::C, NB = Sh::NB, BUF = (R + C) * 64;
    constexpr int G = (R + C) / 32;            // loads of a wave and tile
    constexpr int A = RT / 2, B = CT / 2;      // a wave's 16 x 16 tiles
    static_assert(RT % 2 == 0 && CT % (EPI ? 4 : 2) == 0, "halves");
    static_assert(NB >= 3 && G * (NB - 1) < 64, "loads that can be counted");
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, gq = lane >> 4, wr = wid >> 1, wc = wid & 1;
    BatchTile t;
    if (!batch_tile<R, C>(p, &t)) return;
    const int K = p.K, nt = t.stages, turn = batch_turn(p, t);
    // rows behind the last one come as zeros; a load takes 8 rows, a stage's start and
    // a load's rows are scalars
    const int w0 = batch_row<C, EPI>(t.n0, 0), at = ((lane & 7) ^ (lane >> 3)) * 16;
    const LdsSource xs = lds_source(p.x + (long)t.m0 * K,
                                    (u32)min(p.M - t.m0, R) * K * 2);
    const LdsSource ws = lds_source(p.w + (long)w0 * K,
                                    min((long)(p.N - w0) * K * 2, 0xffffffffl));
    const u32 lane_at = (u32)(lane >> 3) * K * 2 + at;
    u32 rows[G];
#pragma unroll
    for (int i = 0; i < G; ++i) {
        const int row = (i * 4 + wid) * 8;
        rows[i] = (u32)(row < R ? row : batch_row<C, EPI>(t.n0, row - R) - w0) * K * 2;
    }
    const u32 first = t.k0 * 2, behind = first + nt * 128;
    u32 stage = first + turn * 128;
    auto issue = [&](int buf) {                // the next tile
#pragma unroll
        for (int i = 0; i < G; ++i) {
            bf16_t* dst = lds + buf * BUF + (i * 4 + wid) * 512;
            if ((i * 4 + wid) * 8 < R) load_lds16(xs, lane_at, rows[i] + stage, dst);
            else load_lds16<ONCE>(ws, lane_at, rows[i] + stage, dst);
        }
        stage += 128;
        if (stage == behind) stage = first;
    };
    // a wave's columns; with gates, the second half of its tiles are the ups
    auto col_tile = [&](int b) {
        return !EPI ? wc * B + b
                    : b % (B / 2) + wc * (B / 2) + (b < B / 2 ? 0 : CT / 2);
    };
    f32x4 acc[A][B];
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
        for (int b = 0; b < B; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 xf[2][A], wf[2][B];
    auto read = [&](int buf, int c) {          // half c of a tile
        const bf16_t* s = lds + buf * BUF + ((c * 4 + gq) ^ (fr & 7)) * 8;
#pragma unroll
        for (int b = 0; b < B; ++b)
            wf[c][b] =
                *(const bf16x8*)(s + (R + col_tile(b) * 16 + fr) * 64);
#pragma unroll
        for (int a = 0; a < A; ++a)
            xf[c][a] = *(const bf16x8*)(s + ((wr * A + a) * 16 + fr) * 64);
    };
    // W's rows are the products' rows, so that a lane has 4 columns of a row
    auto multiply = [&](int c) {
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int b = 0; b < B; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    wf[c][b], xf[c][a], acc[a][b], 0, 0, 0);
    };
    auto spread = [] {                         // reads between the products
        constexpr int EACH = A * B / (A + B) > 0 ? A * B / (A + B) : 1;
#pragma unroll
        for (int i = 0; i < A + B; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x008, EACH, 0);
        }
    };

#pragma unroll
    for (int u = 0; u < NB; ++u)
        if (u < nt) issue(u);
    if (nt < NB) {                             // all of K is under way
        WAIT_LOADS(0);
        lds_barrier();
        for (int kt = 0; kt < nt; ++kt) {
            read(kt, 0);
            read(kt, 1);
            multiply(0);
            multiply(1);
        }
    } else {
        WAIT_LOADS(G * (NB - 1));
        lds_barrier();
        read(0, 0);
        int buf = 0;
        for (int kt = NB; kt < nt; ++kt) {
            const int next = buf + 1 == NB ? 0 : buf + 1;
            read(buf, 1);
            multiply(0);
            spread();
            WAIT_LOADS(G * (NB - 2));
            lds_barrier();
            issue(buf);
            read(next, 0);
            multiply(1);
            spread();
            buf = next;
        }
        auto last = [&](auto behind, auto&& rest) {    // tiles behind this one
            constexpr int L = behind.value;
            const int next = buf + 1 == NB ? 0 : buf + 1;
            read(buf, 1);
            multiply(0);
            spread();
            if constexpr (L > 0) {
                WAIT_LOADS(G * (L - 1));
                lds_barrier();
                read(next, 0);
            }
            multiply(1);
            buf = next;
            if constexpr (L > 0)
                rest(std::integral_constant<int, L - 1>(), rest);
        };
        last(std::integral_constant<int, NB - 1>(), last);
    }

#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int m = t.m0 + (wr * A + a) * 16 + fr;
        if (m >= p.M) continue;
        batch_store<B, EPI>(
            p, t.ks, m, acc[a],
            [&](int b) { return batch_row<C, EPI>(t.n0, col_tile(b) * 16); },
            [&](int b) { return (t.n0 >> 1) + col_tile(b) * 16; });
    }
}

// ===========================================================================
// 256 columns: a vocabulary's scores of up to 160 rows.
//
// 4 waves load, and 8 multiply, 2 by 4: with a wave a SIMD that does both, as above, the
// products wait while the CU's queue of loads is full, a stage's time is the sum of the
// two (1.9 us for 160 rows, .6 of them products), and a round's stores and first loads are
// on top. Here the ring runs on from one tile to the next under the stores, a block
// stays for its tiles, and the waves meet once a stage: the next one is there, the one
// before is free. What is left to gain was in the stores: 160 rows without them 129 us,
// with stores of half lines 166, of whole ones (turn_tiles) 164, of these past the
// caches, as W goes, 152 (half ones past them 160). W's way from memory bounds it; the
// products take 105 us alone. The token pick behind it then reads from memory: from
// COLS_PAST bytes of scores on a step and its pick are faster so by 1 to 2 % where tokens
// are drawn, and where the highest are taken at most 2 % slower; with fewer rows by
// less, and slower by more (128256 x 3072, a step of 4 layers with the pick, us, through
// the caches and past them, drawn; highest: 16 rows 410, 407; 439, 447, 24 488, 485; 516,
// 523, 48 509, 499; 531, 533, 128 673, 659; 689, 686). Parts of K are read next. 128256
// columns, us, k_gemm_tile in 256 columns and this:
//   rows   24           64           96           128          160
//   K 3072 130 -> 126   143 -> 129   158 -> 135   173 -> 142   184 -> 152
//   K 2048                           106 -> 96                 129 -> 104
// ===========================================================================
#define COLS_PAST 20000000l

template <int RT>
struct GemmCols {
    static constexpr int R = RT * 16, C = 256, THREADS = 768;
    static constexpr int STAGE = (R + C) * 128;         // bytes
    static constexpr int NB = 160 * 1024 / STAGE, BYTES = NB * STAGE;
};

// PAST: scores past the caches. (Not by a branch: the compiler makes one store of two
// that differ in that alone.)
template <int RT, bool ONCE, bool PAST>
__global__ void __launch_bounds__(768, 3)
k_gemm_cols(const BatchArgs p) {
    typedef GemmCols<RT> Sh;
    constexpr int R = Sh::R, C = Sh::C, NB = Sh::NB, BUF = (R + C) * 64;
    constexpr int G = (R + C) / 32;            // loads of a wave and stage
    constexpr int A = RT / 2, B = 4;           // a wave's 16 x 16 tiles
    static_assert(RT % 2 == 0 && NB >= 3 && NB <= 4 && G * (NB - 1) < 64,
                  "loads that can be counted");
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    const int lane = threadIdx.x & 63, K = p.K;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // an XCD's tiles follow each other, a block's are `stride` apart
    const int total = p.N / C * p.splitk * p.rblocks, each = (total + 7) >> 3;
    const int first = (int)(blockIdx.x & 7) * each + (int)(blockIdx.x >> 3);
    const int last = min(total, ((int)(blockIdx.x & 7) + 1) * each);
    const int stride = (int)(gridDim.x >> 3);
    if (first >= last) return;

    if (wid >= 8) {                            // the loads
        const int v = wid - 8, lr = lane >> 3;
        const u32 lane_at = (u32)lr * K * 2 + ((lane & 7) ^ lr) * 16;
        int item = first, left = 0;            // the tile to load, its stages
        u32 stage = 0, begin = 0, behind = 0;
        LdsSource xs, ws;
        auto aim = [&] {
            const BatchTile t = batch_place<R, C>(p, item);
            xs = lds_source(p.x + (long)t.m0 * K, (u32)min(p.M - t.m0, R) * K * 2);
            ws = lds_source(p.w + (long)t.n0 * K, (u32)C * K * 2);
            begin = t.k0 * 2;
            behind = begin + t.stages * 128;
            stage = begin + batch_turn(p, t) * 128;
            left = t.stages;
        };
        auto issue = [&](int buf) {
#pragma unroll
            for (int i = 0; i < G; ++i) {
                const int row = (i * 4 + v) * 8;
                bf16_t* dst = lds + buf * BUF + (i * 4 + v) * 512;
                if (row < R) load_lds16(xs, lane_at, (u32)row * K * 2 + stage, dst);
                else load_lds16<ONCE>(ws, lane_at, (u32)(row - R) * K * 2 + stage, dst);
            }
            stage += 128;
            if (stage == behind) stage = begin;
            if (--left == 0) {
                item += stride;
                if (item < last) aim();
            }
        };
        aim();
        int ahead = 0, buf = 0;                // stages under way, next buffer
        for (; ahead < NB - 1 && item < last; ++ahead) {
            issue(buf);
            buf = buf + 1 == NB ? 0 : buf + 1;
        }
        while (ahead) {                        // the oldest one is there
            if (ahead == NB - 1) WAIT_LOADS(G * (NB - 2));
            else if (NB > 3 && ahead == 2) WAIT_LOADS(G);
            else WAIT_LOADS(0);
            lds_barrier();
            --ahead;
            if (item < last) {
                issue(buf);
                buf = buf + 1 == NB ? 0 : buf + 1;
                ++ahead;
            }
        }
        return;
    }

    const int fr = lane & 15, gq = lane >> 4, wr = wid >> 2, wc = wid & 3;
    int buf = 0;
    for (int item = first; item < last; item += stride) {
        const BatchTile t = batch_place<R, C>(p, item);
        f32x4 acc[A][B];
#pragma unroll
        for (int a = 0; a < A; ++a)
#pragma unroll
            for (int b = 0; b < B; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
        for (int kt = 0; kt < t.stages; ++kt) {
            lds_barrier();
            bf16x8 xf[2][A], wf[2][B];
#pragma unroll
            for (int c = 0; c < 2; ++c) {
                const bf16_t* s = lds + buf * BUF + ((c * 4 + gq) ^ (fr & 7)) * 8 +
                                  fr * 64;
#pragma unroll
                for (int b = 0; b < B; ++b)
                    wf[c][b] = *(const bf16x8*)(s + (R + (wc * B + b) * 16) * 64);
#pragma unroll
                for (int a = 0; a < A; ++a)
                    xf[c][a] = *(const bf16x8*)(s + (wr * A + a) * 1024);
            }
#pragma unroll
            for (int c = 0; c < 2; ++c)
#pragma unroll
                for (int a = 0; a < A; ++a)
#pragma unroll
                    for (int b = 0; b < B; ++b)
                        acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                            wf[c][b], xf[c][a], acc[a][b], 0, 0, 0);
            buf = buf + 1 == NB ? 0 : buf + 1;
        }
#pragma unroll
        for (int a = 0; a < A; ++a) {
            turn_tiles(acc[a]);
            const int n = t.n0 + (wc * B + (fr >> 2)) * 16 + gq * 4;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int m = t.m0 + (wr * A + a) * 16 + j * 4 + (fr & 3);
                if (m >= p.M) continue;
                f32x4 v = acc[a][j];
                if (p.splitk == 1)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = bf2f(f2bf(v[r]));
                if (p.splitk == 1 && p.out)
                    *(u32x2*)(p.out + (long)m * p.N + n) =
                        (u32x2){pack2(v[0], v[1]), pack2(v[2], v[3])};
                else {
                    f32x4* to = (f32x4*)(p.ws + ((long)t.ks * p.M + m) * p.N + n);
                    if constexpr (PAST) __builtin_nontemporal_store(v, to);
                    else *to = v;
                }
            }
        }
    }
}

// ===========================================================================
// More than 64 rows a block.
//
// A wave that issues a load waits while the CU's queue of loads is full, and with
// these products it mostly is. So 4 waves load and 4 multiply, and they meet once a
// stage of 64 k: the next one is there, the last one's buffer is free. x comes by
// stages, NX - 1 ahead, W by pairs of stages, whose lines are neighbours in memory,
// LEAD or one less ahead.
// The multiplying waves are 2 by 2: halves of the rows, and of each stage's k (so a
// piece of x is read from LDS once, of W twice), or, where the sums would not fit into
// 256 registers, of the columns. They have W's pieces of two stages in registers, and
// x's too (TWICE), or those of a row of tiles anew as soon as it is multiplied.
// Against k_gemm_tile with as many rows, whose 4 waves do both (us, 2 GB of weights in
// turn, parts of K without what adds them up, each at its best tiling):
//   rows        96              160             256
//   5120x3072   11.2 -> 11.0    14.4 -> 13.2    17.2 -> 16.3
//   3072x8192   14.6 -> 14.1    18.0 -> 17.7    22.7 -> 21.0
//   12288x3072  20.3 -> 19.7    23.7 -> 22.5    29.4 -> 27.5
//   16384x3072  27.4 -> 26.2    35.3 -> 30.9    37.9 -> 33.7 (gated)
//   128256x3072  184 ->  179     212 ->  200     246 ->  230
// 48 columns, for which the halves of k are needed: 160 rows of 3072 x 3072 11.5 -> 11.0.
// ===========================================================================
template <int RT, int CT>
struct GemmFed {
    static constexpr int R = RT * 16, C = CT * 16, THREADS = 512;
    static constexpr int ring_w(int nx) { return nx % 2 ? nx + 1 : nx + 2; }
    static constexpr int bytes(int nx) { return (R * nx + C * ring_w(nx)) * 128; }
    static constexpr int ring() {
        int n = 8;
        while (n > 3 && bytes(n) > 160 * 1024) --n;
        return n;
    }
    static constexpr int NX = ring(), NW = ring_w(NX), BYTES = bytes(NX);
    static constexpr bool BY_K = RT / 2 * CT <= 36;
};

template <int RT, int CT, int EPI, bool ONCE>
__global__ void __launch_bounds__(512, 2)
k_gemm_fed(const BatchArgs p) {
    typedef GemmFed<RT, CT> Sh;
    constexpr int R = Sh::R, C = Sh::C, NX = Sh::NX, NW = Sh::NW, LEAD = NW - 2;
    constexpr int GX = RT / 2, GW = CT;        // a wave's loads: a stage's x, a pair's W
    constexpr bool BY_K = Sh::BY_K;
    constexpr int A = RT / 2, B = BY_K ? CT : CT / 2;   // a wave's 16 x 16 tiles
    static_assert(RT % 2 == 0 && (BY_K || CT % 2 == 0) && (!EPI || B % 2 == 0),
                  "halves");
    static_assert(Sh::BYTES <= 160 * 1024 && (!BY_K || Sh::BYTES >= RT * CT * 1024),
                  "rings, and sums that meet, fit into LDS");
    static_assert(GX * (NX - 2) + GW * ((NX - 1) / 2) < 64, "that can be counted");
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    bf16_t* const ldw = lds + NX * R * 64;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    BatchTile t;
    if (!batch_tile<R, C>(p, &t)) return;
    const int K = p.K, nt = t.stages;

    if (wid >= 4) {                            // the loads
        const int v = wid - 4, lr = lane >> 3, at = ((lane & 7) ^ lr) * 8 + t.k0;
        const int turn = batch_turn(p, t) & ~1;    // (nt is even if not 0)
        const bf16_t *sx[GX], *sw[GW];
#pragma unroll
        for (int i = 0; i < GX; ++i)
            sx[i] = p.x + at +
                    (long)min(t.m0 + (i * 4 + v) * 8 + lr, p.M - 1) * K;
#pragma unroll
        for (int i = 0; i < GW; ++i)           // waves 1 and 3: the second stage's
            sw[i] = p.w + at + (long)batch_row<C, EPI>(
                                   t.n0, (i * 2 + (v >> 1)) * 8 + lr) * K;
        int bx = 0, bw = 0, ix = 0, iw = 0;    // next buffers and stages
        auto load_x = [&] {
            if (ix >= nt) return;
            const int s = ix + turn - (ix + turn >= nt ? nt : 0);
#pragma unroll
            for (int i = 0; i < GX; ++i)
                load_lds16(sx[i] + s * 64, lds + (bx * R + (i * 4 + v) * 8) * 64);
            bx = bx + 1 == NX ? 0 : bx + 1;
            ++ix;
        };
        auto load_w = [&] {
            if (iw >= nt) return;
            const int half = v & 1;            // (behind the last stage: it again)
            const int s = min(iw + turn - (iw + turn >= nt ? nt : 0) + half, nt - 1);
#pragma unroll
            for (int i = 0; i < GW; ++i) {
                bf16_t* dst = ldw + ((bw + half) * C + (i * 2 + (v >> 1)) * 8) * 64;
                if (ONCE) load_lds16_once(sw[i] + s * 64, dst);
                else load_lds16(sw[i] + s * 64, dst);
            }
            bw = bw + 2 == NW ? 0 : bw + 2;
            iw += 2;
        };
        // a stage's W is on its way no later than its x
#pragma unroll 1
        for (int s = 0; s < NX - 1; ++s) {
            if (s == 0 || s % 2 == (NX % 2 == 0)) load_w();
            load_x();
        }
        auto step = [&](int i, auto even) {    // stage i + 1 comes, i is free
            // loads behind those of x of stage i + 1, if there are all of them
            constexpr int PAIRS = NX % 2 == 0 ? (NX - 2) / 2
                                  : even.value ? (NX - 1) / 2 : (NX - 3) / 2;
            const int behind = nt - 2 - i;     // stages (of which W counts not here)
            if (i + LEAD < nt) WAIT_LOADS(GX * (NX - 2) + GW * PAIRS);
            else if (NX >= 5 && behind >= 3) WAIT_LOADS(GX * 3);
            else if (NX >= 4 && behind >= 2) WAIT_LOADS(GX * 2);
            else if (behind >= 1) WAIT_LOADS(GX);
            else WAIT_LOADS(0);
            lds_barrier();
            if (!even.value) load_w();
            load_x();
        };
        int i = -1;
        for (; i + 2 < nt; i += 2) {
            step(i, std::false_type());
            step(i + 1, std::true_type());
        }
        if (i + 1 < nt) step(i, std::false_type());
        if (BY_K) {
            lds_barrier();                     // (those of batch_join)
            lds_barrier();
        }
        return;
    }

    const int fr = lane & 15, gq = lane >> 4, wr = wid >> 1, wc = wid & 1;
    constexpr bool TWICE = A * B <= 24;
    constexpr int XS = TWICE ? 2 : 1, H = A / 2;
    f32x4 acc[A][B];
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
        for (int b = 0; b < B; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    bf16x8 xf[XS][A], wf[2][B];
    // columns of a wave's tiles; with gates, the second half of them are the ups
    auto col_tile = [&](int b) {
        return BY_K ? b : !EPI ? wc * B + b
                    : b % (B / 2) + wc * (B / 2) + (b < B / 2 ? 0 : CT / 2);
    };
    int bx = 0, bw = 0;
    auto place = [&](int h) { return ((h * 4 + gq) ^ (fr & 7)) * 8 + fr * 64; };
    auto read_w = [&](int c, int h, int b) {   // to set c, of the stage's half h
        wf[c][b] = *(const bf16x8*)(ldw + bw * C * 64 + place(h) +
                                    col_tile(b) * 1024);
    };
    auto read_x = [&](int c, int h, int a) {
        xf[c % XS][a] = *(const bf16x8*)(lds + bx * R * 64 + place(h) +
                                         (wr * A + a) * 1024);
    };
    // W's rows are the products' rows, so that a lane has 4 columns of a row
    auto row = [&](int c, int a) {
#pragma unroll
        for (int b = 0; b < B; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                wf[c][b], xf[c % XS][a], acc[a][b], 0, 0, 0);
    };
    // Products of set c, under them reads of half h to the other one: of the next
    // stage, if it starts there.
    auto part = [&](int c, int h, auto starts) {
        constexpr int FIRST = TWICE ? 0 : H;   // rows of tiles ahead of the barrier
#pragma unroll
        for (int a = 0; a < FIRST; ++a) row(c, a);
        if constexpr (decltype(starts)::value) {
            bx = bx + 1 == NX ? 0 : bx + 1;
            bw = bw + 1 == NW ? 0 : bw + 1;
            lds_barrier();
        }
        if constexpr (TWICE) {
#pragma unroll
            for (int b = 0; b < B; ++b) read_w(c ^ 1, h, b);
#pragma unroll
            for (int a = 0; a < A; ++a) read_x(c ^ 1, h, a);
#pragma unroll
            for (int a = 0; a < A; ++a) row(c, a);
            constexpr int EACH = A * B / (A + B);
#pragma unroll
            for (int i = 0; i < A + B; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, EACH > 0 ? EACH : 1, 0);
            }
        } else {
            constexpr int Q = A - H, EACH = (H + B + Q - 1) / Q;
#pragma unroll
            for (int j = 0; j < Q; ++j) {
#pragma unroll
                for (int i = j * EACH; i < (j + 1) * EACH; ++i) {
                    if (i < H) read_x(0, h, i);
                    else if (i < H + B) read_w(c ^ 1, h, i - H);
                }
                row(c, H + j);
                __builtin_amdgcn_sched_barrier(0);
                read_x(0, h, H + j);
            }
        }
    };
    const int half = BY_K ? wc : 0;
    lds_barrier();
#pragma unroll
    for (int b = 0; b < B; ++b) read_w(0, half, b);
#pragma unroll
    for (int a = 0; a < A; ++a) read_x(0, half, a);
    if constexpr (BY_K) {
        int i = 1;
#pragma unroll 1
        for (; i + 1 < nt; i += 2) {
            part(0, wc, std::true_type());
            part(1, wc, std::true_type());
        }
        if (i < nt) {
            part(0, wc, std::true_type());
#pragma unroll
            for (int b = 0; b < B; ++b) wf[0][b] = wf[1][b];
            if constexpr (TWICE)
#pragma unroll
                for (int a = 0; a < A; ++a) xf[0][a] = xf[1][a];
        }
#pragma unroll
        for (int a = 0; a < A; ++a) row(0, a);
        batch_join<A, B, C, EPI>(p, t, t.m0 + wr * A * 16, wc, acc,
                                 (f32x4*)lds + wr * A * B * 64 + lane);
    } else {
#pragma unroll 1
        for (int i = 1; i < nt; ++i) {
            part(0, 1, std::false_type());
            part(1, 0, std::true_type());
        }
        part(0, 1, std::false_type());
#pragma unroll
        for (int a = 0; a < A; ++a) row(1, a);
#pragma unroll
        for (int a = 0; a < A; ++a) {
            const int m = t.m0 + (wr * A + a) * 16 + fr;
            if (m >= p.M) continue;
            batch_store<B, EPI>(
                p, t.ks, m, acc[a],
                [&](int b) { return batch_row<C, EPI>(t.n0, col_tile(b) * 16); },
                [&](int b) { return (t.n0 >> 1) + col_tile(b) * 16; });
        }
    }
}
