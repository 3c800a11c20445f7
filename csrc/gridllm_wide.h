// Many-row GEMM: out[M,N] = x[M,K] @ W[N,K]^T (bf16 I/O, f32 sums), for prompts
// and the largest decode batches.
//
// Block: 8 waves, 2 by 4, one block a CU; a wave has A by B MFMA tiles of 16 x 16.
// Stages of 64 k of x and W come by loads into LDS, whose 16-byte pieces are
// XOR-swizzled by their rows through the addresses (no bank conflicts), into rings
// of NB stages. A wave takes its pieces of a half of a stage at once, ahead of the
// products of the half before. So a stage's buffer is free after the first quarter
// of its products, and filled again in the other three: a load has 1.25 to 1.5
// stages' time (NB = 2) to arrive, and they are issued at the rate at which the CU
// takes them; two barriers a stage. Measured at 8192^3, 256 x 256: 797 us with one
// barrier, all of a stage's loads at once behind it and a block for each tile, 744
// now (1477 TFLOP/s; the library 695 to 720). What bounds it is power: cycles are
// the same without the loads (81 % of them with an MFMA in each SIMD), and the clock
// goes from 2.25 to 1.65 GHz with them. With the library's 32 x 32 products: 5 %
// slower, more ring for x alone: no change.
//
// Blocks stay for several tiles: the ring runs on from one to the next, under the
// stores (16 bytes a lane: W's rows are laid into LDS in an order that gives a lane
// 8 columns that follow each other). A tile's last stage reads the next one's first
// pieces, as every stage does, and a tile's first products add to nothing, in a copy of
// the stage (4096 x 16384 x 3072 309 -> 302 us, 3072 x 6144 x 3072 in 192 x 192 105 ->
// 103, 2048 x 3072 x 3072 in 192 x 128 66 -> 62.5; gated units of 192 x 256 261 -> 253).
// What is left of a tile's end is its stores: all CUs' at once, they take 15 of 302 us
// (measured with stores that stay in L2), and starting CUs or XCDs 1 to 6 us apart
// changes nothing.
// Tiles of an XCD are neighbours, in groups of 4
// rows of tiles, so that what its 32 CUs read at a time fits in its L2: 8000 x 16384
// x 3072 617 us in groups of 8, 600 of 4.
//
// A number of tiles that leaves the last round of CUs half empty costs a whole one:
// the first `full` tiles are of shape S, the others of the half as large S2
// (2731 x 8192 x 2048: 92 us in 2 rounds of 256 x 256, 80 with the rest halved).
//
// EPI 1: W rows in groups of 64 gate | 64 up; stores the gated unit [M, N / 2] of
// the results rounded to bf16, as a library product and the unit behind it have it.
// Sums go over all of K in order, as the library's do but for those of its tiles
// whose K it cuts, so that more than 99.9 % of results are the same to the bit.
// EPI 2: the result, rounded to bf16, as f32 (a vocabulary's scores); with one tile of
// rows, which reads W once, past the Infinity Cache (see load_lds16_once; 256 rows of
// 128256 x 3072 in a step 207 -> 201 us, and the step's other kernels find theirs
// there: 4 layers 880 -> 861), and stores go past the caches, too, in whole lines (256
// rows 200 -> 194, 192 198 -> 181; a step of 256 rows with the token pick behind it, which
// then reads them from memory: drawn tokens 852 -> 840, the highest 860 -> 858). More
// tiles of rows read W again, and would wait for memory where the Infinity Cache has it
// (us, through it and past it, 128256 x 3072: 257 rows 300, 361, 512 444, 481, 1024 886,
// 936; 300 of 151936 x 896 131, 155).
// EPI 3: squared ReLU. EPI 4: W rows in turns of 16 gate | 16 up, [M, N / 2].
// Rows past M and N are read as zeros by the buffer descriptors' bounds, and so are
// the stages past the last tile: a wave's offset is the end of the matrix at most,
// and a lane's is added to it.
// Constraints: N % 8 == 0 (EPI 1: 128), K % 64 == 0, K >= 256, x and W of less than
// WIDE_BYTES.
#pragma once

#include "gridllm_tiles.h"

#define WIDE_BYTES 0xe0000000L         // (so that offsets fit into 32 bits)

struct WideArgs {
    void* out;
    const bf16_t *x, *w;
    int M, N, K;
    GluParams glu;
};

// A tile: its first row, the row behind its last one, its first column, and the row
// of W where its matrix starts.
struct WideTile {
    int m0, end, n0, w0;
};

// Where rows come from and go to. GATHER: x's rows are looked up one by one. ONCE: W's
// are read once, and past the Infinity Cache.
template <bool O>
struct DenseRows {
    static constexpr bool GATHER = false, ONCE = O;
    DEV_INLINE int from(int m) const { return m; }
    DEV_INLINE long to(int m) const { return m; }
    DEV_INLINE float weight(int m) const { return 1.f; }
};

template <int A_, int B_, int NB_>
struct WideShape {
    static constexpr int A = A_, B = B_, NB = NB_, R = A * 32, C = B * 64;
    static constexpr int BYTES = NB * (R + C) * 128;
};
struct NoShape {
    static constexpr int R = 0, BYTES = 0;
};

// Tiles item, item + stride, ... < last, as place says; wrows: of W.
template <class S, int EPI, class Place, class Rows>
DEV_INLINE void wide_tiles(const WideArgs& p, bf16_t* lds, int item, int last,
                           int stride, Place place, int wrows,
                           const Rows rows) {
#ifdef __HIP_DEVICE_COMPILE__          // (the host has no buffer descriptors)
    constexpr int A = S::A, B = S::B, NB = S::NB, R = S::R, C = S::C;
    constexpr int BUF = (R + C) * 64, G = (R + C) / 64;  // loads of a wave, stage
    constexpr bool PLAIN = EPI == 4;            // W's rows are in order
    constexpr int STORES = EPI == 1 ? A * B / 4 : EPI == 2 ? A * B
                           : PLAIN ? A * B / 2 : A * ((B + 1) / 2);
    constexpr int GX = Rows::GATHER ? R / 64 : 1;
    constexpr int L1 = G / 4, L2 = 2 * L1;      // loads behind quarters 2 and 3
    static_assert(A % 2 == 0 && (EPI != 1 || B % 4 == 0) &&
                  ((EPI != 2 && !PLAIN) || B % 2 == 0), "halves");
    static_assert((NB - 2) * G + L2 + STORES < 64, "that can be counted");
    if (item >= last) return;
    const int M = p.M, N = p.N, K = p.K, nt = K >> 6;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, gq = lane >> 4, wr = wid >> 2, wc = wid & 3;
    const auto xr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)p.x, 0, (int)((u32)M * K * 2), 0x00020000);
    const auto wrs = __builtin_amdgcn_make_buffer_rsrc(
        (void*)p.w, 0, (int)((u32)wrows * K * 2), 0x00020000);

    // A load takes 8 rows of the stage to LDS in the order of lanes. Row j of W's
    // tile b is column 8 (j / 4) + j % 4, + 4 for an odd b, of the two tiles' 32 (a
    // last, single tile: j), or of two tiles of gates, and of ups.
    const int lr = lane >> 3, at = ((lane & 7) ^ lr) * 16;
    int vx[GX], vw;                             // a lane's offsets, with k
    u32 so[G];                                  // the wave's, of its rows
    auto tile_of = [&](int i) {                 // W's tile in a wave's load i
        return ((i * 8 + wid) * 8 - R) % (B * 16) >> 4;
    };
    auto aim = [&](int it) {
        const WideTile t = place(it);
        const int m0 = t.m0, n0 = t.n0;
        if constexpr (!Rows::GATHER) vx[0] = lr * K * 2 + at;
        vw = (PLAIN ? lr : (lr >> 2) * 8 + (lr & 3)) * K * 2 + at;
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const int row = (i * 8 + wid) * 8;
            int r = min(m0 + row, M);
            if (Rows::GATHER && i * 64 < R) {
                vx[i % GX] = (u32)rows.from(min(m0 + row + lr, t.end - 1)) * K *
                                 2 + at;
                r = 0;
            }
            if (i * 64 >= R) {
                const int v = (row - R) / (B * 16), b = tile_of(i), j = row & 15;
                const int c = B % 2 && b == B - 1 ? j
                                                  : (j >> 2) * 8 + (b & 1) * 4;
                r = n0 + (PLAIN ? row - R : v * B * 16 + (b >> 1) * 32 + c);
                if (EPI == 1) {
                    const int o = (n0 >> 1) + v * B * 8 +
                                  (b % (B / 2) >> 1) * 32 + c;
                    r = (o >> 6) * 128 + (o & 63) + (b >= B / 2 ? 64 : 0);
                }
                r = min(t.w0 + r, wrows);
            }
            so[i] = (u32)r * K * 2;             // (the end, at most)
        }
    };
    auto issue = [&](int buf, int i) {
        const auto dst = (__attribute__((address_space(3))) unsigned int*)(
            lds + buf * BUF + (i * 8 + wid) * 512);
        const int v = !Rows::GATHER && B % 2 && tile_of(i) == B - 1 ? vx[0] : vw;
        if (i * 64 < R)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xr, dst, 16, vx[i % GX],
                                                     so[i], 0, 0);
        else if (Rows::ONCE)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, dst, 16, v, so[i], 0, 2);
        else
            __builtin_amdgcn_raw_ptr_buffer_load_lds(wrs, dst, 16, v, so[i], 0, 0);
        if (i + 1 == G) {
#pragma unroll
            for (int k = 0; k < GX; ++k) vx[k] += 128;
            vw += 128;
        }
    };

    f32x4 acc[A][B];
    bf16x8 xf[2][A], wf[2][B];
    auto read = [&](int buf, int c, int i) {    // piece i of half c of a stage
        const bf16_t* t = lds + buf * BUF + ((c * 4 + gq) ^ (fr & 7)) * 8 +
                          fr * 64;
        if (i < B)
            wf[c][i] = *(const bf16x8*)(t + (R + (wc * B + i) * 16) * 64);
        else
            xf[c][i - B] = *(const bf16x8*)(t + (wr * A + i - B) * 1024);
    };
    // Products of half c and half of its rows of tiles, from a0 on, between them
    // the pieces of half rc of rbuf (ahead of the last products) and loads l0 ..
    // l1 - 1 into lbuf. first: the first products of a tile.
    auto quarter = [&](auto first, int c, int a0, int rbuf, int rc, bool reads,
                       int lbuf, int l0, int l1) {
        constexpr int Q = A / 2, PER = (A + B + Q - 2) / (Q - 1);
        const int each = (l1 - l0 + Q - 1) / Q;
#pragma unroll
        for (int j = 0; j < Q; ++j) {
#pragma unroll
            for (int i = j * PER; i < (j + 1) * PER; ++i)
                if (reads && i < A + B) read(rbuf, rc, i);
#pragma unroll
            for (int i = l0 + j * each; i < l0 + (j + 1) * each; ++i)
                if (i < l1) issue(lbuf, i);
#pragma unroll
            for (int b = 0; b < B; ++b)
                acc[a0 + j][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    wf[c][b], xf[c][a0 + j],
                    decltype(first)::value ? (f32x4){0.f, 0.f, 0.f, 0.f}
                                           : acc[a0 + j][b], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    };
    int buf = 0;
    // fresh: the next stage's loads are older than the stores of the tile before
    auto stage = [&](bool fresh, auto first) {
        const std::false_type no;
        const int next = buf + 1 == NB ? 0 : buf + 1;
        quarter(first, 0, 0, buf, 1, true, 0, 0, 0);
        lds_barrier();                          // all have this stage
        quarter(first, 0, A / 2, 0, 0, false, buf, 0, L1);
        quarter(no, 1, 0, 0, 0, false, buf, L1, L2);
        if (fresh) WAIT_LOADS((NB - 2) * G + L2 + STORES);
        else WAIT_LOADS((NB - 2) * G + L2);
        lds_barrier();                          // the next one is there
        quarter(no, 1, A / 2, next, 0, true, buf, L2, G);
        buf = next;
    };

    aim(item);
#pragma unroll
    for (int u = 0; u < NB; ++u)
#pragma unroll
        for (int i = 0; i < G; ++i) issue(u, i);
    WAIT_LOADS(G * (NB - 1));
    lds_barrier();
    bool stored = false;                        // all of the tile before
#pragma unroll
    for (int i = 0; i < A + B; ++i) read(buf, 0, i);
    for (; item < last; item += stride) {
        const WideTile t = place(item);
        const int m0 = t.m0, n0 = t.n0;
        auto ahead = [&](int kt) {
            if (kt != nt - NB) return;          // loads go on to the next tile
            if (item + stride < last) aim(item + stride);
            else
#pragma unroll
                for (int i = 0; i < G; ++i)
                    so[i] = (u32)(i * 64 < R ? M : wrows) * K * 2;
        };
        ahead(0);
        stage(stored, std::true_type());
#pragma unroll 1
        for (int kt = 1; kt < nt; ++kt) {
            ahead(kt);
            stage(kt < NB - 1 && stored, std::false_type());
        }
        // lane holds row fr and columns gq * 4 + 0 .. 3 of each tile
#pragma unroll
        for (int a = 0; a < A; ++a) {
            if constexpr (EPI == 2) {          // (tile b: 4 of each 8 of its pair's)
                static_assert(B == 4, "tiles to turn");
                f32x4 v[4];
#pragma unroll
                for (int b = 0; b < 4; ++b)
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[b][r] = (float)(__bf16)acc[a][b][r];
                turn_tiles(v);
                const int n = n0 + wc * 64 + (fr >> 3) * 32 + gq * 8 +
                              (fr >> 2 & 1) * 4;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int m = m0 + (wr * A + a) * 16 + j * 4 + (fr & 3);
                    if (m >= t.end || n >= N) continue;
                    f32x4* to = (f32x4*)((float*)p.out + rows.to(m) * N + n);
                    if (Rows::ONCE) __builtin_nontemporal_store(v[j], to);
                    else *to = v[j];
                }
                continue;
            }
            const int m = m0 + (wr * A + a) * 16 + fr;
            if (m >= t.end) continue;
            const int ld = EPI == 1 || EPI == 4 ? N >> 1 : N;
            const long at = rows.to(m) * ld;
            const int nw = EPI == 1 ? (n0 >> 1) + wc * B * 8
                : EPI == 4 ? (n0 >> 1) + wc * B * 8 : n0 + wc * B * 16;
            if constexpr (PLAIN) {
                const float wi = rows.weight(m);
#pragma unroll
                for (int b = 0; b < B; b += 2) {
                    const int n = nw + b * 8 + gq * 4;
                    if (n >= ld) continue;
                    float f[4], u[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        f[r] = wi * acc[a][b][r];
                        u[r] = wi * acc[a][(b + 1) % B][r];
                    }
                    glu_units(f, f, u, p.glu);
                    st4((bf16_t*)p.out + at + n, f);
                }
                continue;
            }
#pragma unroll
            for (int b = 0; b + 1 < (EPI == 1 ? B / 2 : B); b += 2) {
                const int n = nw + b * 16 + gq * 8;
                if (n >= ld) continue;
                float f[8], u[8];
#pragma unroll
                for (int r = 0; r < 8; ++r) {
                    f[r] = acc[a][b + (r >> 2)][r & 3];
                    if (EPI == 1) u[r] = acc[a][b + (r >> 2) + B / 2][r & 3];
                    if (EPI == 3) f[r] = fmaxf(f[r], 0.f) * fmaxf(f[r], 0.f);
                }
                if constexpr (EPI == 1) {
                    round8(f);
                    round8(u);
                    glu_units(f, f, u, p.glu);
                }
                *(bf16x8*)((bf16_t*)p.out + at + n) = to_bf16x8(f);
            }
            if constexpr (B % 2 && EPI == 0) {
                const int n = nw + (B - 1) * 16 + gq * 4;
                if (n >= ld) continue;
                bf16x4 v;
#pragma unroll
                for (int r = 0; r < 4; ++r) v[r] = (__bf16)acc[a][B - 1][r];
                *(bf16x4*)((bf16_t*)p.out + at + n) = v;
            }
        }
        stored = m0 + R <= t.end && n0 + C <= N;
    }
    WAIT_LOADS(0);                              // (of nothing, into LDS)
    lds_barrier();
#endif
}

template <class S, class S2, int EPI, bool ONCE>
__global__ void __launch_bounds__(512, 2)
k_gemm_wide(const WideArgs p, int full) {
    extern __shared__ __attribute__((aligned(16))) bf16_t lds[];
    const int rb = (p.M + S::R - 1) / S::R, cb = (p.N + S::C - 1) / S::C;
    const int xcd = blockIdx.x & 7, at = (int)(blockIdx.x >> 3);
    const int stride = (int)(gridDim.x >> 3);
    auto place = [&](int it) {
        const int group = it / (4 * cb), in = it - group * 4 * cb;
        const int rows = min(4, rb - group * 4);
        return WideTile{(group * 4 + in % rows) * S::R, p.M, in / rows * S::C, 0};
    };
    const int each = (full + 7) >> 3;           // tiles of an XCD
    wide_tiles<S, EPI>(p, lds, xcd * each + at, min(full, (xcd + 1) * each),
                       stride, place, p.N, DenseRows<ONCE>());
    if constexpr (S2::R > 0) {
        static_assert(S2::R * 2 == S::R && S2::C == S::C, "halves");
        const int rest = (rb * cb - full) * 2, each = (rest + 7) >> 3;
        wide_tiles<S2, EPI>(
            p, lds, xcd * each + at, min(rest, (xcd + 1) * each), stride,
            [&](int it) {
                WideTile t = place(full + (it >> 1));
                t.m0 += (it & 1) * S2::R;
                return t;
            }, p.N, DenseRows<ONCE>());
    }
}

// Shapes by number, their sizes, and what they take, in us: a stage (`idle` of it
// with one tile on the chip, as a whole round takes), a tile beside it (`glu` more
// for the unit), a launch. Fitted to 330 to 1550 timings each over the products of
// the models here and 257 to 8192 rows; later ones, of more products, are 3 to 4 %
// longer, with a standard deviation of 4 to 6 %. Gated units, both shapes, to 435 of
// these others: the faster shape in all but 1.7 % of sizes, where the other one is 2 to 4 %
// faster (before, in 6.1 %, and up to 17).
struct WideTimes {
    int rows, cols;
    float stage, idle, tile, glu, launch;
};
static constexpr WideTimes kWide[] = {
    {256, 256, 1.350f, .660f, 3.82f, 1.49f, 4.7f},      // rest in halves
    {192, 192, .885f, .720f, 2.23f, 0.f, 5.4f},
    {256, 192, 1.090f, .716f, 2.91f, 0.f, 5.2f},
    {192, 128, .648f, .713f, .77f, 0.f, 5.0f},
    {192, 256, 1.190f, .755f, 0.f, 1.33f, 5.5f},        // gated units, f32
};
static constexpr WideTimes kWideHalf = {128, 256, .801f, .712f, 1.67f, 1.75f,
                                        0.f};
static constexpr int kWideShapes = 5;
typedef WideShape<8, 4, 2> Wide256;
typedef WideShape<4, 4, 3> WideHalf;

static bool wide_fits(int M, int N, int K, int epi, int shape) {
    if (shape < 0 || shape >= kWideShapes || M < 1 || N < 1 || K < 256) return false;
    if (K % 64 || N % (epi == 1 ? 128 : 8)) return false;
    if ((long)M * K * 2 > WIDE_BYTES || (long)N * K * 2 > WIDE_BYTES ||
        K > 1 << 20) return false;
    return epi == 0 ? shape < 4 : shape == 0 || shape == 4;
}

static float wide_rounds(const WideTimes& t, int K, int epi, int tiles) {
    const int whole = tiles / 256, some = tiles % 256, nt = K / 64;
    const float over = t.tile + (epi == 1 ? t.glu : 0.f);
    return whole * (nt * t.stage + over) +
           (some ? nt * t.stage * (t.idle + (1 - t.idle) * some / 256.f) + over
                 : 0.f);
}

// The fastest shape for a product by these times, and of how many whole tiles.
static float wide_best(int M, int N, int K, int epi, int* shape, int* full) {
    float best = INFINITY;
    for (int s = 0; s < kWideShapes; ++s) {
        if (!wide_fits(M, N, K, epi, s)) continue;
        const WideTimes& t = kWide[s];
        const long tiles = (long)((M + t.rows - 1) / t.rows) *
                           ((N + t.cols - 1) / t.cols);
        if (tiles > 1 << 24) continue;
        const int total = (int)tiles;
        const float us = t.launch + wide_rounds(t, K, epi, total);
        if (us < best) { best = us; *shape = s; *full = total; }
        if (s != 0 || total % 256 == 0) continue;
        const int head = total / 256 * 256;
        const float mixed = t.launch + wide_rounds(t, K, epi, head) +
                            kWideHalf.launch +
                            wide_rounds(kWideHalf, K, epi, (total - head) * 2);
        if (mixed < best) { best = mixed; *shape = s; *full = head; }
    }
    return best;
}
