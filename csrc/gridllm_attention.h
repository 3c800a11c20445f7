// Attention kernel templates, shared by the contiguous slot cache and the
// paged cache: where a block of keys lies comes from a KV policy.
#pragma once

#include "gridllm_tiles.h"

#include <type_traits>

// Where 64 keys (aligned to 64) of a sequence's kv head start, in elements.
// Caches of contiguous slots: [slots, Hk, Smax, D].
template <int D>
struct SlotKV {
    const bf16_t* k;
    const bf16_t* v;
    int Hk, Smax;
    DEV_INLINE long off(int slot, int hk, int key) const {
        return (((long)slot * Hk + hk) * Smax + key) * D;
    }
    struct Walk {
        DEV_INLINE long operator()(const SlotKV& kv, int slot, int hk, int key) {
            return kv.off(slot, hk, key);
        }
    };
};

// Caches of pages of 64 keys: [pages, Hk, 64, D]; table[slot][i] is the page
// of keys 64 i .. 64 i + 63.
#define KV_PAGE 64
template <int D>
struct PagedKV {
    const bf16_t* k;
    const bf16_t* v;
    const int* table;
    int Hk, per_slot;
    DEV_INLINE long off(int slot, int hk, int key) const {
        const int page = table[(long)slot * per_slot + (key / KV_PAGE)];
        return (((long)page * Hk + hk) * KV_PAGE + key % KV_PAGE) * D;
    }
    // The same for keys in order: lanes hold the numbers of 64 pages, since a load for
    // each would be waited for, and all loads of keys that are under way with it
    struct Walk {
        int pages = 0, first = -1;
        DEV_INLINE long operator()(const PagedKV& kv, int slot, int hk, int key) {
            const int page = key / KV_PAGE;
            if (page >> 6 != first) {
                first = page >> 6;
                pages = kv.table[(long)slot * kv.per_slot +
                                 min(first * 64 + (int)(threadIdx.x & 63),
                                     kv.per_slot - 1)];
            }
            const int at = __builtin_amdgcn_readlane(pages, page & 63);
            return (((long)at * kv.Hk + hk) * KV_PAGE + key % KV_PAGE) * D;
        }
    };
};

// Which keys up to its own a query sees. Kernels walk blocks of keys by number
// (decode) or by first key (prefill) and leave out what no row sees.
struct AllKeys {
    DEV_INLINE int blocks(int seq) const { return (seq + 63) >> 6; }
    DEV_INLINE int start(int b, int seq) const { return b << 6; }
    DEV_INLINE int skip(int k0, int q0) const { return k0; }
    DEV_INLINE bool sees(int q, int key) const { return true; }
    // whether all queries up to q see the 64 keys from `key` on, as far as
    // they are not ahead of them
    DEV_INLINE bool sees_tile(int q, int key) const { return true; }
};

// The last `size` keys, its own included, and the first `keep`.
struct WindowKeys {
    int size, keep;
    // blocks of 64 that hold kept keys, and the first one of the window behind
    // them, for the last of seq positions
    DEV_INLINE int kept(int seq) const { return (min(keep, seq) + 63) >> 6; }
    DEV_INLINE int window(int seq) const {
        return max(kept(seq), max(0, seq - size) >> 6);
    }
    DEV_INLINE int blocks(int seq) const {
        return kept(seq) + ((seq + 63) >> 6) - window(seq);
    }
    DEV_INLINE int start(int b, int seq) const {
        const int k = kept(seq);
        return (b < k ? b : window(seq) + b - k) << 6;
    }
    // first key, from k0 on, of a tile of 64 that rows from q0 on may see
    DEV_INLINE int skip(int k0, int q0) const {
        return k0 < keep ? k0 : max(k0, max(0, q0 - size + 1) & ~63);
    }
    DEV_INLINE bool sees(int q, int key) const {
        return q - key < size || key < keep;
    }
    DEV_INLINE bool sees_tile(int q, int key) const {
        return q - key < size || key + 63 < keep;
    }
};

// What happens to a head's sums before they are stored. `sink` (nullable, one
// per query head) adds exp(sink) to the softmax denominator; `gate` (nullable,
// row stride gate_ld) multiplies the output by its sigmoid: one per query
// head, or (gate_el) one per element; so does `scale`. out_ld: row stride of
// the output, 0 if the heads fill a row.
struct HeadEpilogue {
    const float* sink;
    const bf16_t* gate;
    int gate_ld;
    int gate_el = 0;
    float scale = 1.f;
    int out_ld = 0;
    DEV_INLINE long at(long row, int head, int Hq, int D) const {
        return row * (out_ld ? out_ld : Hq * D) + head * D;
    }
    DEV_INLINE float element(int row, int col) const {
        if (!gate_el) return 1.f;
        return 1.f / (1.f + __expf(-bf2f(gate[(long)row * gate_ld + col])));
    }
    // M, L: running maximum and sum of the log2-domain softmax. Returns the
    // factor for the accumulated values.
    DEV_INLINE float factor(int row, int head, float M, float L) const {
        float f = 1.f;
        if (sink) {
            const float s2 = sink[head] * LOG2E;
            const float m2 = fmaxf(M, s2);
            f = (M == -INFINITY) ? 0.f : exp2f(M - m2);
            L = L * f + exp2f(s2 - m2);
        }
        f = L > 0.f ? f / L * scale : 0.f;
        if (gate && !gate_el)
            f /= 1.f + __expf(-bf2f(gate[(long)row * gate_ld + head]));
        return f;
    }
};

// ===========================================================================
// GQA decode attention (flash-decode style).
//   q:   [B, Hq, D] bf16 (one new token per sequence)
//   kc/vc: bf16 caches
//   seqlen: [B] int32 (number of valid keys, including the current token)
//   rows: [B] {row, keys, slot, -} in the order in which rows' blocks start, or null:
//         in that of the batch. With the longest first the last blocks to start are
//         short (us, cache of 8 heads of 128, rows as they come and sorted): 24 of 1000
//         to 6000 keys 72.0, 65.5, 64 of 333 to 2000 66.3, 60.6, 160 of 170 to 1000
//         76.8, 66.3, 256 of 64 to 384 49.3, 44.8, 8 of 500 to 3000 22.0, 21.4
//   out: [B, Hq, D] bf16
//   ws (nsplit>1): f32 [B, Hq, nsplit, D+2]  (unnormalized acc, m, l)
//
// Block = 4 waves, one block per (b, hk, split). Waves take turns at steps of
// KS = 4096 / D keys, whose K and V (8 KB each) they load into registers one
// step ahead: K as MFMA operands (scores of all G = Hq/Hk query heads at once,
// S = mfma(A=Q, B=K)), V row-wise, 16 bytes a lane, for f32 sums in the vector
// unit; weights stay f32 and pass through LDS. The 4 waves combine in LDS.
// Bound by HBM and, for few keys, by the chain load - scores - weights - sums.
// 24 heads of 128 over 8, before (a key row per lane, f32 scores, waves waiting
// for their own loads) and now: 24 rows of up to 6000 keys 193 -> 70 us
// (5.1 TB/s), 256 of up to 384 99 -> 41 us (5.9 TB/s), one of 900 17 -> 9 us, in
// a loop; among a step's other kernels the first two take 66 and 5, and 53.
// V's loads go past the caches; K's, of half a cache line each, do not (both
// halves would fetch it: 24 rows 73 us).
// mfma_f32_16x16x32_bf16:
//   A[i][k]: lane l holds i = l&15, k = (l>>4)*8 + 0..7
//   B[k][j]: lane l holds j = l&15, same k chunk
//   D[i][j]: lane l holds j = l&15, i = (l>>4)*4 + reg
// Constraints: D in {64, 128, 256}; G <= 8.
// Own: where a row's queries, new key and value come from. StoredQueries: q, and the
// cache has the other two. Else the block makes them (own(row, head, turned, column,
// position, lo, hi) gives 8 columns and those D / 2 further on), keeps them in LDS, and
// one of the row's blocks of a kv head writes them to the cache (a row without keys has
// no place there).
// ===========================================================================
struct StoredQueries {
    static constexpr bool MADE = false;
};

#define MAXG 8
#define MAX_SPLIT 64

// The softmax's reference moves only when a maximum grows by more than
// 2^MAX_LAG: weights are at most that, their sums are f32.
#define MAX_LAG 8.f

template <int N>                       // x of the lane N further on in its 16
DEV_INLINE float rotate16(float x) {
    return __uint_as_float(__builtin_amdgcn_mov_dpp(
        (int)__float_as_uint(x), 0x120 + N, 0xf, 0xf, true));
}
DEV_INLINE float max_of16(float x) {
    x = fmaxf(x, rotate16<8>(x));
    x = fmaxf(x, rotate16<4>(x));
    x = fmaxf(x, rotate16<2>(x));
    return fmaxf(x, rotate16<1>(x));
}
DEV_INLINE float sum_of16(float x) {
    x += rotate16<8>(x);
    x += rotate16<4>(x);
    x += rotate16<2>(x);
    return x + rotate16<1>(x);
}

// Steps of a row and of one of its splits: at least one for each wave.
DEV_INLINE int split_steps(int steps, int nsplit) {
    return max((steps + nsplit - 1) / nsplit, 4);
}

// A kv head with more than MAXG query heads is served by `ngrp` blocks of G
// query heads each. Sequence lengths are given as seqlen + seq_add.
template <int D, int G, class KV, class Keys, class Own = StoredQueries>
__global__ void __launch_bounds__(256, 2)
k_attn_decode(bf16_t* __restrict__ out, const bf16_t* __restrict__ q,
              const KV kv,
              const int* __restrict__ seqlen, int seq_add,
              const int* __restrict__ slot_map,
              const int4* __restrict__ rows, float* __restrict__ ws,
              int ngrp, int nsplit, float scale, const HeadEpilogue epi,
              const Keys keys, const Own own = Own()) {
    constexpr int KS = 4096 / D;           // keys of a step
    constexpr int SPB = 64 / KS;           // steps of a block of 64 keys
    constexpr int KT = KS / 16, ND = D / 32;
    constexpr int LV = D / 8;              // lanes of a V row
    constexpr int R = G < 4 ? G : 4;       // heads of a lane
    const int Hg = kv.Hk * ngrp;
    const int split = blockIdx.x % nsplit;
    const int hg = (blockIdx.x / nsplit) % Hg;
    const int hk = hg / ngrp;
    int b = blockIdx.x / (nsplit * Hg), bc = b, seq;  // row, its slot, its keys
    int place = 0;                                    // and (own) rotary position
    if (rows) {
        const int4 r = rows[b];
        b = r.x;
        seq = r.y;
        bc = r.z;
        place = r.w;
    } else {
        if (slot_map) bc = slot_map[b];
        seq = seqlen[b] + seq_add;
        if constexpr (Own::MADE) place = own.pos[b];
    }
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int Hq = Hg * G;

    __shared__ __attribute__((aligned(16))) float p_lds[4][G][KS];
    __shared__ float red[4][G * D];
    __shared__ float wml[4][G][2];         // per-wave m, l
    // the row's queries, key and value
    __shared__ __attribute__((aligned(16))) bf16_t made[Own::MADE ? (G + 2) * D : 8];

    const int blocks = keys.blocks(seq);
    const int steps = blocks <= 0 ? 0 : (blocks - 1) * SPB +
        (seq - keys.start(blocks - 1, seq) + KS - 1) / KS;
    const int per = split_steps(steps, nsplit);
    const int end = min(steps, split * per + per);
    int cur = split * per + wid;
    if (split && split * per >= steps) {   // nothing left for this split
        if (threadIdx.x < G) {
            float* wsp = ws + (((long)b * Hq + hg * G + threadIdx.x) * nsplit +
                               split) * (D + 2);
            wsp[D] = -INFINITY;
            wsp[D + 1] = 0.f;
        }
        return;
    }

    const int fr = lane & 15, kg = (lane >> 4) * 8;
    bf16x8 qf[ND];                         // head fr (or the last one)
    auto load_q = [&](const bf16_t* heads) {
        const bf16_t* qr = heads + min(fr, G - 1) * D + kg;
#pragma unroll
        for (int s = 0; s < ND; ++s) qf[s] = *(const bf16x8*)(qr + s * 32);
    };
    if constexpr (!Own::MADE) load_q(q + ((long)b * Hq + hg * G) * D);
    const float scale2 = scale * LOG2E;    // log2-domain softmax

    const int rg = lane / LV, d8 = (lane % LV) * 8;
    bf16x8 kf[KT][ND];
    uint4 vf[8];
    auto first_key = [&](int st) {
        return keys.start(st / SPB, seq) + st % SPB * KS;
    };
    // rows behind the last key repeat it
    auto start_of = [&](int st) {
        const int k0 = first_key(st);
        return kv.off(bc, hk, k0 & ~63) + (k0 & 63) * D;
    };
    // K and V past the Infinity Cache (see load_lds16_once): with weights that go past
    // it and K that does not, K's part of it is slower than memory (256 rows of up to
    // 384 keys 56 us, 51; 64 of up to 2000 in pages 87, 63). A row's four loads follow
    // each other, so that both halves of a line come at once.
    auto load_k = [&](int st, long at) {
        const int last = seq - 1 - first_key(st);
        const bf16_t* p = kv.k + at + kg;
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            const bf16_t* r = p + min(t * 16 + fr, last) * D;
#pragma unroll
            for (int s = 0; s < ND; ++s)
                kf[t][s] = __builtin_nontemporal_load(
                    (const bf16x8*)(r + s * 32));
        }
    };
    typedef __attribute__((ext_vector_type(4))) u32 u32x4;
    auto load_v = [&](int st, long at) {
        const int last = seq - 1 - first_key(st);
        const bf16_t* p = kv.v + at + d8;
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const u32x4 x = __builtin_nontemporal_load(
                (const u32x4*)(p + min(rg * 8 + j, last) * D));
            vf[j] = make_uint4(x[0], x[1], x[2], x[3]);
        }
    };

    float m[R], l[R];                      // of heads (lane >> 4) * 4 + r
    float facc[G][8];                      // sums over this lane's V rows
#pragma unroll
    for (int r = 0; r < R; ++r) {
        m[r] = -1e30f;                     // finite: nothing seen weighs 0
        l[r] = 0.f;
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < 8; ++i) facc[g][i] = 0.f;

    auto step = [&](int st, auto MORE) {
        long next = 0;
        if constexpr (decltype(MORE)::value) next = start_of(st + 4);
        if constexpr (Own::MADE && !decltype(MORE)::value) {
            if (st + 1 == steps) {         // the new key, which the cache may not have
                const int last = seq - 1 - first_key(st);
#pragma unroll
                for (int c = 0; c < ND; ++c) {
                    const bf16x8 k = *(const bf16x8*)(made + G * D + kg + c * 32);
#pragma unroll
                    for (int t = 0; t < KT; ++t)
                        if (t * 16 + fr >= last) kf[t][c] = k;
                }
                const bf16x8 v = *(const bf16x8*)(made + (G + 1) * D + d8);
#pragma unroll
                for (int j = 0; j < 8; ++j)
                    if (rg * 8 + j >= last) vf[j] = __builtin_bit_cast(uint4, v);
            }
        }
        f32x4 s[KT];
#pragma unroll
        for (int t = 0; t < KT; ++t) {
            s[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int c = 0; c < ND; ++c)
                s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    qf[c], kf[t][c], s[t], 0, 0, 0);
        }
        if constexpr (decltype(MORE)::value) load_k(st + 4, next);
        const int k0 = first_key(st);
        float mx[R];
        bool move = false;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            mx[r] = -FLT_MAX;
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                const int key = k0 + t * 16 + fr;
                s[t][r] = key < seq && keys.sees(seq - 1, key)
                    ? s[t][r] * scale2 : -INFINITY;
                mx[r] = fmaxf(mx[r], s[t][r]);
            }
            mx[r] = max_of16(mx[r]);
            move |= mx[r] > m[r] + MAX_LAG;
        }
        if (__any(move)) {
            float alpha[R];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const float mn = mx[r] > m[r] + MAX_LAG ? mx[r] : m[r];
                alpha[r] = exp2f(m[r] - mn);
                l[r] *= alpha[r];
                m[r] = mn;
            }
#pragma unroll
            for (int g = 0; g < G; ++g) {
                const float a = __uint_as_float(__builtin_amdgcn_readlane(
                    __float_as_uint(alpha[g & 3]), g >> 2 << 4));
#pragma unroll
                for (int i = 0; i < 8; ++i) facc[g][i] *= a;
            }
        }
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const int head = (lane >> 4) * 4 + r;
#pragma unroll
            for (int t = 0; t < KT; ++t) {
                const float p = fast_exp2(s[t][r] - m[r]);
                l[r] += p;
                if (head < G) p_lds[wid][head][t * 16 + fr] = p;
            }
        }
        // this wave's weights alone
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        float p[G][8];
#pragma unroll
        for (int g = 0; g < G; ++g) ld8(&p_lds[wid][g][rg * 8], p[g]);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            float v[8];
            unpack8(vf[j], v);
#pragma unroll
            for (int g = 0; g < G; ++g)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    facc[g][i] = fmaf(p[g][j], v[i], facc[g][i]);
        }
        if constexpr (decltype(MORE)::value) load_v(st + 4, next);
        asm volatile("" ::: "memory");     // weights are read
    };
    // the last wave makes the row ahead of its own loads, under the others'
    if constexpr (Own::MADE) {
        constexpr int L = D / 16;          // lanes of a head
        for (int at = lane; wid == 3 && at < (G + 2) * L; at += 64) {
            const int i = at / L, c = at % L * 8;
            const int head = i < G ? hg * G + i : Hq + (i - G) * kv.Hk + hk;
            uint4 lo, hi;
            own(b, head, i <= G, c, place, lo, hi);
            *(uint4*)(made + i * D + c) = lo;
            *(uint4*)(made + i * D + c + D / 2) = hi;
            if (i >= G && steps && end == steps && hg % ngrp == 0) {
                bf16_t* to = (bf16_t*)(i == G ? kv.k : kv.v) +
                             kv.off(bc, hk, seq - 1) + c;
                *(uint4*)to = lo;
                *(uint4*)(to + D / 2) = hi;
            }
        }
    }
    if (cur < end) {
        const long at = start_of(cur);
        load_k(cur, at);
        load_v(cur, at);
    }
    if constexpr (Own::MADE) {
        lds_barrier();                     // (K and V stay under way)
        load_q(made);
    }
    if (cur < end) {
        for (; cur + 4 < end; cur += 4) step(cur, std::true_type());
        step(cur, std::false_type());
    }

    // total the lanes' V rows and keys, then the waves
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int off = 32; off >= LV; off >>= 1)
                facc[g][i] += __shfl_xor(facc[g][i], off, WAVE);
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int head = (lane >> 4) * 4 + r;
        l[r] = sum_of16(l[r]);
        if (fr == 0 && head < G) {
            wml[wid][head][0] = m[r];
            wml[wid][head][1] = l[r];
        }
    }
    if (lane < LV)
#pragma unroll
        for (int g = 0; g < G; ++g) st8(&red[wid][g * D + d8], facc[g]);
    __syncthreads();
    for (int i = threadIdx.x; i < G * D; i += 256) {
        const int g = i / D, d = i % D;
        float M = wml[0][g][0], a = 0.f, L = 0.f;
#pragma unroll
        for (int w = 1; w < 4; ++w) M = fmaxf(M, wml[w][g][0]);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            const float f = exp2f(wml[w][g][0] - M);
            a += red[w][i] * f;
            L += wml[w][g][1] * f;
        }
        if (nsplit == 1) {
            out[epi.at(b, hg * G + g, Hq, D) + d] =
                f2bf(a * epi.factor(b, hg * G + g, M, L) *
                     epi.element(b, (hg * G + g) * D + d));
        } else {
            float* wsp = ws + (((long)b * Hq + hg * G + g) * nsplit + split) *
                              (D + 2);
            wsp[d] = a;
            if (d == 0) {
                wsp[D] = M;
                wsp[D + 1] = L;
            }
        }
    }
}

// Combine split-S partials: a block of 256 per (row, head); nsplit <=
// MAX_SPLIT. Splits that had no keys hold a maximum of -inf and no sums.
template <int D>
__global__ void __launch_bounds__(256)
k_attn_combine(bf16_t* __restrict__ out, const float* __restrict__ ws,
               int Hq, int nsplit, const HeadEpilogue epi) {
    constexpr int NG = 256 / D;               // splits side by side
    __shared__ float part[NG > 1 ? NG - 1 : 1][D];
    const long bh = blockIdx.x;               // b*Hq + hq
    const int d = threadIdx.x % D, grp = threadIdx.x / D;
    const int lane = threadIdx.x & 63;
    const float* base = ws + bh * (long)nsplit * (D + 2);
    float ms = -INFINITY, ls = 0.f;
    if (lane < nsplit) {
        ms = base[lane * (D + 2) + D];
        ls = base[lane * (D + 2) + D + 1];
    }
    const float M = wave_reduce_max(ms);
    const float f = ms == -INFINITY ? 0.f : exp2f(ms - M);
    const float den = wave_reduce_sum(ls * f);
    const int used = __popcll(__ballot(ms != -INFINITY));   // the first ones
    float num = 0.f;
#pragma unroll 8
    for (int s = grp; s < used; s += NG)
        num = fmaf(__shfl(f, s, WAVE), base[s * (D + 2) + d], num);
    if (NG > 1) {
        if (grp) part[grp - 1][d] = num;
        __syncthreads();
        if (grp) return;
#pragma unroll
        for (int g = 0; g < NG - 1; ++g) num += part[g][d];
    }
    const int b = (int)(bh / Hq), h = (int)(bh % Hq);
    out[epi.at(b, h, Hq, D) + d] =
        f2bf(num * epi.factor(b, h, M, den) * epi.element(b, h * D + d));
}

// ===========================================================================
// GQA prefill attention — flash-style on MFMA (bf16), reads K/V straight
// from the cache.
//   q:   [T, Hq, D] bf16 (roped)
//   out: [T, Hq, D] bf16
// Workgroup = 4 waves; wave w owns 32 q-rows of ONE q-head. K/V are walked in
// tiles of 64 keys, loaded straight into LDS one tile ahead.
//
// S^T = mfma(A=K, B=Q) puts a q-row's scores in ONE lane pair, so the softmax
// row-reduce stays in registers; the weights become the B operand of
// O^T = mfma(A=V^T, B=P) by one swap of lane halves, and V^T comes from LDS by
// transposing reads. The softmax's reference moves only when a row's maximum
// grows by more than 2^MAX_LAG (weights are at most that, sums are f32).
//
// 8000 tokens, 24 heads of 128 over 8: 383 us, 1026 TFLOP/s of the pairs that are
// seen (1889 us with one 32-key tile at a time, V transposed by stores into LDS and K
// read from L2 by every wave; 432 with waits for all reads of LDS, and heads one after
// the other); 8 prompts of up to 1300 79 -> 62, 3500 in pages 116 -> 94. Matrix cores
// are busy half of the time, at a clock of 1.94 GHz (2.05 when they were 44 %: power),
// vector unit (half of it the exponentials) and LDS some 40 %, one wave's phases after
// each other; two waves share a SIMD. Tiles of 32 keys with three waves a SIMD,
// working on three tiles at once by software, and two groups of four waves that take
// turns at products and at the softmax, were slower (the last 412 us).
// mfma_f32_32x32x16_bf16:
//   A[i][k]: lane l holds i = l&31, k = (l>>5)*8 + 0..7
//   B[k][j]: lane l holds j = l&31, same k chunk
//   C/D[i][j]: col j = l&31, row i = (reg&3) + 8*(reg>>2) + 4*(l>>5)
// Constraints: D in {64, 128, 256}; Hq % Hk == 0.
// ===========================================================================
// LDS elements of a block: two tiles of keys and values.
template <int D>
constexpr int prefill_lds() { return 2 * 64 * 2 * D; }

// Scheduling of N LDS reads that feed one MFMA each: AHEAD of them in flight.
// (Left alone the compiler reads two, waits for both, and so on: the LDS
// latency eight times in a row.)
template <int N, int AHEAD>
DEV_INLINE void reads_ahead() {
    __builtin_amdgcn_sched_group_barrier(0x100, AHEAD, 0);
#pragma unroll
    for (int i = 0; i < N - AHEAD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
}

DEV_INLINE bool prefill_item(int ntiles, int Hq, int* tile, int* head) {
    return prefill_place(blockIdx.x, ntiles, Hq, tile, head);
}
static inline unsigned prefill_grid(long ntiles, long Hq) {
    return (unsigned)((ntiles * Hq + 7) / 8 * 8);
}

// One tile of 128 q-rows of one q-head for one sequence. q0 = its first row;
// row0 = row of q[0] in the epilogue's gate.
template <int D, class KV, class Keys = AllKeys>
__device__ __forceinline__ void
attn_prefill_tile(bf16_t* __restrict__ out, const bf16_t* __restrict__ q,
                  const KV& kv, int T, int Hq, int G, int hq, int slot,
                  int s_total, int causal_off, float scale, int q0,
                  bf16_t* lds, const HeadEpilogue& epi, int row0,
                  const Keys keys = Keys()) {
    constexpr int NS = D / 16;     // 16-wide d slices (QK^T fragments)
    constexpr int NT = D / 32;     // 32-wide d tiles (output / V^T)
    constexpr int VT = NT < 4 ? NT : 4;
    constexpr int CPR = D / 8;     // 16-byte chunks per row
    constexpr int LOADS = 64 * CPR / 256;    // of K, and of V, per thread
    constexpr int TILE = 2 * 64 * D;

    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int hi = lane >> 5;
    const int ln = lane & 31;
    const int hk = hq / G;
    const int qw = q0 + wid * 32;

    // Q fragments: lane holds Q[row][s*16 + hi*8 + 0..7] (B operand). Scores
    // are scaled by |scale|; its sign goes into q.
    bf16x8 qf[NS];
    {
        const bf16_t* qrow =
            q + ((long)min(qw + ln, T - 1) * Hq + hq) * D + hi * 8;
#pragma unroll
        for (int s = 0; s < NS; ++s) qf[s] = *(const bf16x8*)(qrow + s * 16);
        if (scale < 0.f)
#pragma unroll
            for (int s = 0; s < NS; ++s) qf[s] = -qf[s];
    }
    const float scale2 = fabsf(scale) * LOG2E;      // log2-domain softmax

    // A thread loads 16-byte chunks of rows trow, trow + 256 / CPR, ... K's
    // chunks are XORed with the row's low bits: 8 rows at one column then lie
    // in 8 different chunks. V's by 4 times those of 4 rows (D = 64, whose rows
    // fill half the banks: of every second row), so that the 4 rows x 4 chunks
    // of a transposing read fill the banks (with K's swizzle they shared a
    // quarter of them: 10 % of the kernel). The low bits are the same in all of
    // a thread's rows.
    const int trow = threadIdx.x / CPR, tcol = threadIdx.x % CPR;
    const int kcol = (tcol ^ (trow & 7)) * 8;
    const int vcol = (tcol ^ (CPR > 8 ? (trow & 3) << 2 : (trow & 2) << 1)) * 8;
    // keys from k0 on, which lie together; rows behind the last key are zeros
    const u32 ko = (trow * D + kcol) * 2, vo = (trow * D + vcol) * 2;
    auto issue = [&](int k0, long at, bf16_t* to) {
        const u32 bytes = min(s_total - k0, 64) * D * 2;
        const LdsSource ks = lds_source(kv.k + at, bytes);
        const LdsSource vs = lds_source(kv.v + at, bytes);
        bf16_t* tw = to + wid * 512;
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
            load_lds16(ks, ko, i * 4096, tw + i * 2048);
            load_lds16(vs, vo, i * 4096, tw + TILE / 2 + i * 2048);
        }
    };

    // Where a lane reads, of a tile's first rows: K by the swizzle of its row
    // (the low bits of the chunk number; the others are the slice's), V by
    // transposing reads of rows l % 16 / 4, whose swizzle exchanges 32-wide
    // tiles.
    int kat[4], vat[VT];
#pragma unroll
    for (int s = 0; s < 4; ++s)
        kat[s] = ln * D + ((s * 2 + hi) ^ (ln & 7)) * 8;
    const int vr = (lane & 15) >> 2;
#pragma unroll
    for (int t = 0; t < VT; ++t)
        vat[t] = (hi * 8 + vr) * D + (t ^ (CPR > 8 ? vr : vr >> 1)) * 32 +
                 (lane & 16) + (lane & 3) * 4;

    const int q_abs = causal_off + qw + ln;
    float m = -1e30f, l = 0.f;          // finite: nothing seen weighs 0
    f32x16 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[t][r] = 0.f;

    // One tile in LDS; MASK: some of its keys are not seen by all rows.
    auto step = [&](const bf16_t* kt, int kc, auto MASK) {
        constexpr bool mask = decltype(MASK)::value;
        const bf16_t* vt = kt + TILE / 2;
        f32x16 sv[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) sv[u][r] = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s)
#pragma unroll
            for (int u = 0; u < 2; ++u)
                sv[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                    *(const bf16x8*)(kt + kat[s & 3] + u * 32 * D +
                                     (s >> 2) * 64), qf[s], sv[u], 0, 0, 0);
        reads_ahead<2 * NS, 4>();
        __builtin_amdgcn_sched_barrier(0);

        float mx = -FLT_MAX;
        u32 seen = 0;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                if constexpr (mask) {
                    const int key = kc + u * 32 + (r & 3) + 8 * (r >> 2) +
                                    4 * hi;
                    const bool ok = key < s_total && key <= q_abs &&
                                    keys.sees(q_abs, key);
                    seen |= (u32)ok << (u * 16 + r);
                    mx = fmaxf(mx, ok ? sv[u][r] : -FLT_MAX);
                } else {
                    mx = fmaxf(mx, sv[u][r]);
                }
            }
        mx = max_across32(mx) * scale2;
        if (__any(mx > m + MAX_LAG)) {
            const float mn = mx > m + MAX_LAG ? mx : m;
            const float alpha = fast_exp2(m - mn);
            l *= alpha;
            m = mn;
#pragma unroll
            for (int t = 0; t < NT; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[t][r] *= alpha;
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            float ls = 0.f;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                float w = fast_exp2(fmaf(sv[u][r], scale2, -m));
                if constexpr (mask)
                    w = seen >> (u * 16 + r) & 1 ? w : 0.f;
                sv[u][r] = w;
                ls += w;
            }
            l += ls;
#pragma unroll
            for (int s = 0; s < 2; ++s) {
                // lane half hi holds keys 8 g + 4 hi + 0..3; it needs
                // 8 hi + 0..7
                u32 w[4];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const int o = 8 * s + 2 * i;
                    const u32x2 x = __builtin_amdgcn_permlane32_swap(
                        pack2(sv[u][o], sv[u][o + 1]),
                        pack2(sv[u][o + 4], sv[u][o + 5]), false, false);
                    w[i] = x[0];
                    w[2 + i] = x[1];
                }
                bf16x8 pf;
                __builtin_memcpy(&pf, w, 16);
                // O^T += V^T P
#pragma unroll
                for (int t = 0; t < NT; ++t) {
                    bf16x8 v;
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const bf16x4 x = read_transposed(
                            vt + vat[t % VT] + (u * 32 + s * 16 + j * 4) * D +
                            t / VT * VT * 32);
#pragma unroll
                        for (int i = 0; i < 4; ++i) v[j * 4 + i] = x[i];
                    }
                    acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                        v, pf, acc[t], 0, 0, 0);
                }
            }
        }
    };

    const int kmax = min(s_total, causal_off + q0 + 128);
    const int qfirst = causal_off + q0;
    int k0 = keys.skip(0, qfirst), buf = 0;
    typename KV::Walk place;
    if (k0 < kmax) issue(k0, place(kv, slot, hk, k0), lds);
    // (or the compiler waits for q in each step, and for the next tile with it)
#pragma unroll
    for (int s = 0; s < NS; ++s) asm volatile("" : "+v"(qf[s]));
    // all rows of the block see the whole tile
    auto whole = [&] {
        return k0 + 63 <= qfirst && k0 + 63 < s_total &&
               keys.sees_tile(qfirst + 127, k0);
    };
    auto walk = [&](auto MASK) {
        const int kc = k0;
        const bf16_t* kt = lds + buf * TILE;
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();              // tile is there, the other one is free
        buf ^= 1;
        k0 = keys.skip(k0 + 64, qfirst);
        if (k0 < kmax) issue(k0, place(kv, slot, hk, k0), lds + buf * TILE);
        if (!decltype(MASK)::value || kc <= causal_off + qw + 31)
            step(kt, kc, MASK);     // else ahead of all of the wave's rows
    };
    // two loops, so that sums stay in their registers
    while (k0 < kmax) {
        while (k0 < kmax && whole()) walk(std::false_type());
        while (k0 < kmax && !whole()) walk(std::true_type());
    }

    // ---- normalize + store: lane holds O^T[*][q=ln] — one q-row --------
    l += __shfl_xor(l, 32, WAVE);
    if (qw + ln < T) {
        const int r = qw + ln;
        const float inv = epi.factor(row0 + r, hq, m, l);
        bf16_t* orow = out + epi.at(r, hq, Hq, D);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int d = t * 32 + 8 * g + 4 * hi;
                float f[4];
#pragma unroll
                for (int i = 0; i < 4; ++i) f[i] = acc[t][4 * g + i] * inv;
                if (epi.gate_el) {
                    float z[4];
                    ld4(epi.gate + (long)(row0 + r) * epi.gate_ld + hq * D + d,
                        z);
#pragma unroll
                    for (int i = 0; i < 4; ++i) f[i] /= 1.f + __expf(-z[i]);
                }
                st4(orow + d, f);
            }
        }
    }
}
