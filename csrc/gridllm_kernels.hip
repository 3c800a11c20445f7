// GridLLM-AMD CDNA4 (gfx950 / MI355X) kernels.
//
// Hand-written HIP for the decode/prefill hot path of the in-process engine
// that replaces the reference's external Ollama dependency
// (reference: client/src/services/OllamaService.ts — an HTTP adapter; the
// compute it delegated lives here instead).
//
// Design notes:
//  * wave64; all bf16 I/O is loaded vectorized (uint4 = 16 B = 8 bf16),
//    compute in f32; MFMA (mfma_f32_16x16x32/32x32x16_bf16) for the
//    matmul-shaped kernels (prefill attention, projection GEMMs).
//  * memory-bound ops target the HBM3E roofline (~6.3 TB/s achievable);
//    decode projections are bound by streaming W, or a CU's loads of x and W:
//    k_gemm_rows loads straight into MFMA operands, k_gemm_tile and k_gemm_fed
//    move both through rings in LDS.
//  * attention decode: 4-wave workgroup per (batch, kv_head, split), K and V
//    streamed through registers; split-S partials where B*Hk is small.
//  * exported as extern "C" with an explicit hipStream_t so launches are
//    capturable in hipGraphs from the Python host layer (ctypes binding —
//    no torch C++ ABI dependency, no hipify, no CUDA shims).
//
// Build: hipcc --offload-arch=gfx950 -O3 -shared -fPIC

#include "gridllm_attention.h"
#include "gridllm_batch.h"
#include "gridllm_wide.h"

// ===========================================================================
// RMSNorm (optionally fused residual add):
//   if res_in:  z = x + res_in; res_out = z  else z = x
//   y = z * rsqrt(mean(z^2) + eps) * w
// x,y,w,res: bf16. One workgroup (256 thr) per row; H % 8 == 0.
// A row stays in registers between the two passes (NV chunks a thread, or
// NV = 0: rows of any length, read twice): 8000 rows of 3072 with a residual 38
// -> 33 us, 6 TB/s.
// ===========================================================================

// Rows that are normed: stored ones, or f32 partial sums `stride` apart of a
// product whose K is in parts, rounded as its result would be.
struct StoredRow {
    const bf16_t* x;
    DEV_INLINE uint4 operator()(long c) const { return ((const uint4*)x)[c]; }
    DEV_INLINE void two(long c, long d, uint4& lo, uint4& hi) const {
        lo = (*this)(c);
        hi = (*this)(d);
    }
};
struct SummedRow {
    const float* ws;
    long stride;
    int parts;
    DEV_INLINE uint4 operator()(long c) const {
        float f[8] = {};
#pragma unroll 4
        for (int k = 0; k < parts; ++k) {
            float a[8];
            ld8(ws + k * stride + c * 8, a);
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] += a[i];
        }
        return pack8(f);
    }
    // (up to eight parts of two places at a time: one after the other they would wait
    // two to four times)
    DEV_INLINE void two(long c, long d, uint4& lo, uint4& hi) const {
        float f[8] = {}, g[8] = {};
#pragma unroll 1
        for (int k0 = 0; k0 < parts; k0 += 8) {
            float a[8][8], b[8][8];
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (k0 + k >= parts) break;
                ld8(ws + (k0 + k) * stride + c * 8, a[k]);
                ld8(ws + (k0 + k) * stride + d * 8, b[k]);
            }
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                if (k0 + k >= parts) break;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    f[i] += a[k][i];
                    g[i] += b[k][i];
                }
            }
        }
        lo = pack8(f);
        hi = pack8(g);
    }
};

// (rr, ro: a residual that is added, and the sum; SummedRow has one, or NV > 0.) NV
// turns of THREADS threads have the row, and all loads are on their way at once,
// the weights', too. In a graph, rows of 3072 with a residual, us: 1 row 3.3 with 256
// threads and the weights loaded after the sum, now 2.6; 256 rows 3.8 and 3.2; 8000
// rows 30.1 and 29.6. None of 2304 to 8192 columns and 1 to 8192 rows got slower.
template <int NV, int THREADS, class Row>
DEV_INLINE void rmsnorm_row(bf16_t* yr, const Row x, const bf16_t* w,
                            const bf16_t* rr, bf16_t* ro, int H, float eps,
                            float* red) {
    const int nchunk = H >> 3;  // uint4 chunks
    uint4 z[NV ? NV : 1];       // of this thread, rounded as they are stored
    uint4 g[NV ? NV : 1];
    float ss = 0.f;
    auto first = [&](int c) {
        uint4 v = x(c);
        float f[8];
        unpack8(v, f);
        if (rr) {
            float b[8];
            unpack8(((const uint4*)rr)[c], b);
#pragma unroll
            for (int i = 0; i < 8; ++i) f[i] += b[i];
            v = pack8(f);
            ((uint4*)ro)[c] = v;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += f[i] * f[i];
        return v;
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int c = threadIdx.x + k * THREADS;
            if (c < nchunk) {
                g[k] = ((const uint4*)w)[c];
                z[k] = first(c);
            }
        }
    } else {
        for (int c = threadIdx.x; c < nchunk; c += THREADS) first(c);
    }
    const float scale =
        rsqrtf(block_sum<THREADS>(ss, red) / (float)H + eps);
    auto second = [&](int c, const uint4 zv, const uint4 gv) {
        float f[8], b[8];
        unpack8(zv, f);
        unpack8(gv, b);
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = f[i] * scale * b[i];
        ((uint4*)yr)[c] = pack8(f);
    };
    if constexpr (NV > 0) {
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            const int c = threadIdx.x + k * THREADS;
            if (c < nchunk) second(c, z[k], g[k]);
        }
    } else {
        for (int c = threadIdx.x; c < nchunk; c += THREADS)
            second(c, rr ? ((const uint4*)ro)[c] : x(c), ((const uint4*)w)[c]);
    }
}

template <int NV, int THREADS>
__global__ void __launch_bounds__(THREADS)
k_rmsnorm(bf16_t* __restrict__ y, const bf16_t* __restrict__ x,
          const bf16_t* __restrict__ w, const bf16_t* __restrict__ res_in,
          bf16_t* __restrict__ res_out, int H, float eps) {
    __shared__ float red[8];
    const long at = blockIdx.x * (long)H;
    rmsnorm_row<NV, THREADS>(y + at, StoredRow{x + at}, w, res_in ? res_in + at : nullptr,
                    res_out ? res_out + at : nullptr, H, eps, red);
}

// The same behind a product whose K is in parts: their sums are taken here, which
// spares a launch and the result's way through memory. With the product: 24 rows
// of 3072, K = 3072 in 5 parts 12.1 -> 11.2 us; 45 rows of 2048, K = 2048 in 4
// 10.5 -> 8.5; 256 rows of 3072, K = 8192 in 4 33.1 -> 29.9.
template <int NV, int THREADS>
__global__ void __launch_bounds__(THREADS)
k_rmsnorm_parts(bf16_t* __restrict__ y, const float* __restrict__ ws, int parts,
                const bf16_t* __restrict__ w, const bf16_t* __restrict__ res_in,
                bf16_t* __restrict__ res_out, int H, float eps) {
    __shared__ float red[8];
    const long at = blockIdx.x * (long)H;
    rmsnorm_row<NV, THREADS>(y + at, SummedRow{ws + at, gridDim.x * (long)H, parts}, w,
                    res_in + at, res_out + at, H, eps, red);
}

// ===========================================================================
// Start and end of a decode step: see gl_decode_start and
// gl_advance_lengths, which stand for the dozen index kernels of 4 us each that
// a step had. A slot that there is not ends the program, as an index does that
// torch finds out of bounds, before anything is read or counted by it.
// ===========================================================================
// rows (B <= ROWS_ORDERED): {row, keys, slot, rotary position}, the longest first and
// equal ones in the batch's order, as attention's blocks start. Four lanes count the
// rows that are ahead of one, by LDS: in the launch that there is anyway, 5.8 us for 256
// rows (4.7 without; 12.7 by a lane a row).
#define ROWS_ORDERED 1024
__global__ void __launch_bounds__(256)
k_decode_positions(int* __restrict__ pos, int* __restrict__ slot_t,
                   int* __restrict__ pos_rope, int* __restrict__ attn_seq,
                   int4* __restrict__ rows, const int* __restrict__ seq_lens,
                   const int* __restrict__ rope_off,
                   const int* __restrict__ slot_map, int B, int slots,
                   int Smax) {
    typedef __attribute__((ext_vector_type(4))) int i32x4;
    __shared__ __attribute__((aligned(16))) int lens[ROWS_ORDERED];
    const int i = blockIdx.x * 64 + (threadIdx.x >> 2), part = threadIdx.x & 3;
    const int s = i < B ? slot_map[i] : 0;
    if ((unsigned)s >= (unsigned)slots) __builtin_trap();
    const int p = seq_lens[s], all = (B + 15) & ~15;
    if (rows)
        for (int j = threadIdx.x; j < all; j += 256) {
            const int t = j < B ? slot_map[j] : -1;
            lens[j] = (unsigned)t < (unsigned)slots ? seq_lens[t] : INT_MIN;
        }
    if (i < B && part == 0) {
        pos[i] = p;
        if (slot_t) slot_t[i] = s * Smax + p;
        if (attn_seq) attn_seq[i] = p + 1;
        if (pos_rope) pos_rope[i] = p + rope_off[s];
    }
    if (!rows) return;
    __syncthreads();
    int ahead = 0;
#pragma unroll 4
    for (int j = part * 4; j < all; j += 16) {
        const i32x4 m = *(const i32x4*)(lens + j);
#pragma unroll
        for (int k = 0; k < 4; ++k) ahead += m[k] > p || (m[k] == p && j + k < i);
    }
    ahead += __shfl_xor(ahead, 1, WAVE);
    ahead += __shfl_xor(ahead, 2, WAVE);
    if (i < B && part == 0)
        rows[ahead] = make_int4(i, p + 1, s, rope_off ? p + rope_off[s] : p);
}

__global__ void __launch_bounds__(256)
k_advance_lengths(int* __restrict__ seq_lens, const int* __restrict__ slot_map,
                  int B, int slots) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= B) return;
    const int s = slot_map[i];
    if ((unsigned)s >= (unsigned)slots) __builtin_trap();
    atomicAdd(seq_lens + s, 1);
}

// A prompt's positions start .. start + T - 1 and places in its slot; and, when
// it has been run, the slot's length and (if it started anew) rotary offset.
__global__ void __launch_bounds__(256)
k_prompt_positions(int* __restrict__ pos, int* __restrict__ slot_t, int slot,
                   int start, int T, int Smax) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i < T) {
        pos[i] = start + i;
        slot_t[i] = slot * Smax + start + i;
    }
}

__global__ void k_prompt_end(int* __restrict__ seq_lens,
                             int* __restrict__ rope_off, int slot, int start,
                             int T) {
    seq_lens[slot] = start + T;
    if (start == 0) rope_off[slot] = 0;
}

// The same for B new sequences, and their rows `lasts` of x, one behind the other
// (out null: none of them). Bound by the launch, so there is one: torch needs five
// (a conversion, two scatters, a gather and an upload of 64-bit indices). With the
// indices' one copy instead of four 4 prompts of 60 tokens (16 layers of 2048) take
// 397 us for 424, 8 of 300 (28 of 3072) 1320 for 1347. A slot or row that there is
// not ends the program.
__global__ void __launch_bounds__(256)
k_prompts_end(int* __restrict__ seq_lens, int* __restrict__ rope_off,
              const int* __restrict__ of_slots, const int* __restrict__ lens,
              int slots, uint4* __restrict__ out, const uint4* __restrict__ x,
              const int* __restrict__ lasts, int rows, int pieces) {
    const int b = blockIdx.x, s = of_slots[b];
    if ((unsigned)s >= (unsigned)slots) __builtin_trap();
    if (threadIdx.x == 0) {
        seq_lens[s] = lens[b];
        rope_off[s] = 0;
    }
    if (!out) return;
    const int r = lasts[b] < 0 ? lasts[b] + rows : lasts[b];
    if ((unsigned)r >= (unsigned)rows) __builtin_trap();
    for (int c = threadIdx.x; c < pieces; c += 256)
        out[(long)b * pieces + c] = x[(long)r * pieces + c];
}

// x = emb[token], y = rmsnorm(x) * w: one block per row. Tokens count from the
// end if negative; others than the table has end the program, as an index does
// that a lookup by torch finds out of bounds.
template <int NV, int THREADS>
__global__ void __launch_bounds__(THREADS)
k_embed_norm(bf16_t* __restrict__ x, bf16_t* __restrict__ y,
             const bf16_t* __restrict__ emb,
             const long long* __restrict__ tokens,
             const bf16_t* __restrict__ w, int H, int vocab, float eps) {
    __shared__ float red[8];
    long long t = tokens[blockIdx.x];
    if (t < 0) t += vocab;
    if (t < 0 || t >= vocab) __builtin_trap();
    const long at = blockIdx.x * (long)H;
    const bf16_t* row = emb + t * H;
    for (int c = threadIdx.x; c < H >> 3; c += THREADS)
        ((uint4*)(x + at))[c] = ((const uint4*)row)[c];
    rmsnorm_row<NV, THREADS>(y + at, StoredRow{row}, w, nullptr, nullptr, H, eps, red);
}

// ===========================================================================
// RoPE (neox/llama split-half layout), in-place on q and k.
//   q: [T, Hq, D]  k: [T, Hk, D]  (bf16)
//   cos/sin: [max_seq, D/2] (f32, host-precomputed table)
//   pos: [T] int32 absolute positions
// Pair (t, h, i): (a,b) = (x[i], x[i+D/2]) -> (a*c - b*s, a*s + b*c)
// Thread handles 2 consecutive pairs (4 B loads both halves).
// ===========================================================================

__global__ void __launch_bounds__(256)
k_rope(bf16_t* __restrict__ q, bf16_t* __restrict__ k,
       const float* __restrict__ cost, const float* __restrict__ sint,
       const int* __restrict__ pos, int T, int Hq, int Hk, int D) {
    const int half = D >> 1;
    const int pairs2 = half >> 1;             // 2-pair work items per head
    const long total = (long)T * (Hq + Hk) * pairs2;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total;
         idx += gridDim.x * 256L) {
        int p2 = (int)(idx % pairs2);
        long th = idx / pairs2;
        int h = (int)(th % (Hq + Hk));
        int t = (int)(th / (Hq + Hk));
        bf16_t* base = (h < Hq) ? q + ((long)t * Hq + h) * D
                                : k + ((long)t * Hk + (h - Hq)) * D;
        const int i = p2 * 2;
        const int p = pos[t];
        const float2 c = ((const float2*)(cost + (long)p * half))[p2];
        const float2 s = ((const float2*)(sint + (long)p * half))[p2];
        u32 lo = *(u32*)(base + i);           // 2 bf16: x[i], x[i+1]
        u32 hi = *(u32*)(base + half + i);    // 2 bf16: x[i+half], x[i+half+1]
        float a0 = __uint_as_float((lo & 0xffffu) << 16);
        float a1 = __uint_as_float(lo & 0xffff0000u);
        float b0 = __uint_as_float((hi & 0xffffu) << 16);
        float b1 = __uint_as_float(hi & 0xffff0000u);
        float r0 = a0 * c.x - b0 * s.x, r1 = a1 * c.y - b1 * s.y;
        float q0 = a0 * s.x + b0 * c.x, q1 = a1 * s.y + b1 * c.y;
        *(u32*)(base + i) = (u32)f2bf(r0) | ((u32)f2bf(r1) << 16);
        *(u32*)(base + half + i) = (u32)f2bf(q0) | ((u32)f2bf(q1) << 16);
    }
}

// ===========================================================================
// Gated linear unit: out[n, F] = act(gateup[n, 0:F], gateup[n, F:2F])  (bf16)
// Fused epilogue for the gate/up projection (one GEMM outputs [n, 2F]).
// ===========================================================================

__global__ void __launch_bounds__(256)
k_swiglu(bf16_t* __restrict__ out, const bf16_t* __restrict__ gateup,
         long n, int F, const GluParams glu) {
    const int fc = F >> 3;                    // uint4 chunks per half-row
    const long total = n * fc;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total;
         idx += gridDim.x * 256L) {
        long r = idx / fc;
        int c = (int)(idx % fc);
        const uint4 gv = ((const uint4*)(gateup + r * 2L * F))[c];
        const uint4 uv = ((const uint4*)(gateup + r * 2L * F + F))[c];
        float g[8], u[8];
        unpack8(gv, g);
        unpack8(uv, u);
        glu_units(g, g, u, glu);
        ((uint4*)(out + r * (long)F))[c] = pack8(g);
    }
}

// ===========================================================================
// Fused RoPE + KV-cache write (the per-layer attention prologue).
//   qkv: [N, (Hq+2*Hk)*D] bf16 — the raw fused-QKV GEMM output (row-dense),
//   bias: [(Hq+2*Hk)*D] bf16, added to it (rounded, as a sum of its own), or null;
//   q_out: [N, Hq, D] roped q; k is roped and written straight into kcache,
//   v copied into vcache (slot[n] = cache_slot*Smax + pos).
// Replaces {2x contiguous-copy, rope, kv_append} = 4 kernels + one HBM
// round trip per layer. One workgroup (64 thr) per (token, head).
// ===========================================================================

__global__ void __launch_bounds__(64)
k_rope_kv(const bf16_t* __restrict__ qkv, bf16_t* __restrict__ q_out,
          bf16_t* __restrict__ kc, bf16_t* __restrict__ vc,
          const float* __restrict__ cost, const float* __restrict__ sint,
          const int* __restrict__ pos, const int* __restrict__ slot,
          const bf16_t* __restrict__ bias, int Hq, int Hk, int D, int Smax) {
    const int nh = Hq + Hk;
    const int n = blockIdx.x / nh;
    const int h = blockIdx.x % nh;
    const int W = (Hq + 2 * Hk) * D;
    const int half = D >> 1;
    const int p = pos[n];
    const float* crow = cost + (long)p * half;
    const float* srow = sint + (long)p * half;

    const bf16_t* src;
    auto biased = [&](bf16_t v, int at) {
        return bias ? f2bf(bf2f(v) + bf2f(bias[at])) : v;
    };
    bf16_t* dst;
    if (h < Hq) {
        src = qkv + (long)n * W + h * D;
        dst = q_out + ((long)n * Hq + h) * D;
    } else {
        const int hk = h - Hq;
        src = qkv + (long)n * W + (Hq + hk) * D;
        const long sl = slot[n];
        const long b = sl / Smax, pp = sl % Smax;
        dst = kc + (((b * Hk + hk) * Smax) + pp) * D;
        // copy v row (no rope)
        const bf16_t* vsrc = qkv + (long)n * W + (Hq + Hk + hk) * D;
        bf16_t* vdst = vc + (((b * Hk + hk) * Smax) + pp) * D;
        for (int i = threadIdx.x; i < D; i += 64)
            vdst[i] = biased(vsrc[i], (Hq + Hk + hk) * D + i);
    }
    for (int i = threadIdx.x; i < half; i += 64) {
        float a = bf2f(biased(src[i], h * D + i));
        float b = bf2f(biased(src[i + half], h * D + i + half));
        float c = crow[i], s = srow[i];
        dst[i] = f2bf(a * c - b * s);
        dst[i + half] = f2bf(a * s + b * c);
    }
}

// The same, 8 pairs a lane: half / 8 lanes turn a q or k head (two 16-byte
// loads and stores), as many copy a v head; heads of all tokens lie one after
// the other over the lanes. D % 16 == 0 and rows at 16 bytes. 8000 tokens of
// 24 + 8 + 8 heads of 128: 83 us (2 TB/s) with a wave per head and 2-byte
// accesses, 31 us (5.2 TB/s) now. Rows may be a product's partial sums (SummedRow),
// which spares the kernel that adds them up (four layers of llama3.2:1b, 45
// tokens 323 -> 316 us).
template <class Row>
DEV_INLINE void turned8(const Row& rows, long src, int half, const bf16_t* bias,
                        bool turn, const float* cos_, const float* sin_, uint4& lo,
                        uint4& hi) {
    rows.two(src, src + (half >> 3), lo, hi);
    if (bias) {
        float a[8], b[8];
        unpack8(lo, a);
        ld8(bias, b);
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] += b[k];
        lo = pack8(a);
        unpack8(hi, a);
        ld8(bias + half, b);
#pragma unroll
        for (int k = 0; k < 8; ++k) a[k] += b[k];
        hi = pack8(a);
    }
    if (turn) {
        float a[8], b[8], co[8], si[8];
        ld8(cos_, co);
        ld8(sin_, si);
        unpack8(lo, a);
        unpack8(hi, b);
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float u = a[k], v = b[k];
            a[k] = u * co[k] - v * si[k];
            b[k] = u * si[k] + v * co[k];
        }
        lo = pack8(a);
        hi = pack8(b);
    }
}

template <class Row>
__global__ void __launch_bounds__(256)
k_rope_kv8(const Row rows, bf16_t* __restrict__ q_out,
           bf16_t* __restrict__ kc, bf16_t* __restrict__ vc,
           const float* __restrict__ cost, const float* __restrict__ sint,
           const int* __restrict__ pos, const int* __restrict__ slot,
           const bf16_t* __restrict__ bias, int N, int Hq, int Hk, int D,
           int Smax) {
    const int half = D >> 1, lanes = half >> 3, heads = Hq + 2 * Hk;
    const long i = blockIdx.x * 256L + threadIdx.x;
    const long item = i / lanes;
    if (item >= (long)N * heads) return;
    const int c = (int)(i % lanes) * 8;
    const int n = (int)(item / heads), h = (int)(item % heads);
    const long at = h < Hq + Hk ? (long)pos[n] * half + c : 0;
    uint4 lo, hi;
    turned8(rows, (item * D + c) >> 3, half, bias ? bias + h * D + c : nullptr,
            h < Hq + Hk, cost + at, sint + at, lo, hi);
    bf16_t* dst;
    if (h < Hq) {
        dst = q_out + ((long)n * Hq + h) * D + c;
    } else {
        const int s = slot[n], b = s / Smax, p = s - b * Smax;
        const int hk = h < Hq + Hk ? h - Hq : h - Hq - Hk;
        dst = (h < Hq + Hk ? kc : vc) + (((long)b * Hk + hk) * Smax + p) * D +
              c;
    }
    *(uint4*)dst = lo;
    *(uint4*)(dst + half) = hi;
}

// A decode row's queries, key and value for k_attn_decode (see Own there), in place of
// that kernel ahead of it: a launch less a layer. The last wave makes them under the
// others' loads of keys (all of them behind their own: 256 rows of up to 384 keys 54, now
// 48; 53 with the kernel ahead). A decode step of 256 rows, 4 layers, 840 -> 805 us.
template <int D, class Row>
struct TurnedHeads {
    static constexpr bool MADE = true;
    Row rows;
    const float *cos_, *sin_;
    const int* pos;
    const bf16_t* bias;
    int heads;                         // queries', keys' and values'
    DEV_INLINE void operator()(int row, int head, bool turn, int c, int place,
                               uint4& lo, uint4& hi) const {
        const long at = (long)place * (D / 2) + c;
        turned8(rows, (((long)row * heads + head) * D + c) >> 3, D / 2,
                bias ? bias + head * D + c : nullptr, turn, cos_ + at, sin_ + at, lo,
                hi);
    }
};

// ===========================================================================
// KV-cache append.
//   kc/vc: [B, Hk, Smax, D] bf16;  kn/vn: [N, Hk, D];  slot[N] = b*Smax + pos
// One workgroup (64 thr) per (token, kv-head); copies both K and V rows.
// ===========================================================================

__global__ void __launch_bounds__(64)
k_kv_append(bf16_t* __restrict__ kc, bf16_t* __restrict__ vc,
            const bf16_t* __restrict__ kn, const bf16_t* __restrict__ vn,
            const int* __restrict__ slot, int Hk, int D, int Smax) {
    const int n = blockIdx.x / Hk;
    const int h = blockIdx.x % Hk;
    const long sl = slot[n];
    const long b = sl / Smax, p = sl % Smax;
    const long dst = ((b * Hk + h) * Smax + p) * D;
    const long src = ((long)n * Hk + h) * D;
    const int nu = D >> 1;                    // u32 chunks
    for (int i = threadIdx.x; i < nu; i += 64) {
        ((u32*)(kc + dst))[i] = ((const u32*)(kn + src))[i];
        ((u32*)(vc + dst))[i] = ((const u32*)(vn + src))[i];
    }
}

// ===========================================================================
// Skinny-M weight-streaming GEMM:  out[M,N] = x[M,K] @ W[N,K]^T   (bf16 I/O)
//
// The decode-path projection GEMMs (M = batch <= 256, W = torch linear
// weight, row-major [N,K]) are HBM-bound on W. hipBLASLt reaches only ~40%
// of the roofline on these shapes (profiles/r01_decode_profile.md), so this
// kernel streams W once, straight into MFMA B
// fragments — both operands are k-contiguous, so fragments load directly
// from HBM/L2 with no LDS staging (M <= 256 by 16-row MFMA tiles).
//
// mfma_f32_16x16x32_bf16 lane mapping used here:
//   A[i][k]: lane l holds rows i = l&15, k = (l>>4)*8 + 0..7  (8 bf16 = 16 B)
//   B[k][j]: lane l holds col  j = l&15, same k chunk
//   D[i][j]: col j = l&15, row i = (l>>4)*4 + reg
// Block = 4 waves; each wave owns 16 output columns (BN = 64 per block);
// grid = (N/64) * splitk, k-slices 32-aligned; splitk > 1 accumulates f32
// partials in ws, combined by k_gemm_combine.
// Constraints: N % 64 == 0, K % 32 == 0, M <= 16*MT.
// ===========================================================================

template <int MT>
__global__ void __launch_bounds__(256, 2)
k_gemm_skinny(bf16_t* __restrict__ out, float* __restrict__ ws,
              const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
              int M, int N, int K, int splitk, int kslice) {
    // Occupancy-first design: the grid is (N/64) * splitk blocks with
    // kslice a small multiple of 256, so 2-8 blocks share each CU and TLP
    // hides the weight-stream latency (one wave per SIMD cannot — measured).
    // Per 256-k sub-slice the body is straight-line: issue all 8 B chunks
    // (16 B/lane, k-contiguous; not nontemporal: a load takes half a cache
    // line, 24 rows of 9216 x 3072 in 8 parts 22.2 -> 19.6 us), stage the x
    // panel into LDS coalesced
    // (XOR-swizzled), barrier, 8 x MT MFMAs off ds_read_b128 fragments.
    const int lane = threadIdx.x & 63;
    const int wid = threadIdx.x >> 6;
    const int ks = blockIdx.x % splitk;
    const int ntile = blockIdx.x / splitk;
    const int n0 = ntile * 64 + wid * 16;       // this wave's column base
    const int k0 = ks * kslice;
    const int k1 = min(K, k0 + kslice);
    const int fr = lane & 15;                   // fragment row (A) / col (B)
    const int kg = (lane >> 4) * 8;             // k sub-chunk

    constexpr int KS = 256;                     // k per staged panel
    constexpr int ROWS = MT * 16;
    __shared__ __attribute__((aligned(16))) bf16_t xs[ROWS * KS];
    const int swz = (fr & 15) << 4;

    f32x4 acc[MT];
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};

    const bf16_t* wrow = w + (long)(n0 + fr) * K + kg;

    for (int kp = k0; kp < k1; kp += KS) {
        const int nch = min(KS, k1 - kp) >> 5;  // 32-k chunks (8 when full)
        // all B chunks of this panel in flight first (branchless clamp)
        const int kcl = k1 - 32;
        bf16x8 bb[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
            bb[u] = *(const bf16x8*)(wrow + min(kp + u * 32, kcl));
        // stage x[*, kp:kp+KS] -> LDS: thread c covers (row=c/32, kc=c%32);
        // 32 lanes read one row's 512 B contiguously; swizzled ds_write_b128
        if (kp > k0) __syncthreads();           // previous panel fully read
#pragma unroll
        for (int i = 0; i < MT * 2; ++i) {
            const int c = (int)threadIdx.x + i * 256;
            const int row = c >> 5;
            const int kc = c & 31;
            const uint4 v = *(const uint4*)(
                x + (long)min(row, M - 1) * K
                + min((long)kp + kc * 8, (long)K - 8));
            const int byte = ((row * KS + kc * 8) * 2) ^ ((row & 15) << 4);
            *(uint4*)((char*)xs + byte) = v;
        }
        __syncthreads();
        // 8 chunks x MT MFMAs; full panels take the unguarded fast path
        if (nch == 8) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int row = t * 16 + fr;
                    const int byte = ((row * KS + u * 32 + kg) * 2) ^ swz;
                    const bf16x8 a = *(const bf16x8*)((const char*)xs + byte);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        a, bb[u], acc[t], 0, 0, 0);
                }
            }
        } else {
            for (int u = 0; u < nch; ++u) {
                const bf16x8 b = bb[u];
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    const int row = t * 16 + fr;
                    const int byte = ((row * KS + u * 32 + kg) * 2) ^ swz;
                    const bf16x8 a = *(const bf16x8*)((const char*)xs + byte);
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        a, b, acc[t], 0, 0, 0);
                }
            }
        }
    }

    const int orow = (lane >> 4) * 4;           // D rows this lane holds
    const int ocol = n0 + fr;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = t * 16 + orow + r;
            if (m < M) {
                if (splitk == 1) {
                    out[(long)m * N + ocol] = f2bf(acc[t][r]);
                } else {
                    ws[((long)ks * M + m) * N + ocol] = acc[t][r];
                }
            }
        }
    }
}

// ===========================================================================
// Few-row GEMM: out[M,N] = x[M,K] @ W[N,K]^T (bf16 I/O, f32 sums), M <= 16.
//
// Bound by streaming W, and for weights of a few MB by how soon all of it is on
// its way: a block takes 16 columns over all of K, its 8 waves a part of K
// each, whose loads start a batch of U chunks ahead, straight into MFMA
// operands. The waves' sums meet in LDS, so there is no second kernel and no
// workspace, which is what makes it the fastest for up to 20 MB of W with up to 4
// rows while K is 4096 or less, and 10 MB with 16 while it is 3072 or less (one row,
// k_gemm_tile's best split behind it: 2048 x 2048 5.7 us, 7.0; 3072 x 3072 6.7, 7.9;
// larger W streams faster there: 5120 x 3072 11.1, 9.7; longer K keeps a block at it:
// 2048 x 8192 13.0, 10.7; 16 rows of 2048 x 2048 7.2, 7.6, of 3072 x 3072 9.9, 8.3).
// Every block reads all of x, which for 16 rows costs as much as W. A gated unit's two
// columns halve its rate: it has those that no tiling fits. W's loads are plain: each takes half a cache
// line of a row, and past the caches (nontemporal) both halves fetch it: 8.0, 11.1, 16.6
// and 24.3 us.
// mfma_f32_16x16x32_bf16: A = x rows, B = W rows (k-contiguous both).
// GLU: W rows in groups of 64 gate | 64 up; a block takes 16 of each and
// stores the gated unit [M, N / 2].
// Constraints: N % 16 == 0 (GLU: N % 128 == 0), K % 32 == 0.
// ===========================================================================
template <int GLU>
__global__ void __launch_bounds__(512, 2)
k_gemm_rows(bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
            const bf16_t* __restrict__ w, int M, int N, int K,
            const GluParams glu) {
    constexpr int WAVES = 8, U = 4, NC = GLU ? 2 : 1;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, kg = (lane >> 4) * 8;
    const int n0 = GLU ? (blockIdx.x >> 2) * 128 + (blockIdx.x & 3) * 16
                       : blockIdx.x * 16;
    const int chunks = K >> 5;
    const int per = (chunks + WAVES - 1) / WAVES;
    const int c0 = wid * per, c1 = min(chunks, c0 + per);

    const bf16_t* wp[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i)
        wp[i] = w + (long)(n0 + i * 64 + fr) * K + kg;
    const bf16_t* xp = x + (long)min(fr, M - 1) * K + kg;

    f32x4 acc[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) acc[i] = (f32x4){0.f, 0.f, 0.f, 0.f};

    bf16x8 a0[U], b0[U][NC], a1[U], b1[U][NC];
    // chunks behind the last repeat it, and are not added
    auto load = [&](bf16x8 (&a)[U], bf16x8 (&b)[U][NC], int c) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int at = min(c + u, c1 - 1) * 32;
#pragma unroll
            for (int i = 0; i < NC; ++i)
                b[u][i] = *(const bf16x8*)(wp[i] + at);
            a[u] = *(const bf16x8*)(xp + at);
        }
    };
    auto add = [&](bf16x8 (&a)[U], bf16x8 (&b)[U][NC]) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < NC; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a[u], b[u][i], acc[i], 0, 0, 0);
    };
    // the last batch, the only one that may be short: the loop has no guards
    auto add_some = [&](bf16x8 (&a)[U], bf16x8 (&b)[U][NC], int n) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (u >= n) break;
#pragma unroll
            for (int i = 0; i < NC; ++i)
                acc[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    a[u], b[u][i], acc[i], 0, 0, 0);
        }
    };
    int c = c0, left = c1 - c0;
    if (left > 0) {
        load(a0, b0, c);
        while (left > 2 * U) {
            load(a1, b1, c + U);
            add(a0, b0);
            load(a0, b0, c + 2 * U);
            add(a1, b1);
            c += 2 * U;
            left -= 2 * U;
        }
        if (left > U) {
            load(a1, b1, c + U);
            add(a0, b0);
            add_some(a1, b1, left - U);
        } else {
            add_some(a0, b0, left);
        }
    }

    // the waves' sums; lane holds row (l >> 4) * 4 + r, column l & 15
    __shared__ f32x4 red[WAVES][NC][64];
#pragma unroll
    for (int i = 0; i < NC; ++i) red[wid][i][lane] = acc[i];
    __syncthreads();
    if (wid) return;
    f32x4 s[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        s[i] = red[0][i][lane];
#pragma unroll
        for (int v = 1; v < WAVES; ++v) s[i] += red[v][i][lane];
    }
    const int col = GLU ? (blockIdx.x >> 2) * 64 + (blockIdx.x & 3) * 16 + fr
                        : n0 + fr;
    float y[4], u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        y[r] = s[0][r];
        u[r] = s[NC - 1][r];
    }
    if (GLU) glu_units(y, y, u, glu);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        const int m = (lane >> 4) * 4 + r;
        if (m < M) out[(long)m * (GLU ? N >> 1 : N) + col] = f2bf(y[r]);
    }
}

// A kernel with more LDS than the default limit asks for it, once.
template <auto Kernel>
static int allow_lds(int bytes) {
    static const hipError_t e = hipFuncSetAttribute(
        (const void*)Kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
        bytes);
    return (int)e;
}

// Whether W, in parts of kslice of K, is read past the Infinity Cache: with one block of
// rows, or with two or three if it is little, in parts so short that these read it
// nearly at one time. (Time through the cache of that past it, mean of 28 such tilings
// 1.02, of 20 with longer parts 1.00, of 43 with more blocks of rows .97, of 148 with
// larger W .96. See gridllm_batch.h.)
static bool tile_once(int M, int N, int K, int rows, int kslice) {
    const int blocks = (M + rows - 1) / rows;
    return blocks == 1 ||
           (blocks < 4 && (long)N * K <= 8000000 && kslice < 1536);
}

template <int RT, int CT, int EPI, bool ONCE = false, bool PAST = false>
static int launch_gemm_tile(hipStream_t st, BatchArgs p) {
    constexpr bool both = RT <= 4;              // waves load and multiply
    typedef std::conditional_t<CT == 16, GemmCols<RT>, std::conditional_t<
        both, GemmTile<RT, CT>, GemmFed<RT, CT>>> Sh;
    if constexpr (both || CT == 16)
        if (p.K > BATCH_K)                      // (see there)
            return launch_gemm_tile<RT < 6 ? 6 : RT, CT == 16 ? 8 : CT, EPI>(st, p);
    p.rblocks = (p.M + Sh::R - 1) / Sh::R;
    if constexpr (!ONCE)
        if (tile_once(p.M, p.N, p.K, Sh::R, p.kslice))
            return launch_gemm_tile<RT, CT, EPI, true>(st, p);
    if constexpr (CT == 16 && ONCE && !PAST)
        if (p.splitk == 1 && (long)p.M * p.N * 4 >= COLS_PAST)
            return launch_gemm_tile<RT, CT, EPI, ONCE, true>(st, p);
    constexpr auto kernel = [] {
        if constexpr (CT == 16) return k_gemm_cols<RT, ONCE, PAST>;
        else if constexpr (both) return k_gemm_tile<RT, CT, EPI, ONCE>;
        else return k_gemm_fed<RT, CT, EPI, ONCE>;
    }();
    const int e = allow_lds<kernel>(Sh::BYTES);
    if (e) return e;
    const long total = (long)(p.N / Sh::C) * p.splitk * p.rblocks;
    const long each = (total + 7) / 8;         // (256 columns: blocks stay)
    kernel<<<(unsigned)(8 * (CT == 16 ? min(each, 32l) : each)), Sh::THREADS,
             Sh::BYTES, st>>>(p);
    LAUNCH_CHECK();
    return 0;
}

template <class S, class S2, int EPI, bool ONCE = false>
static int launch_gemm_wide(hipStream_t st, const WideArgs& p, int full) {
    if constexpr (EPI == 2 && !ONCE)
        if (p.M <= S::R) return launch_gemm_wide<S, S2, EPI, true>(st, p, full);
    constexpr int bytes = S::BYTES > S2::BYTES ? S::BYTES : S2::BYTES;
    constexpr auto kernel = k_gemm_wide<S, S2, EPI, ONCE>;
    const int e = allow_lds<kernel>(bytes);
    if (e) return e;
    const int total = (p.M + S::R - 1) / S::R * ((p.N + S::C - 1) / S::C);
    full = S2::R ? min(full, total) : total;
    const int most = max(full, (total - full) * 2);     // blocks' tiles
    kernel<<<8 * min((most + 7) / 8, 32), 512, bytes, st>>>(p, full);
    LAUNCH_CHECK();
    return 0;
}

// Combine split-K slabs of an INTERLEAVED gate/up projection with the
// SwiGLU epilogue applied during the combine: out[M, N/2] bf16.
__global__ void __launch_bounds__(256)
k_gemm_combine_swiglu(bf16_t* __restrict__ out, const float* __restrict__ ws,
                      int M, int N, int splitk, const GluParams glu) {
    const int no = N >> 1;
    const long mn = (long)M * N, total = (long)M * (no >> 2);
    for (long i = blockIdx.x * 256L + threadIdx.x; i < total;
         i += gridDim.x * 256L) {
        const long m = i / (no >> 2);
        const int j = (int)(i % (no >> 2)) * 4;        // output column
        const float* p = ws + m * N + (j >> 6) * 128 + (j & 63);
        float g[4] = {}, u[4] = {};
#pragma unroll 4
        for (int k = 0; k < splitk; ++k) {
            float a[4], b[4];
            ld4(p + k * mn, a);
            ld4(p + k * mn + 64, b);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                g[e] += a[e];
                u[e] += b[e];
            }
        }
        glu_units(g, g, u, glu);
        st4(out + m * (long)no + j, g);
    }
}

// SwiGLU over an INTERLEAVED gate/up activation (128-col groups
// [64 gate | 64 up]) — the library-GEMM fallback path for interleaved
// weights: out[n, F] from gu[n, 2F].
__global__ void __launch_bounds__(256)
k_swiglu_il(bf16_t* __restrict__ out, const bf16_t* __restrict__ gu,
            long n, int F, const GluParams glu) {
    const int fc = F >> 3;                        // 8-col units per out row
    const long total = n * fc;
    for (long idx = blockIdx.x * 256L + threadIdx.x; idx < total;
         idx += gridDim.x * 256L) {
        const long r = idx / fc;
        const int j = (int)(idx % fc) * 8;
        const int grp = j >> 6, win = j & 63;
        const bf16_t* base = gu + r * 2L * F + grp * 128 + win;
        uint4 gv = *(const uint4*)base;
        uint4 uv = *(const uint4*)(base + 64);
        float g[8], u[8];
        unpack8(gv, g);
        unpack8(uv, u);
        glu_units(g, g, u, glu);
        ((uint4*)(out + r * (long)F))[j >> 3] = pack8(g);
    }
}

// Combine split-K f32 partials -> bf16 out. Grid-stride over M*N/8 uint4s.
__global__ void __launch_bounds__(256)
k_gemm_combine(bf16_t* __restrict__ out, const float* __restrict__ ws,
               long mn, int splitk) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i * 4 < mn;
         i += gridDim.x * 256L) {
        float4 s = ((const float4*)ws)[i];
#pragma unroll 4
        for (int k = 1; k < splitk; ++k) {
            float4 v = ((const float4*)(ws + (long)k * mn))[i];
            s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
        }
        u32 lo = (u32)f2bf(s.x) | ((u32)f2bf(s.y) << 16);
        u32 hi = (u32)f2bf(s.z) | ((u32)f2bf(s.w) << 16);
        ((uint2*)out)[i] = make_uint2(lo, hi);
    }
}

template <int D>
__global__ void __launch_bounds__(256, 2)
k_attn_prefill(bf16_t* __restrict__ out, const bf16_t* __restrict__ q,
               const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc,
               int T, int Hq, int G, int Hk, int Smax, int slot,
               int s_total, int causal_off, float scale) {
    __shared__ __attribute__((aligned(16))) bf16_t lds[prefill_lds<D>()];
    int tile, hq;
    if (!prefill_item((T + 127) / 128, Hq, &tile, &hq)) return;
    const SlotKV<D> kv{kc, vc, Hk, Smax};
    const HeadEpilogue epi{nullptr, nullptr, 0};
    attn_prefill_tile<D>(out, q, kv, T, Hq, G, hq, slot, s_total,
                            causal_off, scale, tile * 128, lds, epi, 0);
}

// ===========================================================================
// Varlen BATCHED prefill: one launch covers MANY fresh sequences.
//   meta[tile] = {q_off, len, slot, q0}: a tile is rows
//   [q0, q0+128) of the sequence packed at q_off in q/out, against KV slot
//   `slot` with s_total = len, causal_off = 0.
// Motivation: admission batches ran attention per sequence and layer from
// Python — 52k host launches, 36 ms per 32-prompt admission. One meta-driven
// launch per layer removes the loop and fills the chip (ntiles * Hq blocks).
// ===========================================================================
template <int D>
__global__ void __launch_bounds__(256, 2)
k_attn_prefill_batch(bf16_t* __restrict__ out, const bf16_t* __restrict__ q,
                     const bf16_t* __restrict__ kc,
                     const bf16_t* __restrict__ vc,
                     const int4* __restrict__ meta, int ntiles, int Hq, int G,
                     int Hk, int Smax, float scale) {
    __shared__ __attribute__((aligned(16))) bf16_t lds[prefill_lds<D>()];
    int tile, hq;
    if (!prefill_item(ntiles, Hq, &tile, &hq)) return;
    const int4 m = meta[tile];
    const SlotKV<D> kv{kc, vc, Hk, Smax};
    const HeadEpilogue epi{nullptr, nullptr, 0};
    attn_prefill_tile<D>(out + (long)m.x * Hq * D, q + (long)m.x * Hq * D,
                            kv, m.y, Hq, G, hq, m.z, m.y, /*causal_off=*/0,
                            scale, m.w, lds, epi, 0);
}

template <int MT>
static void launch_gemm_skinny(hipStream_t st, bf16_t* out, float* ws,
                               const bf16_t* x, const bf16_t* w, int M, int N,
                               int K, int splitk, int kslice) {
    dim3 grid((unsigned)((N / 64) * splitk)), blk(256);
    k_gemm_skinny<MT><<<grid, blk, 0, st>>>(out, ws, x, w, M, N, K, splitk,
                                            kslice);
}

// ===========================================================================
// Fused sampling: Gumbel-argmax token pick for the no-filter path
// (temperature + optional seed).
// RNG contract matches gridllm_amd/engine/sampler.py exactly: noise is a
// pure function of (key, candidate index) via the same splitmix64
// constants with torch's ARITHMETIC int64 shifts (emulated on unsigned),
// u = ((z>>38)&0xFFFFFF)/2^24 clamped to [1e-6, 1-1e-6], g=-log(-log u).
// key==0 marks a greedy row: no noise (sampler.py greedy_mask semantics).
// Ties pick the lowest index (torch.argmax first-max rule).
//
// A row is cut into S segments of a block each, so that few rows fill the chip
// too; their picks meet in the slot's marks, or a second kernel picks among them.
// Bound by the vector unit: the hash's second product (three of 32 bits: its upper
// half is what is used; the first one is a sum, see hash_of), beside which all that
// is done for each element of a long segment is a bound of its noise, one logarithm by
// the hardware. What a block then looks at are the batches of 8 whose largest bound is
// next to its largest, and after these whatever is not below the best of them: exactly,
// but for elements that the hardware's two logarithms put clearly behind. The picked one
// is among them. A segment of three batches a lane or less is looked at right away:
// bounds are two meetings of the block more (in a graph, us, looked at and with bounds:
// 1 row 7.2, 9.3, 20 11.1, 13.3, 34 13.7, 14.5, 40 15.3, 15.3; two kernels that look at
// all 8.3, 11.2, 13.3, 14.5). Rows of 128256, us, with two logarithms for each element,
// exact values in each step of a wave and a second kernel, and now: 64 rows 18.3, 17.8,
// 149 33.9, 26.9, 512 80.6, 57.6; called one by one, 1 row 13.3, 10.0 (the host's time).
// Masked candidates cost no logarithm: 20, 64 and 512 rows of one candidate 10.7, 15.8
// and 56 (13.8, 25.4 and 142 with exact values of all; bounds alone, behind which all of
// a masked segment was looked at, 26.6, 45 and 257). Of 64 rows' 17.8 some 10 are a
// launch, the loads of a key, the exact values and the two atomics of a block, and .3 the
// look for rows of the same slot; slots' marks in one line had 20 rows take 5 more.
// ===========================================================================
struct Pick {
    float val;
    int at;
};
DEV_INLINE bool better(float v, int i, const Pick& p) {
    return v > p.val || (v == p.val && i < p.at);
}
DEV_INLINE Pick wave_pick(Pick p) {
#pragma unroll
    for (int off = 32; off; off >>= 1) {
        const float v = __shfl_xor(p.val, off, WAVE);
        const int i = __shfl_xor(p.at, off, WAVE);
        if (better(v, i, p)) p = Pick{v, i};
    }
    return p;
}

// Keys of a step: given, or (keys null) made from a slot's seed and number of
// draws as sampler.py does.
struct SampleKeys {
    const long long* keys;
    const float* temps;            // by row, or by slot if slots is there
    const long long* slots;
    const long long* seeds;
    long long* draws;
    const long long* nongreedy;
    unsigned long long count;      // of slots
    DEV_INLINE unsigned long long key(int row) const {
        if (!slots) return (unsigned long long)keys[row];
        const long long s = slots[row];
        const unsigned long long k =
            ((unsigned long long)seeds[s] * 6364136223846793005ull +
             (unsigned long long)(draws[s] + 1) * 1442695040888963407ull) &
            0x7fffffffffffffffull;
        return k * (unsigned long long)nongreedy[s];
    }
    DEV_INLINE float temp(int row) const {
        return temps[slots ? slots[row] : row];
    }
};

// The hash's upper half of candidate i from (i ^ key) * NOISE. With the bits of i in
// two parts that is a sum of two products, one of which all of a wave's lanes have,
// and the other one all chunks of 256.
#define NOISE 0x9E3779B97F4A7C15ull
DEV_INLINE u32 hash_of(unsigned long long z) {
    z ^= (unsigned long long)((long long)z >> 29);  // arithmetic >>
    // z *= 0xBF58476D1CE4E5B9; z ^= z >> 32: their upper half
    const u32 lo = (u32)z, top = (u32)(z >> 32);
    const u32 h = __umulhi(lo, 0x1CE4E5B9u) + lo * 0xBF58476Du +
                  top * 0x1CE4E5B9u;
    return h ^ (u32)((int)h >> 31);
}
DEV_INLINE float noise_of(u32 h) {
    const float u = (float)(h >> 6 & 0xFFFFFFu) * (1.0f / 16777216.0f);
    return fminf(fmaxf(u, 1e-6f), (float)(1.0 - 1e-6));  // rounded like torch
}
// The noise and c, or more: -log(-log u) <= -log(1 - u), and 1 - u is w 2^-24 at
// least (15 for where u is clamped). c has the 24 log 2.
#define LN2 0.6931472f
DEV_INLINE float bounded(u32 h, float c) {
    const float w = fmaxf((float)(~h >> 6 & 0xFFFFFFu), 15.f);
    return fmaf(__builtin_amdgcn_logf(w), -LN2, c);
}

// The picks of a row's blocks meet in two words of its slot's cache line, which are 0
// between calls: the largest pick, as a number whose order is that of better(), and how many
// there have been. The last block stores the row's token and counts its draw. All that
// blocks tell each other goes through these atomics, a block's second one behind the
// answer to its first, so that there is nothing to release. A slot is in one call at a
// time, as its draws are.
#define MARK 16
DEV_INLINE void meet(const Pick p, int* token, unsigned long long* mark,
                     long long* draws, int blocks) {
    const u32 v = __float_as_uint(p.val + 0.f);          // (no -0)
    unsigned long long best = p.at == 2147483647 ? 0 :
        (unsigned long long)(v >> 31 ? ~v : v | 0x80000000u) << 32 | ~(u32)p.at;
    if (blocks > 1) {
        const unsigned long long was = atomicMax(mark, best);
        asm volatile("s_waitcnt vmcnt(0)" :: "v"(was) : "memory");
        if (atomicAdd(mark + 1, 1ull) != blocks - 1) return;
        best = atomicExch(mark, 0ull);
        atomicExch(mark + 1, 0ull);
    }
    *token = best ? ~(u32)best : 0;                      // all -inf -> 0
    *draws += 1;
}

// What is clearly less than x, which may be infinite.
DEV_INLINE float below(float x, float by) {
    x = fminf(x, 3e38f);
    return x - by - 1e-5f * fabsf(x);
}

// Rows that name one slot can neither meet in its mark nor count its draw before the
// others have read it: a block takes all of them, one after the other, each element by
// its exact value. Others leave them.
DEV_INLINE void sample_same(int* out, const float* logits, const SampleKeys& how,
                            int row, int rows, int v, Pick* part) {
    const long long slot = how.slots[row];
    for (int r = 0; r < row; ++r)
        if (how.slots[r] == slot) return;
    const unsigned long long key = how.key(row);
    const float t = how.temp(row);
    for (int r = row; r < rows; ++r) {
        if (how.slots[r] != slot) continue;
        Pick best{-INFINITY, 2147483647};
        for (int i = threadIdx.x; i < v; i += 256) {
            float val = logits[(long)r * v + i] / t;
            if (key != 0ull)
                val += -logf(-logf(noise_of(
                    hash_of(((unsigned long long)i ^ key) * NOISE))));
            if (better(val, i, best)) best = Pick{val, i};
        }
        best = wave_pick(best);
        if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = best;
        __syncthreads();
        if (threadIdx.x == 0) {
            for (int k = 1; k < 4; ++k)
                if (better(part[k].val, part[k].at, best)) best = part[k];
            out[r] = best.val == -INFINITY ? 0 : best.at;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0) how.draws[slot] += 1;
}

// Candidates of a lane: 4 that follow each other in each of two chunks of 256.
__global__ void __launch_bounds__(256)
k_sample_gumbel(Pick* __restrict__ ws, int* __restrict__ out,
                unsigned long long* __restrict__ marks,
                const float* __restrict__ logits, const SampleKeys how, int v,
                int segments) {
    constexpr int E = 8;
    const int row = blockIdx.x / segments, seg = blockIdx.x % segments;
    const float* x = logits + (long)row * v;
    const int per = ((v + segments - 1) / segments + 255) & ~255;
    const int i0 = seg * per, i1 = min(v, i0 + per);
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const bool wide = (v & 3) == 0;    // rows start at 16 bytes
    auto load = [&](int base, float* f) {
#pragma unroll
        for (int c = 0; c < E; c += 4) {
            const int i = base + c * 64 + lane * 4;
            if (wide && i + 4 <= i1) {
                ld4(x + i, f + c);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    f[c + e] = i + e < i1 ? x[i + e] : -INFINITY;
            }
        }
    };
    const int first = i0 + wid * 512;
    float f[E], ahead[E];
    load(first, ahead);                // (no later than the row's slot)
    const long long slot = how.slots ? how.slots[row] : 0;
    if (how.slots && (unsigned long long)slot >= how.count) __builtin_trap();
    const int rows = (int)gridDim.x / segments, r0 = min((int)threadIdx.x, rows - 1);
    const long long other = marks ? how.slots[r0] : 0;  // (looked at later)
    const unsigned long long key = how.key(row);
    const float t = how.temp(row), rt = 1.f / t;
    unsigned long long low[4];
#pragma unroll
    for (int e = 0; e < 4; ++e)
        low[e] = ((lane * 4 + e) ^ (key & 255)) * NOISE;
    auto hash = [&](int base, int e) {
        const unsigned long long chunk = base + (e >> 2) * 256;
        return hash_of((chunk ^ (key & ~255ull)) * NOISE + low[e & 3]);
    };

    // bounds of all: a lane's largest batch, and the largest of its other ones
    float most = -INFINITY, next = -INFINITY;
    int at_most = first;
    const bool fair = __builtin_amdgcn_readfirstlane(fabsf(rt) <= FLT_MAX);
    const bool bounds = fair && per > 6144;
    const float least = fair ? -FLT_MAX : -INFINITY;    // behind it masked ones alone
    for (int base = first; bounds && base < i1; base += 2048) {
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = ahead[e];
        load(base + 2048, ahead);
        float m = -INFINITY;
        if (key != 0ull) {             // (around the elements: they overlap)
#pragma unroll
            for (int e = 0; e < E; ++e)
                m = fmaxf(m, bounded(hash(base, e), fmaf(f[e], rt, 24 * LN2)));
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) m = fmaxf(m, f[e] * rt);
        }
        next = fmaxf(next, fminf(m, most));
        if (m > most) {
            most = m;
            at_most = base;
        }
    }

    bool same = marks && other == slot && r0 != row;    // another row has the slot
    if (marks)
        for (int r = threadIdx.x + 256; r < rows; r += 256)
            same |= how.slots[r] == slot && r != row;
    same = __any(same);

    // Exact values of a batch's elements, but for those that the hardware's logarithms
    // put behind the best of the wave, and for masked ones.
    Pick best{-INFINITY, 2147483647};
    auto look = [&](int base, bool mine) {
        float g[E], u[E], a[E], lim = best.val;
        auto at = [&](int e) { return base + (e >> 2) * 256 + lane * 4 + (e & 3); };
        if (bounds || base != first) load(mine ? base : i1, ahead);
#pragma unroll
        for (int e = 0; e < E; ++e) {
            g[e] = ahead[e];
            u[e] = 0.f;
            a[e] = g[e] * rt;
            if (key != 0ull) {
                u[e] = noise_of(hash(base, e));     // (lanes' batches may differ)
                // log2 by the hardware: good to 1e-3 here, below u = 0.999
                a[e] -= LN2 * __builtin_amdgcn_logf(
                    -LN2 * __builtin_amdgcn_logf(u[e]));
            }
            if (mine && u[e] <= 0.999f) lim = fmaxf(lim, a[e]);
        }
        lim = fmaxf(below(max_across16(max_of16(lim)), 0.05f), least);
        u32 left = 0;
#pragma unroll
        for (int e = 0; e < E; ++e)        // (so that NaN and +inf are)
            if (mine && at(e) < i1 && !(a[e] < lim && u[e] <= 0.999f))
                left |= 1u << e;
#pragma unroll 1
        while (__any(left != 0)) {
            const int at_e = left ? __ffs((int)left) - 1 : 0;
            float x_e = g[0], u_e = u[0];
#pragma unroll
            for (int e = 1; e < E; ++e)
                if (e == at_e) {
                    x_e = g[e];
                    u_e = u[e];
                }
            float val = x_e / t;
            if (key != 0ull) val += -logf(-logf(u_e));
            if (left && better(val, at(at_e), best)) best = Pick{val, at(at_e)};
            left &= left - 1;
        }
    };
    __shared__ float bound[4];
    __shared__ Pick part[4];
    __shared__ int twice[4];
    // first the batches next to the largest bound; the best of these says what else
    // may be it: other lanes' largest batches, and all of lanes with another large one
    bool near = true, mine = true, more = !bounds;
    bool masked = false;               // all of the segment
    int base = at_most, behind = bounds ? -1 : first + 2048;
    if (bounds) {
        float top = max_across16(max_of16(most));
        if (lane == 0) bound[wid] = top;
        __syncthreads();
        top = fmaxf(fmaxf(bound[0], bound[1]), fmaxf(bound[2], bound[3]));
        near = !(most < below(top, 0.1f));
        masked = !(top > -INFINITY);
        mine = near && !masked;
    }
    for (;;) {
        if (__any(mine)) look(base, mine);
        if (behind < 0) {
            const Pick w = wave_pick(best);
            __syncthreads();
            if (lane == 0) bound[wid] = w.val;
            __syncthreads();
            const float lim = below(
                fmaxf(fmaxf(bound[0], bound[1]), fmaxf(bound[2], bound[3])), 1e-4f);
            more = !masked && !(next < lim);
            mine = !near && !(most < lim);
            behind = first;
            continue;
        }
        if (!__any(more) || behind >= i1) break;
        mine = more;
        base = behind;
        behind += 2048;
    }
    best = wave_pick(best);
    if (lane == 0) {
        part[wid] = best;
        twice[wid] = same;
    }
    __syncthreads();
    if (twice[0] | twice[1] | twice[2] | twice[3]) {
        if (seg == 0) sample_same(out, logits, how, row, rows, v, part);
        return;
    }
    if (threadIdx.x == 0) {
        for (int k = 1; k < 4; ++k)
            if (better(part[k].val, part[k].at, best)) best = part[k];
        if (best.val == -INFINITY) best.at = 2147483647;    // (not all were looked at)
        if (marks) meet(best, out + row, marks + MARK * slot, how.draws + slot,
                        segments);
        else ws[blockIdx.x] = best;
    }
}

// One wave per row; counts the draw of the row's slot.
__global__ void __launch_bounds__(64)
k_sample_pick(int* __restrict__ out, const Pick* __restrict__ ws,
              const SampleKeys how, int segments) {
    const int row = blockIdx.x;
    Pick best{-INFINITY, 2147483647};
    for (int s = threadIdx.x; s < segments; s += 64) {
        const Pick p = ws[(long)row * segments + s];
        if (better(p.val, p.at, best)) best = p;
    }
    best = wave_pick(best);
    if (threadIdx.x) return;
    out[row] = best.at == 2147483647 ? 0 : best.at;      // all -inf -> 0
    if (how.slots) how.draws[how.slots[row]] += 1;
}

// ===========================================================================
// Host-callable entry points (extern "C", explicit stream — ctypes-bound).
// All return hipError_t as int (0 == success); callers must check.
// ===========================================================================

template <int D, class Own>
static int launch_attn_decode(hipStream_t st, bf16_t* out, const bf16_t* q,
                              const bf16_t* kc, const bf16_t* vc,
                              const int* seqlen, const int* slot_map,
                              const int4* rows, float* ws, int B, int Hk, int G,
                              int Smax, int nsplit, float scale, const Own own) {
    dim3 grid((unsigned)(B * Hk * nsplit));
    const SlotKV<D> kv{kc, vc, Hk, Smax};
    const HeadEpilogue epi{nullptr, nullptr, 0};
    switch (G) {   // compile-time G keeps softmax state in registers
#define CASE_G(GG) \
        case GG: k_attn_decode<D, GG><<<grid, dim3(256), 0, st>>>( \
                out, q, kv, seqlen, 0, slot_map, rows, ws, 1, nsplit, scale, \
                epi, AllKeys(), own); \
            break;
        CASE_G(1) CASE_G(2) CASE_G(3) CASE_G(4)
        CASE_G(5) CASE_G(6) CASE_G(7) CASE_G(8)
#undef CASE_G
        default: return -102;
    }
    LAUNCH_CHECK();
    if (nsplit > 1) {
        k_attn_combine<D><<<dim3((unsigned)(B * Hk * G)), dim3(256), 0, st>>>(
            out, ws, Hk * G, nsplit, epi);
        LAUNCH_CHECK();
    }
    return 0;
}

extern "C" {

int gl_rmsnorm(void* stream, void* y, const void* x, const void* w,
               const void* res_in, void* res_out, long n, int h, float eps) {
    if (h % 8 != 0 || (res_in && !res_out)) return -100;
#define GO(NV, THREADS) k_rmsnorm<NV, THREADS> \
        <<<dim3((unsigned)n), dim3(THREADS), 0, (hipStream_t)stream>>>( \
        (bf16_t*)y, (const bf16_t*)x, (const bf16_t*)w, \
        (const bf16_t*)res_in, (bf16_t*)res_out, h, eps)
    if (h <= 2048) GO(1, 256);
    else if (h <= 4096) GO(1, 512);
    else if (h <= 8192) GO(2, 512);
    else GO(0, 256);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gl_rmsnorm_parts(void* stream, void* y, const void* ws, int parts,
                     const void* w, const void* res_in, void* res_out, int n,
                     int h, float eps) {
    if (h % 8 || n < 1 || parts < 1 || !res_in || !res_out) return -100;
#define GO(NV, THREADS) k_rmsnorm_parts<NV, THREADS> \
        <<<dim3((unsigned)n), dim3(THREADS), 0, (hipStream_t)stream>>>( \
        (bf16_t*)y, (const float*)ws, parts, (const bf16_t*)w, \
        (const bf16_t*)res_in, (bf16_t*)res_out, h, eps)
    if (h <= 2048) GO(1, 256);
    else if (h <= 4096) GO(1, 512);
    else if (h <= 8192) GO(2, 512);
    else GO(0, 256);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

// What a decode step starts with. Per batch row: position, place in the cache,
// rotary position and number of keys of its slot. slots: of seq_lens and
// rope_off. slot_t, pos_rope, attn_seq and rope_off may be null.
// rows (nullable): see k_decode_positions
int gl_decode_start(void* stream, void* pos, void* slot_t, void* pos_rope,
                    void* attn_seq, void* rows, const void* seq_lens,
                    const void* rope_off, const void* slot_map, int B, int slots,
                    int Smax) {
    if (slots < 1 || (pos_rope && !rope_off) ||
        (rows && (B > ROWS_ORDERED || (unsigned long)rows % 16))) return -100;
    if (B < 1) return 0;
    k_decode_positions<<<dim3((B + 63) / 64), dim3(256), 0,
                         (hipStream_t)stream>>>(
        (int*)pos, (int*)slot_t, (int*)pos_rope, (int*)attn_seq, (int4*)rows,
        (const int*)seq_lens, (const int*)rope_off, (const int*)slot_map, B,
        slots, Smax);
    LAUNCH_CHECK();
    return 0;
}

// What it ends with: the rows' slots are one longer (rows may share a slot).
int gl_advance_lengths(void* stream, void* seq_lens, const void* slot_map,
                       int B, int slots) {
    if (slots < 1) return -100;
    if (B < 1) return 0;
    k_advance_lengths<<<dim3((B + 255) / 256), dim3(256), 0,
                        (hipStream_t)stream>>>(
        (int*)seq_lens, (const int*)slot_map, B, slots);
    LAUNCH_CHECK();
    return 0;
}

int gl_prompt_positions(void* stream, void* pos, void* slot_t, int slot,
                        int start, int T, int Smax) {
    if (T < 1 || slot < 0 || start < 0) return -100;
    k_prompt_positions<<<dim3((T + 255) / 256), dim3(256), 0,
                         (hipStream_t)stream>>>(
        (int*)pos, (int*)slot_t, slot, start, T, Smax);
    LAUNCH_CHECK();
    return 0;
}

int gl_prompt_end(void* stream, void* seq_lens, void* rope_off, int slot,
                  int start, int T) {
    if (slot < 0 || start < 0) return -100;
    k_prompt_end<<<dim3(1), dim3(1), 0, (hipStream_t)stream>>>(
        (int*)seq_lens, (int*)rope_off, slot, start, T);
    LAUNCH_CHECK();
    return 0;
}

int gl_prompts_end(void* stream, void* seq_lens, void* rope_off,
                   const void* of_slots, const void* lens, int B, int slots,
                   void* out, const void* x, const void* lasts, int rows, int H) {
    if (B < 1 || slots < 1 || (out && (H < 8 || H % 8 || rows < 1 || !x ||
                                       !lasts))) return -100;
    k_prompts_end<<<dim3((unsigned)B), dim3(256), 0, (hipStream_t)stream>>>(
        (int*)seq_lens, (int*)rope_off, (const int*)of_slots, (const int*)lens,
        slots, (uint4*)out, (const uint4*)x, (const int*)lasts, rows, H / 8);
    LAUNCH_CHECK();
    return 0;
}

int gl_embed_norm(void* stream, void* x, void* y, const void* emb,
                  const void* tokens, const void* w, long n, int h, int vocab,
                  float eps) {
    if (h % 8 != 0 || vocab < 1) return -100;
    if (n < 1) return 0;
#define GO(NV, THREADS) k_embed_norm<NV, THREADS> \
        <<<dim3((unsigned)n), dim3(THREADS), 0, (hipStream_t)stream>>>( \
        (bf16_t*)x, (bf16_t*)y, (const bf16_t*)emb, \
        (const long long*)tokens, (const bf16_t*)w, h, vocab, eps)
    if (h <= 2048) GO(1, 256);
    else if (h <= 4096) GO(1, 512);
    else if (h <= 8192) GO(2, 512);
    else GO(0, 256);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gl_rope(void* stream, void* q, void* k, const void* cost, const void* sint,
            const void* pos, int T, int Hq, int Hk, int D) {
    if (D % 4 != 0) return -100;
    long total = (long)T * (Hq + Hk) * (D / 4);
    int grid = (int)min((total + 255) / 256, (long)2048);
    if (grid == 0) return 0;
    k_rope<<<dim3(grid), dim3(256), 0, (hipStream_t)stream>>>(
        (bf16_t*)q, (bf16_t*)k, (const float*)cost, (const float*)sint,
        (const int*)pos, T, Hq, Hk, D);
    LAUNCH_CHECK();
    return 0;
}

int gl_swiglu(void* stream, void* out, const void* gateup, long n, int f,
              float alpha, float limit, float shift, float cubic) {
    if (f % 8 != 0) return -100;
    long total = n * (f / 8);
    int grid = (int)min((total + 255) / 256, (long)2048);
    if (grid == 0) return 0;
    k_swiglu<<<dim3(grid), dim3(256), 0, (hipStream_t)stream>>>(
        (bf16_t*)out, (const bf16_t*)gateup, n, f,
        GluParams{alpha, limit, shift, cubic});
    LAUNCH_CHECK();
    return 0;
}

int gl_kv_append(void* stream, void* kc, void* vc, const void* kn,
                 const void* vn, const void* slot, int n, int hk, int d,
                 int smax) {
    if (d % 2 != 0 || n == 0) return (d % 2) ? -100 : 0;
    k_kv_append<<<dim3(n * hk), dim3(64), 0, (hipStream_t)stream>>>(
        (bf16_t*)kc, (bf16_t*)vc, (const bf16_t*)kn, (const bf16_t*)vn,
        (const int*)slot, hk, d, smax);
    LAUNCH_CHECK();
    return 0;
}

// parts > 0: qkv is f32 sums [parts, N, (Hq + 2 Hk) D] (D % 16 == 0, all at 16
// bytes).
int gl_rope_kv(void* stream, const void* qkv, int parts, void* q_out, void* kc,
               void* vc, const void* cost, const void* sint, const void* pos,
               const void* slot, const void* bias, int N, int Hq, int Hk, int D,
               int Smax) {
    if (D % 4 != 0 || N == 0) return (D % 4) ? -100 : 0;
    const unsigned long ptrs = (unsigned long)qkv | (unsigned long)q_out |
        (unsigned long)kc | (unsigned long)vc | (unsigned long)cost |
        (unsigned long)sint | (unsigned long)bias;
    if (D % 16 == 0 && ptrs % 16 == 0) {
        const long heads = Hq + 2 * Hk, items = N * heads * (D / 16);
        const SummedRow sums{(const float*)qkv, N * heads * D, parts};
#define GO(rows) k_rope_kv8<<<dim3((unsigned)((items + 255) / 256)), \
            dim3(256), 0, (hipStream_t)stream>>>( \
            rows, (bf16_t*)q_out, (bf16_t*)kc, (bf16_t*)vc, \
            (const float*)cost, (const float*)sint, (const int*)pos, \
            (const int*)slot, (const bf16_t*)bias, N, Hq, Hk, D, Smax)
        if (parts > 0) GO(sums);
        else GO(StoredRow{(const bf16_t*)qkv});
#undef GO
        LAUNCH_CHECK();
        return 0;
    }
    if (parts > 0) return -100;
    k_rope_kv<<<dim3((unsigned)(N * (Hq + Hk))), dim3(64), 0,
                (hipStream_t)stream>>>(
        (const bf16_t*)qkv, (bf16_t*)q_out, (bf16_t*)kc, (bf16_t*)vc,
        (const float*)cost, (const float*)sint, (const int*)pos,
        (const int*)slot, (const bf16_t*)bias, Hq, Hk, D, Smax);
    LAUNCH_CHECK();
    return 0;
}

int gl_attn_decode(void* stream, void* out, const void* q, const void* kc,
                   const void* vc, const void* seqlen, const void* slot_map,
                   const void* rows, void* ws, int B, int Hq,
                   int Hk, int D, int Smax, int nsplit, float scale) {
    if ((unsigned long)rows % 16 || Hq < 1 || Hk < 1 || Hq % Hk != 0 ||
        Hq / Hk > MAXG || nsplit < 1 || nsplit > MAX_SPLIT || (nsplit > 1 && !ws))
        return -100;
    const int G = Hq / Hk;
    hipStream_t st = (hipStream_t)stream;
#define GO(DD) return launch_attn_decode<DD>( \
        st, (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kc, (const bf16_t*)vc, \
        (const int*)seqlen, (const int*)slot_map, (const int4*)rows, (float*)ws, B, \
        Hk, G, Smax, nsplit, scale, StoredQueries())
    if (D == 128) GO(128);
    if (D == 64) GO(64);
#undef GO
    return -101;
}

// The same of rows of a product [B][(Hq + 2 Hk) D], or its f32 sums in parts (> 0): q and
// k are turned by cost and sint at pos (rows' own, if there are rows), k and v written
// to the cache as key seqlen - 1.
int gl_rope_attn_decode(void* stream, void* out, const void* qkv, int parts,
                        void* kc, void* vc, const void* cost, const void* sint,
                        const void* pos, const void* bias, const void* seqlen,
                        const void* slot_map, const void* rows, void* ws, int B,
                        int Hq, int Hk, int D, int Smax, int nsplit, float scale) {
    const unsigned long ptrs = (unsigned long)qkv | (unsigned long)kc |
        (unsigned long)vc | (unsigned long)cost | (unsigned long)sint |
        (unsigned long)bias | (unsigned long)rows;
    if (ptrs % 16 || B < 1 || Hq < 1 || Hk < 1 || Hq % Hk != 0 || Hq / Hk > MAXG ||
        nsplit < 1 || nsplit > MAX_SPLIT || (nsplit > 1 && !ws) || parts < 0)
        return -100;
    const int G = Hq / Hk;
    const int heads = Hq + 2 * Hk;
#define GO(DD, Row, ...) return launch_attn_decode<DD>( \
        (hipStream_t)stream, (bf16_t*)out, (const bf16_t*)nullptr, \
        (const bf16_t*)kc, (const bf16_t*)vc, (const int*)seqlen, \
        (const int*)slot_map, (const int4*)rows, (float*)ws, B, Hk, G, Smax, nsplit, \
        scale, TurnedHeads<DD, Row>{__VA_ARGS__, (const float*)cost, \
        (const float*)sint, (const int*)pos, (const bf16_t*)bias, heads})
#define PICK(DD) do { \
        if (parts) GO(DD, SummedRow, SummedRow{(const float*)qkv, \
                                               (long)B * heads * DD, parts}); \
        else GO(DD, StoredRow, StoredRow{(const bf16_t*)qkv}); } while (0)
    if (D == 128) PICK(128);
    if (D == 64) PICK(64);
#undef PICK
#undef GO
    return -101;
}

int gl_gemm_skinny(void* stream, void* out, void* ws, const void* x,
                   const void* w, int M, int N, int K, int splitk,
                   int kslice) {
    if (N % 64 != 0 || K % 32 != 0 || kslice % 32 != 0) return -100;
    hipStream_t st = (hipStream_t)stream;
    const int mt = (M + 15) / 16;
#define CASE_MT(T) else if (mt <= T) launch_gemm_skinny<T>( \
        st, (bf16_t*)out, (float*)ws, (const bf16_t*)x, (const bf16_t*)w, \
        M, N, K, splitk, kslice)
    if (false) {}
    CASE_MT(1); CASE_MT(2); CASE_MT(3); CASE_MT(4); CASE_MT(6); CASE_MT(8);
    CASE_MT(12); CASE_MT(16);
    else return -103;
#undef CASE_MT
    LAUNCH_CHECK();
    if (splitk > 1) {
        long mn = (long)M * N;
        long chunks = (mn + 3) / 4;
        int grid = (int)min((chunks + 255) / 256, (long)2048);
        k_gemm_combine<<<dim3(grid), dim3(256), 0, st>>>(
            (bf16_t*)out, (const float*)ws, mn, splitk);
        LAUNCH_CHECK();
    }
    return 0;
}

int gl_gemm_rows(void* stream, void* out, const void* x, const void* w, int M,
                 int N, int K, int fuse_glu, float alpha, float limit,
                 float shift, float cubic) {
    if (M < 1 || M > 16 || K < 32 || K % 32 || N % (fuse_glu ? 128 : 16))
        return -100;
    const GluParams glu{alpha, limit, shift, cubic};
    hipStream_t st = (hipStream_t)stream;
    if (fuse_glu)
        k_gemm_rows<1><<<dim3((unsigned)(N / 32)), dim3(512), 0, st>>>(
            (bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, M, N, K, glu);
    else
        k_gemm_rows<0><<<dim3((unsigned)(N / 16)), dim3(512), 0, st>>>(
            (bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, M, N, K, glu);
    LAUNCH_CHECK();
    return 0;
}

int gl_gemm_tile(void* stream, void* out, void* ws, const void* x,
                 const void* w, int M, int N, int K, int splitk, int kslice,
                 int rows, int cols, int fuse_swiglu, float alpha,
                 float limit, float shift, float cubic) {
    const GluParams glu{alpha, limit, shift, cubic};
    if (M < 1 || K < 1 || K % 64 || kslice < 64 || kslice % 64 || N < 1 ||
        cols < 1 || N % cols || (fuse_swiglu && N % 128) || splitk < 1 ||
        (long)(splitk - 1) * kslice >= K || (long)splitk * kslice < K ||
        (splitk > 1 && !ws) || (!out && (!ws || fuse_swiglu))) return -100;
    const BatchArgs p{(bf16_t*)out, (float*)ws, (const bf16_t*)x,
                      (const bf16_t*)w, M, N, K, splitk, kslice, 0, glu};
    hipStream_t st = (hipStream_t)stream;
    int e = -103;
#define GO(RT, CT, EPI) \
    if (rows == RT * 16 && cols == CT * 16 && !fuse_swiglu == !EPI) \
        e = launch_gemm_tile<RT, CT, EPI>(st, p)
#define COLS(RT) GO(RT, 4, 0); GO(RT, 6, 0); GO(RT, 8, 0); GO(RT, 4, 1); \
    GO(RT, 8, 1)
    GO(6, 3, 0); GO(8, 3, 0); GO(10, 3, 0); GO(12, 3, 0); GO(16, 3, 0);
    GO(2, 16, 0); GO(4, 16, 0); GO(6, 16, 0); GO(8, 16, 0); GO(10, 16, 0);
    COLS(2); COLS(4); COLS(6); COLS(8); COLS(10); COLS(12); COLS(16);
#undef COLS
#undef GO
    if (e || splitk == 1 || !out) return e;    // (no out: ws is wanted)
    const long quads = (long)M * (fuse_swiglu ? N >> 3 : N >> 2);
    const int grid = (int)min((quads + 255) / 256, (long)2048);
    if (fuse_swiglu)
        k_gemm_combine_swiglu<<<dim3(grid), dim3(256), 0, st>>>(
            (bf16_t*)out, (const float*)ws, M, N, splitk, glu);
    else
        k_gemm_combine<<<dim3(grid), dim3(256), 0, st>>>(
            (bf16_t*)out, (const float*)ws, (long)M * N, splitk);
    LAUNCH_CHECK();
    return 0;
}

int gl_gemm_tile_once(int M, int N, int K, int rows, int kslice) {
    return rows < 1 ? -100 : tile_once(M, N, K, rows, kslice);
}

// shape: one of kWide; full: of its tiles, the others are halved (shape 0). epi: as
// in gridllm_wide.h.
int gl_gemm_wide(void* stream, void* out, const void* x, const void* w, int M,
                 int N, int K, int shape, int full, int epi, float alpha,
                 float limit, float shift, float cubic) {
    const unsigned long ptrs = (unsigned long)out | (unsigned long)x |
        (unsigned long)w;
    if (epi < 0 || epi > 2 || full < 0 || ptrs % 16 ||
        !wide_fits(M, N, K, epi, shape)) return -100;
    const WideArgs p{out, (const bf16_t*)x, (const bf16_t*)w, M, N, K,
                     GluParams{alpha, limit, shift, cubic}};
    hipStream_t st = (hipStream_t)stream;
    typedef WideShape<6, 4, 2> Wide192;
    switch (shape * 3 + epi) {
        case 0: return launch_gemm_wide<Wide256, WideHalf, 0>(st, p, full);
        case 1: return launch_gemm_wide<Wide256, WideHalf, 1>(st, p, full);
        case 2: return launch_gemm_wide<Wide256, WideHalf, 2>(st, p, full);
        case 3: return launch_gemm_wide<WideShape<6, 3, 3>, NoShape, 0>(
                st, p, full);
        case 6: return launch_gemm_wide<WideShape<8, 3, 2>, NoShape, 0>(
                st, p, full);
        case 9: return launch_gemm_wide<WideShape<6, 2, 4>, NoShape, 0>(
                st, p, full);
        case 13: return launch_gemm_wide<Wide192, NoShape, 1>(st, p, full);
        case 14: return launch_gemm_wide<Wide192, NoShape, 2>(st, p, full);
    }
    return -103;
}

// What to run a product of more than 256 rows by: plan[0] 0 the library, 1
// gl_gemm_tile by rows plan[1], columns plan[2], parts plan[3], 2 gl_gemm_wide by
// shape plan[1] and full plan[2]. The times are those of wide_best and of _tile_us
// in hip_ops.py, which holds up to 1200 rows too. Over 2712 random sizes of the models
// here, of 257 to 8192 rows and more than 21 us, what is picked takes .973 of the
// library's time in the mean; what is run here, in the mean and at most: tiles .90 and
// 1.24 of it, 256 x 256 .95, 1.12, 192 x 192 .93, 1.29, 256 x 192 .91, 1.05, 192 x 128
// .97, 1.51.
//   Gated units are always done here: the library's needs another pass (16384 x 3072,
//   272 rows 48 -> 38 us by tiles; 2731 338 -> 220).
//   K from 4096 on with up to 1200 rows: tiles with K in parts (300 x 2048 x 8192 34 ->
//   25, 512 x 3072 x 12288 74 -> 47, 1200 x 3072 x 8192 75 -> 65). Shorter K: tiles
//   where they are one round of CUs, three quarters of it or more (300 x 12288 x 3072
//   43 -> 33, 800 x 3072 x 3072 30 -> 26, 1024 x 5120 x 3072 42 -> 40; two rounds, 640
//   x 12288 x 3072, take 63 us, the library 54; 160 tiles, 1200 x 4096 x 3072, 45, 40).
//   21 us and less: what a call to the library costs the host, and twice what one
//   here does (four layers of 0.5b, 260 tokens, are bound by that).
//   Longer ones go here where a shape's tiles fill their last round of CUs as the
// library's do not: 256 x 256 one that is .6 full at most, as its halves fill one (rows
// of more than 4096 with one or two rounds before, and that one .37 to .5 full: outside
// of that 1.0 to 1.1 of the library's time in the mean); 192 x 192 none or .8 of one
// behind full rounds, .85 alone; 256 x 192 .6 behind two or more; 192 x 128 .85 alone,
// .75 behind two, none behind one or three (.75 and more behind one or three: 1.07 to
// 1.28).
//   whole: not in parts of K, and gated units by k_gemm_wide, whose sums and roundings
// are the library's but where that cuts K itself (more than 99.9 % of results are the
// same to the bit). Where a model makes much of a rounding (a sequence's first token
// has one key, and a head's norm behind it leaves the sign of q . k alone), single
// values then hardly depend on what runs them; against 64 bits both are alike.
//   epi: as of gl_gemm_wide, which has not each shape for each. Scores in f32 (2) go
// as a plain product does if its shape has them (0), else by the library and a pass
// to f32: by shape 4 350 x 32000 x 2048 takes 58 us, 62 by the library, but 300 x
// 32064 x 3072 81, 79, and 513 x 32000 x 4096 178, 156.
int gl_gemm_plan(int M, int N, int K, int epi, int whole, int* plan) {
    plan[0] = plan[1] = plan[2] = plan[3] = 0;
    if (epi < 0 || epi > 2) return -100;
    const bool fuse_glu = epi == 1;
    int shape = 0, full = 0, way = 0;
    bool fills = false;                        // blocks of tiles: one round of CUs
    float best = wide_best(M, N, K, fuse_glu ? 1 : 0, &shape, &full);
    if (best < INFINITY) {
        way = 2;
        plan[1] = shape;
        plan[2] = full;
    }
    const int heights[] = {96, 128, 160, 192, 256};
    const int widths[] = {64, 96, 128};
    if (!whole && M > 0 && M <= 1200 && N > 0 && K > 0 && K % 64 == 0 &&
        !(fuse_glu && N % 128)) {
        for (int rows : heights) for (int cols : widths) {
            if (N % cols || (fuse_glu && cols == 96)) continue;
            const long tiles = (long)((M + rows - 1) / rows) * (N / cols);
            if (tiles > 512) continue;
            const int most = max(1, min((int)(256 / tiles), K / 384));
            for (int parts : {1, (most + 1) / 2, most}) {
                const int slice = ((K + parts - 1) / parts + 63) / 64 * 64;
                const int n = (K + slice - 1) / slice;
                const float area = (float)rows * cols;
                float us = 3.9f + (tiles * n + 255) / 256 *
                    (3.f + slice * (rows * 1.42e-5f + cols * 3.2e-5f +
                                    area * 1.09e-7f) +
                     (fuse_glu ? area * 5.8e-5f : 0.f));
                if (n > 1) us += (float)n * M * N * 2.4e-6f;
                if (us >= best) continue;
                best = us;
                way = 1;
                fills = tiles * n >= 192 && tiles * n <= 256;
                plan[1] = rows;
                plan[2] = cols;
                plan[3] = n;
            }
        }
    }
    bool here = fuse_glu || best <= 21.f || (way == 1 && (K >= 4096 || fills));
    if (way == 2) {
        const WideTimes& t = kWide[plan[1]];
        const long tiles = (long)((M + t.rows - 1) / t.rows) *
                           ((N + t.cols - 1) / t.cols);
        const long some = tiles % 256, rounds = tiles / 256;   // full ones
        if (plan[1] == 0)
            here |= rounds > 0 && some > 0 &&
                    (K <= 4096 ? some <= 154
                               : rounds < 3 && some >= 96 && some <= 128);
        else if (plan[1] == 1)
            here |= rounds > 0 ? some == 0 || some >= 204 : some >= 218;
        else if (plan[1] == 2)
            here |= rounds > 1 && some >= 160;
        else
            here |= rounds % 2 ? rounds < 4 && some == 0
                    : rounds == 0 ? some >= 218 : rounds == 2 && some >= 192;
        if (epi == 2 && plan[1] != 0) here = false;
    }
    plan[0] = here ? way : 0;
    return 0;
}

// keys [b] and temps [b]; or, with slots [b], temps, seeds, draws and nongreedy
// by slot (`count` of them), of which draws are advanced. ws: 8 bytes per row and
// segment.
int gl_sample_gumbel(void* stream, void* out, void* ws, const void* logits,
                     const void* keys, const void* temps, const void* slots,
                     const void* seeds, void* draws, const void* nongreedy,
                     int b, int v, int segments, int count) {
    if (segments < 1 || (slots ? count < 1 || !seeds || !draws || !nongreedy
                               : !keys)) return -100;
    if (b <= 0) return 0;
    const SampleKeys how{(const long long*)keys, (const float*)temps,
                         (const long long*)slots, (const long long*)seeds,
                         (long long*)draws, (const long long*)nongreedy,
                         (unsigned long long)count};
    hipStream_t st = (hipStream_t)stream;
    k_sample_gumbel<<<dim3((unsigned)(b * segments)), dim3(256), 0, st>>>(
        (Pick*)ws, nullptr, nullptr, (const float*)logits, how, v, segments);
    LAUNCH_CHECK();
    k_sample_pick<<<dim3((unsigned)b), dim3(64), 0, st>>>(
        (int*)out, (const Pick*)ws, how, segments);
    LAUNCH_CHECK();
    return 0;
}

// By slot, in one launch: marks 128 bytes per slot, 0 (and left so).
int gl_sample_slots(void* stream, void* out, const void* logits,
                    const void* temps, const void* slots, const void* seeds,
                    void* draws, const void* nongreedy, void* marks, int b, int v,
                    int segments, int count) {
    if (segments < 1 || count < 1 || v < 1 || !slots || !seeds || !draws ||
        !nongreedy || !marks) return -100;
    if (b <= 0) return 0;
    const SampleKeys how{nullptr, (const float*)temps, (const long long*)slots,
                         (const long long*)seeds, (long long*)draws,
                         (const long long*)nongreedy, (unsigned long long)count};
    k_sample_gumbel<<<dim3((unsigned)(b * segments)), dim3(256), 0,
                      (hipStream_t)stream>>>(
        nullptr, (int*)out, (unsigned long long*)marks, (const float*)logits, how, v,
        segments);
    LAUNCH_CHECK();
    return 0;
}

int gl_swiglu_il(void* stream, void* out, const void* gu, long n, int f,
                 float alpha, float limit, float shift, float cubic) {
    if (f % 64 != 0) return -100;
    hipStream_t st = (hipStream_t)stream;
    long total = n * (f >> 3);
    int grid = (int)min((total + 255) / 256, (long)4096);
    k_swiglu_il<<<dim3(grid), dim3(256), 0, st>>>(
        (bf16_t*)out, (const bf16_t*)gu, n, f,
        GluParams{alpha, limit, shift, cubic});
    LAUNCH_CHECK();
    return 0;
}

// The tile and head of a prefill block: place[0], place[1] (1 if it has none).
int gl_prefill_place(int block, int ntiles, int Hq, int* place) {
    return !prefill_place(block, ntiles, Hq, place, place + 1);
}

int gl_attn_prefill(void* stream, void* out, const void* q, const void* kc,
                    const void* vc, int T, int Hq, int Hk, int D, int Smax,
                    int slot, int s_total, int causal_off, float scale) {
    hipStream_t st = (hipStream_t)stream;
    if (Hq % Hk) return -110;
    const int G = Hq / Hk;
    if (T < 1) return -100;
    dim3 grid(prefill_grid((T + 127) / 128, Hq)), blk(256);
    if (D == 128)
        k_attn_prefill<128><<<grid, blk, 0, st>>>(
            (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kc,
            (const bf16_t*)vc, T, Hq, G, Hk, Smax, slot, s_total,
            causal_off, scale);
    else if (D == 64)
        k_attn_prefill<64><<<grid, blk, 0, st>>>(
            (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kc,
            (const bf16_t*)vc, T, Hq, G, Hk, Smax, slot, s_total,
            causal_off, scale);
    else
        return -111;
    LAUNCH_CHECK();
    return 0;
}

int gl_attn_prefill_batch(void* stream, void* out, const void* q,
                          const void* kc, const void* vc, const void* meta,
                          int ntiles, int Hq, int Hk, int D, int Smax,
                          float scale) {
    hipStream_t st = (hipStream_t)stream;
    if (Hq % Hk) return -110;
    const int G = Hq / Hk;
    if (ntiles < 1) return -100;
    dim3 grid(prefill_grid(ntiles, Hq)), blk(256);
    if (D == 128)
        k_attn_prefill_batch<128><<<grid, blk, 0, st>>>(
            (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kc,
            (const bf16_t*)vc, (const int4*)meta, ntiles, Hq, G, Hk, Smax,
            scale);
    else if (D == 64)
        k_attn_prefill_batch<64><<<grid, blk, 0, st>>>(
            (bf16_t*)out, (const bf16_t*)q, (const bf16_t*)kc,
            (const bf16_t*)vc, (const int4*)meta, ntiles, Hq, G, Hk, Smax,
            scale);
    else
        return -111;
    LAUNCH_CHECK();
    return 0;
}

// A prompt's layer (Llama family): its launches one behind the other, 4 us of the
// host each, where calls from Python take 7 to 13 with their tensors and checks
// (four layers of llama3.2:1b, 45 tokens, were bound by that).
struct LayerProduct {
    long long kind, a, b, c;       // 0 k_gemm_rows; 1 k_gemm_tile: rows, columns, parts;
};                                 // 2 k_gemm_wide: shape, whole tiles
struct PromptLayer {
    // normed rows and residuals [T, H] in and out, and behind the attention
    void *normed, *resid, *mid_normed, *mid_resid;
    void *qkv, *q, *attn, *act, *y, *ws;       // working space; ws: f32 parts
    const void *wqkv, *bqkv, *wo, *wgateup, *wdown, *mlp_norm, *next_norm;
    void *kc, *vc;
    const void *cost, *sint, *pos, *places, *meta;     // meta: of several prompts
    long long T, H, Hq, Hk, D, F, Smax, slot, start, tiles;
    LayerProduct p_qkv, p_o, p_gateup, p_down;
};

static int layer_product(void* st, const LayerProduct& p, void* out, void* ws,
                         const void* x, const void* w, int M, int N, int K,
                         int glu) {
    const GluParams u{1.f, INFINITY, 0.f, 0.f};
    if (p.kind == 0)
        return gl_gemm_rows(st, out, x, w, M, N, K, glu, u.alpha, u.limit,
                            u.shift, u.cubic);
    if (p.kind == 1) {
        if (p.c < 1) return -100;
        const int slice = ((K + (int)p.c - 1) / (int)p.c + 63) / 64 * 64;
        return gl_gemm_tile(st, out, ws, x, w, M, N, K, (K + slice - 1) / slice,
                            slice, (int)p.a, (int)p.b, glu, u.alpha, u.limit,
                            u.shift, u.cubic);
    }
    return gl_gemm_wide(st, out, x, w, M, N, K, (int)p.a, (int)p.b, glu, u.alpha,
                        u.limit, u.shift, u.cubic);
}

// A product's parts of K that what follows adds up; 0: none, or one.
static int layer_parts(const LayerProduct& p, int K) {
    if (p.kind != 1 || p.c < 2 || K <= 64) return 0;
    const int slice = ((K + (int)p.c - 1) / (int)p.c + 63) / 64 * 64;
    return (K + slice - 1) / slice;
}

// (rmsnorm(y) * weight, y) of y = x w^T + resid
static int layer_joined(void* st, const LayerProduct& p, const PromptLayer& l,
                        const void* x, const void* w, int K, const void* weight,
                        const void* resid, void* normed, void* sum, float eps) {
    const int T = (int)l.T, H = (int)l.H;
    const int parts = H % 8 ? 0 : layer_parts(p, K);
    const int e = layer_product(st, p, parts ? nullptr : l.y, l.ws, x, w, T, H, K,
                                0);
    if (e) return e;
    if (!parts)
        return gl_rmsnorm(st, normed, l.y, weight, resid, sum, T, H, eps);
    return gl_rmsnorm_parts(st, normed, l.ws, parts, weight, resid, sum, T, H,
                            eps);
}

int gl_prompt_layer(void* st, const void* layer, float scale, float eps) {
    const PromptLayer& l = *(const PromptLayer*)layer;
    const int T = (int)l.T, H = (int)l.H, Hq = (int)l.Hq, Hk = (int)l.Hk;
    const int D = (int)l.D, Smax = (int)l.Smax;
    const int parts = layer_parts(l.p_qkv, H);
    int e = layer_product(st, l.p_qkv, parts ? nullptr : l.qkv, l.ws, l.normed,
                          l.wqkv, T, (Hq + 2 * Hk) * D, H, 0);
    if (!e) e = gl_rope_kv(st, parts ? l.ws : l.qkv, parts, l.q, l.kc, l.vc,
                           l.cost, l.sint, l.pos, l.places, l.bqkv, T, Hq, Hk, D,
                           Smax);
    if (!e) e = l.meta
        ? gl_attn_prefill_batch(st, l.attn, l.q, l.kc, l.vc, l.meta,
                                (int)l.tiles, Hq, Hk, D, Smax, scale)
        : gl_attn_prefill(st, l.attn, l.q, l.kc, l.vc, T, Hq, Hk, D, Smax,
                          (int)l.slot, (int)l.start + T, (int)l.start, scale);
    if (!e) e = layer_joined(st, l.p_o, l, l.attn, l.wo, Hq * D, l.mlp_norm,
                             l.resid, l.mid_normed, l.mid_resid, eps);
    if (!e) e = layer_product(st, l.p_gateup, l.act, l.ws, l.mid_normed,
                              l.wgateup, T, 2 * (int)l.F, H, 1);
    if (!e) e = layer_joined(st, l.p_down, l, l.act, l.wdown, (int)l.F,
                             l.next_norm, l.mid_resid, l.normed, l.resid, eps);
    return e;
}

int gl_device_sync() { return (int)hipDeviceSynchronize(); }

}  // extern "C"
