// gfx950 kernels of the layer-list models: a decoder whose layers each name a
// mixer (grouped softmax attention over a paged cache, latent or talking-heads
// attention, mLSTM, gated linear or lightning attention with a matrix memory
// per sequence, or two of these side by side) and a feed-forward (dense gated,
// dense with PolyNorm, or routed experts, with a shared one beside them).
// Latent attention is in gridllm_latent.hip, talking heads in gridllm_talk.hip.
//
// Conventions
//  * T is the element type of activations, weights and the KV cache: bf16, or
//    f32 for the exact mode. The residual stream, norms, scores, gates, router
//    logits and recurrent state are f32 in both.
//  * Widths and head sizes are padded by the host to multiples of 64 with zero
//    weights, so rows are 16-byte aligned and padding stays zero; the true
//    sizes enter only where a mean is taken.
//  * The tokens of a step are ordered decode rows first (one token of a
//    sequence each), then the prompt portions, each a contiguous segment.
//
// Exported extern "C" with an explicit stream; nothing here allocates.

#include "gridllm_attention.h"
#include "gridllm_tiles.h"
#include "gridllm_wide.h"

// ===========================================================================
// x = embed[token], f32, plus pos_table[position] if there is one, then its
// norm if there are norm weights; xb = the same in T
// ===========================================================================
template <class T>
__global__ void __launch_bounds__(256)
k_embed(float* __restrict__ x, T* __restrict__ xb,
        const T* __restrict__ emb, const T* __restrict__ ptab,
        const long long* __restrict__ tok, const int* __restrict__ pos,
        const float* __restrict__ w, float w_off, int W, int Wtrue, float eps,
        int vocab, int max_pos) {
    __shared__ float red[4];
    const long n = blockIdx.x;
    const long t = min(max(tok[n], 0ll), (long long)vocab - 1);
    const long p = ptab ? min(max(pos[n], 0), max_pos - 1) : 0;
    auto row = [&](int c, float* a) {
        ld8(emb + t * W + c, a);
        if (!ptab) return;
        float b[8];
        ld8(ptab + p * W + c, b);
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] += b[i];
    };
    float rs = 1.f;
    if (w) {
        float ss = 0.f;
        for (int c = threadIdx.x * 8; c < W; c += 2048) {
            float a[8];
            row(c, a);
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += a[i] * a[i];
        }
        rs = 1.f / sqrtf(block_sum(ss, red) / (float)Wtrue + eps);
    }
    for (int c = threadIdx.x * 8; c < W; c += 2048) {
        float a[8];
        row(c, a);
        if (w) {
            float g[8];
            ld8(w + c, g);
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] *= rs * (w_off + g[i]);
        }
        st8(x + n * W + c, a);
        if (xb) st8(xb + n * W + c, a);
    }
}

// ===========================================================================
// Norm of a sublayer's output, added to the residual:
//   x += y * (1 / sqrt(mean(y^2) + eps)) * (w_off + w);  xb = T(x)
// TOP > 0 (routed experts): y is sum_k wt[n, k] * ye[n * top + k].
// W <= 8192 (a row is kept in registers); the mean is over Wtrue elements.
// ===========================================================================
// 8 columns of a sublayer's output. A pair of weight zero has no row (its
// expert is an identity).
template <class T, bool MOE>
DEV_INLINE void sublayer8(const T* y, const float* wt, int top, long n, int W,
                          int c, float* v) {
    if (!MOE) {
        ld8(y + n * W + c, v);
        return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.f;
    for (int k0 = 0; k0 < top; k0 += 4) {       // 4 rows in flight
        float f[4][8], g[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const long r = n * top + min(k0 + k, top - 1);
            g[k] = k0 + k < top ? wt[r] : 0.f;
            if (g[k] != 0.f) ld8(y + r * W + c, f[k]);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k)
            if (g[k] != 0.f)
#pragma unroll
                for (int i = 0; i < 8; ++i) v[i] += g[k] * f[k][i];
    }
}

// What y is: a sublayer's output, a row per (token, expert), or partial sums
enum { PLAIN, PAIRS, PARTS };

// NV turns of THREADS threads have a row; x and the weights are loaded ahead of the
// sum. In a graph, rows of 3072, us: 45 rows with 4 parts 4.2 with 256 threads and
// both loaded after it, now 3.3; 256 rows 4.9 and 4.2; 5991 rows, no parts, 33.8 and
// 33.4. Of 2304 to 8192 columns, up to 1000 rows 1.0 to 1.25 times as fast, 2048 of 4096
// and of 6144 .96, 8192 .99 to 1.17.
template <class T, int KIND, int NV, int THREADS>
__global__ void __launch_bounds__(THREADS)
k_post_norm(float* __restrict__ x, T* __restrict__ xb,
            const void* __restrict__ y, const float* __restrict__ wt, int top,
            const float* __restrict__ w, float w_off, int W, int Wtrue,
            float eps) {
    __shared__ float red[8];
    const long n = blockIdx.x;
    float v[NV][8], a[NV][8], g[NV][8];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * THREADS + threadIdx.x) * 8;
        if (c < W) {
            ld8(x + n * W + c, a[j]);
            ld8(w + c, g[j]);
            if (KIND == PARTS)
                summed8((const float*)y, top, n, gridDim.x, W, c, v[j]);
            else
                sublayer8<T, KIND == PAIRS>((const T*)y, wt, top, n, W, c,
                                            v[j]);
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += v[j][i] * v[j][i];
        }
    }
    const float rs =
        1.f / sqrtf(block_sum<THREADS>(ss, red) / (float)Wtrue + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * THREADS + threadIdx.x) * 8;
        if (c < W) {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                a[j][i] += v[j][i] * rs * (w_off + g[j][i]);
            st8(x + n * W + c, a[j]);
            if (xb) st8(xb + n * W + c, a[j]);
        }
    }
}

// ===========================================================================
// Norm behind the sum, and the average over depth:
//   r = norm(alpha * x + y) * (w_off + w)       r: the (sub)layer's result
//   hist null:  x' = r
//   otherwise:  x' = sum_{j < nh} coef[j] hist[j] + coef[nh] r, and r is
//               kept as hist[nh] if `keep`. hist: f32 [layers + 1][N][W]
//   xb = T(x'). The row x may be x' or a row of hist.
// With experts y is their weighted sum plus ident[n] * x (the weight of the
// identity experts, which return the sublayer's input).
// ===========================================================================
template <class T, bool MOE>
__global__ void __launch_bounds__(256)
k_sum_norm(float* xo, T* __restrict__ xb, const float* x,
           const T* __restrict__ y, const float* __restrict__ wt, int top,
           const float* __restrict__ ident, const float* __restrict__ w,
           float w_off, float alpha, float* hist,
           const float* __restrict__ coef, int nh, int keep, long N, int W,
           int Wtrue, float eps) {
    __shared__ float red[4];
    const long n = blockIdx.x;
    if (MOE && ident) alpha += ident[n];
    float v[4][8];
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = (j * 256 + threadIdx.x) * 8;
        if (c < W) {
            float a[8];
            sublayer8<T, MOE>(y, wt, top, n, W, c, v[j]);
            ld8(x + n * W + c, a);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                v[j][i] += alpha * a[i];
                ss += v[j][i] * v[j][i];
            }
        }
    }
    const float rs = 1.f / sqrtf(block_sum(ss, red) / (float)Wtrue + eps);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = (j * 256 + threadIdx.x) * 8;
        if (c < W) {
            float g[8];
            ld8(w + c, g);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[j][i] *= rs * (w_off + g[i]);
            if (hist) {
                if (keep) st8(hist + (nh * N + n) * W + c, v[j]);
                const float cr = coef[nh];
#pragma unroll
                for (int i = 0; i < 8; ++i) v[j][i] *= cr;
                for (int l0 = 0; l0 < nh; l0 += 4) {    // 4 rows in flight
                    float f[4][8];
#pragma unroll
                    for (int l = 0; l < 4; ++l)
                        ld8(hist + (min(l0 + l, nh - 1) * N + n) * W + c, f[l]);
#pragma unroll
                    for (int l = 0; l < 4; ++l) {
                        const float cl = l0 + l < nh ? coef[l0 + l] : 0.f;
#pragma unroll
                        for (int i = 0; i < 8; ++i) v[j][i] += cl * f[l][i];
                    }
                }
            }
            st8(xo + n * W + c, v[j]);
            if (xb) st8(xb + n * W + c, v[j]);
        }
    }
}

// out[r] = norm(x[rows[r]]) in T; rows null = identity
template <class T>
__global__ void __launch_bounds__(256)
k_norm_rows(T* __restrict__ out, const float* __restrict__ x,
            const int* __restrict__ rows, const float* __restrict__ w,
            float w_off, int W, int Wtrue, float eps) {
    __shared__ float red[4];
    const long n = rows ? rows[blockIdx.x] : blockIdx.x;
    float ss = 0.f;
    for (int c = threadIdx.x * 8; c < W; c += 2048) {
        float a[8];
        ld8(x + n * W + c, a);
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += a[i] * a[i];
    }
    const float rs = 1.f / sqrtf(block_sum(ss, red) / (float)Wtrue + eps);
    for (int c = threadIdx.x * 8; c < W; c += 2048) {
        float a[8], g[8];
        ld8(x + n * W + c, a);
        ld8(w + c, g);
#pragma unroll
        for (int i = 0; i < 8; ++i) a[i] *= rs * (w_off + g[i]);
        st8(out + (long)blockIdx.x * W + c, a);
    }
}

// ===========================================================================
// Norm in groups: a row's `groups` equal consecutive parts, each divided by
// its own root mean square, times w (no offset).
//   ADD:  x += norm(y) * wy;  out = norm(x) * w, if there is an out
//   else: out[r] = norm(x[rows[r]]) * w
// Columns from Wtrue on carry zeros. Squares are summed in pieces of GR columns
// (the largest power of two up to 8 that divides a group), which meet in LDS:
// group sums come out the same in every run. W <= 8192.
// ===========================================================================
struct Groups {
    int count, size;
};

// v holds a thread's columns, 8 from (j * threads + its number) * 8 on for each j;
// factors 1 / rms by group into rs
template <int NV, int GR>
DEV_INLINE void group_factors(const float (&v)[NV][8], float* part, float* rs,
                              int W, const Groups gp, float eps) {
    __syncthreads();                       // part and rs are free
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * blockDim.x + threadIdx.x) * 8;
        if (c < W)
#pragma unroll
            for (int i = 0; i < 8; i += GR) {
                float s = 0.f;
#pragma unroll
                for (int k = 0; k < GR; ++k) s += v[j][i + k] * v[j][i + k];
                part[(c + i) / GR] = s;
            }
    }
    __syncthreads();
    const int lane = threadIdx.x & 63, n = gp.size / GR;
    for (int g = threadIdx.x >> 6; g < gp.count; g += blockDim.x >> 6) {
        float s = 0.f;
        for (int i = lane; i < n; i += 64) s += part[g * n + i];
        s = wave_reduce_sum(s);
        if (lane == 0) rs[g] = 1.f / sqrtf(s / (float)gp.size + eps);
    }
    __syncthreads();
}

// f *= rs of each column's group
template <int GR>
DEV_INLINE void scale_groups(float (&f)[8], const float* rs, int c,
                             const Groups gp) {
#pragma unroll
    for (int i = 0; i < 8; i += GR) {
        const float r = rs[min((c + i) / gp.size, gp.count - 1)];
#pragma unroll
        for (int k = 0; k < GR; ++k) f[i + k] *= r;
    }
}

// parts > 0: y is f32 partial sums. A thread has 8 NV columns, and all its loads are
// on their way at once, but for the weights of two turns, whose registers would have a
// SIMD hold fewer waves (8192 rows of 5120 in groups of 128: 157 us with them ahead, 116
// behind the sums; 1024 20.8, 19.9; one 7.6 either way). Bound by the loads and the
// sums' steps: 160 rows of 3072 with 2 and 8 parts 7.6 us with 256 threads a row and
// weights read after the sums, now 5.7.
template <class T, bool ADD, int GR, int NV>
__global__ void __launch_bounds__(512)
k_group_norm(T* __restrict__ out, float* __restrict__ x,
             const void* __restrict__ y, int parts,
             const int* __restrict__ rows,
             const float* __restrict__ wy, const float* __restrict__ w, int W,
             const Groups gp, float eps) {
    extern __shared__ float part[];        // W / GR, then a factor per group
    float* const rs = part + W / GR;
    const long n = !ADD && rows ? rows[blockIdx.x] : blockIdx.x;
    float v[NV][8], a[NV][8], gy[NV][8], g[NV][8];
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * blockDim.x + threadIdx.x) * 8;
        if (c >= W) continue;
        ld8(x + n * W + c, a[j]);
        if (NV == 1 && ADD) ld8(wy + c, gy[j]);
        if (NV == 1 && out) ld8(w + c, g[j]);
        if (ADD && parts)
            summed8((const float*)y, parts, n, gridDim.x, W, c, v[j]);
        else if (ADD)
            ld8((const T*)y + n * W + c, v[j]);
    }
    if (ADD) {
        group_factors<NV, GR>(v, part, rs, W, gp, eps);
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (j * blockDim.x + threadIdx.x) * 8;
            if (c >= W) continue;
            if (NV > 1) ld8(wy + c, gy[j]);
            scale_groups<GR>(v[j], rs, c, gp);
#pragma unroll
            for (int i = 0; i < 8; ++i) a[j][i] += v[j][i] * gy[j][i];
            st8(x + n * W + c, a[j]);
        }
        if (!out) return;
    }
    group_factors<NV, GR>(a, part, rs, W, gp, eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * blockDim.x + threadIdx.x) * 8;
        if (c >= W) continue;
        if (NV > 1) ld8(w + c, g[j]);
        scale_groups<GR>(a[j], rs, c, gp);
#pragma unroll
        for (int i = 0; i < 8; ++i) a[j][i] *= g[j][i];
        st8(out + (long)blockIdx.x * W + c, a[j]);
    }
}

// ===========================================================================
// Hyper-connections: ns residual streams x_s, f32 [N][ns][W].
//   start: x_s = embed[token] * scale for all s
//   join:  x_t = sum_s mix[s][t] x_s + put[t] y, all from the old ones
// and what the next sublayer reads, if there is one:
//   h = T(norm(sum_s in[s] x_s) * w)
// hc holds mix [from][to], then put. y is a sublayer's output; with experts
// (top > 0) the sum of a token's pairs, and `extra` adds a row times the
// sigmoid of a number per token. S: ns rounded up to a power of two. W <= 2048
// NV; the mean is over Wtrue elements.
// ===========================================================================
template <class T, int NV>
DEV_INLINE void store_normed(T* h, const float u[NV][8], const float* w,
                             long n, int W, int Wtrue, float eps, float* red) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < NV; ++j)
        if ((j * 256 + threadIdx.x) * 8 < W)
#pragma unroll
            for (int i = 0; i < 8; ++i) ss += u[j][i] * u[j][i];
    const float rs = 1.f / sqrtf(block_sum(ss, red) / (float)Wtrue + eps);
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * 256 + threadIdx.x) * 8;
        if (c < W) {
            float g[8];
            ld8(w + c, g);
#pragma unroll
            for (int i = 0; i < 8; ++i) g[i] *= u[j][i] * rs;
            st8(h + n * W + c, g);
        }
    }
}

template <class T>
__global__ void __launch_bounds__(256)
k_streams_start(float* __restrict__ x, T* __restrict__ h,
                const T* __restrict__ emb, const long long* __restrict__ tok,
                float scale, const float* __restrict__ in,
                const float* __restrict__ w, int ns, int W, int Wtrue,
                float eps, int vocab) {
    __shared__ float red[4];
    const long n = blockIdx.x;
    const long t = min(max(tok[n], 0ll), (long long)vocab - 1);
    float total = 0.f, u[4][8];
    for (int s = 0; s < ns; ++s) total += in[s];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = (j * 256 + threadIdx.x) * 8;
        if (c < W) {
            float a[8];
            ld8(emb + t * W + c, a);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                a[i] *= scale;
                u[j][i] = total * a[i];
            }
            for (int s = 0; s < ns; ++s) st8(x + (n * ns + s) * W + c, a);
        }
    }
    store_normed<T, 4>(h, u, w, n, W, Wtrue, eps, red);
}

template <class T, int S, int NV, bool MOE>
__global__ void __launch_bounds__(256)
k_streams_join(float* __restrict__ x, T* __restrict__ h,
               const T* __restrict__ y, int top, const T* __restrict__ extra,
               const float* __restrict__ extra_z, int extra_ld,
               const float* __restrict__ hc, const float* __restrict__ in,
               const float* __restrict__ w, int ns, int W, int Wtrue,
               float eps) {
    constexpr bool AHEAD = S * NV <= 8;     // all loads ahead of the stores
    constexpr int NX = AHEAD ? NV : 1;
    __shared__ float red[4];
    const long n = blockIdx.x;
    float* xr = x + n * ns * W;
    const float ge = MOE && extra ? sigmoidf_(extra_z[n * extra_ld]) : 0.f;
    float a[NX][S][8], v[NX][8], u[NV][8];
    auto load = [&](int j, int c) {
#pragma unroll
        for (int s = 0; s < S; ++s)
            if (s < ns) ld8(xr + (long)s * W + c, a[j][s]);
        if (!MOE) {
            ld8(y + n * W + c, v[j]);
            return;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) v[j][i] = 0.f;
        for (int k0 = 0; k0 < top; k0 += 4) {       // 4 rows in flight
            float f[4][8];
#pragma unroll
            for (int k = 0; k < 4; ++k)
                ld8(y + (n * top + min(k0 + k, top - 1)) * W + c, f[k]);
#pragma unroll
            for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    v[j][i] += k0 + k < top ? f[k][i] : 0.f;
        }
        if (extra) {
            float f[8];
            ld8(extra + n * W + c, f);
#pragma unroll
            for (int i = 0; i < 8; ++i) v[j][i] += ge * f[i];
        }
    };
    if (AHEAD)
#pragma unroll
        for (int j = 0; j < NV; ++j) {
            const int c = (j * 256 + threadIdx.x) * 8;
            if (c < W) load(j % NX, c);
        }
#pragma unroll
    for (int j = 0; j < NV; ++j) {
        const int c = (j * 256 + threadIdx.x) * 8, jx = j % NX;
        if (c < W) {
            if (!AHEAD) load(jx, c);
#pragma unroll
            for (int i = 0; i < 8; ++i) u[j][i] = 0.f;
#pragma unroll
            for (int t = 0; t < S; ++t) {
                if (t >= ns) continue;
                const float put = hc[ns * ns + t], read = h ? in[t] : 0.f;
                float r[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) r[i] = put * v[jx][i];
#pragma unroll
                for (int s = 0; s < S; ++s) {
                    if (s >= ns) continue;
                    const float m = hc[s * ns + t];
#pragma unroll
                    for (int i = 0; i < 8; ++i) r[i] += m * a[jx][s][i];
                }
#pragma unroll
                for (int i = 0; i < 8; ++i) u[j][i] += read * r[i];
                st8(xr + (long)t * W + c, r);
            }
        }
    }
    if (h) store_normed<T, NV>(h, u, w, n, W, Wtrue, eps, red);
}

// out[r] = norm(sum_s x_s[rows[r]]) * w; rows null = identity
template <class T>
__global__ void __launch_bounds__(256)
k_streams_norm(T* __restrict__ out, const float* __restrict__ x,
               const int* __restrict__ rows, const float* __restrict__ w,
               int ns, int W, int Wtrue, float eps) {
    __shared__ float red[4];
    const long n = rows ? rows[blockIdx.x] : blockIdx.x;
    float u[4][8];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int c = (j * 256 + threadIdx.x) * 8;
#pragma unroll
        for (int i = 0; i < 8; ++i) u[j][i] = 0.f;
        if (c < W)
            for (int s = 0; s < ns; ++s) {
                float a[8];
                ld8(x + (n * ns + s) * W + c, a);
#pragma unroll
                for (int i = 0; i < 8; ++i) u[j][i] += a[i];
            }
    }
    store_normed<T, 4>(out, u, w, blockIdx.x, W, Wtrue, eps, red);
}

// ===========================================================================
// PolyNorm: out = c0 N(z) + c1 N(z^2) + c2 N(z^3) + c3, powers by element, N
// dividing a row by its root mean square over Ftrue elements (columns behind
// them are zero). NV > 0: a row of up to NV * THREADS * 8 columns stays in registers.
// Bound by its loads and steps. With 256 and 512 threads, in a graph, us: 160 rows of
// 12288 5.7 and 4.6, 4096 rows 35.4 and 34.1; of 4096 columns 3.8 and 3.4, but 16.0 and
// 18.0. Between 4096 and 6144 columns two turns of 512 threads are mostly empty, which
// many rows show: 5120 columns, 160 rows 3.8 and 3.5, 512 4.4 and 4.7, 8192 34.0 and 41.3.
// ===========================================================================
template <class T, int NV, int THREADS>
__global__ void __launch_bounds__(THREADS)
k_poly_norm(T* __restrict__ out, const T* __restrict__ z,
            const float* __restrict__ coef, int F, int Ftrue, float eps) {
    __shared__ float red[3][8];
    constexpr int KEEP = NV ? NV : 1;
    const long n = blockIdx.x;
    float v[KEEP][8], ss[3] = {0.f, 0.f, 0.f};
    auto add = [&](const float* f) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float q = f[i] * f[i];
            ss[0] += q;
            ss[1] += q * q;
            ss[2] += q * q * q;
        }
    };
    if (NV) {
#pragma unroll
        for (int j = 0; j < KEEP; ++j) {
            const int c = (j * THREADS + threadIdx.x) * 8;
            if (c < F) {
                ld8(z + n * F + c, v[j]);
                add(v[j]);
            }
        }
    } else {
        for (int c = threadIdx.x * 8; c < F; c += THREADS * 8) {
            ld8(z + n * F + c, v[0]);
            add(v[0]);
        }
    }
    float k[3];
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        const float s = wave_reduce_sum(ss[i]);
        if ((threadIdx.x & 63) == 0) red[i][threadIdx.x >> 6] = s;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 3; ++i) {
        float s = red[i][0];
#pragma unroll
        for (int v = 1; v < THREADS / 64; ++v) s += red[i][v];
        k[i] = coef[i] / sqrtf(s / (float)Ftrue + eps);
    }
    const float k3 = coef[3];
    auto put = [&](float* f, int c) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
            f[i] = k3 + f[i] * (k[0] + f[i] * (k[1] + f[i] * k[2]));
        st8(out + n * F + c, f);
    };
    if (NV) {
#pragma unroll
        for (int j = 0; j < KEEP; ++j) {
            const int c = (j * THREADS + threadIdx.x) * 8;
            if (c < F) put(v[j], c);
        }
    } else {
        for (int c = threadIdx.x * 8; c < F; c += THREADS * 8) {
            ld8(z + n * F + c, v[0]);
            put(v[0], c);
        }
    }
}

// out = glu(gu[:, :F], gu[:, F:]), f32
__global__ void __launch_bounds__(256)
k_glu_f32(float* __restrict__ out, const float* __restrict__ gu, long n,
          int F, const GluParams p) {
    for (long i = blockIdx.x * 256L + threadIdx.x; i < n * F;
         i += gridDim.x * 256L) {
        const long r = i / F, c = i % F;
        float g = fminf(gu[r * 2 * F + c], p.limit);
        float u = fminf(fmaxf(gu[r * 2 * F + F + c], -p.limit), p.limit);
        const float z = p.alpha * g * (1.f + p.cubic * g * g);
        out[i] = g / (1.f + expf(-z)) * (u + p.shift);
    }
}

// ===========================================================================
// Projection to a few f32 outputs (router logits, recurrence gates):
//   out[n, j] = sum_k x[n, k] w[j, k] + bias[j], bf16 inputs, f32 result.
// One block per 16 rows x 16 NT outputs; its 8 waves split K and add up in
// LDS, each with U steps of loads in flight. Fragments load straight from
// memory (both operands are k-contiguous). K % 32 == 0.
// ===========================================================================
template <int NT>
__global__ void __launch_bounds__(512)
k_proj_f32(float* __restrict__ out, const bf16_t* __restrict__ x,
           const bf16_t* __restrict__ w, const float* __restrict__ bias,
           int M, int N, int K) {
    constexpr int U = NT == 1 ? 6 : 4;
    __shared__ float red[8][16][16 * NT + 1];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int fr = lane & 15, kg = (lane >> 4) * 8;
    const int m0 = blockIdx.x * 16, n0 = blockIdx.y * 16 * NT;
    const bf16_t* xr = x + (long)min(m0 + fr, M - 1) * K + kg;
    const bf16_t* wr[NT];
    f32x4 acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        wr[t] = w + (long)min(n0 + t * 16 + fr, N - 1) * K + kg;
        acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    }
    const int steps = K >> 5;
    for (int s0 = wid; s0 < steps; s0 += 8 * U) {
        bf16x8 a[U], b[U][NT];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = min(s0 + u * 8, steps - 1);
            a[u] = *(const bf16x8*)(xr + s * 32);
#pragma unroll
            for (int t = 0; t < NT; ++t)
                b[u][t] = *(const bf16x8*)(wr[t] + s * 32);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (s0 + u * 8 < steps)
#pragma unroll
                for (int t = 0; t < NT; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        a[u], b[u][t], acc[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
            red[wid][(lane >> 4) * 4 + r][t * 16 + fr] = acc[t][r];
    __syncthreads();
    for (int e = threadIdx.x; e < 256 * NT; e += 512) {
        const int i = e / (16 * NT), j = e % (16 * NT);
        if (m0 + i >= M || n0 + j >= N) continue;
        float v = bias ? bias[n0 + j] : 0.f;
#pragma unroll
        for (int k = 0; k < 8; ++k) v += red[k][i][j];
        out[(long)(m0 + i) * N + n0 + j] = v;
    }
}

// ===========================================================================
// Attention prologue: rotated (if there are tables) unit-RMS q and k (no
// weight), query temperature, and the write of k and v into the paged cache,
// from one projection row
//   [H*P q | G*P k | G*P v | ...], row stride ld.
// temperature(p) = 1 + coef * ln(floor((p + 1) / every) + 1).
// P / 8 lanes per head. Further waves put SiLU on act_n columns from act_0 on,
// in place (q, k and v of a recurrence in the same row).
// ===========================================================================
template <class T, int P>
__global__ void __launch_bounds__(256)
k_qknorm_kv(T* __restrict__ qkv, T* __restrict__ q_out,
            T* __restrict__ kc, T* __restrict__ vc,
            const int* __restrict__ table, int per_slot,
            const int* __restrict__ pos, const int* __restrict__ slot,
            int N, int H, int G, int ld_, int dim, float eps, float coef,
            int every, const Rotation rot, int act_0, int act_n) {
    constexpr int LPH = P / 8, HW = 64 / LPH;
    const int nh = H + 2 * G;
    const int groups = (nh + HW - 1) / HW, per = groups + (act_n + 511) / 512;
    const long item = blockIdx.x * 4L + (threadIdx.x >> 6);
    if (item >= (long)N * per) return;
    const int n = (int)(item / per), it = (int)(item % per);
    const int lane = threadIdx.x & 63;
    float f[8];
    if (it >= groups) {
        const int c = (it - groups) * 512 + lane * 8;
        if (c >= act_n) return;
        T* z = qkv + (long)n * ld_ + act_0 + c;
        ld8(z, f);
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] *= sigmoidf_(f[i]);
        st8(z, f);
        return;
    }
    const int h = it * HW + lane / LPH, c = (lane % LPH) * 8;
    if (h >= nh) return;
    ld8(qkv + (long)n * ld_ + (long)h * P + c, f);
    const int p = pos[n];
    T* dst;
    if (h < H) {
        dst = q_out + ((long)n * H + h) * P;
    } else {
        const int blk = p / KV_PAGE;
        if (blk >= per_slot) return;
        const int hk = (h - H) % G;
        const long page = table[(long)slot[n] * per_slot + blk];
        dst = (h < H + G ? kc : vc) +
              ((page * G + hk) * KV_PAGE + p % KV_PAGE) * P;
    }
    if (h < H + G) {
        if (c < 2 * rot.half) rotate8(f, c, p, rot);
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < 8; ++i) ss += f[i] * f[i];
#pragma unroll
        for (int off = LPH / 2; off > 0; off >>= 1)
            ss += __shfl_xor(ss, off, WAVE);
        float s = 1.f / sqrtf(ss / (float)dim + eps);
        if (h < H) s *= 1.f + coef * logf((float)((p + 1) / every) + 1.f);
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] *= s;
    }
    st8(dst + c, f);
}

// Varlen prefill over the paged cache. meta row (8 ints): {q_off, len, slot,
// q0, start}: rows [q0, q0 + 128) of the portion packed at q_off, whose first
// token stands at position `start`.
template <int D, class Keys>
__global__ void __launch_bounds__(256, D > 128 ? 1 : 2)
k_paged_prefill(bf16_t* __restrict__ out, const bf16_t* __restrict__ q,
                const PagedKV<D> kv, const int* __restrict__ meta, int ntiles,
                int Hq, int G, float scale, const HeadEpilogue epi,
                const Keys keys) {
    __shared__ __attribute__((aligned(16))) bf16_t lds[prefill_lds<D>()];
    int tile, hq;
    if (!prefill_item(ntiles, Hq, &tile, &hq)) return;
    const int* m = meta + tile * 8;
    const int q_off = m[0], len = m[1], start = m[4];
    attn_prefill_tile<D>(out + epi.at(q_off, 0, Hq, D),
                            q + (long)q_off * Hq * D, kv, len, Hq, G, hq, m[2],
                            start + len, start, scale, m[3], lds, epi, q_off,
                            keys);
}

// Exact mode: one block per (row, query head), f32 cache, any position.
template <int P>
__global__ void __launch_bounds__(256)
k_attn_rows_f32(float* __restrict__ out, const float* __restrict__ q,
                const float* __restrict__ kc, const float* __restrict__ vc,
                const int* __restrict__ table, int per_slot,
                const int* __restrict__ pos, const int* __restrict__ slot,
                int H, int G, float scale, const float* __restrict__ sink,
                const float* __restrict__ gate, int gate_ld, int gate_el,
                float oscale, int out_ld, const WindowKeys keys) {
    const int n = blockIdx.x / H, h = blockIdx.x % H;
    const int hk = h / (H / G);
    const int* tab = table + (long)slot[n] * per_slot;
    const int seq = min(pos[n] + 1, per_slot * KV_PAGE);
    __shared__ float qs[P], sc[256], red[4], acc_s[256];
    for (int i = threadIdx.x; i < P; i += 256)
        qs[i] = q[((long)n * H + h) * P + i];
    __syncthreads();
    constexpr int NG = 256 / P;
    const int c = threadIdx.x % P, grp = threadIdx.x / P;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    float m = sink ? sink[h] : -INFINITY, l = sink ? 1.f : 0.f, acc = 0.f;
    for (int k0 = keys.skip(0, seq - 1); k0 < seq;
         k0 = keys.skip(k0 + 256, seq - 1)) {
        const int j = k0 + threadIdx.x;
        const bool seen = j < seq && keys.sees(seq - 1, j);
        float s = -INFINITY;
        if (seen) {
            const float* kr = kc + (((long)tab[j / KV_PAGE] * G + hk) * KV_PAGE
                                    + j % KV_PAGE) * P;
            s = 0.f;
            for (int i = 0; i < P; i += 4) {
                const float4 kv = *(const float4*)(kr + i);
                s += kv.x * qs[i] + kv.y * qs[i + 1] + kv.z * qs[i + 2] +
                     kv.w * qs[i + 3];
            }
            s *= scale;
        }
        float mx = wave_reduce_max(s);
        if (lane == 0) red[wid] = mx;
        __syncthreads();
        mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
        const float mn = fmaxf(m, mx);
        const float alpha = (m == -INFINITY) ? 0.f : expf(m - mn);
        const float p = seen ? expf(s - mn) : 0.f;
        sc[threadIdx.x] = p;
        m = mn;
        __syncthreads();                       // red read, sc written
        const float ps = wave_reduce_sum(p);
        if (lane == 0) red[wid] = ps;
        acc *= alpha;
        const int jn = min(256, seq - k0);
        for (int t = grp; t < jn; t += NG) {
            const int jj = k0 + t;
            acc += sc[t] * vc[(((long)tab[jj / KV_PAGE] * G + hk) * KV_PAGE +
                               jj % KV_PAGE) * P + c];
        }
        __syncthreads();
        l = l * alpha + red[0] + red[1] + red[2] + red[3];
        __syncthreads();
    }
    acc_s[threadIdx.x] = acc;
    __syncthreads();
    if (threadIdx.x < P) {
        float a = 0.f;
        for (int g = 0; g < NG; ++g) a += acc_s[g * P + threadIdx.x];
        float f = l > 0.f ? oscale / l : 0.f;
        if (gate)
            f *= sigmoidf_(gate[(long)n * gate_ld +
                                (gate_el ? h * P + threadIdx.x : h)]);
        out[(long)n * out_ld + h * P + threadIdx.x] = a * f;
    }
}

// ===========================================================================
// mLSTM: matrix memory with exponential gates, per head
//   i = cap tanh(zi / cap);  f = logsigmoid(cap tanh(zf / cap))
//   m' = max(f + m, i);  keep = exp(f + m - m');  put = exp(i - m')
//   S = keep S + put v k^T;  n = keep n + put k
//   o = S q / (max(|n . q|, exp(-m')) + 1e-6),  q scaled by dim^-1/2
// The state of a slot is f32 [H][DV + 1][DK]: row r < DV is S[:, r] over the
// key dimension, and row DV is n, which is the memory of the constant value
// 1, so one update serves both. m is f32 [H]. A segment that starts at
// position 0 takes the state as zero whatever the slot holds.
// Projection row: [H*DK q | H*DK k | H*DV v | H*DV out gate | ...], stride ld;
// gate row: [H zi | H zf], f32, biases included.
// ===========================================================================
DEV_INLINE void mlstm_gates(const float* gr, int h, int H, float cap,
                            float& i, float& f) {
    i = cap * tanhf(gr[h] / cap);
    const float z = cap * tanhf(gr[H + h] / cap);
    f = log_sigmoid(z);
}

// seg (int4): {first token, length, slot, start position}; null: row r is a
// segment of one token at pos[r] of slot[r].
DEV_INLINE int4 segment(const int4* seg, const int* pos, const int* slot,
                        int r) {
    if (seg) return seg[r];
    return make_int4(r, 1, slot[r], pos[r]);
}

// Token by token. Block = (segment, head, `rpb` state rows); LPR lanes hold
// one row of DK as NJ float4 each, and a wave works on 64 / LPR rows at once,
// U of them in flight. The other kinds have neither an input gate nor a
// normaliser row (S is [H][DV][DK]): their memory decays per key channel, gr
// being the logarithm of the decay, f32 [n][H*DK] (gated linear attention), or
// by a constant per head, gr f32 [H] (lightning attention).
// Bound by reading and writing the states: past the caches both ways, and ahead of the
// gates, queries and keys (ONCE), where all of a step's recurrent layers have REC_ONCE of
// them or more (the Infinity Cache is 256 MB): a layer then finds little of what it wrote
// a step before, and the step's other data stays. Below, states stay from step to step.
// The line is where whole models change sides; a step with and without ONCE, us, by MB:
//   birepel:3b, five layers of 12 x 128 x 257  126 1480, 1492, 189 1538, 1527, 253 1577,
//     1612, 505 1772, 1801
//   maferax:5b, six of 12 x 128 x 256  151 1936, 1945, 189 2004, 1999, 226 2064, 2090,
//     302 2144, 2211
//   zinavik:4b, eight  151 2114, 2126, 201 2370, 2395, 302 2484, 2530, 805 2975, 3026
//   two of birepel's five, in three layers  152 482, 463, 202 526, 504, 227 524, 522, 253
//     547, 550, 404 653, 669, 808 932, 963; 202 MB of several batches in turn 530, 548
// 32 rows a block; 64: 49.9 us a call of 64 sequences, not 47.0.
#define REC_ONCE 200000000l
enum Rec { MLSTM = 0, CHANNELS = 1, CONSTANT = 2 };

template <class T, int LPR, int NJ, int KIND, bool ONCE>
__global__ void __launch_bounds__(256)
k_rec_step(float* __restrict__ o, float* __restrict__ S,
           const float* __restrict__ mst, const T* __restrict__ qkv,
           const float* __restrict__ gr, const int4* __restrict__ segs,
           const int* __restrict__ pos, const int* __restrict__ slot,
           int H, int DK, int DV, int ld_, float qscale, float cap,
           int rpb) {
    constexpr int RW = 64 / LPR;
    constexpr int U = NJ == 1 ? 4 : 2;
    constexpr bool CH = KIND == CHANNELS, GATED = KIND == MLSTM;
    const int R = GATED ? DV + 1 : DV;
    const int4 sg = segment(segs, pos, slot, blockIdx.x);
    const int h = blockIdx.y;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int c0 = (lane % LPR) * 4, rl = lane / LPR;
    const int rbeg = blockIdx.z * rpb, rend = min(R, rbeg + rpb);
    float* Sb = S + ((long)sg.z * H + h) * R * DK;
    f32x4 s[U][NJ];
    auto load_rows = [&](int r0, bool fresh) {
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int j = 0; j < NJ; ++j) {
                const int r = r0 + u * RW + rl, c = c0 + j * LPR * 4;
                s[u][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
                if (fresh || r >= rend || c >= DK) continue;
                const f32x4* from = (const f32x4*)(Sb + (long)r * DK + c);
                s[u][j] = ONCE ? __builtin_nontemporal_load(from) : *from;
            }
    };
    float m = !GATED || sg.w == 0 ? 0.f : mst[(long)sg.z * H + h];
    for (int t = 0; t < sg.y; ++t) {
        const long n = sg.x + t;
        const bool fresh = sg.w + t == 0;
        int r0 = rbeg + wid * RW * U;
        if (ONCE) load_rows(r0, fresh);
        float keep1 = KIND == CONSTANT ? gr[h] : 0.f, put = 1.f;
        if (GATED) {
            float gi, gf;
            mlstm_gates(gr + n * 2 * H, h, H, cap, gi, gf);
            const float mn = fmaxf(gf + m, gi);
            keep1 = expf(gf + m - mn);
            put = expf(gi - mn);
            m = mn;
        }
        const T* row = qkv + n * ld_;
        float qv[NJ][4], kv[NJ][4], keep[CH ? NJ : 1][4];
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
            const int c = c0 + j * LPR * 4;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const bool in = c < DK;
                qv[j][i] = in ? ld(row + h * DK + c + i) * qscale : 0.f;
                kv[j][i] = in ? ld(row + (H + h) * DK + c + i) * put : 0.f;
                if (CH)
                    keep[j][i] =
                        in ? expf(gr[n * H * DK + h * DK + c + i]) : 0.f;
            }
        }
        auto kept = [&](int j, int i) { return CH ? keep[j][i] : keep1; };
        const T* vrow = row + 2 * H * DK + h * DV;
        while (r0 < rend) {
            if (!ONCE) load_rows(r0, fresh);
            float v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int r = r0 + u * RW + rl;
                v[u] = r < DV ? ld(vrow + r) : 1.f;
                if (r >= rend) v[u] = 0.f;
            }
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int r = r0 + u * RW + rl;
                float a = 0.f;
#pragma unroll
                for (int j = 0; j < NJ; ++j) {
                    const int c = c0 + j * LPR * 4;
                    f32x4 z = s[u][j];
                    z.x = kept(j, 0) * z.x + kv[j][0] * v[u];
                    z.y = kept(j, 1) * z.y + kv[j][1] * v[u];
                    z.z = kept(j, 2) * z.z + kv[j][2] * v[u];
                    z.w = kept(j, 3) * z.w + kv[j][3] * v[u];
                    a += z.x * qv[j][0] + z.y * qv[j][1] + z.z * qv[j][2] +
                         z.w * qv[j][3];
                    if (r >= rend || c >= DK) continue;
                    f32x4* to = (f32x4*)(Sb + (long)r * DK + c);
                    if (ONCE) __builtin_nontemporal_store(z, to);
                    else *to = z;
                }
#pragma unroll
                for (int off = LPR / 2; off > 0; off >>= 1)
                    a += __shfl_xor(a, off, WAVE);
                if (lane % LPR == 0 && r < rend)
                    o[(n * H + h) * (DV + 4) + r] = a;
            }
            r0 += 4 * RW * U;
            if (ONCE) load_rows(r0, fresh);
        }
    }
}

// o (f32 rows of DV + 4 per token and head: DV sums, n . q, padding)
// -> T out[n, H*DV]: unit RMS per head, times norm, times sigmoid of the
// output gate. Items [0, nseg) are segments of the token-by-token kernel, whose
// o still lacks its denominator and whose m is advanced here; the nplain
// tokens from plain0 on are finished sums. One wave per (item, head). With
// SILU the gate multiplies by itself times its sigmoid.
template <class T, bool SILU>
__global__ void __launch_bounds__(256)
k_rec_out(T* __restrict__ out, const float* __restrict__ o,
            float* __restrict__ mst, const T* __restrict__ qkv,
            const float* __restrict__ gr, const int4* __restrict__ segs,
            const int* __restrict__ pos, const int* __restrict__ slot,
            const float* __restrict__ norm, int nseg, int plain0, int nplain,
            int H, int DK, int DV, int ld_, int dvtrue, float cap,
            float eps) {
    const long item = blockIdx.x * 4L + (threadIdx.x >> 6);
    if (item >= (long)(nseg + nplain) * H) return;
    const int it = (int)(item / H), h = (int)(item % H);
    const int lane = threadIdx.x & 63;
    int4 sg;
    float m = 0.f;
    const bool is_seg = it < nseg;
    if (is_seg) {
        sg = segment(segs, pos, slot, it);
        if (sg.w != 0) m = mst[(long)sg.z * H + h];
    } else {
        sg = make_int4(plain0 + it - nseg, 1, 0, 0);
    }
    for (int t = 0; t < sg.y; ++t) {
        const long n = sg.x + t;
        const float* ob = o + (n * H + h) * (DV + 4);
        float inv = 1.f;
        if (is_seg) {
            float gi, gf;
            mlstm_gates(gr + n * 2 * H, h, H, cap, gi, gf);
            m = fmaxf(gf + m, gi);
            inv = 1.f / (fmaxf(fabsf(ob[DV]), expf(-m)) + 1e-6f);
        }
        float ss = 0.f;
        for (int c = lane * 4; c < DV; c += 256) {
            const float4 v = *(const float4*)(ob + c);
            ss += (v.x * v.x + v.y * v.y + v.z * v.z + v.w * v.w) * inv * inv;
        }
        const float rs =
            inv / sqrtf(wave_reduce_sum(ss) / (float)dvtrue + eps);
        const T* g = qkv + n * ld_ + (long)H * (2 * DK + DV) + (long)h * DV;
        T* dst = out + (n * H + h) * DV;
        for (int c = lane * 4; c < DV; c += 256) {
            const float4 v = *(const float4*)(ob + c);
            const float4 w = *(const float4*)(norm + h * DV + c);
            float z[4];
            ld4(g + c, z);
#pragma unroll
            for (int i = 0; i < 4; ++i)
                z[i] = sigmoidf_(z[i]) * (SILU ? z[i] : 1.f);
            const float r[4] = {v.x * rs * w.x * z[0], v.y * rs * w.y * z[1],
                                v.z * rs * w.z * z[2], v.w * rs * w.w * z[3]};
            st4(dst + c, r);
        }
    }
    if (is_seg && lane == 0) mst[(long)sg.z * H + h] = m;
}

// The same for heads that are normed together and have no denominators
// (lightning attention): one block per token, out rows of stride out_ld. NV > 0:
// a row of up to NV * 1024 columns stays in registers.
template <class T, int NV>
__global__ void __launch_bounds__(256)
k_rec_row_out(T* __restrict__ out, const float* __restrict__ o,
              const T* __restrict__ gate, const float* __restrict__ norm,
              int H, int DV, int ld_, int out_ld, int true_cols, float eps) {
    __shared__ float red[4];
    constexpr int KEEP = NV ? NV : 1;
    const long n = blockIdx.x;
    const int cols = H * DV;
    const float* ob = o + n * H * (DV + 4);
    float v[KEEP][4], ss = 0.f;
    auto load = [&](int c, float* f) {
        ld4(ob + (c / DV) * (DV + 4) + c % DV, f);
    };
    auto add = [&](const float* f) {
        ss += f[0] * f[0] + f[1] * f[1] + f[2] * f[2] + f[3] * f[3];
    };
    if (NV) {
#pragma unroll
        for (int j = 0; j < KEEP; ++j) {
            const int c = (j * 256 + threadIdx.x) * 4;
            if (c < cols) {
                load(c, v[j]);
                add(v[j]);
            }
        }
    } else {
        for (int c = threadIdx.x * 4; c < cols; c += 1024) {
            load(c, v[0]);
            add(v[0]);
        }
    }
    const float rs = 1.f / sqrtf(block_sum(ss, red) / (float)true_cols + eps);
    auto put = [&](int c, float* f) {
        float z[4], w[4];
        ld4(gate + n * ld_ + c, z);
        ld4(norm + c, w);
#pragma unroll
        for (int i = 0; i < 4; ++i) f[i] *= rs * w[i] * sigmoidf_(z[i]);
        st4(out + n * out_ld + c, f);
    };
    if (NV) {
#pragma unroll
        for (int j = 0; j < KEEP; ++j) {
            const int c = (j * 256 + threadIdx.x) * 4;
            if (c < cols) put(c, v[j]);
        }
    } else {
        for (int c = threadIdx.x * 4; c < cols; c += 1024) {
            load(c, v[0]);
            put(c, v[0]);
        }
    }
}

// ---------------------------------------------------------------------------
// Prompt portions in chunks of 64 tokens. With F_t the running sum of f
// inside a chunk, a_s = i_s - F_s and M_t = max(m_in, max_{s<=t} a_s):
//   m_t = F_t + M_t
//   S_t = exp(m_in - M_t) S_in + sum_{s<=t} exp(a_s - M_t) v_s k_s^T
// so the state that enters each chunk (one chunk after the other, in registers)
// and the outputs (all chunks at once) separate, both on the matrix cores. Where a
// product takes f32 factors (state, weighted keys) they are split into two bf16
// parts.
//
// chunk (int4): {first token, length, segment, -}
// seg   (int4): {slot, start position, first chunk, chunks}
// dS: [chunks][H][DV + 1][DK], the entering states as (hi | lo << 16) bf16 pairs.
// scal: f32 [chunks][H][4] = {max a, F total, m of the slot before the step, -}.
// ---------------------------------------------------------------------------
#define MCH 64

// Lightning attention (CONST) is the case i = 0, f the same for every token: m
// then stays 0. It has no normaliser and no head norm; gr is f by head, f32
// [H]. Score weights are (hi, lo) pairs of bf16, too.

// running sum of f, a, running max of a; lane = token, wave-wide
template <bool CONST>
DEV_INLINE void chunk_scan(const float* gr, int tok0, int clen, int h, int H,
                           float cap, float& F, float& a, float& amax) {
    const int t = threadIdx.x & 63;
    float gi = -INFINITY, gf = 0.f;
    if (t < clen) {
        if (CONST) {
            gi = 0.f;
            gf = gr[h];
        } else {
            mlstm_gates(gr + (long)(tok0 + t) * 2 * H, h, H, cap, gi, gf);
        }
    }
    F = gf;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float u = __shfl_up(F, off, WAVE);
        if (t >= off) F += u;
    }
    a = gi - F;
    amax = a;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const float u = __shfl_up(amax, off, WAVE);
        if (t >= off) amax = fmaxf(amax, u);
    }
}

// Places in LDS of 16-byte pieces c, swapped by the row so that 16 lanes' rows
// do not meet in a bank: of 64 f32, of 64 bf16, and of `cols` bf16 that are read
// transposed, where 4 rows' pairs of pieces have to lie apart.
DEV_INLINE int at_f32(int row, int c) { return row * 64 + (c ^ (row & 15)) * 4; }
DEV_INLINE int at_bf16(int row, int c) { return row * 64 + (c ^ (row & 7)) * 8; }
DEV_INLINE int at_cols(int row, int c, int cols) {
    return row * cols + (c ^ ((row & 3) << 1 | (row >> 2 & 1))) * 8;
}

// The tokens' values, up to 256 columns of them, on their way to LDS
template <int TOKENS = 64>
DEV_INLINE void load_values(bf16_t* vs, const bf16_t* v, long ld_, int last,
                            int cols) {
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int i = 0; i < cols / 32 * TOKENS / 64; ++i) {
        const int pc = i * 256 + threadIdx.x, row = pc / (cols / 8);
        const int c = at_cols(row, pc % (cols / 8), cols) / 8 -
                      row * (cols / 8);
        load_lds16(v + min(row, last) * ld_ + c * 8,
                   vs + (i * 256 + wid * 64) * 8);
    }
}

// Values (16 columns from `col` on, as the products' rows) of 32 tokens.
DEV_INLINE bf16x8 value_piece(const bf16_t* vs, int ks, int col, int cols) {
    const int lane = threadIdx.x & 63, fr = lane & 15, gq = lane >> 4;
    const int d = col + (fr & 3) * 4;
    bf16x8 v;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const int row = ks * 32 + gq * 8 + (fr >> 2) + j * 4;
        const bf16x4 x =
            read_transposed(vs + at_cols(row, d >> 3, cols) + (d & 7));
#pragma unroll
        for (int i = 0; i < 4; ++i) v[j * 4 + i] = x[i];
    }
    return v;
}

// Of each chunk and head: the weights exp(a - max a) of its keys, f32 [64] at w, and
// of scal max a, F total and m of the slot before the step. A wave has a head.
template <bool CONST>
__global__ void __launch_bounds__(256)
k_mlstm_weights(float* __restrict__ w, float* __restrict__ scal,
                const float* __restrict__ mst, const float* __restrict__ gr,
                const int4* __restrict__ chunks, const int4* __restrict__ segs,
                int H, float cap) {
    const int4 ch = chunks[blockIdx.x];
    const int h = blockIdx.y * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (h >= H) return;
    float F, a, amax;
    chunk_scan<CONST>(gr, ch.x, ch.y, h, H, cap, F, a, amax);
    const float A = __shfl(amax, 63, WAVE);
    const long at = (long)blockIdx.x * H + h;
    w[at * 64 + lane] = lane < ch.y ? expf(a - A) : 0.f;
    if (lane == 63) {
        const int4 sg = segs[ch.z];
        scal[at * 4] = A;
        scal[at * 4 + 1] = F;
        scal[at * 4 + 2] = CONST || sg.y == 0 ? 0.f : mst[(long)sg.x * H + h];
    }
}

// The state that enters each chunk of a prompt portion, left in dS as (hi | lo << 16)
// bf16 pairs; the slot's state is advanced. Block = (segment, head, 32 key channels
// and NK * 64 value columns), and the state stays in registers from chunk to chunk: a
// wave has NK * 16 by 16. A chunk's operands are loaded two chunks ahead.
// Bound by a step's instructions and latencies (.8 us a chunk) where a segment is
// long, by the stores where there are many. 45 chunks of 4 segments, 12 heads of 128
// x 256: 58 us when the chunks' own contributions were written first, read and
// added up by a second kernel; now 35, with operands that the Infinity Cache has. In a
// step it has most of them, and they take 34; with all from memory, 51. (256 threads,
// each with twice the keys: 34, but 54 instead of 44 for one segment of 3500.) With what
// is ahead of it and the outputs, mLSTM's 55 chunks of one segment: 127 us before, now
// 105; of 4 heads, whose blocks are 64, 76 and 78.
// KIND: gated linear attention's decays by channel (b), or weights and sums of
// k_mlstm_weights, where the slot's m is advanced too; mLSTM's normaliser, the row
// behind the value columns, is the product of the keys with ones.
#define STATE_K 32
enum { STATE_GLA, STATE_MLSTM, STATE_CONST };
// a thread's token in a chunk: b and the last token's, or its weight, max a and F total
template <bool GLA> struct TokenWeights { f32x4 b, bT; };
template <> struct TokenWeights<false> { float w, A, F; };
template <int KIND, int NK>
__global__ void __launch_bounds__(512)
k_chunk_states(u32* __restrict__ dS, float* __restrict__ S,
               const float* __restrict__ scal, float* __restrict__ m_in,
               float* __restrict__ mst, const bf16_t* __restrict__ qkv,
               const float* __restrict__ b, const int4* __restrict__ chunks,
               const int4* __restrict__ segs, int nseg, int H, int DK, int DV,
               int ld_) {
    constexpr bool GLA = KIND == STATE_GLA, NORM = KIND == STATE_MLSTM;
    constexpr int VW = 64 * NK;
    __shared__ __attribute__((aligned(16))) bf16_t vs[64 * VW];
    __shared__ __attribute__((aligned(16))) bf16_t kh[64 * STATE_K];
    __shared__ __attribute__((aligned(16))) bf16_t kl[64 * STATE_K];
    __shared__ __attribute__((aligned(16))) float keep[STATE_K];
    // (the grid's x is a multiple of 8, so that an XCD has all of a head's blocks)
    if ((int)blockIdx.x >= nseg * H) return;
    const int h = blockIdx.x % H, nd = DK / STATE_K;
    const int d0 = (int)blockIdx.y % nd * STATE_K;
    const int v0 = (int)blockIdx.y / nd * VW;
    const int lane = threadIdx.x & 63, fr = lane & 15, gq = lane >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int kcol = NK == 1 ? wid >> 2 << 4 : 0;
    const int vcol = NK == 1 ? (wid & 3) << 4 : wid << 4;
    const int4 sg = segs[blockIdx.x / H];
    const int first = chunks[sg.z].x;
    const int4 end = chunks[sg.z + sg.w - 1];
    const int n = end.x + end.y - first;           // tokens
    const int t = threadIdx.x >> 3, c = threadIdx.x & 7;   // token, piece of its row
    const long C = (long)H * DK;
    const bf16_t* kp = qkv + (long)first * ld_ + C + h * DK + d0 + c * 4;
    const bf16_t* vp = qkv + (long)first * ld_ + 2 * C + h * DV + v0 + c * 8;
    const float* bp = GLA ? b + (long)first * C + h * DK + d0 + c * 4
                          : b + ((long)sg.z * H + h) * 64 + t;
    const float* const sp = scal + ((long)sg.z * H + h) * 4;
    float m = GLA ? 0.f : sp[2];
    const bool leads = blockIdx.y == 0 && threadIdx.x == 0;
    struct Piece { f32x2 k; f32x4 v[NK]; TokenWeights<GLA> w; } pieces[2];
    auto load = [&](Piece& p, int at) {
        const long row = min(at * 64 + t, n - 1);
        p.k = *(const f32x2*)(kp + row * ld_);
#pragma unroll
        for (int i = 0; i < NK; ++i)
            p.v[i] = *(const f32x4*)(vp + row * ld_ + i * 64);
        if constexpr (GLA) {
            p.w.b = *(const f32x4*)(bp + row * C);
            p.w.bT = *(const f32x4*)(bp + min(at * 64 + 63, n - 1) * C);
        } else {
            const long to = min(at, sg.w - 1);
            p.w.w = bp[to * H * 64];
            p.w.A = sp[to * H * 4];
            p.w.F = sp[to * H * 4 + 1];
        }
    };
    // (so that nothing of it is waited for earlier)
    auto wait = [](Piece& p) {
        asm volatile("" : "+v"(p.k), "+v"(p.v[0]), "+v"(p.v[NK - 1]));
        if constexpr (GLA)
            asm volatile("" : "+v"(p.w.b), "+v"(p.w.bT));
        else
            asm volatile("" : "+v"(p.w.w));
    };
    // places of 16-byte pieces among 32 columns, for reads as value_piece's
    auto at32 = [](int row, int c) {
        return row * STATE_K + (c ^ (row >> 2 & 2)) * 8;
    };
    auto key_piece = [&](const bf16_t* keys, int ks, int i0) {
        const int d = kcol + i0 * 16 + (fr & 3) * 4;
        bf16x8 v;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int row = ks * 32 + gq * 8 + (fr >> 2) + j * 4;
            const bf16x4 x =
                read_transposed(keys + at32(row, d >> 3) + (d & 7));
#pragma unroll
            for (int i = 0; i < 4; ++i) v[j * 4 + i] = x[i];
        }
        return v;
    };
    const long own = (long)(v0 + vcol + fr) * DK + d0 + kcol + gq * 4;
    const long size = (long)(NORM ? DV + 1 : DV) * DK;
    float* Sb = S + ((long)sg.x * H + h) * size + own;
    u32* Db = dS + ((long)sg.z * H + h) * size + own;
    f32x4 acc[NK];
#pragma unroll
    for (int d = 0; d < NK; ++d) {
        acc[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
        if (sg.y != 0) acc[d] = *(const f32x4*)(Sb + d * 16);
    }
    // The normaliser: the waves of the first 16 columns have it, lanes 0 of 16 store.
    const long below = (long)(DV - fr) * DK;
    const bool norms = NORM && v0 + vcol == 0;
    f32x4 den[NK];
    if (norms)
#pragma unroll
        for (int d = 0; d < NK; ++d) {
            den[d] = (f32x4){0.f, 0.f, 0.f, 0.f};
            if (sg.y != 0) den[d] = *(const f32x4*)(Sb + below + d * 16);
        }
    bf16x8 ones;
#pragma unroll
    for (int i = 0; i < 8; ++i) ones[i] = (__bf16)1.f;
    auto packed = [](f32x4 x) {
        uint4 pk;
        u32* pp = (u32*)&pk;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const bf16_t hi = f2bf(x[r]);
            pp[r] = (u32)hi | ((u32)f2bf(x[r] - bf2f(hi)) << 16);
        }
        return pk;
    };
    auto step = [&](Piece& p, int at) {
        lds_barrier();                             // the last chunk's are read
        wait(p);
        float f[4], stay = 0.f, w[4];
        const bool in = at * 64 + t < n;
        if constexpr (GLA) {
#pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = __expf(p.w.bT[i] - p.w.b[i]);
            if (t == 0)
#pragma unroll
                for (int i = 0; i < 4; ++i) keep[c * 4 + i] = __expf(p.w.bT[i]);
        } else {
            const float M = fmaxf(m, p.w.A);
            if (leads) m_in[(sg.z + at) * (long)H + h] = m;
            stay = expf(m - M);
            w[0] = w[1] = w[2] = w[3] = expf(p.w.A - M) * p.w.w;
            m = p.w.F + M;
        }
        ld4((const bf16_t*)&p.k, f);
        bf16x4 hi, lo;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float x = f[i] * (in ? w[i] : 0.f);
            hi[i] = (__bf16)x;
            lo[i] = (__bf16)(x - (float)hi[i]);
        }
        const int to = at32(t, c >> 1) + (c & 1) * 4;
        *(bf16x4*)(kh + to) = hi;
        *(bf16x4*)(kl + to) = lo;
#pragma unroll
        for (int i = 0; i < NK; ++i)
            *(f32x4*)(vs + at_cols(t, i * 8 + c, VW)) = p.v[i];
        lds_barrier();
        load(p, at + 2);
        bf16x8 v[2], k[2][NK][2];
        f32x4 kept[NK];
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            v[ks] = value_piece(vs, ks, vcol, VW);
#pragma unroll
            for (int d = 0; d < NK; ++d) {
                k[ks][d][0] = key_piece(kh, ks, d);
                k[ks][d][1] = key_piece(kl, ks, d);
            }
        }
#pragma unroll
        for (int d = 0; d < NK; ++d)
            kept[d] = GLA ? *(const f32x4*)(keep + kcol + d * 16 + gq * 4)
                          : (f32x4){stay, stay, stay, stay};
        __builtin_amdgcn_sched_barrier(0);         // all on their way
#pragma unroll
        for (int d = 0; d < NK; ++d) {
            *(uint4*)(Db + at * (H * size) + d * 16) = packed(acc[d]);
            acc[d] *= kept[d];
        }
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int d = 0; d < NK; ++d)
                    acc[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        k[ks][d][i], v[ks], acc[d], 0, 0, 0);
        if (!norms) return;
#pragma unroll
        for (int d = 0; d < NK; ++d) {
            if (fr == 0)
                *(uint4*)(Db + at * (H * size) + below + d * 16) =
                    packed(den[d]);
            den[d] *= kept[d];
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int i = 0; i < 2; ++i)
                    den[d] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        k[ks][d][i], ones, den[d], 0, 0, 0);
        }
    };
    load(pieces[0], 0);
    load(pieces[1], 1);
    wait(pieces[0]);               // (else each turn waits as the first one must)
    wait(pieces[1]);
    for (int at = 0;;) {
        step(pieces[0], at);
        if (++at >= sg.w) break;
        step(pieces[1], at);
        if (++at >= sg.w) break;
    }
#pragma unroll
    for (int d = 0; d < NK; ++d) {
        *(f32x4*)(Sb + d * 16) = acc[d];
        if (norms && fr == 0) *(f32x4*)(Sb + below + d * 16) = den[d];
    }
    if (NORM && leads) mst[(long)sg.x * H + h] = m;
}

// 8 (hi | lo << 16) pairs -> the two bf16 fragments
DEV_INLINE void split8(const u32* p, bf16x8& hi, bf16x8& lo) {
    const uint4 x = ((const uint4*)p)[0], y = ((const uint4*)p)[1];
    uint4 a, b;
    a.x = (x.x & 0xffffu) | (x.y << 16);  b.x = (x.x >> 16) | (x.y & 0xffff0000u);
    a.y = (x.z & 0xffffu) | (x.w << 16);  b.y = (x.z >> 16) | (x.w & 0xffff0000u);
    a.z = (y.x & 0xffffu) | (y.y << 16);  b.z = (y.x >> 16) | (y.y & 0xffff0000u);
    a.w = (y.z & 0xffffu) | (y.w << 16);  b.w = (y.z >> 16) | (y.w & 0xffff0000u);
    hi = *(bf16x8*)&a;
    lo = *(bf16x8*)&b;
}

// Output gates of a chunk, for lane = 4 columns c * 64 + wid * 16 + gq * 4 + r of
// tokens rt * 16 + fr: on their way ahead of the last products.
template <int RT>
DEV_INLINE void load_gates(uint2 (&z)[4][RT], const bf16_t* gate, long ld_,
                           int last, int DV) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c * 64 < DV)
                z[c][rt] = *(const uint2*)(
                    gate + min(rt * 16 + (lane & 15), last) * ld_ + c * 64 +
                    wid * 16 + (lane >> 4) * 4);
}

// A chunk's outputs, laid out as its gates, with all of the head's columns in the
// block: unit RMS, times norm, times the gate's sigmoid (SILU: and the gate).
// red: f32 [4][RT * 16] in LDS.
template <bool SILU, int RT>
DEV_INLINE void store_normed(bf16_t* out, const f32x4 (&acc)[4][RT],
                             float* red, const uint2 (&gates)[4][RT],
                             long out_ld, const float* norm, int len, int DV,
                             int dvtrue, float eps) {
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int fr = lane & 15, gq = lane >> 4, col0 = wid * 16 + gq * 4;
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        float ss = 0.f;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c * 64 < DV)
#pragma unroll
                for (int r = 0; r < 4; ++r) ss += acc[c][rt][r] * acc[c][rt][r];
        ss += __shfl_xor(ss, 16, WAVE);
        ss += __shfl_xor(ss, 32, WAVE);
        if (gq == 0) red[(wid * RT + rt) * 16 + fr] = ss;
    }
    float w[4][4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
        if (c * 64 < DV) ld4(norm + c * 64 + col0, w[c]);
    __syncthreads();
#pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int t = rt * 16 + fr;
        const float ss = red[t] + red[RT * 16 + t] + red[RT * 32 + t] +
                         red[RT * 48 + t];
        const float rs = 1.f / sqrtf(ss / (float)dvtrue + eps);
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c * 64 >= DV) continue;
            float z[4];
            ld4((const bf16_t*)&gates[c][rt], z);
#pragma unroll
            for (int r = 0; r < 4; ++r)
                z[r] = acc[c][rt][r] * rs * w[c][r] *
                       (sigmoidf_(z[r]) * (SILU ? z[r] : 1.f));
            if (t < len) st4(out + t * out_ld + c * 64 + col0, z);
        }
    }
}

// Block = (chunk, head, 256 value columns). Scores: a wave owns 16 tokens;
// outputs: every fourth 16 columns for all 64, so that the state is read once.
// Queries and keys come through LDS, 64 channels ahead of their use. With all of a
// head's columns here (out), the head's norm and gate follow at once; out and
// CONST exclude each other. Bound by its instructions, as k_gla_chunk_out: 3500
// tokens, 12 heads of 128 x 256: 92 us with tokens split over the waves and 128 columns
// a block, and 28 of the norm behind it, now 66 (some 8 of it the gates' exponentials,
// which are not the hardware's: those are off by 6e-8 |z|).
template <bool CONST>
__global__ void __launch_bounds__(256, 2)
k_mlstm_chunk_out(float* __restrict__ o, bf16_t* __restrict__ out,
                  const float* __restrict__ dS,
                  const float* __restrict__ ms,
                  const bf16_t* __restrict__ qkv,
                  const float* __restrict__ gr,
                  const int4* __restrict__ chunks,
                  const float* __restrict__ norm, int H, int DK, int DV,
                  int ld_, float qscale, float cap, int dvtrue, float eps) {
    __shared__ __attribute__((aligned(16))) bf16_t vs[64 * 256];
    __shared__ __attribute__((aligned(16))) bf16_t qk[2][2][64 * 64];
    __shared__ float sa[MCH], sM[MCH], sm[MCH], sin_[MCH], snq[MCH], sden[MCH];
    const int4 ch = chunks[blockIdx.x];
    const int h = blockIdx.y, v0 = blockIdx.z * 256, nv = min(256, DV - v0);
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, gq = lane >> 4, r0 = wid * 16, last = ch.y - 1;
    const u32* Sb = (const u32*)dS +
                    ((long)blockIdx.x * H + h) * (CONST ? DV : DV + 1) * DK;
    const u32* nb = Sb + (long)DV * DK + gq * 8;       // the normaliser's row
    Sb += (long)(v0 + r0 + fr) * DK + gq * 8;
    const bf16_t* qh = qkv + (long)ch.x * ld_ + h * DK;

    auto issue = [&](int buf, int k0) {    // queries and keys of 64 channels
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const int pc = i * 256 + threadIdx.x, row = pc >> 3;
            const bf16_t* src = qh + (long)min(row, last) * ld_ + k0 +
                                ((pc & 7) ^ (row & 7)) * 8;
            load_lds16(src, qk[buf][0] + (i * 256 + wid * 64) * 8);
            load_lds16(src + (long)H * DK,
                       qk[buf][1] + (i * 256 + wid * 64) * 8);
        }
    };
    uint4 st[2][4][2];
    auto load_state = [&](int k0, int ks, int c) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            st[ks][c][i] = *(const uint4*)(Sb + (long)c * 64 * DK + k0 +
                                           ks * 32 + i * 4);
    };
    uint4 nw[2][2];
    auto load_norm = [&](int k0) {
        if (CONST) return;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i)
                nw[ks][i] = *(const uint4*)(nb + k0 + ks * 32 + i * 4);
    };
    issue(0, 0);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c * 64 < nv) load_state(0, ks, c);
    load_norm(0);
    load_values(vs, qkv + (long)ch.x * ld_ + 2l * H * DK + h * DV + v0, ld_,
                last, nv);
    if (wid == 0) {
        float F, a, amax;
        chunk_scan<CONST>(gr, ch.x, ch.y, h, H, cap, F, a, amax);
        const float m_in = ms[(long)blockIdx.x * H + h];
        const float M = fmaxf(m_in, amax);
        sa[lane] = a;
        sM[lane] = M;
        sm[lane] = F + M;
        sin_[lane] = expf(m_in - M);
    }

    // ---- scores of this wave's tokens against the chunk's keys, n . q, and
    // what the entering state gives
    f32x4 sc[4], acc[4][4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        sc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[j][c] = sc[j];
    }
    float nq = 0.f;
    int buf = 0;
    for (int k0 = 0; k0 < DK; k0 += 64, buf ^= 1) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();                 // they are there, the others are free
        const bool more = k0 + 64 < DK;
        if (more) issue(buf ^ 1, k0 + 64);
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            const int c8 = ks * 4 + gq;
            bf16x8 q[4];
#pragma unroll
            for (int rt = 0; rt < 4; ++rt)
                q[rt] = *(const bf16x8*)(
                    qk[buf][0] + at_bf16(rt * 16 + fr, c8));
            const bf16x8 own =
                *(const bf16x8*)(qk[buf][0] + at_bf16(r0 + fr, c8));
#pragma unroll
            for (int j = 0; j < 4; ++j)
                if (j <= wid)
                    sc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        own,
                        *(const bf16x8*)(qk[buf][1] +
                                         at_bf16(j * 16 + fr, c8)),
                        sc[j], 0, 0, 0);
            if (!CONST) {
                float qf[8];
                unpack8(*(const uint4*)&own, qf);
                const u32* np = (const u32*)nw[ks];
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    nq += qf[i] * (__uint_as_float(np[i] << 16) +
                                   __uint_as_float(np[i] & 0xffff0000u));
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (c * 64 >= nv) continue;
                bf16x8 sh, sl;
                split8((const u32*)st[ks][c], sh, sl);
                if (more) load_state(k0 + 64, ks, c);
#pragma unroll
                for (int rt = 0; rt < 4; ++rt) {
                    acc[c][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        sh, q[rt], acc[c][rt], 0, 0, 0);
                    acc[c][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        sl, q[rt], acc[c][rt], 0, 0, 0);
                }
            }
        }
        if (more) load_norm(k0 + 64);
    }
    uint2 gates[4][4];
    if (out)
        load_gates(gates, qkv + (long)ch.x * ld_ + 2l * H * DK + (long)H * DV +
                              h * DV, ld_, last, DV);
    if (!CONST) {
        nq += __shfl_xor(nq, 16, WAVE);
        nq += __shfl_xor(nq, 32, WAVE);
        if (lane < 16) snq[r0 + lane] = nq;
    }
    lds_barrier();                     // queries and keys have been read
    bf16_t* const ps = qk[0][0];
    bf16_t* const pl = qk[0][1];
    float den[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if (j > (wid | 1)) continue;
        const int key = j * 16 + fr;
        const float ak = sa[key];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = r0 + gq * 4 + r;
            const float p = (key <= row && key < ch.y)
                ? sc[j][r] * qscale * expf(ak - sM[row]) : 0.f;
            den[r] += p;
            const int at = at_bf16(row, key >> 3) + (key & 7);
            ps[at] = f2bf(p);
            if (CONST) pl[at] = f2bf(p - bf2f(f2bf(p)));
        }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
#pragma unroll
        for (int off = 8; off > 0; off >>= 1)
            den[r] += __shfl_xor(den[r], off, WAVE);
        if (fr == 0) sden[r0 + gq * 4 + r] = den[r];
    }
    lds_barrier();
    float inv[4];
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
        const int t = rt * 16 + fr;
        const float in = sin_[t] * qscale;
        inv[rt] = 1.f;
        if (!CONST) {
            const float d = sden[t] + in * snq[t];
            inv[rt] = 1.f / (fmaxf(fabsf(d), expf(-sm[t])) + 1e-6f);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[c][rt][r] *= in;
    }
    // ---- the chunk's own values
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
        bf16x8 hi[4], lo[4];
#pragma unroll
        for (int rt = ks * 2; rt < 4; ++rt) {
            const int at = at_bf16(rt * 16 + fr, ks * 4 + gq);
            hi[rt] = *(const bf16x8*)(ps + at);
            if (CONST) lo[rt] = *(const bf16x8*)(pl + at);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (c * 64 >= nv) continue;
            const bf16x8 v = value_piece(vs, ks, c * 64 + r0, nv);
#pragma unroll
            for (int rt = ks * 2; rt < 4; ++rt) {
                acc[c][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    v, hi[rt], acc[c][rt], 0, 0, 0);
                if (CONST)
                    acc[c][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        v, lo[rt], acc[c][rt], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[c][rt][r] *= inv[rt];
    if (out) {
        store_normed<false>(
            out + ((long)ch.x * H + h) * DV, acc, (float*)qk[1][0], gates,
            (long)H * DV, norm + h * DV, ch.y, DV, dvtrue, eps);
        return;
    }
#pragma unroll
    for (int rt = 0; rt < 4; ++rt) {
        const int t = rt * 16 + fr;
        if (t > last) continue;
        float* ob = o + ((long)(ch.x + t) * H + h) * (DV + 4) + v0 + r0 +
                    gq * 4;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c * 64 < nv) *(f32x4*)(ob + c * 64) = acc[c][rt];
    }
}

// ===========================================================================
// Gated linear attention: S_t = diag(a_t) S_{t-1} + k_t v_t^T, o_t = S_t^T q_t
// with a_t = sigmoid(z_t)^(1 / tau) per key channel, q scaled by dim^-1/2.
// b holds the running sum of log a inside a chunk, f32 [n][H*DK] (a decode row
// is a chunk of its own). State and projection rows are laid out as mLSTM's,
// without the normaliser row.
// ===========================================================================

// log a of 16 tokens for 16 NT channels: z = W2 u + bias with w = W2^T, f32 [R][C],
// by the matrix cores' f32 products. A lane has 4 tokens, (lane / 16) * 4 on, of
// channels c0 + n * 16 + lane % 16.
template <int NT>
DEV_INLINE void log_decays(f32x4 (&z)[NT], const float* u, const float* w,
                           const float* bias, int last, int c0, int R, int C,
                           float inv_tau) {
    const int fr = threadIdx.x & 15, gq = (threadIdx.x & 63) >> 4;
    const float* ur = u + (long)min(fr, last) * R;
    int c[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
        c[n] = min(c0 + n * 16 + fr, C - 1);
        const float b0 = bias[c[n]];
        z[n] = (f32x4){b0, b0, b0, b0};
    }
    for (int rb = 0; rb < R; rb += 16) {
        float a[4], v[4][NT];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int k = rb + j * 4 + gq;
            a[j] = k < R ? ur[k] : 0.f;
#pragma unroll
            for (int n = 0; n < NT; ++n)
                v[j][n] = k < R ? w[(long)k * C + c[n]] : 0.f;
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int n = 0; n < NT; ++n)
                z[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[j], v[j][n], z[n],
                                                            0, 0, 0);
    }
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) z[n][r] = log_sigmoid(z[n][r]) * inv_tau;
}

// b for 64 channels, of 16 of the first nd tokens, chunks of their own (a wave has
// 16 channels), or of one chunk ({first token, length, ..}; a wave has 16 tokens,
// whose sums meet in LDS). Bound by the logarithms: 2730 tokens, 1536 channels, rank
// 16: 34 us with log1pf and u in scalar registers, which are too few for 16 tokens
// (25 without log1pf), now 13.7.
__global__ void __launch_bounds__(256)
k_gla_decay(float* __restrict__ b, const float* __restrict__ u,
            const float* __restrict__ w, const float* __restrict__ bias,
            const int4* __restrict__ chunks, int nd, int R, int C,
            float inv_tau) {
    __shared__ float sums[4][64];
    const int it = blockIdx.x, singles = (nd + 15) / 16;
    const int fr = threadIdx.x & 15, gq = (threadIdx.x & 63) >> 4;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c0 = blockIdx.y * 64;
    if (it < singles) {
        const int left = nd - it * 16, c = c0 + wid * 16 + fr;
        f32x4 z[1];
        log_decays(z, u + (long)it * 16 * R, w, bias, left - 1, c0 + wid * 16,
                   R, C, inv_tau);
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (c < C && gq * 4 + r < left)
                b[(it * 16l + gq * 4 + r) * C + c] = z[0][r];
        return;
    }
    const int4 ch = chunks[it - singles];
    const int t0 = min(wid * 16, ch.y - 1);
    f32x4 z[4];
    log_decays(z, u + (long)(ch.x + t0) * R, w, bias, ch.y - 1 - t0, c0, R, C,
               inv_tau);
    float ahead[4];                    // of the wave's tokens before the lane's
#pragma unroll
    for (int n = 0; n < 4; ++n) {
#pragma unroll
        for (int r = 1; r < 4; ++r) z[n][r] += z[n][r - 1];
        float sum = z[n][3];
        float up = __shfl_up(sum, 16, WAVE);
        if (gq >= 1) sum += up;
        up = __shfl_up(sum, 32, WAVE);
        if (gq >= 2) sum += up;
        up = __shfl_up(sum, 16, WAVE);
        ahead[n] = gq ? up : 0.f;
        if (gq == 3) sums[wid][n * 16 + fr] = sum;
    }
    __syncthreads();
#pragma unroll
    for (int n = 0; n < 4; ++n) {
        const int c = c0 + n * 16 + fr;
        for (int v = 0; v < wid; ++v) ahead[n] += sums[v][n * 16 + fr];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int t = wid * 16 + gq * 4 + r;
            if (c < C && t < ch.y)
                b[(long)(ch.x + t) * C + c] = z[n][r] + ahead[n];
        }
    }
}

// Prompt portions in chunks of 64 tokens, as mLSTM's: with b_t the sum of log
// decays up to token t and T the last token,
//   S_t = diag(exp(b_t)) S_in + sum_{s<=t} diag(exp(b_t - b_s)) k_s v_s^T
// Decays enter products as differences that are never positive where the span
// is unbounded, and as (hi, lo) pairs of bf16.
DEV_INLINE void split_bf16(float x, bf16_t& hi, bf16_t& lo) {
    hi = f2bf(x);
    lo = f2bf(x - bf2f(hi));
}

// 8 values f[i] exp(e[i]) as the (hi, lo) pair of bf16 fragments
DEV_INLINE void decayed8(const bf16_t* p, const float* e, bf16x8& hi,
                         bf16x8& lo) {
    float f[8];
    ld8(p, f);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float x = f[i] * __expf(e[i]);
        hi[i] = (__bf16)x;
        lo[i] = (__bf16)(x - (float)hi[i]);
    }
}

// hi . hi + hi . lo + lo . hi
DEV_INLINE f32x4 mfma_split(bf16x8 ah, bf16x8 al, bf16x8 bh, bf16x8 bl,
                            f32x4 c) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh, c, 0, 0, 0);
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl, c, 0, 0, 0);
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh, c, 0, 0, 0);
}

// Block = (chunk, head, 256 value columns, half): 32 of the chunk's tokens, against
// its keys up to them (HALF 1: the later ones and all 64 keys). Scores: a wave has 16
// tokens and every other 32 channels; two waves' sums meet in LDS. They refer to b at
// the end of the 16 tokens before: queries then decay by exp(b_t - ref) and older keys
// by exp(ref - b_s), both at most 1. Keys of the same 16 tokens grow by exp(ref - b_s)
// instead, unless a channel loses so much in 16 tokens that this could overflow; then
// these scores are taken pair by pair. Outputs: a wave owns every fourth 16 columns for
// all 32 tokens; decayed queries and scores meet in LDS. With all of a head's columns
// here (out), the head's norm and gate follow at once.
// Bound by waiting (53 % of a wave's time) and its instructions (35 % of a SIMD's). With
// all 64 tokens in a block, two a CU, a wave having one to four tiles of keys: 540 of
// them, 12 heads of 128 x 256, took three turns of 17 us, 59 in all. 1080 of 32 tokens,
// three a CU, their waves with 3 or 4 tiles (1 or 2): 49, and with the two of a chunk on
// one XCD 48. Four a CU with 112 bytes spilled: 56; the state loaded earlier, into
// registers that spill: 53.
#define GLA_SPAN 60.f
template <int HALF, bool FULL>
DEV_INLINE void gla_out(float* lds, float* o, bf16_t* out,
                        const float* dS, const bf16_t* qkv, const float* b,
                        const int4 ch, const float* norm, int at, int v0, int H, int DK,
                        int DV, int ld_, float qscale, int dvtrue, float eps) {
    constexpr int T0 = HALF * 32, KT = 2 + HALF * 2;   // first token, tiles of keys
    // keys, queries and decayed queries, then values
    bf16_t* const vs = (bf16_t*)lds;
    float* const bs = lds + 24 * 256;
    bf16_t* const ks_ = vs;
    bf16_t* const qr = vs + 64 * 64;
    bf16_t* const qs[2] = {vs + 96 * 64, vs + 128 * 64};
    const int h = blockIdx.y, nv = FULL ? 256 : min(256, DV - v0);
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, gq = lane >> 4;
    const int rt0 = wid & 1, half = wid >> 1, r0 = T0 + rt0 * 16;
    const long C = (long)H * DK;
    const int last = ch.y - 1;
    const float* bh = b + (long)ch.x * C + h * DK;     // row t at t * C
    const bf16_t* qh = qkv + (long)ch.x * ld_ + h * DK;
    const bf16_t* kh = qh + C;
    const float* ref = r0 ? bh + min(r0 - 1, last) * C : nullptr;
    const LdsSource states =
        lds_source(dS + ((long)at * H + h) * DV * DK, (u32)DV * DK * 4);
    const u32 state_at = (u32)(v0 + wid * 16 + fr) * DK * 4 + gq * 32;

    // b, queries and keys of 64 channels; behind the last ones nothing is read
    const u32 bbytes = (u32)(last * C + DK) * 4;
    const u32 qbytes = (u32)(last * (long)ld_ + C + DK) * 2;
    const LdsSource bsrc = lds_source(bh, bbytes), qsrc = lds_source(qh, qbytes);
    u32 bat[KT], qat, kat[KT / 2];
#pragma unroll
    for (int i = 0; i < KT; ++i) {
        const int pc = i * 256 + threadIdx.x, row = pc >> 4;
        bat[i] = (u32)(min(row, last) * C) * 4 + ((pc & 15) ^ (row & 15)) * 16;
    }
    {
        const int row = threadIdx.x >> 3, c = ((threadIdx.x & 7) ^ (row & 7)) * 16;
        qat = (u32)min(T0 + row, last) * ld_ * 2 + c;
#pragma unroll
        for (int i = 0; i < KT / 2; ++i)
            kat[i] = (u32)min(i * 32 + row, last) * ld_ * 2 + c;
    }
    auto issue = [&](int k0) {
        const bool any = k0 < DK;
        const u32 at = any ? k0 * 4 : bbytes, qa = any ? k0 * 2 : qbytes;
#pragma unroll
        for (int i = 0; i < KT; ++i)
            load_lds16(bsrc, bat[i], at, (bf16_t*)(bs + (i * 256 + wid * 64) * 4));
        load_lds16(qsrc, qat, qa, qr + wid * 64 * 8);
#pragma unroll
        for (int i = 0; i < KT / 2; ++i)
            load_lds16(qsrc, kat[i], qa + (u32)C * 2, ks_ + (i * 256 + wid * 64) * 8);
    };
    u32x4 st[4][2];
    auto load_state = [&](int k0, int ks, int c) {
#pragma unroll
        for (int i = 0; i < 2; ++i)
            st[c][i] = load16(states, state_at,
                                  (c * 64 * DK + k0 + ks * 32 + i * 4) * 4);
    };
    // ---- does a channel lose too much within these 16 tokens?
    float span = 0.f;
    for (int c = lane; c < DK; c += 64)
        span = fmaxf(span, (ref ? ref[c] : 0.f) -
                               bh[min(r0 + 15, last) * C + c]);
    issue(0);
    const bool pairwise = wave_reduce_max(span) > GLA_SPAN;

    // scores, and what the entering state gives
    const int own = T0 / 16 + rt0, jmax = pairwise ? own - 1 : own;
    f32x4 sc[KT], acc[4][2];
#pragma unroll
    for (int j = 0; j < KT; ++j) sc[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) acc[c][rt] = (f32x4){0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < DK; k0 += 64) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        {                                          // queries for the state
            const int t = threadIdx.x >> 3, c = threadIdx.x & 7;
            float e[8];
            ld4(bs + at_f32(T0 + t, c * 2), e);
            ld4(bs + at_f32(T0 + t, c * 2 + 1), e + 4);
            bf16x8 hi, lo;
            decayed8(qr + at_bf16(t, c), e, hi, lo);
            *(bf16x8*)(qs[0] + at_bf16(t, c)) = hi;
            *(bf16x8*)(qs[1] + at_bf16(t, c)) = lo;
        }
        {
            const int c = half * 4 + gq;
            // (rows behind the last hold its b; places in tiles of 16 rows)
            const int b0 = at_f32(fr, c * 2), b1 = at_f32(fr, c * 2 + 1);
            float rf[8], e[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) rf[i] = 0.f;
            if (r0) {
                ld4(bs + at_f32(r0 - 1, c * 2), rf);
                ld4(bs + at_f32(r0 - 1, c * 2 + 1), rf + 4);
            }
            ld4(bs + r0 * 64 + b0, e);
            ld4(bs + r0 * 64 + b1, e + 4);
#pragma unroll
            for (int i = 0; i < 8; ++i) e[i] -= rf[i];
            bf16x8 ah, al;
            decayed8(qr + rt0 * 1024 + at_bf16(fr, c), e, ah, al);
#pragma unroll
            for (int j = 0; j < KT; ++j) {
                if (j > jmax) continue;
                ld4(bs + j * 1024 + b0, e);
                ld4(bs + j * 1024 + b1, e + 4);
#pragma unroll
                for (int i = 0; i < 8; ++i) e[i] = rf[i] - e[i];
                bf16x8 th, tl;
                decayed8(ks_ + j * 1024 + at_bf16(fr, c), e, th, tl);
                sc[j] = mfma_split(ah, al, th, tl, sc[j]);
            }
        }
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (FULL || c * 64 < nv) load_state(k0, 0, c);
        lds_barrier();
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 hi[2], lo[2];
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                const int at = at_bf16(rt * 16 + fr, ks * 4 + gq);
                hi[rt] = *(const bf16x8*)(qs[0] + at);
                lo[rt] = *(const bf16x8*)(qs[1] + at);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (!FULL && c * 64 >= nv) continue;
                bf16x8 sh, sl;
                split8((const u32*)st[c], sh, sl);
                if (ks == 0) load_state(k0, 1, c);
#pragma unroll
                for (int rt = 0; rt < 2; ++rt)
                    acc[c][rt] = mfma_split(sh, sl, hi[rt], lo[rt],
                                            acc[c][rt]);
            }
            if (ks == 0) issue(k0 + 64);
        }
    }
    WAIT_LOADS(0);                     // (zeros, of the last turn)
    if (pairwise && half == 0) {
        const int s = min(r0 + fr, last);
        const bf16_t* kr = kh + (long)s * ld_;
        const float* bk = bh + s * C;
        f32x4 d = {0.f, 0.f, 0.f, 0.f};
        for (int c = 0; c < DK; c += 4) {
            float kf[4], e[4];
            ld4(kr + c, kf);
            ld4(bk + c, e);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int t = min(r0 + gq * 4 + r, last);
                float qf[4], f[4];
                ld4(qh + (long)t * ld_ + c, qf);
                ld4(bh + t * C + c, f);
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    d[r] += qf[i] * kf[i] * __expf(fminf(f[i] - e[i], 0.f));
            }
        }
#pragma unroll
        for (int j = 0; j < KT; ++j)
            if (j == own) sc[j] = d;
    }
    uint2 gates[4][2];
    if (out)
        load_gates(gates, qkv + (long)(ch.x + T0) * ld_ + 2 * C + (long)H * DV +
                              h * DV, ld_, last - T0, DV);
    lds_barrier();                     // keys, queries and b have been read
    load_values<KT * 16>(vs, qkv + (long)ch.x * ld_ + 2 * C + h * DV + v0, ld_,
                         last, nv);
    f32x4* const meet = (f32x4*)(lds + 32 * 256) + rt0 * 256 + lane;
    bf16_t* const ph = vs + 256 * 64;
    bf16_t* const pl = ph + 32 * 64;
#pragma unroll
    for (int j = 0; j < KT; ++j)       // the other one's tiles
        if ((j & 1) != half) meet[j * 64] = sc[j];
    lds_barrier();
#pragma unroll
    for (int j = 0; j < KT; ++j)
        if ((j & 1) == half) sc[j] += meet[j * 64];
    lds_barrier();
#pragma unroll
    for (int j = 0; j < KT; ++j) {
        if ((j & 1) != half) continue;
        const int key = j * 16 + fr;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = rt0 * 16 + gq * 4 + r;
            const float p =
                key <= T0 + row && key <= last ? sc[j][r] * qscale : 0.f;
            const int at = at_bf16(row, key >> 3) + (key & 7);
            split_bf16(p, ph[at], pl[at]);
        }
    }
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
        for (int rt = 0; rt < 2; ++rt)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[c][rt][r] *= qscale;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    lds_barrier();
    // the chunk's own values
#pragma unroll
    for (int ks = 0; ks < KT / 2; ++ks) {
        bf16x8 hi[2], lo[2];
#pragma unroll
        for (int rt = 0; rt < 2; ++rt) {
            const int at = at_bf16(rt * 16 + fr, ks * 4 + gq);
            hi[rt] = *(const bf16x8*)(ph + at);
            lo[rt] = *(const bf16x8*)(pl + at);
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) {
            if (!FULL && c * 64 >= nv) continue;
            const bf16x8 v = value_piece(vs, ks, c * 64 + wid * 16, nv);
#pragma unroll
            for (int rt = 0; rt < 2; ++rt) {
                acc[c][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    v, hi[rt], acc[c][rt], 0, 0, 0);
                acc[c][rt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                    v, lo[rt], acc[c][rt], 0, 0, 0);
            }
        }
    }
    if (out) {
        lds_barrier();                 // values have been read
        store_normed<true>(
            out + ((long)(ch.x + T0) * H + h) * DV, acc, lds, gates,
            (long)H * DV, norm + h * DV, ch.y - T0, DV, dvtrue, eps);
        return;
    }
#pragma unroll
    for (int rt = 0; rt < 2; ++rt) {
        const int t = T0 + rt * 16 + fr;
        if (t > last) continue;
        float* ob = o + ((long)(ch.x + t) * H + h) * (DV + 4) + v0 + wid * 16 +
                    gq * 4;
#pragma unroll
        for (int c = 0; c < 4; ++c)
            if (c * 64 < nv)
                *(f32x4*)(ob + c * 64) = acc[c][rt];
    }
}

__global__ void __launch_bounds__(256, 3)
k_gla_chunk_out(float* __restrict__ o, bf16_t* __restrict__ out,
                const float* __restrict__ dS, const bf16_t* __restrict__ qkv,
                const float* __restrict__ b, const int4* __restrict__ chunks,
                const float* __restrict__ norm, int nchunks, int H, int DK, int DV,
                int ld_, float qscale, int dvtrue, float eps) {
    __shared__ __attribute__((aligned(16))) float lds[40 * 256];
    // (the two halves 8 blocks apart: on one XCD, whose L2 has the state)
    const int x = blockIdx.x, at = (x >> 4) * 8 + (x & 7);
    if (at >= nchunks) return;
    const int4 ch = chunks[at];
    const bool late = !(x & 8);
    const int v0 = blockIdx.z * 256;
#define GO(...) gla_out<__VA_ARGS__>(lds, o, out, dS, qkv, b, ch, norm, at, v0, H, DK, \
                                     DV, ld_, qscale, dvtrue, eps)
    if (late && ch.y <= 32) return;
    if (DV - v0 >= 256) { if (late) GO(1, true); else GO(0, true); }
    else { if (late) GO(1, false); else GO(0, false); }
#undef GO
}

// ===========================================================================
// Routed experts.
//   route:   top experts of every token by f32 logits (ties: lower index),
//            their weights, by softmax or (plain) sigmoids; counts per expert
//            and each pair's rank. The choice may add a correction per expert
//            to the softmax scores and be confined to the best of equal groups;
//            router outputs beyond the experts are identities, whose weights
//            are summed up apart
//   scatter: pairs (token * top + k) sorted by expert, and the tile list
//            {expert, first sorted row, rows, -}; entry max_tiles holds the
//            number of tiles
//   gemm:    rows of one expert against its weights, once for the up
//            projection (gathers token rows, times the pairs' weights if these
//            go with the input; squared ReLU or a gated unit) and once for the
//            down projection (writes each pair's row back in pair order)
// The (weighted) sum over a token's pairs is taken in k_post_norm, k_sum_norm
// or k_streams_join.
// ===========================================================================
//
// Pairs in the order of their experts, and the list of tiles: by block `part` of
// those of THREADS that share the pairs, from the counts of E experts that have
// weights.
template <int THREADS, int MAX>
DEV_INLINE void moe_order(int part, int* sorted, int4* tiles, const int* idx,
                          const int* rank, const int* counts, int pairs, int E,
                          int bm, int max_tiles) {
    __shared__ int off[MAX + 1], toff[MAX + 1];
    for (int e = threadIdx.x; e < E; e += THREADS) off[e + 1] = counts[e];
    if (threadIdx.x == 0) off[0] = toff[0] = 0;
    __syncthreads();
    if (threadIdx.x < 64) {            // one wave scans, 64 experts a turn
        int base = 0, tbase = 0;
        for (int e0 = 0; e0 < E; e0 += 64) {
            const int e = e0 + threadIdx.x;
            int c = e < E ? off[e + 1] : 0;
            int t = (c + bm - 1) / bm;
#pragma unroll
            for (int s = 1; s < 64; s <<= 1) {
                const int a = __shfl_up(c, s, WAVE);
                const int b = __shfl_up(t, s, WAVE);
                if ((int)threadIdx.x >= s) { c += a; t += b; }
            }
            if (e < E) { off[e + 1] = base + c; toff[e + 1] = tbase + t; }
            base += __shfl(c, 63, WAVE);
            tbase += __shfl(t, 63, WAVE);
        }
    }
    __syncthreads();
    const int i = part * THREADS + threadIdx.x;
    if (i < pairs && idx[i] < E) {
        const int at = off[idx[i]] + rank[i];
        if (at >= 0 && at < pairs) sorted[at] = i;
    }
    if (part == 0) {
        for (int e = threadIdx.x; e < E; e += THREADS) {
            const int n = off[e + 1] - off[e];
            for (int t = 0; t * bm < n; ++t)
                if (toff[e] + t < max_tiles)
                    tiles[toff[e] + t] = make_int4(e, off[e] + t * bm,
                                                   min(bm, n - t * bm), 0);
        }
        if (threadIdx.x == 0)
            tiles[max_tiles] = make_int4(min(toff[E], max_tiles), 0, 0, 0);
    }
}

// A wave routes `tpw` tokens, one expert per lane and VPL experts deep. The
// place of an expert among a token's logits is the number of larger ones, so
// the chosen fall out of one pass over the lanes. Counts are gathered per
// block in LDS and added up once per block and expert.
// ALONE: one block of 16 waves has all tokens, and orders the pairs too, so that
// few rows, which launches bound, need no zeros and no second kernel (1 row of 64
// experts, 8 of them chosen, with the products 34.4 -> 31.5 us).
template <int VPL, bool ALONE>
__global__ void __launch_bounds__(ALONE ? 1024 : 256)
k_moe_route(int* __restrict__ idx, float* __restrict__ wt,
            int* __restrict__ rank, int* __restrict__ counts,
            const float* __restrict__ z, int ldz,
            const float* __restrict__ corr, float* __restrict__ ident, int N,
            int E, int experts, int top, int groups, int keep, float eps,
            float scale, int sigmoid, int tpw, int* __restrict__ sorted,
            int4* __restrict__ tiles, int bm, int max_tiles) {
    constexpr int WAVES = ALONE ? 16 : 4, THREADS = WAVES * 64;
    __shared__ int cnt[VPL * 64], base[VPL * 64];
    __shared__ float cs[WAVES][VPL * 64], gm[WAVES][VPL * 64];
    for (int e = threadIdx.x; e < VPL * 64; e += THREADS) cnt[e] = 0;
    __syncthreads();
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int n0 = (blockIdx.x * WAVES + wid) * tpw;
    for (int n = n0; n < min(N, n0 + tpw); ++n) {
        float v[VPL], s[VPL];          // choice score, score
        int place[VPL];
        float mx = -INFINITY;
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            const int e = i * 64 + lane;
            v[i] = e < E ? z[(long)n * ldz + e] : -INFINITY;
            if (v[i] != v[i]) v[i] = -INFINITY;   // keeps the choice in range
            place[i] = 0;
            mx = fmaxf(mx, v[i]);
        }
        mx = wave_reduce_max(mx);
        float total = 0.f;
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            s[i] = i * 64 + lane >= E ? 0.f
                   : sigmoid ? sigmoidf_(v[i]) : expf(v[i] - mx);
            total += s[i];
        }
        total = sigmoid ? 1.f : wave_reduce_sum(total);
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            const int e = i * 64 + lane;
            s[i] /= total;
            if (corr && e < E) {
                v[i] = s[i] + corr[e];
                if (v[i] != v[i]) v[i] = -INFINITY;
            }
        }
        if (groups > 1) {
            // a group's score is its largest; the others' experts drop out
            const int gs = E / groups;
            asm volatile("" ::: "memory");
#pragma unroll
            for (int i = 0; i < VPL; ++i) cs[wid][i * 64 + lane] = v[i];
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own wave's
            for (int g = lane; g < groups; g += 64) {
                float a = -INFINITY;
#pragma unroll 4
                for (int j = 0; j < gs; ++j) a = fmaxf(a, cs[wid][g * gs + j]);
                gm[wid][g] = a;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
            for (int i = 0; i < VPL; ++i) {
                const int e = i * 64 + lane;
                if (e >= E) continue;
                const int own = e / gs;
                const float a = gm[wid][own];
                int ahead = 0;
#pragma unroll 4
                for (int g = 0; g < groups; ++g) {
                    const float b = gm[wid][g];
                    ahead += b > a || (b == a && g < own);
                }
                if (ahead >= keep) v[i] = -INFINITY;
            }
        }
#pragma unroll
        for (int j = 0; j < VPL; ++j) {
            const int last = min(64, E - j * 64);
#pragma unroll 8
            for (int l = 0; l < last; ++l) {
                const float o = __uint_as_float(
                    __builtin_amdgcn_readlane(__float_as_uint(v[j]), l));
#pragma unroll
                for (int i = 0; i < VPL; ++i)
                    place[i] += i > j ? o >= v[i] : i < j ? o > v[i]
                        : o > v[i] || (o == v[i] && l < lane);
            }
        }
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < VPL; ++i)
            sum += place[i] < top && i * 64 + lane < E ? s[i] : 0.f;
        sum = wave_reduce_sum(sum);
        float same = 0.f;
#pragma unroll
        for (int i = 0; i < VPL; ++i) {
            const int e = i * 64 + lane;
            if (place[i] >= top || e >= E) continue;
            const long at = (long)n * top + place[i];
            const float w = sigmoid ? s[i] : s[i] / (sum + eps) * scale;
            idx[at] = e;
            wt[at] = e < experts ? w : 0.f;
            if (e >= experts) same += w;
            rank[at] = atomicAdd(cnt + e, 1);       // within the block
        }
        if (ident) {
            same = wave_reduce_sum(same);
            if (lane == 0) ident[n] = same;
        }
    }
    __syncthreads();
    if constexpr (ALONE) {
        moe_order<THREADS, VPL * 64>(0, sorted, tiles, idx, rank, cnt, N * top,
                                     experts, bm, max_tiles);
        return;
    }
    for (int e = threadIdx.x; e < E; e += 256)
        base[e] = cnt[e] ? atomicAdd(counts + e, cnt[e]) : 0;
    __syncthreads();
    const long p0 = (long)blockIdx.x * 4 * tpw * top;
    const long p1 = min((long)N * top, p0 + 4L * tpw * top);
    for (long at = p0 + threadIdx.x; at < p1; at += 256)
        rank[at] += base[idx[at]];
}

__global__ void __launch_bounds__(256)
k_moe_scatter(int* __restrict__ sorted, int4* __restrict__ tiles,
              const int* __restrict__ idx, const int* __restrict__ rank,
              const int* __restrict__ counts, int pairs, int E, int bm,
              int max_tiles) {
    moe_order<256, 1024>(blockIdx.x, sorted, tiles, idx, rank, counts, pairs, E,
                         bm, max_tiles);
}

DEV_INLINE float sq_relu(float v) {
    v = fmaxf(v, 0.f);
    return v * v;
}

// Work item of this block: tiles of neighbouring numbers (the columns of one
// row tile, then the next row tile of the expert) go to the same XCD, whose L2
// then holds the rows and weights they share. Blocks are dealt to the 8 XCDs
// in turn, and only the tiles in use are counted. Returns false if none is
// left for the block.
DEV_INLINE bool moe_work(const int4* tiles, int max_tiles, int ntn, int4& tl,
                         int& nt) {
    const int total = tiles[max_tiles].x * ntn;
    const int per = (total + 7) >> 3;
    const int i = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
    if ((int)(blockIdx.x >> 3) >= per || i >= total) return false;
    tl = tiles[i / ntn];
    nt = i % ntn;
    return true;
}

// R rows x 128 columns per block, 4 waves of R / 2 x 64, both
// operands through LDS by global_load_lds (source addresses pre-swizzled so
// that the lane-linear image reads back without bank conflicts), NB buffers.
// With few rows per expert the same pipeline streams the weights, in tiles of 32
// rows with 3 buffers: 48 rows in all, 64 experts, 160 -> 155 us; 12 rows gated 199 ->
// 168 (a CU's loads queue up, and of 128 rows as many are x's as W's). Weights go past
// the Infinity Cache (see load_lds16_once): 48 rows with the same 805 MB call after call,
// of which part then stays there, 150 -> 131; three sets of them in turn 151 -> 131. (8
// experts of 320 x 512, all of which would: 150 rows 27.0 -> 28.3.)
// ACT != 0 (up projection): row r of the tile is token sorted[row0 + r] / top,
// output in sorted order through squared ReLU (1) or, with weight rows in turns
// of 16 gate | 16 up, the gated unit `glu` in N / 2 columns (2); pw (nullable):
// a weight per pair on the unit's input. ACT 0: row r is sorted row row0 + r and
// its output goes to pair order. The MFMA computes W x^T, so a lane ends up with
// 4 neighbouring columns of one row.
// K % 64 == 0, N % 64 == 0 (ACT 2: N % 128 == 0).
template <int ACT, int NB, int R>
__global__ void __launch_bounds__(256, 2)
k_moe_gemm(bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
           const bf16_t* __restrict__ w, const int4* __restrict__ tiles,
           const int* __restrict__ sorted, int top, int N, int K, int ntn,
           int max_tiles, const GluParams glu, const float* __restrict__ pw) {
    constexpr int BK = 64, TB = (R + 128) * BK, GL = (R + 128) / 32;
    constexpr int A = R / 32;
    constexpr bool UP = ACT != 0;
    const int NO = ACT == 2 ? N / 2 : N;
    __shared__ __attribute__((aligned(16))) bf16_t lds[NB * TB];
    int4 tl;
    int nti;
    if (!moe_work(tiles, max_tiles, ntn, tl, nti)) return;
    const int n0 = nti * 128;
    const int lane = threadIdx.x & 63;
    const int wid = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int fr = lane & 15, kg = (lane >> 4) * 8;
    const int lrow = lane >> 3, lkb = (lane & 7) * 16;
    const char* src[GL];
#pragma unroll
    for (int i = 0; i < GL; ++i) {     // pieces of 8 rows: A of x, 4 of w
        const int row = (i < A ? wid * A + i : wid * 4 + i - A) * 8 + lrow;
        const bf16_t* p;
        if (i < A) {
            const int r = tl.y + min(row, tl.z - 1);
            p = x + (long)(UP ? sorted[r] / top : r) * K;
        } else {
            p = w + ((long)tl.x * N + min(n0 + row, N - 1)) * K;
        }
        src[i] = (const char*)p + (lkb ^ ((row & 7) << 4));
    }
    auto issue = [&](int buf, int kt) {
#pragma unroll
        for (int i = 0; i < GL; ++i) {
            const int piece = i < A ? wid * A + i : 4 * A + wid * 4 + i - A;
            const bf16_t* from = (const bf16_t*)(src[i] + (long)kt * BK * 2);
            if (i < A) load_lds16(from, lds + buf * TB + piece * 512);
            else load_lds16_once(from, lds + buf * TB + piece * 512);
        }
    };
    f32x4 acc[A][4];
#pragma unroll
    for (int a = 0; a < A; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int nt = K / BK;
    const int wr = (wid >> 1) * (R / 2), wc = (wid & 1) * 64;
#pragma unroll
    for (int u = 0; u < NB - 1; ++u)
        if (u < nt) issue(u, u);
    for (int kt = 0; kt < nt; ++kt) {
        if (kt + NB - 1 < nt)
            asm volatile("s_waitcnt vmcnt(%0)" :: "i"(GL * (NB - 2)) : "memory");
        else
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        if (kt + NB - 1 < nt) issue((kt + NB - 1) % NB, kt + NB - 1);
        const char* xb = (const char*)(lds + (kt % NB) * TB);
        const char* wb = xb + R * BK * 2;
#pragma unroll
        for (int kc = 0; kc < 2; ++kc) {
            bf16x8 b[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const int row = wc + c * 16 + fr;
                b[c] = *(const bf16x8*)(wb + row * 128 +
                    (((kc * 32 + kg) * 2) ^ ((row & 7) << 4)));
            }
#pragma unroll
            for (int a = 0; a < A; ++a) {
                const int row = wr + a * 16 + fr;
                const bf16x8 av = *(const bf16x8*)(xb + row * 128 +
                    (((kc * 32 + kg) * 2) ^ ((row & 7) << 4)));
#pragma unroll
                for (int c = 0; c < 4; ++c)
                    acc[a][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        b[c], av, acc[a][c], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int a = 0; a < A; ++a) {
        const int m = wr + a * 16 + fr;
        if (m >= tl.z) continue;
        bf16_t* orow = out + (UP ? (long)tl.y + m : sorted[tl.y + m]) *
                                 (long)NO;
        const float wi = ACT == 2 && pw ? pw[sorted[tl.y + m]] : 1.f;
#pragma unroll
        for (int c = 0; c < 4; c += ACT == 2 ? 2 : 1) {
            const int n = (ACT == 2 ? (n0 + wc + c * 16) / 2
                                    : n0 + wc + c * 16) + (lane >> 4) * 4;
            float f[4], u[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                f[r] = ACT == 2 ? wi * acc[a][c][r]
                     : ACT == 1 ? sq_relu(acc[a][c][r]) : acc[a][c][r];
                u[r] = wi * acc[a][(c + 1) & 3][r];
            }
            if (ACT == 2) glu_units(f, f, u, glu);
            if (n < NO) st4(orow + n, f);
        }
    }
}

// Many rows per expert: by k_gemm_wide's tiles, S::R rows of the list's by S::C
// columns, blocks of one a CU that take them in turn. 4096 tokens, 64 experts of 3072
// x 1024, 8 of them chosen 621 -> 493 us for both products (840 TFLOP/s; the tile
// lists' last tiles are half empty), gated, 7 762 -> 575; bound as k_gemm_wide.
// ONCE: tiles of 128 rows are for experts that mostly have one. 150, 256, 512 and 700
// tokens of 64 experts, 8 of them chosen, us: 162, 169, 184 and 192 with weights that
// stay in the Infinity Cache, 147, 152, 165 and 167 with such that go past it.
template <bool O>
struct ExpertRows {
    static constexpr bool GATHER = true, ONCE = O;
    const int* sorted;
    const float* pw;
    int top;                       // up: x's rows are tokens'; 0: down
    DEV_INLINE int from(int m) const { return top ? sorted[m] / top : m; }
    DEV_INLINE long to(int m) const { return top ? m : sorted[m]; }
    DEV_INLINE float weight(int m) const { return pw ? pw[sorted[m]] : 1.f; }
};

template <class S, int ACT>
__global__ void __launch_bounds__(512, 2)
k_moe_wide(const WideArgs p, const int4* __restrict__ tiles,
           const int* __restrict__ sorted, int top, int experts, int max_tiles,
           const float* __restrict__ pw) {
    extern __shared__ __attribute__((aligned(16))) bf16_t wide_lds[];
    const int cb = (p.N + S::C - 1) / S::C, items = tiles[max_tiles].x * cb;
    const int xcd = blockIdx.x & 7, at = (int)(blockIdx.x >> 3);
    const int each = (items + 7) >> 3;          // tiles of an XCD
    wide_tiles<S, ACT == 2 ? 4 : ACT ? 3 : 0>(
        p, wide_lds, xcd * each + at, min(items, (xcd + 1) * each),
        (int)(gridDim.x >> 3), [&](int it) {
            const int4 tl = tiles[it / cb];
            return WideTile{tl.y, tl.y + tl.z, it % cb * S::C, tl.x * p.N};
        }, experts * p.N, ExpertRows<S::R == 128>{sorted, pw, ACT ? top : 0});
}

// A few rows: up to 16 against 16 columns per block, K split over the 4 waves,
// so that a handful of experts still fills the chip. (16 output columns: 32
// weight rows if gated.)
template <int ACT>
__global__ void __launch_bounds__(256)
k_moe_gemm_few(bf16_t* __restrict__ out, const bf16_t* __restrict__ x,
               const bf16_t* __restrict__ w, const int4* __restrict__ tiles,
               const int* __restrict__ sorted, int top, int N, int K,
               int ntn, int max_tiles, const GluParams glu,
               const float* __restrict__ pw) {
    constexpr int U = 8, NW = ACT == 2 ? 2 : 1;
    constexpr bool UP = ACT != 0;
    __shared__ __attribute__((aligned(16))) float red[NW][4][16][20];
    int4 tl;
    int nti;
    if (!moe_work(tiles, max_tiles, ntn, tl, nti)) return;
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    const int fr = lane & 15, kg = (lane >> 4) * 8;
    const int n0 = nti * 16 * NW;
    const bf16_t* wr = w + ((long)tl.x * N + n0 + fr) * K + kg;
    const int r = tl.y + min(fr, tl.z - 1);
    const bf16_t* xr = x + (long)(UP ? sorted[r] / top : r) * K + kg;
    f32x4 acc[NW];
#pragma unroll
    for (int t = 0; t < NW; ++t) acc[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
    const int steps = K >> 5;
    for (int s0 = 0; s0 < steps; s0 += 4 * U) {
        // a wave takes two neighbouring steps, whose loads share cache lines
        auto step = [&](int u) { return s0 + ((u >> 1) * 4 + wid) * 2 + (u & 1); };
        bf16x8 a[U], b[U][NW];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int s = min(step(u), steps - 1);
#pragma unroll
            for (int t = 0; t < NW; ++t)
                b[u][t] = *(const bf16x8*)(wr + (long)t * 16 * K + s * 32);
            a[u] = *(const bf16x8*)(xr + s * 32);
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (step(u) < steps)
#pragma unroll
                for (int t = 0; t < NW; ++t)
                    acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
                        b[u][t], a[u], acc[t], 0, 0, 0);
    }
#pragma unroll
    for (int t = 0; t < NW; ++t)
        *(f32x4*)&red[t][wid][fr][(lane >> 4) * 4] = acc[t];
    __syncthreads();
    const int m = threadIdx.x >> 4, c = threadIdx.x & 15;
    if (m >= tl.z) return;
    float v[NW];
#pragma unroll
    for (int t = 0; t < NW; ++t)
        v[t] = red[t][0][m][c] + red[t][1][m][c] + red[t][2][m][c] +
               red[t][3][m][c];
    const float wi = ACT == 2 && pw ? pw[sorted[tl.y + m]] : 1.f;
    float y[1] = {ACT == 2 ? wi * v[0] : ACT == 1 ? sq_relu(v[0]) : v[0]};
    const float u[1] = {wi * v[NW - 1]};
    if (ACT == 2) glu_units(y, y, u, glu);
    out[(UP ? (long)tl.y + m : sorted[tl.y + m]) * (long)(N / NW) + nti * 16 +
        c] = f2bf(y[0]);
}

// Exact mode: 16 rows x 64 weight rows per block, f32 products.
template <int ACT>
__global__ void __launch_bounds__(256)
k_moe_gemm_f32(float* __restrict__ out, const float* __restrict__ x,
               const float* __restrict__ w, const int4* __restrict__ tiles,
               const int* __restrict__ sorted, int top, int N, int K,
               int ntn, int max_tiles, const GluParams glu,
               const float* __restrict__ pw) {
    constexpr bool UP = ACT != 0;
    __shared__ float xs[16][33], ws[64][33];
    int4 tl;
    int nti;
    if (!moe_work(tiles, max_tiles, ntn, tl, nti)) return;
    const int n0 = nti * 64;
    const int col = threadIdx.x & 63, r4 = (threadIdx.x >> 6) * 4;
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < K; k0 += 32) {
        for (int i = threadIdx.x; i < 16 * 32; i += 256) {
            const int r = tl.y + min(i >> 5, tl.z - 1);
            xs[i >> 5][i & 31] =
                x[(long)(UP ? sorted[r] / top : r) * K + k0 + (i & 31)];
        }
        for (int i = threadIdx.x; i < 64 * 32; i += 256)
            ws[i >> 5][i & 31] =
                w[((long)tl.x * N + n0 + (i >> 5)) * K + k0 + (i & 31)];
        __syncthreads();
#pragma unroll
        for (int k = 0; k < 32; ++k) {
            const float wv = ws[col][k];
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[r] += xs[r4 + r][k] * wv;
        }
        __syncthreads();
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float v = ACT == 1 ? sq_relu(acc[r]) : acc[r];
        if (ACT == 2) {
            if (pw) v *= pw[sorted[tl.y + min(r4 + r, tl.z - 1)]];
            const float u = fminf(fmaxf(__shfl_down(v, 16, WAVE), -glu.limit),
                                  glu.limit);
            v = fminf(v, glu.limit);
            const float z = glu.alpha * v * (1.f + glu.cubic * v * v);
            v = v / (1.f + expf(-z)) * (u + glu.shift);
        }
        if (r4 + r >= tl.z) continue;
        const long dst = UP ? tl.y + r4 + r : sorted[tl.y + r4 + r];
        if (ACT != 2)
            out[dst * N + n0 + col] = v;
        else if (!(col & 16))
            out[dst * (N / 2) + n0 / 2 + (col & 32) / 2 + (col & 15)] = v;
    }
}

// ===========================================================================
// Entry points. f32 != 0 selects the exact mode. 0 = success.
// ===========================================================================
typedef WideShape<4, 4, 3> Moe128;
typedef WideShape<6, 4, 2> Moe192;
typedef WideShape<8, 4, 2> Moe256;

template <class S, int ACT>
static int go_moe_wide(hipStream_t st, const WideArgs& p, const void* tiles,
                       const void* sorted, int top, int experts, int max_tiles,
                       const void* pw) {
    static const hipError_t e = hipFuncSetAttribute(
        (const void*)k_moe_wide<S, ACT>,
        hipFuncAttributeMaxDynamicSharedMemorySize, S::BYTES);
    if (e) return (int)e;
    const long most = (long)max_tiles * ((p.N + S::C - 1) / S::C);
    k_moe_wide<S, ACT><<<(unsigned)(8 * min((most + 7) / 8, 32l)), 512, S::BYTES,
                         st>>>(p, (const int4*)tiles, (const int*)sorted, top,
                               experts, max_tiles, (const float*)pw);
    LAUNCH_CHECK();
    return 0;
}

template <int D, int G>
static void launch_paged_decode(hipStream_t st, void* out, const void* q,
                                const PagedKV<D>& kv, const int* pos,
                                const int* slot, const int4* rows, float* ws,
                                int B, int ngrp, int nsplit, float scale,
                                const HeadEpilogue& epi,
                                const WindowKeys& keys) {
    const dim3 grid((unsigned)(B * kv.Hk * ngrp * nsplit));
    k_attn_decode<D, G><<<grid, dim3(256), 0, st>>>(
        (bf16_t*)out, (const bf16_t*)q, kv, pos, 1, slot, rows, ws, ngrp, nsplit,
        scale, epi, keys);
}

template <int D>
static int paged_decode(hipStream_t st, void* out, const void* q,
                        const void* kc, const void* vc, const int* table,
                        int per_slot, const int* pos, const int* slot,
                        const int4* rows, float* ws, int B, int Hq, int Hk,
                        int nsplit, float scale, const HeadEpilogue& epi,
                        const WindowKeys& keys) {
    const PagedKV<D> kv{(const bf16_t*)kc, (const bf16_t*)vc, table, Hk,
                        per_slot};
    const int per = Hq / Hk;
    int g = per;
    if (g > MAXG) for (g = MAXG; per % g; --g) {}
    switch (g) {
#define CASE_G(GG) case GG: launch_paged_decode<D, GG>(st, out, q, kv, pos, \
        slot, rows, ws, B, per / GG, nsplit, scale, epi, keys); break;
        CASE_G(1) CASE_G(2) CASE_G(3) CASE_G(4)
        CASE_G(5) CASE_G(6) CASE_G(7) CASE_G(8)
#undef CASE_G
        default: return -102;
    }
    LAUNCH_CHECK();
    if (nsplit > 1) {
        k_attn_combine<D><<<dim3((unsigned)(B * Hq)), dim3(256), 0, st>>>(
            (bf16_t*)out, ws, Hq, nsplit, epi);
        LAUNCH_CHECK();
    }
    return 0;
}

// Blocks of 128 value columns weigh keys half as often, and are half as many.
// 128 / 64 columns, 12 heads of 128 x 256, us: segments of 1100, 800, 500 and 331
// tokens (384 blocks of 128) 35 / 41, 12 of 300 40 / 47; one of 3500 (96) 63 / 44.
template <int KIND>
static void chunk_states(hipStream_t st, void* dS, void* S, const void* scal,
                         float* m_in, void* mst, const void* qkv, const void* b,
                         const void* chunks, const void* segs, int nseg, int H,
                         int DK, int DV, int ld_) {
    const bool wide = DV % 128 == 0 &&
                      nseg * H * (DK / STATE_K) * (DV / 128) >= 256;
#define GO(NK) k_chunk_states<KIND, NK><<<dim3((nseg * H + 7) / 8 * 8, \
        DK / STATE_K * (DV / (64 * NK))), 512, 0, st>>>((u32*)dS, (float*)S, \
        (const float*)scal, m_in, (float*)mst, (const bf16_t*)qkv, \
        (const float*)b, (const int4*)chunks, (const int4*)segs, nseg, H, DK, \
        DV, ld_)
    if (wide) GO(2); else GO(1);
#undef GO
}

extern "C" {

int gh_embed(void* stream, int f32, void* x, void* xb, const void* emb,
             const void* ptab, const void* tok, const void* pos,
             const void* w, float w_off, int N, int W, int Wtrue, float eps,
             int vocab, int max_pos) {
    if (W % 64 || N < 1) return -100;
    hipStream_t st_ = (hipStream_t)stream;
#define GO(T) k_embed<T><<<N, 256, 0, st_>>>((float*)x, (T*)xb, \
        (const T*)emb, (const T*)ptab, (const long long*)tok, \
        (const int*)pos, (const float*)w, w_off, W, Wtrue, eps, vocab, max_pos)
    if (f32) GO(float); else GO(bf16_t);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_sum_norm(void* stream, int f32, void* xo, void* xb, const void* x,
                const void* y, const void* wt, int top, const void* ident,
                const void* w, float w_off, float alpha, void* hist,
                const void* coef, int nh, int keep, int N, int W, int Wtrue,
                float eps) {
    if (W % 64 || W > 8192 || N < 1 || (hist && nh < 1)) return -100;
    hipStream_t st_ = (hipStream_t)stream;
#define GO(T, M) k_sum_norm<T, M><<<N, 256, 0, st_>>>((float*)xo, (T*)xb, \
        (const float*)x, (const T*)y, (const float*)wt, top, \
        (const float*)ident, (const float*)w, w_off, alpha, (float*)hist, \
        (const float*)coef, nh, keep, N, W, Wtrue, eps)
    if (f32) { if (wt) GO(float, true); else GO(float, false); }
    else { if (wt) GO(bf16_t, true); else GO(bf16_t, false); }
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_post_norm(void* stream, int f32, void* x, void* xb, const void* y,
                 const void* wt, int top, const void* w, float w_off, int N,
                 int W, int Wtrue, float eps) {
    if (W % 64 || W > 8192 || N < 1) return -100;
    hipStream_t st_ = (hipStream_t)stream;
#define GON(T, M, NV, THREADS) k_post_norm<T, M, NV, THREADS><<<N, THREADS, 0, \
        st_>>>((float*)x, (T*)xb, y, (const float*)wt, top, (const float*)w, \
        w_off, W, Wtrue, eps)
#define GO(T, M) do { if (W <= 2048) GON(T, M, 1, 256); \
        else if (W <= 4096) GON(T, M, 1, 512); else GON(T, M, 2, 512); } while (0)
    if (f32) { if (wt) GO(float, PAIRS); else GO(float, PLAIN); }
    else { if (wt) GO(bf16_t, PAIRS); else GO(bf16_t, PLAIN); }
    LAUNCH_CHECK();
    return 0;
}

// y: f32 partial sums [parts][N][W]
int gh_post_norm_parts(void* stream, void* x, void* xb, const void* y,
                       int parts, const void* w, float w_off, int N, int W,
                       int Wtrue, float eps) {
    if (W % 64 || W > 8192 || N < 1 || parts < 1) return -100;
    const void* const wt = nullptr;
    const int top = parts;
    hipStream_t st_ = (hipStream_t)stream;
    GO(bf16_t, PARTS);
#undef GO
#undef GON
    LAUNCH_CHECK();
    return 0;
}

int gh_norm_rows(void* stream, int f32, void* out, const void* x,
                 const void* rows, const void* w, float w_off, int M, int W,
                 int Wtrue, float eps) {
    if (W % 64 || M < 1) return -100;
    hipStream_t st_ = (hipStream_t)stream;
    if (f32)
        k_norm_rows<float><<<M, 256, 0, st_>>>((float*)out, (const float*)x,
            (const int*)rows, (const float*)w, w_off, W, Wtrue, eps);
    else
        k_norm_rows<bf16_t><<<M, 256, 0, st_>>>((bf16_t*)out, (const float*)x,
            (const int*)rows, (const float*)w, w_off, W, Wtrue, eps);
    LAUNCH_CHECK();
    return 0;
}

int gh_group_norm(void* stream, int f32, void* out, void* x, const void* y,
                  int parts, const void* rows, const void* wy, const void* w,
                  int N, int W, int groups, int size, float eps) {
    if (parts < 0 || (parts && (f32 || !y)) || N < 1 || W % 8 || W > 8192 ||
        groups < 1 || size < 1 ||
        (long)groups * size > W || (!y && !out) || (y && rows)) return -100;
    const int gr = size % 8 == 0 ? 8 : size % 4 == 0 ? 4 : size % 2 ? 1 : 2;
    const int lds = (W / gr + groups) * 4;
    if (lds > 64 * 1024) return -100;
    const Groups gp{groups, size};
    // (256 threads for a row of 6144 in groups of 128: 160 rows 15.5 and not 9.7 us,
    // 4096 rows 73.5 and not 64.7)
    const int threads = W <= 2048 ? 256 : 512;
#define GO(T, A, B) do { if (W <= 4096) GON(T, A, B, 1); else GON(T, A, B, 2); \
        } while (0)
#define GON(T, A, B, NV) k_group_norm<T, A, B, NV><<<N, threads, lds, \
        (hipStream_t)stream>>>((T*)out, (float*)x, y, parts, \
        (const int*)rows, (const float*)wy, (const float*)w, W, gp, eps)
#define PICK(T, A) do { if (gr == 8) GO(T, A, 8); else if (gr == 4) \
        GO(T, A, 4); else if (gr == 2) GO(T, A, 2); else GO(T, A, 1); \
        } while (0)
    if (f32) { if (y) PICK(float, true); else PICK(float, false); }
    else { if (y) PICK(bf16_t, true); else PICK(bf16_t, false); }
#undef PICK
#undef GON
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_poly_norm(void* stream, int f32, void* out, const void* z,
                 const void* coef, int N, int F, int Ftrue, float eps) {
    if (N < 1 || F % 8 || Ftrue < 1 || Ftrue > F) return -100;
#define GO(T, NV, THREADS) k_poly_norm<T, NV, THREADS><<<N, THREADS, 0, \
        (hipStream_t)stream>>>((T*)out, (const T*)z, (const float*)coef, F, \
        Ftrue, eps)
#define PICK(T) do { if (F <= 4096) GO(T, 2, 256); \
        else if (F <= 6144 && N >= 512) GO(T, 3, 256); \
        else if (F <= 8192) GO(T, 2, 512); else if (F <= 16384) GO(T, 4, 512); \
        else GO(T, 0, 512); } while (0)
    if (f32) PICK(float); else PICK(bf16_t);
#undef PICK
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_glu_f32(void* stream, void* out, const void* gu, long n, int F,
               float alpha, float limit, float shift, float cubic) {
    if (n < 1) return -100;
    const int grid = (int)min((n * F + 255) / 256, (long)4096);
    k_glu_f32<<<grid, 256, 0, (hipStream_t)stream>>>(
        (float*)out, (const float*)gu, n, F,
        GluParams{alpha, limit, shift, cubic});
    LAUNCH_CHECK();
    return 0;
}

int gh_proj_f32(void* stream, void* out, const void* x, const void* w,
                const void* bias, int M, int N, int K) {
    if (K % 32 || M < 1 || N < 1) return -100;
    hipStream_t st_ = (hipStream_t)stream;
#define GO(NT) k_proj_f32<NT><<<dim3((M + 15) / 16, \
        (N + 16 * NT - 1) / (16 * NT)), 512, 0, st_>>>((float*)out, \
        (const bf16_t*)x, (const bf16_t*)w, (const float*)bias, M, N, K)
    // few rows: narrow blocks, so that more of them stream the weights
    if (M <= 512 || N <= 16) GO(1);
    else if (N <= 32) GO(2);
    else if ((N + 79) / 80 < (N + 63) / 64) GO(5);
    else GO(4);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_streams_start(void* stream, int f32, void* x, void* h, const void* emb,
                     const void* tok, float scale, const void* in,
                     const void* w, int N, int ns, int W, int Wtrue, float eps,
                     int vocab) {
    if (N < 1 || ns < 1 || W % 64 || W > 8192) return -100;
#define GO(T) k_streams_start<T><<<N, 256, 0, (hipStream_t)stream>>>( \
        (float*)x, (T*)h, (const T*)emb, (const long long*)tok, scale, \
        (const float*)in, (const float*)w, ns, W, Wtrue, eps, vocab)
    if (f32) GO(float); else GO(bf16_t);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

// moe: y holds `top` rows per token, and extra (nullable) one more
int gh_streams_join(void* stream, int f32, int moe, void* x, void* h,
                    const void* y, int top, const void* extra,
                    const void* extra_z, int extra_ld, const void* hc,
                    const void* in, const void* w, int N, int ns, int W,
                    int Wtrue, float eps) {
    if (N < 1 || ns < 1 || ns > 16 || W % 64 || W > 8192 ||
        (moe && top < 1) || (h && !(in && w)) || (extra && !extra_z))
        return -100;
#define GO(T, S, NV, M) k_streams_join<T, S, NV, M><<<N, 256, 0, \
        (hipStream_t)stream>>>((float*)x, (T*)h, (const T*)y, top, \
        (const T*)extra, (const float*)extra_z, extra_ld, (const float*)hc, \
        (const float*)in, (const float*)w, ns, W, Wtrue, eps)
#define PICKV(T, S, M) do { if (W <= 4096) GO(T, S, 2, M); \
        else GO(T, S, 4, M); } while (0)
#define PICK(T, M) do { if (ns == 1) PICKV(T, 1, M); \
        else if (ns == 2) PICKV(T, 2, M); else if (ns <= 4) PICKV(T, 4, M); \
        else if (ns <= 8) GO(T, 8, 4, M); else GO(T, 16, 4, M); } while (0)
    if (f32) { if (moe) PICK(float, true); else PICK(float, false); }
    else { if (moe) PICK(bf16_t, true); else PICK(bf16_t, false); }
#undef PICK
#undef PICKV
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_streams_norm(void* stream, int f32, void* out, const void* x,
                    const void* rows, const void* w, int M, int ns, int W,
                    int Wtrue, float eps) {
    if (M < 1 || ns < 1 || W % 64 || W > 8192) return -100;
#define GO(T) k_streams_norm<T><<<M, 256, 0, (hipStream_t)stream>>>((T*)out, \
        (const float*)x, (const int*)rows, (const float*)w, ns, W, Wtrue, eps)
    if (f32) GO(float); else GO(bf16_t);
#undef GO
    LAUNCH_CHECK();
    return 0;
}

// cos_ and sin_ (nullable): tables of rot_rows x rot_half; act_0, act_n:
// columns that get SiLU in place (which may be all there is: H and G 0)
int gh_qknorm_kv(void* stream, int f32, void* qkv, void* q_out,
                 void* kc, void* vc, const void* table, int per_slot,
                 const void* pos, const void* slot, int N, int H, int G,
                 int P, int ld_, int dim, float eps, float coef, int every,
                 const void* cos_, const void* sin_, int rot_half,
                 int rot_rows, int act_0, int act_n) {
    if (N < 1 || (G ? H % G : H) || every < 1 || rot_half % 4 || 2 * rot_half > P ||
        act_0 % 8 || act_n % 8 || act_0 + act_n > ld_ || ld_ % 8)
        return -100;
    hipStream_t st_ = (hipStream_t)stream;
    const Rotation rot{(const float*)cos_, (const float*)sin_,
                       cos_ ? rot_half : 0, rot_rows};
    const int hw = 512 / P;
    const long per = (H + 2 * G + hw - 1) / hw + (act_n + 511) / 512;
    const unsigned grid = (unsigned)((N * per + 3) / 4);
#define GO(T, PP) k_qknorm_kv<T, PP><<<grid, 256, 0, st_>>>((T*)qkv, \
        (T*)q_out, (T*)kc, (T*)vc, (const int*)table, per_slot, \
        (const int*)pos, (const int*)slot, N, H, G, ld_, dim, eps, coef, \
        every, rot, act_0, act_n)
    if (P == 64) { if (f32) GO(float, 64); else GO(bf16_t, 64); }
    else if (P == 128) { if (f32) GO(float, 128); else GO(bf16_t, 128); }
    else if (P == 256) { if (f32) GO(float, 256); else GO(bf16_t, 256); }
    else return -101;
#undef GO
    LAUNCH_CHECK();
    return 0;
}

// Keys seen: the last `window` (0: all) and the first `keep`. Epilogue: see
// HeadEpilogue
int gh_paged_decode(void* stream, void* out, const void* q, const void* kc,
                    const void* vc, const void* table, int per_slot,
                    const void* pos, const void* slot, const void* rows,
                    void* ws, int B, int Hq, int Hk, int D, int nsplit, float scale,
                    int window, int keep, const void* sink, const void* gate,
                    int gate_ld, int gate_el, float oscale, int out_ld) {
    if (B < 1 || Hq % Hk || nsplit < 1 || nsplit > MAX_SPLIT || window < 0 ||
        keep < 0 || (unsigned long)rows % 16)
        return -100;
    const HeadEpilogue epi{(const float*)sink, (const bf16_t*)gate, gate_ld,
                           gate && gate_el, oscale, out_ld};
    const WindowKeys keys{window ? window : 1 << 30, keep};
    hipStream_t st_ = (hipStream_t)stream;
#define GO(DD) return paged_decode<DD>(st_, out, q, kc, vc, \
        (const int*)table, per_slot, (const int*)pos, (const int*)slot, \
        (const int4*)rows, (float*)ws, B, Hq, Hk, nsplit, scale, epi, keys)
    if (D == 64) GO(64);
    if (D == 128) GO(128);
    if (D == 256) GO(256);
#undef GO
    return -101;
}

int gh_paged_prefill(void* stream, void* out, const void* q, const void* kc,
                     const void* vc, const void* table, int per_slot,
                     const void* meta, int ntiles, int Hq, int Hk, int D,
                     float scale, int window, int keep, const void* sink,
                     const void* gate, int gate_ld, int gate_el, float oscale,
                     int out_ld) {
    if (ntiles < 1 || Hq % Hk || window < 0 || keep < 0 ||
        (gate && gate_el && gate_ld % 4) || out_ld % 4)
        return -100;
    const HeadEpilogue epi{(const float*)sink, (const bf16_t*)gate, gate_ld,
                           gate && gate_el, oscale, out_ld};
    hipStream_t st_ = (hipStream_t)stream;
#define GO(DD, K, ...) k_paged_prefill<DD, K> \
        <<<prefill_grid(ntiles, Hq), 256, 0, st_>>>((bf16_t*)out, \
        (const bf16_t*)q, PagedKV<DD>{(const bf16_t*)kc, (const bf16_t*)vc, \
        (const int*)table, Hk, per_slot}, (const int*)meta, ntiles, Hq, \
        Hq / Hk, scale, epi, K{__VA_ARGS__})
#define PICK(DD) do { if (window) GO(DD, WindowKeys, window, keep); \
        else GO(DD, AllKeys); } while (0)
    if (D == 64) PICK(64);
    else if (D == 128) PICK(128);
    else if (D == 256) PICK(256);
    else return -101;
#undef PICK
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_attn_rows_f32(void* stream, void* out, const void* q, const void* kc,
                     const void* vc, const void* table, int per_slot,
                     const void* pos, const void* slot, int N, int H, int G,
                     int P, float scale, int window, int keep,
                     const void* sink, const void* gate, int gate_ld,
                     int gate_el, float oscale, int out_ld) {
    if (N < 1 || H % G || window < 0 || keep < 0) return -100;
    hipStream_t st_ = (hipStream_t)stream;
    const WindowKeys keys{window ? window : 1 << 30, keep};
#define GO(PP) k_attn_rows_f32<PP><<<(unsigned)((long)N * H), 256, 0, st_>>>( \
        (float*)out, (const float*)q, (const float*)kc, (const float*)vc, \
        (const int*)table, per_slot, (const int*)pos, (const int*)slot, H, G, \
        scale, (const float*)sink, (const float*)gate, gate_ld, gate_el, \
        oscale, out_ld ? out_ld : H * P, keys)
    if (P == 64) GO(64);
    else if (P == 128) GO(128);
    else if (P == 256) GO(256);
    else return -101;
#undef GO
    LAUNCH_CHECK();
    return 0;
}

// kind: Rec. step: bytes of states of all the step's recurrent layers (see k_rec_step)
int gh_rec_step(void* stream, int f32, int kind, void* o, void* S, const void* mst,
                const void* qkv, const void* gr, const void* segs,
                const void* pos, const void* slot, int nseg, int H, int DK,
                int DV, int ld_, float qscale, float cap, int rpb, long step) {
    if (nseg < 1 || DK % 64 || DV % 64 || DK > 1024 || rpb < 1 || kind < 0 ||
        kind > CONSTANT || (kind == MLSTM && !mst))
        return -100;
    hipStream_t st_ = (hipStream_t)stream;
    const dim3 grid((unsigned)nseg, (unsigned)H,
                    (unsigned)((DV + (kind == MLSTM) + rpb - 1) / rpb));
    const bool once = !f32 && step >= REC_ONCE;
#define GO1(T, L, J, C, O) k_rec_step<T, L, J, C, O><<<grid, 256, 0, st_>>>( \
        (float*)o, (float*)S, (const float*)mst, (const T*)qkv, \
        (const float*)gr, (const int4*)segs, (const int*)pos, \
        (const int*)slot, H, DK, DV, ld_, qscale, cap, rpb)
#define GO(T, L, J, C) do { \
        if constexpr (sizeof(T) == 2) { if (once) { GO1(T, L, J, C, true); break; } } \
        GO1(T, L, J, C, false); } while (0)
#define PICK(T, C) do { if (DK <= 64) GO(T, 16, 1, C); \
        else if (DK <= 128) GO(T, 32, 1, C); \
        else if (DK <= 256) GO(T, 64, 1, C); \
        else if (DK <= 512) GO(T, 64, 2, C); else GO(T, 64, 4, C); } while (0)
    if (kind == MLSTM) {
        if (f32) PICK(float, MLSTM); else PICK(bf16_t, MLSTM);
    } else if (kind == CHANNELS) {
        if (f32) PICK(float, CHANNELS); else PICK(bf16_t, CHANNELS);
    } else {
        if (f32) PICK(float, CONSTANT); else PICK(bf16_t, CONSTANT);
    }
#undef PICK
#undef GO
#undef GO1
    LAUNCH_CHECK();
    return 0;
}

int gh_rec_out(void* stream, int f32, int silu, void* out, const void* o,
               void* mst, const void* qkv, const void* gr, const void* segs,
               const void* pos, const void* slot, const void* norm, int nseg,
               int plain0, int nplain, int H, int DK, int DV, int ld_,
               int dvtrue, float cap, float eps) {
    if (nseg + nplain < 1) return -100;
    hipStream_t st_ = (hipStream_t)stream;
    const unsigned grid = (unsigned)(((long)(nseg + nplain) * H + 3) / 4);
#define GO(T, G) k_rec_out<T, G><<<grid, 256, 0, st_>>>((T*)out, \
        (const float*)o, (float*)mst, (const T*)qkv, (const float*)gr, \
        (const int4*)segs, (const int*)pos, (const int*)slot, \
        (const float*)norm, nseg, plain0, nplain, H, DK, DV, ld_, dvtrue, \
        cap, eps)
    if (silu) { if (f32) GO(float, true); else GO(bf16_t, true); }
    else { if (f32) GO(float, false); else GO(bf16_t, false); }
#undef GO
    LAUNCH_CHECK();
    return 0;
}

int gh_rec_row_out(void* stream, int f32, void* out, const void* o,
                   const void* gate, const void* norm, int N, int H, int DV,
                   int ld_, int out_ld, int true_cols, float eps) {
    if (N < 1 || H < 1 || DV % 64 || ld_ % 4 || out_ld % 4 || true_cols < 1)
        return -100;
#define GO(T, NV) k_rec_row_out<T, NV><<<N, 256, 0, (hipStream_t)stream>>>( \
        (T*)out, (const float*)o, (const T*)gate, (const float*)norm, H, DV, \
        ld_, out_ld, true_cols, eps)
#define PICK(T) do { if (H * DV <= 4096) GO(T, 4); \
        else if (H * DV <= 8192) GO(T, 8); else GO(T, 0); } while (0)
    if (f32) PICK(float); else PICK(bf16_t);
#undef PICK
#undef GO
    LAUNCH_CHECK();
    return 0;
}

// constant: lightning attention (gr: log decay by head; mst unused). scal: f32
// [nchunks][H][4], [nchunks][H] and [nchunks][H][64] one behind the other
int gh_mlstm_chunks(void* stream, int constant, void* o, void* out, void* S,
                    void* mst, void* dS, void* scal, const void* qkv,
                    const void* gr, const void* chunks, const void* segs,
                    const void* norm, int nchunks, int nseg, int H, int DK,
                    int DV, int ld_, float qscale, float cap, int dvtrue,
                    float eps) {
    if (nchunks < 1 || nseg < 1 || DK % 64 || DV % 64 || (!constant && !mst) ||
        (out && (constant || DV > 256)))
        return -100;
    hipStream_t st_ = (hipStream_t)stream;
    float* const m_in = (float*)scal + (long)nchunks * H * 4;
    float* const w = m_in + (long)nchunks * H;
#define GO(C) do { \
    k_mlstm_weights<C><<<dim3(nchunks, (H + 3) / 4), 256, 0, st_>>>(w, \
        (float*)scal, (const float*)mst, (const float*)gr, \
        (const int4*)chunks, (const int4*)segs, H, cap); \
    LAUNCH_CHECK(); \
    chunk_states<C ? STATE_CONST : STATE_MLSTM>(st_, dS, S, scal, m_in, mst, \
        qkv, w, chunks, segs, nseg, H, DK, DV, ld_); \
    LAUNCH_CHECK(); \
    k_mlstm_chunk_out<C><<<dim3(nchunks, H, (DV + 255) / 256), 256, 0, \
        st_>>>((float*)o, (bf16_t*)out, (const float*)dS, m_in, \
        (const bf16_t*)qkv, (const float*)gr, \
        (const int4*)chunks, (const float*)norm, H, DK, DV, ld_, qscale, cap, \
        dvtrue, eps); \
    LAUNCH_CHECK(); } while (0)
    if (constant) GO(true); else GO(false);
#undef GO
    return 0;
}

int gh_gla_decay(void* stream, void* b, const void* u, const void* w,
                 const void* bias, const void* chunks, int nd, int nchunks,
                 int R, int C, float inv_tau) {
    if (nd + nchunks < 1 || R < 1 || C < 1) return -100;
    k_gla_decay<<<dim3((nd + 15) / 16 + nchunks, (C + 63) / 64), 256, 0,
                  (hipStream_t)stream>>>((float*)b, (const float*)u,
        (const float*)w, (const float*)bias, (const int4*)chunks, nd, R, C,
        inv_tau);
    LAUNCH_CHECK();
    return 0;
}

int gh_gla_chunks(void* stream, void* o, void* out, void* S, void* dS,
                  const void* qkv, const void* b, const void* chunks,
                  const void* segs, const void* norm, int nchunks, int nseg,
                  int H, int DK, int DV, int ld_, float qscale, int dvtrue,
                  float eps) {
    if (nchunks < 1 || nseg < 1 || DK % 64 || DV % 64 || (out && DV > 256))
        return -100;
    hipStream_t st_ = (hipStream_t)stream;
    chunk_states<STATE_GLA>(st_, dS, S, nullptr, nullptr, nullptr, qkv, b,
                            chunks, segs, nseg, H, DK, DV, ld_);
    LAUNCH_CHECK();
    k_gla_chunk_out<<<dim3((nchunks + 7) / 8 * 16, H, (DV + 255) / 256), 256, 0, st_>>>(
        (float*)o, (bf16_t*)out, (const float*)dS, (const bf16_t*)qkv,
        (const float*)b, (const int4*)chunks, (const float*)norm, nchunks, H, DK,
        DV, ld_, qscale, dvtrue, eps);
    LAUNCH_CHECK();
    return 0;
}

// E router outputs (rows of stride ldz), of which the first `experts` have
// weights. corr (nullable): correction of the choice; ident (nullable): sum of
// a token's weights beyond the experts
int gh_moe_route(void* stream, void* idx, void* wt, void* rank, void* counts,
                 void* sorted, void* tiles, const void* z, int ldz,
                 const void* corr, void* ident, int N, int E, int experts,
                 int top, int groups, int keep, float eps, float scale, int sigmoid, int bm,
                 int max_tiles) {
    if (ldz < E || (sigmoid && (corr || ident))) return -100;
    if (N < 1 || E < 1 || E > 1024 || top < 1 || experts < 1 || experts > E ||
        groups < 1 || E % groups || keep < 1 || keep > groups ||
        top > E / groups * keep)
        return -100;
    hipStream_t st_ = (hipStream_t)stream;
    const long pairs = (long)N * top;
    const bool alone = !counts;
    if (alone && (pairs > 1024 || E > 256)) return -100;
    const int tpw = alone ? (N + 15) / 16 : min(max(N / 2048, 1), 16);
    const unsigned blocks = alone ? 1 : (N + 4 * tpw - 1) / (4 * tpw);
#define GO(V, A) k_moe_route<V, A><<<blocks, A ? 1024 : 256, 0, st_>>>( \
        (int*)idx, (float*)wt, (int*)rank, (int*)counts, (const float*)z, \
        ldz, (const float*)corr, (float*)ident, N, E, experts, top, groups, \
        keep, eps, scale, sigmoid, tpw, (int*)sorted, (int4*)tiles, bm, \
        max_tiles)
    if (E <= 64) { if (alone) GO(1, true); else GO(1, false); }
    else if (E <= 128) { if (alone) GO(2, true); else GO(2, false); }
    else if (E <= 256) { if (alone) GO(4, true); else GO(4, false); }
    else GO(16, false);
#undef GO
    LAUNCH_CHECK();
    if (alone) return 0;
    k_moe_scatter<<<(unsigned)((pairs + 255) / 256), 256, 0, st_>>>(
        (int*)sorted, (int4*)tiles, (const int*)idx, (const int*)rank,
        (const int*)counts, (int)pairs, experts, bm, max_tiles);
    LAUNCH_CHECK();
    return 0;
}

// act: 0 down, 1 up with squared ReLU, 2 gate and up (N weight rows, in turns
// of 16 | 16) with the gated unit's constants; pw (nullable): weights of the
// pairs on its input. bm: rows per tile of the list: 16 (few pairs; the exact
// mode), 32 or 128; or, wide, 128, 192 or 256, with `rows` of x and as many experts
int gh_moe_gemm(void* stream, int f32, int act, void* out, const void* x,
                const void* w, const void* tiles, const void* sorted,
                int top, int N, int K, int bm, int max_tiles, int wide,
                int rows, int experts, float alpha, float limit, float shift, float cubic,
                const void* pw) {
    if (N % (act == 2 ? 128 : 64) || K % 64 || max_tiles < 1 || act < 0 ||
        act > 2)
        return -100;
    const GluParams glu{alpha, limit, shift, cubic};
    hipStream_t st_ = (hipStream_t)stream;
    if (f32) {
        if (bm != 16) return -103;
        const int ntn = N / 64;
        const unsigned grid = (unsigned)((max_tiles * ntn + 7) / 8 * 8);
#define GO(U) k_moe_gemm_f32<U><<<grid, 256, 0, st_>>>((float*)out, \
        (const float*)x, (const float*)w, (const int4*)tiles, \
        (const int*)sorted, top, N, K, ntn, max_tiles, glu, (const float*)pw)
        if (act == 2) GO(2); else if (act) GO(1); else GO(0);
#undef GO
        LAUNCH_CHECK();
        return 0;
    }
#define ARGS (bf16_t*)out, (const bf16_t*)x, (const bf16_t*)w, \
        (const int4*)tiles, (const int*)sorted, top, N, K, ntn, max_tiles, \
        glu, (const float*)pw
    if (wide) {
        if (bm != 128 && bm != 192 && bm != 256) return -103;
        if ((long)experts * N * K * 2 > WIDE_BYTES || K < 256 || experts < 1 ||
            (long)rows * K * 2 > 1l << 30) return -100;
        const WideArgs p{out, (const bf16_t*)x, (const bf16_t*)w, rows, N, K, glu};
#define GO(S) return act == 2 ? go_moe_wide<S, 2>(st_, p, tiles, sorted, top, \
            experts, max_tiles, pw) : act ? go_moe_wide<S, 1>(st_, p, tiles, \
            sorted, top, experts, max_tiles, pw) : go_moe_wide<S, 0>(st_, p, \
            tiles, sorted, top, experts, max_tiles, pw)
        if (bm == 128) GO(Moe128);
        if (bm == 192) GO(Moe192);
        GO(Moe256);
#undef GO
    } else if (bm == 32 || bm == 128) {
        const int ntn = (N + 127) / 128;
        const unsigned grid = (unsigned)((max_tiles * ntn + 7) / 8 * 8);
#define GO(NB, R) do { \
            if (act == 2) k_moe_gemm<2, NB, R><<<grid, 256, 0, st_>>>(ARGS); \
            else if (act) k_moe_gemm<1, NB, R><<<grid, 256, 0, st_>>>(ARGS); \
            else k_moe_gemm<0, NB, R><<<grid, 256, 0, st_>>>(ARGS); } while (0)
        if (bm == 32) GO(3, 32);
        else GO(2, 128);
#undef GO
    } else if (bm == 16) {
        const int ntn = N / (act == 2 ? 32 : 16);
        const unsigned grid = (unsigned)((max_tiles * ntn + 7) / 8 * 8);
        if (act == 2) k_moe_gemm_few<2><<<grid, 256, 0, st_>>>(ARGS);
        else if (act) k_moe_gemm_few<1><<<grid, 256, 0, st_>>>(ARGS);
        else k_moe_gemm_few<0><<<grid, 256, 0, st_>>>(ARGS);
    } else {
        return -103;
    }
#undef ARGS
    LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
