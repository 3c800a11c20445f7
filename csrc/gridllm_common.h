// Helpers shared by the gfx950 kernel sources: bf16 packing, wave
// reductions, MFMA fragment types, and the gated-linear-unit activation.
#pragma once

#include <hip/hip_runtime.h>
#include <math.h>
#include <float.h>

typedef unsigned short bf16_t;
typedef unsigned int u32;

#define WAVE 64
#define DEV_INLINE __device__ __forceinline__

DEV_INLINE float bf2f(bf16_t v) {
    u32 u = ((u32)v) << 16;
    return __uint_as_float(u);
}

// round to nearest even, by the hardware (one instruction; by integers seven)
DEV_INLINE bf16_t f2bf(float f) {
    return __builtin_bit_cast(bf16_t, (__bf16)f);
}

// unpack 8 bf16 from a uint4 into f32[8]
DEV_INLINE void unpack8(const uint4 v, float* f) {
    const u32 w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i]     = __uint_as_float((w[i] & 0xffffu) << 16);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
}

// pack f32[8] -> uint4 of 8 bf16
DEV_INLINE uint4 pack8(const float* f) {
    uint4 v;
    u32* w = (u32*)&v;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        u32 lo = (u32)f2bf(f[2 * i]);
        u32 hi = (u32)f2bf(f[2 * i + 1]);
        w[i] = lo | (hi << 16);
    }
    return v;
}

DEV_INLINE float wave_reduce_sum(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x += __shfl_xor(x, off, WAVE);
    return x;
}

DEV_INLINE float wave_reduce_max(float x) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, WAVE));
    return x;
}

// rows of bf16 or f32 as f32
DEV_INLINE float ld(const bf16_t* p) { return bf2f(*p); }
DEV_INLINE float ld(const float* p) { return *p; }
DEV_INLINE void st(bf16_t* p, float v) { *p = f2bf(v); }
DEV_INLINE void st(float* p, float v) { *p = v; }
DEV_INLINE void ld8(const bf16_t* p, float* f) { unpack8(*(const uint4*)p, f); }
DEV_INLINE void ld8(const float* p, float* f) {
    *(float4*)f = ((const float4*)p)[0];
    *(float4*)(f + 4) = ((const float4*)p)[1];
}
DEV_INLINE void st8(bf16_t* p, const float* f) { *(uint4*)p = pack8(f); }
DEV_INLINE void st8(float* p, const float* f) {
    ((float4*)p)[0] = *(const float4*)f;
    ((float4*)p)[1] = *(const float4*)(f + 4);
}
DEV_INLINE void ld4(const bf16_t* p, float* f) {
    const uint2 v = *(const uint2*)p;
    f[0] = __uint_as_float(v.x << 16);
    f[1] = __uint_as_float(v.x & 0xffff0000u);
    f[2] = __uint_as_float(v.y << 16);
    f[3] = __uint_as_float(v.y & 0xffff0000u);
}
DEV_INLINE void ld4(const float* p, float* f) { *(float4*)f = *(const float4*)p; }
DEV_INLINE void st4(bf16_t* p, const float* f) {
    *(uint2*)p = make_uint2((u32)f2bf(f[0]) | ((u32)f2bf(f[1]) << 16),
                            (u32)f2bf(f[2]) | ((u32)f2bf(f[3]) << 16));
}
DEV_INLINE void st4(float* p, const float* f) { *(float4*)p = *(const float4*)f; }
// 8 columns of a product's output that is still f32 partial sums [parts][N][W] (K
// in parts): added up, and rounded as the product's result would be. Spares that
// product's second launch.
DEV_INLINE void summed8(const float* y, int parts, long n, long N, int W, int c,
                        float* v) {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = 0.f;
#pragma unroll 4
    for (int k = 0; k < parts; ++k) {
        float f[8];
        ld8(y + (k * N + n) * W + c, f);
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] += f[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = bf2f(f2bf(v[i]));
}

// The hardware's reciprocal (1 ulp) and a Newton step, which came out as an exact
// division does for 12 M arguments, in 0.82 of its time. (An infinite sum would
// leave NaN; a NaN has to come through.)
DEV_INLINE float sigmoidf_(float z) {
    const float d = 1.f + expf(-z), r = __builtin_amdgcn_rcpf(d);
    return d > 3e38f ? 0.f : fmaf(fmaf(-d, r, 1.f), r, r);
}

// log(sigmoid(z)) = min(z, 0) - log(1 + E) with E = exp(-|z|), in 0.36 of the time
// that it takes with log1pf: with q = E / (2 + E) <= 1/3
//   log(1 + E) = 2 atanh(q) = 2 (q + q^3 / 3 + q^5 / 5 + ..),
// of which q^17 and beyond are below 2^-29 of it. q is a quotient and its
// remainder. Error against 64 bits: 2.3 units of 2^-24 at most and .56 in root mean
// square for 12 M arguments of 1e-7 to 80, as before.
DEV_INLINE float log_sigmoid(float z) {
#pragma clang fp contract(off)             // q twice: the same, or its rest is wrong
    const float E = expf(-fabsf(z));
    const float d = 2.f + E, dl = E - (d - 2.f);       // d + dl = 2 + E
    const float r = __builtin_amdgcn_rcpf(d), q = E * r, q2 = q * q;
    const float rest = fmaf(-dl, q, fmaf(-d, q, E)) * r;
    float p = 1.f / 15.f;
    p = fmaf(p, q2, 1.f / 13.f);
    p = fmaf(p, q2, 1.f / 11.f);
    p = fmaf(p, q2, 1.f / 9.f);
    p = fmaf(p, q2, 1.f / 7.f);
    p = fmaf(p, q2, 1.f / 5.f);
    p = fmaf(p, q2, 1.f / 3.f);
    return (z > 0.f ? 0.f : z) - 2.f * (q + fmaf(q * q2, p, rest));
}

// sum over a block of THREADS threads; every thread gets it
template <int THREADS = 256>
DEV_INLINE float block_sum(float v, float* red) {
    v = wave_reduce_sum(v);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    v = red[0];
#pragma unroll
    for (int i = 1; i < THREADS / 64; ++i) v += red[i];
    return v;
}

typedef __attribute__((ext_vector_type(8))) __bf16 bf16x8;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(16))) float f32x16;

// Gated linear unit, by its constants:
//   g' = min(g, limit), u' = clamp(u, -limit, limit)
//   y  = g' * sigmoid(alpha * g' * (1 + cubic * g'^2)) * (u' + shift)
// SwiGLU is {alpha 1, limit inf, shift 0, cubic 0}; the tanh form of GELU is
// {2 sqrt(2 / pi), inf, 0, 0.044715}, since (1 + tanh z) / 2 = sigmoid(2 z).
struct GluParams { float alpha, limit, shift, cubic; };

// The hardware's exponential and reciprocal, and a Newton step (see sigmoidf_).
DEV_INLINE float glu_sigmoid(float z) {
    const float d = 1.f + __expf(-z), r = __builtin_amdgcn_rcpf(d);
    return d == INFINITY ? 0.f : fmaf(fmaf(-d, r, 1.f), r, r);
}

// n units; y may be g. With limit inf, cubic 0 and shift 0, by which all lanes branch,
// a unit is 11 instructions, else 19; with an exact division it was 26. The matrix
// cores wait for the units of a product's tile: 4096 x 16384 x 3072, 256 x 256 tiles,
// 308 us with 26 instructions, now 296; K 1024 126, 115.
template <int n>
DEV_INLINE void glu_units(float (&y)[n], const float (&g)[n], const float (&u)[n],
                          const GluParams p) {
    if (p.limit == INFINITY && p.cubic == 0.f && p.shift == 0.f) {
#pragma unroll
        for (int i = 0; i < n; ++i) y[i] = g[i] * glu_sigmoid(p.alpha * g[i]) * u[i];
        return;
    }
#pragma unroll
    for (int i = 0; i < n; ++i) {
        const float a = fminf(g[i], p.limit);
        const float b = fminf(fmaxf(u[i], -p.limit), p.limit);
        y[i] = a * glu_sigmoid(p.alpha * a * (1.f + p.cubic * a * a)) * (b + p.shift);
    }
}

#define LAUNCH_CHECK() do { hipError_t e = hipGetLastError(); \
    if (e != hipSuccess) return (int)e; } while (0)
