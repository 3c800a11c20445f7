// Helpers of the kernels that move 16-bit tiles through LDS into MFMA operands:
// rotation by tables, packing, transposed LDS reads, direct loads into LDS,
// and a barrier that leaves such loads in flight.
#pragma once

#include "gridllm_common.h"

#define PAGE 64
#define LOG2E 1.4426950408889634f

typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
typedef __attribute__((ext_vector_type(2))) unsigned int u32x2;
typedef __attribute__((address_space(3))) bf16x4 lds_bf16x4;

// cos and sin of a position times each pair's frequency: rows of R / 2 values
// (1 and 0 for pairs that are not rotated)
struct Rotation {
    const float* cos_;
    const float* sin_;
    int half, rows;
};

// 16 and 8 bytes of LDS by plain vector types (see load_lds16)
DEV_INLINE void lds_ld4(const float* p, float* f) {
    const f32x4 v = *(const f32x4*)p;
#pragma unroll
    for (int i = 0; i < 4; ++i) f[i] = v[i];
}
DEV_INLINE void lds_st2(bf16_t* p, u32 a, u32 b) { *(u32x2*)p = (u32x2){a, b}; }

// Rotate the neighbouring pairs of 8 coordinates by 4 cosines and sines.
DEV_INLINE void rotate_by(float* f, const float* cos_, const float* sin_) {
    float co[4], si[4];
    lds_ld4(cos_, co);                     // (or of global memory)
    lds_ld4(sin_, si);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float u = f[2 * i], v = f[2 * i + 1];
        f[2 * i] = u * co[i] - v * si[i];
        f[2 * i + 1] = v * co[i] + u * si[i];
    }
}

// The same by the tables; the first is coordinate c of the rotated part.
DEV_INLINE void rotate8(float* f, int c, int p, const Rotation rot) {
    const long at = (long)min(p, rot.rows - 1) * rot.half + c / 2;
    rotate_by(f, rot.cos_ + at, rot.sin_ + at);
}

DEV_INLINE bf16x8 to_bf16x8(const float* f) {
    bf16x8 o;
#pragma unroll
    for (int i = 0; i < 8; ++i) o[i] = (__bf16)f[i];
    return o;
}

// to bf16's values, by two (the compiler converts one at a time)
DEV_INLINE void round8(float (&f)[8]) {
    const bf16x8 b = to_bf16x8(f);
    unpack8(*(const uint4*)&b, f);
}

DEV_INLINE u32 pack2(float a, float b) {
    typedef __attribute__((ext_vector_type(2))) __bf16 bf16x2;
    bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(u32, v);
}

// max over the lanes that differ in bit 5, or bits 4 and 5, of the lane number
DEV_INLINE float max_across32(float x) {
    const u32x2 r = __builtin_amdgcn_permlane32_swap(
        __float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}
DEV_INLINE float max_across16(float x) {
    const u32x2 r = __builtin_amdgcn_permlane16_swap(
        __float_as_uint(x), __float_as_uint(x), false, false);
    return max_across32(fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1])));
}

// 2^x by the hardware instruction (tiny results become 0)
DEV_INLINE float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Products' results as they are stored: a lane has 4 columns of row l % 16 in each of 4
// tiles v[j]. Turned, it has those of rows 4 j + l % 4 in tile l / 4 % 4: a store of 16
// bytes a lane fills whole lines of 4 rows, 256 bytes each, and not half lines of 16.
// (Group k of 4 lanes gets as v[j] what group j had as v[k].)
template <int ROTATE, int GROUPS>
DEV_INLINE float of_group(float mine, float other) {
    return __uint_as_float(__builtin_amdgcn_update_dpp(
        __float_as_uint(mine), __float_as_uint(other), 0x120 + ROTATE, 0xf, GROUPS,
        false));
}
DEV_INLINE void turn_tiles(f32x4 (&v)[4]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        float a[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {          // groups 0 and 2, 1 and 3
            a[j] = of_group<8, 0xc>(v[j][r], v[j + 2][r]);
            a[j + 2] = of_group<8, 0x3>(v[j + 2][r], v[j][r]);
        }
#pragma unroll
        for (int j = 0; j < 4; j += 2) {       // 0 and 1, 2 and 3
            v[j][r] = of_group<4, 0xa>(a[j], a[j + 1]);
            v[j + 1][r] = of_group<12, 0x5>(a[j + 1], a[j]);
        }
    }
}

// 4 x 16 block of 16-bit elements in LDS, read transposed by 16 lanes: lane l
// passes the address of row l / 4, columns 4 (l % 4) .. + 3, and gets column l,
// rows 0 .. 3.
DEV_INLINE bf16x4 read_transposed(const bf16_t* __restrict__ p) {
    return __builtin_amdgcn_ds_read_tr16_b64_v4bf16((lds_bf16x4*)p);
}

// A load into LDS. The compiler has each later access to LDS wait for it, unless
// that access says of what it is: plain vector types, not HIP's structs (float4,
// uint2), and a __restrict__ pointer to a builtin. Kernels with a tile under way
// while they work on another one wait by themselves (WAIT_LOADS).
DEV_INLINE void load_lds16(const bf16_t* src, bf16_t* dst) {
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) unsigned int*)src,
        (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, 0);
}

// The same of what a pass reads once and there is much of (weights, caches): past the
// Infinity Cache. Read through it, more than its 256 MB push each other out, the other
// kernels' data with them, and a next pass finds nothing there; past it, it keeps what
// it has (us, all read in turn: 1600 MB 322, 284; 2400 MB 466, 425; what it would hold
// is 5 % slower: 200 MB 38.8, 40.8). Whole lines of 128 bytes are to be taken.
DEV_INLINE void load_lds16_once(const bf16_t* src, bf16_t* dst) {
    __builtin_amdgcn_global_load_lds(
        (const __attribute__((address_space(1))) unsigned int*)src,
        (__attribute__((address_space(3))) unsigned int*)dst, 16, 0, 2);
}

// The same from `bytes` of memory at p, which all lanes name alike: lane_at and at (a
// scalar) bytes on; what lies behind them comes as zeros. To the compiler's counts
// load_lds16 is an access that may be to LDS itself: with one under way it has a wave
// wait for all of its reads of LDS, where it needs the first (64 x 128 keys and values
// a wave: 20 waits for everything, of 32). With these it waits for that one. Prompt
// attention, 24 heads of 128 over 8: 8000 tokens 432 -> 417 us, 2000 60 -> 55.
#ifdef __HIP_DEVICE_COMPILE__          // (the host has no buffer descriptors)
typedef __amdgpu_buffer_rsrc_t LdsSource;
#else
struct LdsSource {};
#endif
DEV_INLINE LdsSource lds_source(const void* p, u32 bytes) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, (int)bytes, 0x00020000);
#else
    return {};
#endif
}
template <bool ONCE = false>
DEV_INLINE void load_lds16(LdsSource src, u32 lane_at, u32 at, bf16_t* dst) {
#ifdef __HIP_DEVICE_COMPILE__
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        src, (__attribute__((address_space(3))) unsigned int*)dst, 16, lane_at, at, 0,
        ONCE ? 2 : 0);
#endif
}

// 16 bytes of it into registers
typedef __attribute__((ext_vector_type(4))) u32 u32x4;
DEV_INLINE u32x4 load16(LdsSource src, u32 lane_at, u32 at) {
#ifdef __HIP_DEVICE_COMPILE__
    return __builtin_amdgcn_raw_buffer_load_b128(src, lane_at, at, 0);
#else
    return {};
#endif
}

// Waits until no more than n loads or stores of the wave are under way.
#define WAIT_LOADS(n) do { \
        __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | 0xf70); \
        asm volatile("" ::: "memory"); } while (0)

// Barrier that orders LDS accesses alone: loads into LDS stay in flight.
DEV_INLINE void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// Work item of a prefill block: an eighth of all heads' tiles lies on one XCD (blocks
// go round the 8 XCDs), so that heads share their keys in its L2, and of all of these
// later tiles, which see more keys, first. One head's after the other's, the last of
// them started its longest tiles when the others were done (24 heads of 128 over 8,
// 2000 tokens 55 -> 44 us, 3500 100 -> 90, 8000 417 -> 383). False: none.
__host__ DEV_INLINE bool prefill_place(int block, int ntiles, int Hq, int* tile,
                                       int* head) {
    const int total = ntiles * Hq, per = (total + 7) >> 3;
    const int at = block >> 3, i0 = (block & 7) * per, i1 = min(total, i0 + per);
    if (i0 + at >= i1) return false;
    // items i0 .. i1 - 1, head by head: the first one's from turn j0 on, the last
    // one's up to j1; turn j is tile ntiles - 1 - j
    const int h0 = i0 / ntiles, j0 = i0 - h0 * ntiles;
    const int h1 = (i1 - 1) / ntiles, j1 = i1 - h1 * ntiles;
    if (h0 == h1) {
        *head = h0;
        *tile = ntiles - 1 - j0 - at;
        return true;
    }
    // heads of a turn, up to the smaller of j0 and j1, up to the larger, behind it
    const int lo = min(j0, j1), hi = max(j0, j1), whole = h1 - h0 - 1;
    int n = whole + (j0 == 0) + 1, from = 0, r = at;
    if (r >= lo * n) {
        r -= lo * n;
        n = whole + 2 * (j0 <= j1);
        from = lo;
        if (r >= (hi - lo) * n) {
            r -= (hi - lo) * n;
            n = whole + 1;
            from = hi;
        }
    }
    const int j = from + r / n;
    *head = h0 + (j < j0) + r % n;
    *tile = ntiles - 1 - j;
    return true;
}
