/*
 * ckq_device.hpp - gfx950 device helpers shared by the quantized kernels:
 * unaligned 128-bit loads, packed int8 dot, wave64 DPP reductions.
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef uint32_t u32;

/* GGUF blocks are only 2- or 4-byte aligned (Q6_K 210 B, Q8_0 34 B, Q8_K
 * 292 B).  Global loads on gfx950 run in unaligned-access mode, so a packed
 * struct with the true alignment still compiles to one global_load_dwordx4. */
template <int ALIGN> struct __attribute__((packed, aligned(ALIGN))) ckq_v4 { u32 v[4]; };
template <int ALIGN> struct __attribute__((packed, aligned(ALIGN))) ckq_v2 { u32 v[2]; };
template <int ALIGN> struct __attribute__((packed, aligned(ALIGN))) ckq_v1 { u32 v; };

template <int ALIGN, typename T>
__device__ __forceinline__ void ld16(T *dst, const uint8_t *p)
{
    const ckq_v4<ALIGN> t = *reinterpret_cast<const ckq_v4<ALIGN> *>(p);
    dst[0] = (T)t.v[0]; dst[1] = (T)t.v[1]; dst[2] = (T)t.v[2]; dst[3] = (T)t.v[3];
}
template <int ALIGN, typename T>
__device__ __forceinline__ void ld8(T *dst, const uint8_t *p)
{
    const ckq_v2<ALIGN> t = *reinterpret_cast<const ckq_v2<ALIGN> *>(p);
    dst[0] = (T)t.v[0]; dst[1] = (T)t.v[1];
}
template <int ALIGN>
__device__ __forceinline__ u32 ld4(const uint8_t *p)
{
    return reinterpret_cast<const ckq_v1<ALIGN> *>(p)->v;
}
__device__ __forceinline__ u32 ld2(const uint8_t *p)
{
    return *reinterpret_cast<const uint16_t *>(p);
}

/* Four signed int8 products accumulated into int32 (v_dot4_i32_i8). */
__device__ __forceinline__ int dot4(int a, int b, int c) { return __builtin_amdgcn_sdot4(a, b, c, false); }

__device__ __forceinline__ int mul24(int a, int b) { return __mul24(a, b); }

/* IEEE binary16 bit pattern -> fp32 (v_cvt_f32_f16; subnormals preserved). */
__device__ __forceinline__ float h2f(u32 h)
{
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

/* Sign-extend byte `idx` (0..3) of a dword. */
__device__ __forceinline__ int sbyte(u32 v, int idx) { return (int)(v << (24 - 8 * idx)) >> 24; }

/* Wave index as a scalar: lets the compiler keep row indices, row base
 * addresses and loop control in SGPRs (uniform branches, scalar address math). */
__device__ __forceinline__ int wave_in_block() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

/* ---- DPP reductions -------------------------------------------------------
 * Fixed summation tree, so results do not depend on scheduling. */
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_get(float v)
{
    return __builtin_bit_cast(float,
        __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, true));
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ int dpp_get(int v)
{
    return __builtin_amdgcn_update_dpp(0, v, CTRL, ROW_MASK, 0xF, true);
}

/* Sum over groups of LANES consecutive lanes (LANES in 4,8,16,32,64).  The
 * group total ends up in the LAST lane of every group (for 4/8/16 in every
 * lane of the group). */
template <int LANES, typename T>
__device__ __forceinline__ T group_sum(T v)
{
    v += dpp_get<0xB1>(v);                    /* quad_perm [1,0,3,2] */
    v += dpp_get<0x4E>(v);                    /* quad_perm [2,3,0,1] */
    if (LANES >= 8) v += dpp_get<0x141>(v);   /* row_half_mirror */
    if (LANES >= 16) v += dpp_get<0x140>(v);  /* row_mirror */
    if (LANES >= 32) v += dpp_get<0x142, 0xA>(v); /* row_bcast15 into rows 1,3 */
    if (LANES >= 64) v += dpp_get<0x143, 0xC>(v); /* row_bcast31 into rows 2,3 */
    return v;
}

/* Largest of a wave's 64 values, none of them negative, in every lane (through a scalar register); NaNs are passed over
 * as fmaxf does.  Six DPP steps of one VALU instruction and its wait states: the shuffles through LDS that this replaced
 * (ds_bpermute) cost a round trip of some 120 cycles a step, one after another, in kernels that are one chain of
 * latencies when a launch is a single row. */
__device__ __forceinline__ float wave_max(float v)
{
    v = fmaxf(v, dpp_get<0xB1>(v));               /* quad_perm [1,0,3,2] */
    v = fmaxf(v, dpp_get<0x4E>(v));               /* quad_perm [2,3,0,1] */
    v = fmaxf(v, dpp_get<0x141>(v));              /* row_half_mirror */
    v = fmaxf(v, dpp_get<0x140>(v));              /* row_mirror: every lane of a row of 16 has the row's */
    const int i = __builtin_bit_cast(int, v);     /* the four rows, not through row_bcast: an all-NaN row stays NaN */
    const float a = __builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 0)), b = __builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 16));
    const float c = __builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 32)), d = __builtin_bit_cast(float, __builtin_amdgcn_readlane(i, 48));
    return fmaxf(fmaxf(a, b), fmaxf(c, d));
}

/* x86 cvtps2dq + saturating packs (quantize_row_q8_k_sse.c:61-68): round to
 * nearest even; NaN, +-inf and anything outside int32 convert to INT_MIN, which
 * the packs saturate to -128 - also for +inf and for values >= 2^31 (a block of
 * magnitudes below 127/FLT_MAX has an infinite inverse scale). */
__device__ __forceinline__ int rne_sat_i8(float p)
{
    if (!(p < 2147483648.0f)) return -128;     /* NaN, +inf, >= 2^31 */
    const float r = __builtin_rintf(p);
    return (int)fminf(fmaxf(r, -128.0f), 127.0f);
}

/* q = RNE(e * scale) as rne_sat_i8 has it, four to a dword.  Adding 1.5 * 2^23 rounds to the nearest even integer and leaves it in the
 * low bits: a multiplication and an addition a value, and its byte as it is needed, where rne_sat_i8 takes six operations.  That holds
 * for |e * scale| <= 127.x, which is every value unless the block's scale or the value is infinite or NaN; then a result has an
 * exponent other than that of 2^23, and the wave goes through rne_sat_i8. */
template <int N>
__device__ __forceinline__ void q8_round(const float (&e)[N], float scale, u32 (&packed)[N / 4])
{
#pragma clang fp contract(off)
    u32 b[N], any = 0;
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float p = e[i] * scale;
        b[i] = __builtin_bit_cast(u32, p + 12582912.0f);
        any |= b[i];
    }
    if (__builtin_expect(__builtin_amdgcn_ballot_w64((any & 0xB4800000u) != 0) != 0, 0)) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const float p = e[i] * scale;
            b[i] = (u32)rne_sat_i8(p);
        }
    }
#pragma unroll
    for (int k = 0; k < N / 4; ++k)
        packed[k] = __builtin_amdgcn_perm(b[4 * k + 1], b[4 * k], 0x0c0c0400u) | __builtin_amdgcn_perm(b[4 * k + 3], b[4 * k + 2], 0x04000c0cu);
}

/* One wave turns 256 fp32 values (lane l holds elements 4l..4l+3 in e) into
 * the 292-byte Q8_K block at `out` (global or LDS), with the reference's rules
 * (quantize_row_q8_k_sse.c:22-82): the scale comes from the FIRST element of
 * largest magnitude, sign kept, iscale = -127/max, q = RNE(x*iscale)
 * saturated, bsums over 16 elements, d = 1/iscale; an all-zero block is 292
 * zero bytes. */
__device__ __forceinline__ void q8k_quantize_block(const float (&e)[4], int lane, uint8_t *out)
{
    float lmax = 0.0f, smax = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float ax = fabsf(e[i]);
        if (ax > lmax) { lmax = ax; smax = e[i]; }
    }
    /* elements go up with the lane: the first lane that holds the maximum has the first of the largest elements */
    const float amax = wave_max(lmax);
    const int first = __builtin_ctzll(__builtin_amdgcn_ballot_w64(lmax == amax));
    smax = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, smax), first));
    if (amax == 0.0f) {
        reinterpret_cast<u32 *>(out)[lane] = 0;
        if (lane < 9) reinterpret_cast<u32 *>(out)[64 + lane] = 0;
        return;
    }
    const float iscale = -127.0f / smax;
    u32 packed[1];
    q8_round(e, iscale, packed);
    int s = dot4((int)packed[0], 0x01010101, 0);
    reinterpret_cast<u32 *>(out + 4)[lane] = packed[0];
    s = group_sum<4>(s);                       /* 16 consecutive elements = 4 lanes */
    /* two sums a store, so that the block leaves in whole dwords: the host looks for them one by one (ckq_host.c) */
    const u32 pair = ((u32)dpp_get<0x114>(s) & 0xffffu) | ((u32)s << 16);                /* row_shr:4 */
    if ((lane & 7) == 7) reinterpret_cast<u32 *>(out + 260)[lane >> 3] = pair;
    if (lane == 0) *reinterpret_cast<float *>(out) = 1.0f / iscale;
}
