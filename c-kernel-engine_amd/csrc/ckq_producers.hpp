/*
 * ckq_producers.hpp - the activation producers (fp32 -> Q8_K, SiLU(gate)*up ->
 * Q8_K, RMSNorm -> Q8_K) as device functions: the arithmetic of the stand-alone
 * producer kernels of ckq_kernels.hip, kept apart from their launch shapes.
 */
#pragma once
#include "ckq_device.hpp"

/* ---- SiLU(gate) * up as the reference's tile loop evaluates it -------------
 * (fused/prefill_fused_gemm.c:904-906, 1034-1040): g / (1 + expf(-g)), then
 * the product, each operation rounded to fp32.  exp is evaluated in double
 * and rounded once, which agrees with a correctly rounded expf. */
__device__ __forceinline__ float swiglu_value(float g, float u)
{
#pragma clang fp contract(off)
    const float e = (float)exp(-(double)g);
    const float s = g / (1.0f + e);
    return s * u;
}

/* One wave: 256-block `blk` (of bpr per row, rows ldx floats apart) of x, or of SiLU(x) * up, -> the Q8_K block at y + blk * 292.
 * Without SWIGLU rows lie end to end.  Block numbers have 32 bits (2 TB of input): the division by bpr in 64 was a fifth of the kernel's instructions. */
template <bool SWIGLU>
__device__ __forceinline__ void pro_quantize_block(const float *__restrict__ x, const float *__restrict__ up,
                                                   uint8_t *__restrict__ y, u32 blk, u32 bpr, long ldx, int lane)
{
    const size_t src = SWIGLU ? (size_t)(blk / bpr) * ldx + (blk % bpr) * 256u : (size_t)blk * 256u;
    const float4 v = reinterpret_cast<const float4 *>(x + src)[lane];
    float e[4] = {v.x, v.y, v.z, v.w};
    if constexpr (SWIGLU) {
        const float4 w = reinterpret_cast<const float4 *>(up + src)[lane];
        e[0] = swiglu_value(e[0], w.x); e[1] = swiglu_value(e[1], w.y);
        e[2] = swiglu_value(e[2], w.z); e[3] = swiglu_value(e[3], w.w);
    }
    q8k_quantize_block(e, lane, y + (size_t)blk * 292);
}

/* ---- RMSNorm -> Q8_K (reference: src/kernels/fused/rmsnorm_q8_k_fused.c:54-142
 * as an FMA build compiles it) ------------------------------------------------
 * The sum of squares must be the reference's to the bit, or rstd moves by an
 * ulp and quants flip: eight strided lanes (lane j takes x[8i+j]) each a chain
 * of fused multiply-adds, combined as ((l0+l4)+(l1+l5)) + ((l2+l6)+(l3+l7)). */

/* The row lies in LDS chain by chain: element 8 i + j at xs[j * rms_pitch(D) + i], so that a chain is read 16 bytes at a
 * time.  The pitch of D/8 + 8 floats puts the eight chains' reads, and the 64 lanes of a staging store, on different banks
 * (D/8 is a multiple of 32). */
__host__ __device__ __forceinline__ constexpr int rms_pitch(int D) { return D / 8 + 8; }
__host__ __device__ __forceinline__ constexpr size_t rms_lds_bytes(size_t D) { return (8 * (D / 8 + 8) + 8) * sizeof(float); }

/* Lane l of a wave stores elements 4 l .. 4 l + 3 of 256-block b. */
__device__ __forceinline__ void rms_stage(float *xs, int D, int b, int lane, const float4 v)
{
    float *p = xs + 4 * (lane & 1) * rms_pitch(D) + 32 * b + (lane >> 1);
    p[0] = v.x;
    p[rms_pitch(D)] = v.y;
    p[2 * rms_pitch(D)] = v.z;
    p[3 * rms_pitch(D)] = v.w;
}

__device__ __forceinline__ float4 rms_unstage(const float *xs, int D, int b, int lane)
{
    const float *p = xs + 4 * (lane & 1) * rms_pitch(D) + 32 * b + (lane >> 1);
    return make_float4(p[0], p[rms_pitch(D)], p[2 * rms_pitch(D)], p[3 * rms_pitch(D)]);
}

/* Thread j < 8 of the block walks chain j and leaves its sum behind the row.  The chain is serial, one multiply-add
 * after another, and waits for LDS once a 256-block: the compiler moves the reads of the next 32 values to where they are used. */
__device__ __forceinline__ void rms_chain(float *xs, int D, int j)
{
    const float4 *x = reinterpret_cast<const float4 *>(xs + j * rms_pitch(D));
    float acc = 0.0f;
    float4 cur[8], nxt[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) cur[u] = x[u];
    const int nb = D / 256;
    for (int b = 0; b < nb; ++b) {
        const float4 *xn = x + 8 * (b + 1 < nb ? b + 1 : b);
#pragma unroll
        for (int u = 0; u < 8; ++u) nxt[u] = xn[u];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            acc = __fmaf_rn(cur[u].x, cur[u].x, acc);
            acc = __fmaf_rn(cur[u].y, cur[u].y, acc);
            acc = __fmaf_rn(cur[u].z, cur[u].z, acc);
            acc = __fmaf_rn(cur[u].w, cur[u].w, acc);
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) cur[u] = nxt[u];
    }
    xs[8 * rms_pitch(D) + j] = acc;
}

/* The same for rows that share their CU with one other at most.  A multiply-add of the chain takes some eight cycles, and the values should be there
 * before it: 32 are read while the 32 before them are added.  The reads are volatile because the compiler moves ordinary ones to
 * where they are used, as it does above, where every 32 values wait for LDS.  4096 wide, one row 4.2 -> 3.9 us, 256 rows 5.4 -> 5.1, 8192 wide 7.2 -> 6.3; but
 * the 64 registers keep a second block of sixteen waves off the CU (512 rows 6.8 -> 8.5, of eight waves 6.9 -> 6.5).  Sixteen values ahead 4.1 and 6.8; a ring of
 * 32 filled four at a time 4.4 and 7.3; whole waves, a chain to every sixteen lanes that broadcast it their values, 4.4 and 7.0. */
typedef float rms_v4f __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void rms_chain_ahead(float *xs, int D, int j)
{
    typedef const volatile __attribute__((address_space(3))) rms_v4f *lds_ptr;
    const lds_ptr x = (lds_ptr)(const rms_v4f *)(xs + j * rms_pitch(D));
    float acc = 0.0f;
    rms_v4f even[8], odd[8];
    auto load = [&](rms_v4f (&v)[8], int b) {
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = x[8 * b + u];
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const rms_v4f (&v)[8]) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = __builtin_fmaf(v[u][k], v[u][k], acc);
        __builtin_amdgcn_sched_barrier(0);
    };
    const int nb = D / 256;
    load(even, 0);
    int b = 0;
    for (; b + 2 < nb; b += 2) {
        load(odd, b + 1);
        add(even);
        load(even, b + 2);
        add(odd);
    }
    if (b + 1 < nb) load(odd, b + 1);
    add(even);
    if (b + 1 < nb) add(odd);
    xs[8 * rms_pitch(D) + j] = acc;
}

/* rstd from the eight chain sums (every thread derives the same value).
 * sqrtf and '/' are the correctly rounded ones (the __fsqrt_rn intrinsic is not). */
__device__ __forceinline__ float rms_rstd(const float *xs, int D, float eps)
{
    const float4 *l = reinterpret_cast<const float4 *>(xs + 8 * rms_pitch(D));
    const float4 a = l[0], b = l[1];
    const float s04 = a.x + b.x, s15 = a.y + b.y, s26 = a.z + b.z, s37 = a.w + b.w;
    const float sum_sq = (s04 + s15) + (s26 + s37);
    return 1.0f / sqrtf(sum_sq / (float)D + eps);
}

/* One wave: n = (x*rstd)*gamma with two roundings, scale from the largest |n|
 * of the block (unlike quantize_row_q8_k's signed first-largest), iscale =
 * -127/max, d = 1/iscale, q = RNE(n*iscale) saturated; lane l owns 4l..4l+3. */
__device__ __forceinline__ void rms_quant_block(const float4 xv, const float4 gv, float rstd, int lane, uint8_t *out)
{
    const float e[4] = {__fmul_rn(__fmul_rn(xv.x, rstd), gv.x), __fmul_rn(__fmul_rn(xv.y, rstd), gv.y),
                        __fmul_rn(__fmul_rn(xv.z, rstd), gv.z), __fmul_rn(__fmul_rn(xv.w, rstd), gv.w)};
    const float amax = wave_max(fmaxf(fmaxf(fabsf(e[0]), fabsf(e[1])), fmaxf(fabsf(e[2]), fabsf(e[3]))));
    if (amax == 0.0f) {
        reinterpret_cast<u32 *>(out)[lane] = 0;
        if (lane < 9) reinterpret_cast<u32 *>(out)[64 + lane] = 0;
        return;
    }
    const float iscale = __fdiv_rn(-127.0f, amax);
    u32 packed[1];
    q8_round(e, iscale, packed);
    int sum = dot4((int)packed[0], 0x01010101, 0);
    reinterpret_cast<u32 *>(out + 4)[lane] = packed[0];
    sum = group_sum<4>(sum);
    if ((lane & 3) == 3) reinterpret_cast<int16_t *>(out + 260)[lane >> 2] = (int16_t)sum;
    if (lane == 0) *reinterpret_cast<float *>(out) = __fdiv_rn(1.0f, iscale);
}

/* A block of nw waves turns row x (D floats) into its D/256 Q8_K blocks at y.  Wave w owns 256-blocks w, w + nw, ...;
 * the x and gamma of its first GREG blocks are loaded at the start and kept in registers across the chain, so a row of
 * up to GREG * nw blocks costs one round trip to memory.  AHEAD: which form of the chain.  smem: rms_lds_bytes(D). */
template <int GREG, bool AHEAD>
__device__ __forceinline__ void rms_row(const float *__restrict__ x, const float *__restrict__ gamma,
                                        uint8_t *__restrict__ y, int D, float eps, float *xs)
{
    const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_block(), nw = blockDim.x >> 6;
    const int nb = D / 256;
    float4 xv[GREG], gv[GREG];
#pragma unroll
    for (int r = 0; r < GREG; ++r) xv[r] = reinterpret_cast<const float4 *>(x + 256 * min(wave + nw * r, nb - 1))[lane];
#pragma unroll
    for (int r = 0; r < GREG; ++r) gv[r] = reinterpret_cast<const float4 *>(gamma + 256 * min(wave + nw * r, nb - 1))[lane];
#pragma unroll
    for (int r = 0; r < GREG; ++r)
        if (wave + nw * r < nb) rms_stage(xs, D, wave + nw * r, lane, xv[r]);
    for (int b = wave + nw * GREG; b < nb; b += nw) rms_stage(xs, D, b, lane, reinterpret_cast<const float4 *>(x + 256 * b)[lane]);
    __syncthreads();
    if (tid < 8) {
        if constexpr (AHEAD) rms_chain_ahead(xs, D, tid);
        else                 rms_chain(xs, D, tid);
    }
    __syncthreads();
    const float rstd = rms_rstd(xs, D, eps);
#pragma unroll
    for (int r = 0; r < GREG; ++r) {
        const int b = wave + nw * r;
        if (b < nb) rms_quant_block(xv[r], gv[r], rstd, lane, y + (size_t)b * 292);
    }
    for (int b = wave + nw * GREG; b < nb; b += nw)
        rms_quant_block(reinterpret_cast<const float4 *>(x + 256 * b)[lane], reinterpret_cast<const float4 *>(gamma + 256 * b)[lane], rstd, lane,
                        y + (size_t)b * 292);
}
