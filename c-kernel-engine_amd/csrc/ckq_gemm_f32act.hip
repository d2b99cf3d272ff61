/*
 * ckq_gemm_f32act.hip - several tokens of fp32 activations against Q4_K, Q6_K or Q8_0 weights, nothing
 * quantized, on the bf16 matrix cores with fp32 precision.
 *
 *   C[t][n] = sum over scale groups s:  scale(n,s) * sum_{k in s} q(n,k) * x(t,k)  (+ bias[n]);   Q4_K below
 * (reference: gemm_kernels_q4k.c:53-101, gemm_kernels_q6k.c:39-76, gemm_kernels_q8_0.c:254-277, under the token
 * loops of gemm_nt_q4_k / _q6_k / _q8_0).
 *
 * Exactness.  The integers q (4 to 8 bits) are exact in bf16.  An fp32 activation is cut into three bf16 parts,
 * x = hi + mid + lo, each the leading 8 bits of what is left: 24 bits, so the cut is exact (of x 2^24, so that the parts of the
 * smallest numbers are normal too; the scales carry the 2^-24).  Every product of an integer and a part fits fp32, the matrix
 * core adds in fp32, and the scale is applied to the sum of a group in fp32.
 *
 * Precision: rms error against 64 bits no larger than the one-token kernel's (4096 wide, activations of mean 0: Q4_K 1.0e-7
 * against 1.6e-7, Q6_K 1.0e-7 against 1.6e-7, Q8_0 1.0e-7 against 1.25e-7; 11008 wide 1.2 / 1.4 / 1.2e-7 against 1.65 / 1.6 / 1.3e-7;
 * the same for mean 1 and 4).  Three things keep it there:
 * - A weight of Q4_K is s q - m (s = d sc, m = dmin mn, per 32 elements), and s sum(q x) - m sum(x) would cancel after both
 *   sums were rounded (2.4e-7, with activations of mean 1 1.4e-6).  So the integers are centred: c = rint(m / s) brings q - c
 *   around zero, and what is left of the min, m - c s, at most s / 2, multiplies sum(x).
 * - The matrix core cuts off the bits of a sum below its largest term's, towards minus infinity: every sum comes out a little
 *   low, and hundreds of groups add that up (a third of the error at 4096, more than half at 11008).  Every other group
 *   therefore multiplies -x, its scale negated too.
 * - Two groups are added before they meet the running sum, which then takes half as many roundings.
 * Results that are not finite - an activation is not, or is beyond 2^90 or so - are summed again term by term (exact_output),
 * as the kernel for one token forms them.
 *
 * Mapping.  v_mfma_f32_32x32x16_bf16, tokens as rows (A), weight rows as columns (B): a lane holds ONE weight row,
 * so its scale is a register of the lane and one multiply-add per output and group applies it.  A lane (column
 * l % 32, half l / 32) takes the elements its half of the raw bytes holds, straight from memory; the activations are
 * read in the same order, so no byte moves between lanes.  The rest of the min in Q4_K is one more MFMA per group:
 * the lane's share of the group's sum of x against the row's factor, both cut in three.
 *
 * Block = 8 waves on one tile of 32 tokens x 32 R weight rows; the waves cut K into eight contiguous runs and add
 * their partial tiles through LDS, in pairs.  Each wave loads its own activations half a step or a step ahead, a
 * contiguous run per token, and turns them through LDS (a lane loading its own row would touch 64 cache lines per instruction: 40 us
 * instead of 36 at 96 x 4096 x 4096, Q6_K; one token per pass over the weights, as the streaming kernel does it, 245 us);
 * no other wave reads them, so the loop has no barrier.  Cutting the activations in a launch of its own and reading the
 * parts back (6 bytes per element instead of 4) was timed with the cut left out: 96 x 4096 x 4096 Q6_K 32.0 -> 26.7 us, Q8_0 29.3 -> 26.4, of which a launch that cuts
 * takes 2.5 back; not built.
 *
 * Weights.  The address path takes a wave's load in 16 to 22 cycles where quads of lanes read adjacent bytes, in 64 where every lane
 * has a row of its own, and in 160 where the rows' bytes are not on dwords either (measured, 16 bytes a lane, L2).  Q6_K
 * and Q8_0, whose blocks are only 2-byte aligned, therefore come in memory order like the activations (gemm_f32run_kernel, 96 x 4096 x
 * 4096: Q6_K 36.1 -> 31.1 us, Q8_0 36.3 -> 27.6; 200 x 5000 x 8192 Q6_K 207 -> 162, Q8_0 187 -> 145; same bits).  Where a wave's share is
 * shorter than a run (SHORT) that would load the same weights up to four times and wait for them in turn: the block loads them once, all
 * loads under way together, and the smaller tile leaves room for a second block on the CU (Q6_K 75 x 7670 x 512 12.1 -> 10.5 us,
 * 200 x 5000 x 1536 42.1 -> 31.9; a run per wave 14.2 and 42.1).  A row per lane stays (gemm_f32row_kernel) for Q4_K, 16-byte aligned and two
 * loads a step, which loses in memory order (27.5 -> 29.3), and for the sizes named at the launcher.
 *
 * Grid: token groups fastest, so the blocks that share weights run side by side.
 * Bound: VALU issue, on the CUs that have a block.  By the counters at 96 x 4096 x 4096 (two row tiles, 192 blocks) a wave issues 714 / 760 / 519 vector
 * operations per 64 elements in Q4_K / Q6_K / Q8_0: 220-260 cut x, shared by the row tiles, some 60 turn weights and activations
 * through LDS, and per row tile 210-230 / 230 / 110 form the integers and apply the scales, half of them at half rate (conversions, byte permutes).
 * They issue in 78 / 72 / 56 % of the cycles; the matrix cores are busy in 23 / 18 / 20 %, LDS bank conflicts take 0 / 4 / 4 %.  The
 * centring of Q4_K is about 60 of the operations: 96 x 4096 x 4096 23 -> 27 us.
 */
#include "ckq_gemm_common.hpp"
#include "ckq_gemm_f32act.hpp"
#include <type_traits>

namespace {

constexpr int F32_WAVES = 8;
/* factors of the activations and of the scales of group g of a step */
__device__ constexpr float x_up(int g) { return g & 1 ? -16777216.0f : 16777216.0f; }
__device__ constexpr float x_down(int g) { return 1.0f / x_up(g); }

__device__ __forceinline__ u32 pack_bf16(float lo, float hi)      /* two floats whose low 16 bits are to be dropped */
{
    return __builtin_amdgcn_perm(__builtin_bit_cast(u32, hi), __builtin_bit_cast(u32, lo), 0x07060302u);
}

/* eight floats -> their three bf16 parts as MFMA operands (of an infinity or a NaN: NaNs) */
struct Cut { ckq_v4i hi, mid, lo; };
__device__ __forceinline__ float top16(float v) { return __builtin_bit_cast(float, __builtin_bit_cast(u32, v) & 0xffff0000u); }
__device__ __forceinline__ void cut8(const float *x, Cut &c)
{
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        float m[2], l[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const float v = x[2 * i + j];
            m[j] = v - top16(v);
            l[j] = m[j] - top16(m[j]);
        }
        c.hi[i]  = (int)pack_bf16(x[2 * i], x[2 * i + 1]);
        c.mid[i] = (int)pack_bf16(m[0], m[1]);
        c.lo[i]  = (int)pack_bf16(l[0], l[1]);
    }
}

__device__ __forceinline__ ckq_v16f mfma_bf16(ckq_v4i a, ckq_v4i b, ckq_v16f c)
{
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(ckq_v8bf, a), __builtin_bit_cast(ckq_v8bf, b), c, 0, 0, 0);
}

/* Signed byte i of a dword as a float, in one instruction (the compiler extends the byte with an instruction of its own). */
__device__ __forceinline__ float sbyte_f32(u32 v, int i)
{
    float f;
    switch (i) {
    case 0: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_0" : "=v"(f) : "v"(v)); break;
    case 1: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_1" : "=v"(f) : "v"(v)); break;
    case 2: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_2" : "=v"(f) : "v"(v)); break;
    default: asm("v_cvt_f32_i32_sdwa %0, sext(%1) dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:BYTE_3" : "=v"(f) : "v"(v)); break;
    }
    return f;
}

/* Eight signed bytes -> bf16x8 (exact). */
__device__ __forceinline__ ckq_v4i bytes_to_bf16(u32 b0, u32 b1)
{
    ckq_v4i o;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        o[i]     = (int)pack_bf16(sbyte_f32(b0, 2 * i), sbyte_f32(b0, 2 * i + 1));
        o[2 + i] = (int)pack_bf16(sbyte_f32(b1, 2 * i), sbyte_f32(b1, 2 * i + 1));
    }
    return o;
}

/* ---- formats ------------------------------------------------------------------------------------
 * STEP elements of K per step, NG scale groups of 8 * NK elements per lane half in it.
 *   Raw / load      the step's bytes of one weight row that this lane's half decodes: Q4_K from memory, the others from LDS
 *   src_elem(c)     first element of 16-byte chunk c of the activations: of the step (Q4_K, 16 chunks), of its phase p (8)
 *   chunk(g, h, i)  (Q4_K) which chunk holds floats 4 i .. 4 i + 3 of group g for lane half h
 *   RUN, BYTES      steps of a run of weights in LDS and its bytes; LANES lanes bring a row's, one row is PITCH bytes from the next;
 *                   SHIFT: they come from the dword they start in and are shifted into place
 *   operand(g, i)   bf16x8 of the lane's elements 8 i .. 8 i + 7 of group g
 *   scale(g)        fp32 factor of the group; MIN: rest(g), the factor of the group's sum of x
 *   weight(blk, e, i)  element e + i of a block, e a multiple of 16 and i below 16, for exact_output */
struct F32Q4K {
    static constexpr int STEP = 64, NG = 2, NK = 2;
    static constexpr bool MIN = true;
    struct Raw { u32 hdr[4], qs[4]; };
    static __device__ __forceinline__ void load_row(Raw &w, const uint8_t *row, int step, int h, int)
    {
        const uint8_t *blk = row + (u32)(step >> 2) * 144u;
        ld16<4>(w.hdr, blk);
        ld16<4>(w.qs, blk + 16 + 32 * (step & 3) + 16 * h);
    }
    static __device__ __forceinline__ u32 src_elem(int step, int c, int) { return 64u * (u32)step + 4u * c; }
    static __device__ __forceinline__ int chunk(int g, int h, int i) { return 8 * g + 4 * h + i; }
    struct Dec { float s[2], rest[2]; u32 off[2]; };          /* off: 128 - c in every byte */
    static __device__ __forceinline__ void decode(Dec &d, const Raw &w, int step, int)
    {
        u32 sc2, mn2;
        k4_scale_pair(w.hdr[1], w.hdr[2], w.hdr[3], step & 3, &sc2, &mn2);
        const float dd = h2f(w.hdr[0] & 0xffff), dm = h2f(w.hdr[0] >> 16);
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const float m = dm * x_down(g) * (float)((mn2 >> (8 * g)) & 0xff);
            d.s[g] = dd * x_down(g) * (float)((sc2 >> (8 * g)) & 0xff);
            /* 0 to 127, so that q - c is a byte; 0 for a scale of 0 (m / 0 or 0 / 0) and for a min of the other sign */
            float c = __builtin_rintf(m * __builtin_amdgcn_rcpf(d.s[g]));
            c = d.s[g] == 0.0f ? 0.0f : fminf(fmaxf(c, 0.0f), 127.0f);
            d.off[g] = 0x80808080u - __builtin_amdgcn_perm(0u, (u32)c, 0u);
            d.rest[g] = fmaf(-c, d.s[g], m);
        }
    }
    static __device__ __forceinline__ ckq_v4i operand(const Raw &w, const Dec &d, int g, int i)
    {
        u32 v[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const u32 q = g ? w.qs[2 * i + j] >> 4 : w.qs[2 * i + j];
            v[j] = ((q & 0x0f0f0f0fu) + d.off[g]) ^ 0x80808080u;      /* no carries between bytes */
        }
        return bytes_to_bf16(v[0], v[1]);
    }
    static constexpr int BLOCK = 256, WBLOCK = 144;
    static __device__ __forceinline__ float weight(const uint8_t *blk, int e, int i)
    {
        u32 sc2, mn2;
        k4_scale_pair(ld4<4>(blk + 4), ld4<4>(blk + 8), ld4<4>(blk + 12), e >> 6, &sc2, &mn2);
        const int odd = (e >> 5) & 1;
        const float s = h2f(ld2(blk)) * (float)((sc2 >> (8 * odd)) & 0xff), m = h2f(ld2(blk + 2)) * (float)((mn2 >> (8 * odd)) & 0xff);
        const u32 b = blk[16 + 32 * (e >> 6) + (e & 31) + i];
        return s * (float)(odd ? b >> 4 : b & 15u) - m;
    }
};

struct F32Q6K {
    static constexpr int STEP = 64, NG = 4, NK = 1;       /* a step: 16-runs o of the four 32-runs of one 128-half n */
    static constexpr int RUN = 4, BYTES = 210, LANES = 16, PITCH = 240, SHORT_RUNS = 6;
    static constexpr bool SHIFT = true, MIN = false;
    struct Raw { u32 ql0[2], ql1[2], qh[2], sc[2], d; };
    static __device__ __forceinline__ void load_row(Raw &w, const uint8_t *row, int step, int h, int)
    {
        const uint8_t *blk = row + (u32)(step >> 2) * 210u;
        const int n = (step >> 1) & 1, o = step & 1;
        ld8<2>(w.ql0, blk + 64 * n + 16 * o + 8 * h);
        ld8<2>(w.ql1, blk + 64 * n + 32 + 16 * o + 8 * h);
        ld8<2>(w.qh, blk + 128 + 32 * n + 16 * o + 8 * h);
        ld8<2>(w.sc, blk + 192 + 8 * n);
        w.d = ld2(blk + 208);
    }
    static __device__ __forceinline__ u32 src_elem(int step, int c, int)
    {
        return 128u * (u32)(step >> 1) + 16u * (step & 1) + 32u * (c >> 2) + 4u * (c & 3);
    }
    static __device__ __forceinline__ int chunk(int g, int h, int i) { return 4 * g + 2 * h + i; }
    static __device__ __forceinline__ void load(Raw &w, const uint8_t *row, int step, int h)
    {
        const int n = (step >> 1) & 1, o = step & 1;
        auto two = [&](u32 *d, int ofs) {
            const int2 v = *reinterpret_cast<const int2 *>(row + ofs);
            d[0] = (u32)v.x; d[1] = (u32)v.y;
        };
        two(w.ql0, 64 * n + 16 * o + 8 * h);
        two(w.ql1, 64 * n + 32 + 16 * o + 8 * h);
        two(w.qh, 128 + 32 * n + 16 * o + 8 * h);
        two(w.sc, 192 + 8 * n);
        w.d = *reinterpret_cast<const u32 *>(row + 208) & 0xffffu;
    }
    static __device__ __forceinline__ u32 src_elem(int step, int p, int c, int)
    {
        return 128u * (u32)(step >> 1) + 16u * (step & 1) + 32u * (u32)(2 * p + (c >> 2)) + 4u * (u32)(c & 3);
    }
    struct Dec { float s[4]; };
    static __device__ __forceinline__ void decode(Dec &d, const Raw &w, int step, int)
    {
        const float dd = h2f(w.d);
        const int o = step & 1;
#pragma unroll
        for (int g = 0; g < 4; ++g) d.s[g] = dd * x_down(g) * (float)sbyte(w.sc[g >> 1], o + 2 * (g & 1));
    }
    static __device__ __forceinline__ ckq_v4i operand(const Raw &w, const Dec &, int g, int)
    {
        u32 q[2];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const u32 l = (g & 1) ? w.ql1[j] : w.ql0[j];
            const u32 nib = (g >> 1) ? (l >> 4) & 0x0f0f0f0fu : l & 0x0f0f0f0fu;
            const u32 hb = g == 0 ? w.qh[j] << 4 : g == 1 ? w.qh[j] << 2 : g == 2 ? w.qh[j] : w.qh[j] >> 2;
            const u32 v = nib | (hb & 0x30303030u);
            q[j] = ((v | 0x80808080u) - 0x20202020u) ^ 0x80808080u;      /* no borrows between bytes */
        }
        return bytes_to_bf16(q[0], q[1]);
    }
    static constexpr int BLOCK = 256, WBLOCK = 210;
    static __device__ __forceinline__ float weight(const uint8_t *blk, int e, int i)
    {
        const int n = e >> 7, r = (e >> 5) & 3, l = (e & 31) + i;
        const u32 lo = blk[64 * n + 32 * (r & 1) + l], hi = blk[128 + 32 * n + l];
        const int q = (int)(((r >> 1) ? lo >> 4 : lo & 15u) | ((hi >> (2 * r)) & 3u) << 4) - 32;
        return h2f(ld2(blk + 208)) * (float)(int8_t)blk[192 + (e >> 4)] * (float)q;
    }
};

struct F32Q80 {
    static constexpr int STEP = 64, NG = 2, NK = 2;       /* two 32-blocks; the second is missing in the last step of an odd count */
    static constexpr int RUN = 2, BYTES = 136, LANES = 9, PITCH = 144, SHORT_RUNS = 10;
    static constexpr bool SHIFT = false, MIN = false;
    struct Raw { u32 q[2][4]; u32 d[2]; };
    static __device__ __forceinline__ void load_row(Raw &w, const uint8_t *row, int step, int h, int K)
    {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const uint8_t *blk = row + (u32)min(2 * step + g, K / 32 - 1) * 34u;
            w.d[g] = ld2(blk);
            ld16<2>(w.q[g], blk + 2 + 16 * h);
        }
    }
    static __device__ __forceinline__ u32 src_elem(int step, int c, int K)
    {
        return 32u * (u32)min(2 * step + (c >> 3), K / 32 - 1) + 4u * (c & 7);
    }
    static __device__ __forceinline__ int chunk(int g, int h, int i) { return 8 * g + 4 * h + i; }
    static __device__ __forceinline__ void load(Raw &w, const uint8_t *row, int step, int h)
    {
        /* quants of block j start at byte 34 j + 2: two aligned reads around them */
        auto block = [&](auto jc) __attribute__((always_inline)) {
            constexpr int j = decltype(jc)::value, first = (34 * j + 2) / 4, base = first & ~3, sh = (34 * j + 2) & 2, g = j & 1;
            const ckq_v4i a = *reinterpret_cast<const ckq_v4i *>(row + 4 * base + 16 * h), b = *reinterpret_cast<const ckq_v4i *>(row + 4 * base + 16 + 16 * h);
            auto dw = [&](int i) { return (u32)(i < 4 ? a[i] : b[i - 4]); };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int k = first - base + i;
                w.q[g][i] = sh ? __builtin_amdgcn_alignbyte(dw(k + 1), dw(k), 2) : dw(k);
            }
            const u32 d = *reinterpret_cast<const u32 *>(row + ((34 * j) & ~3));
            w.d[g] = (34 * j) & 2 ? d >> 16 : d & 0xffffu;
        };
        if (step & 1) { block(std::integral_constant<int, 2>{}); block(std::integral_constant<int, 3>{}); }
        else          { block(std::integral_constant<int, 0>{}); block(std::integral_constant<int, 1>{}); }
    }
    static __device__ __forceinline__ u32 src_elem(int step, int p, int c, int K) { return 32u * (u32)min(2 * step + p, K / 32 - 1) + 4u * (u32)c; }
    struct Dec { float s[2]; };
    static __device__ __forceinline__ void decode(Dec &d, const Raw &w, int step, int K)
    {
        d.s[0] = h2f(w.d[0]) * x_down(0);
        d.s[1] = 2 * step + 1 < K / 32 ? h2f(w.d[1]) * x_down(1) : 0.0f;
    }
    static __device__ __forceinline__ ckq_v4i operand(const Raw &w, const Dec &, int g, int i)
    {
        return bytes_to_bf16(w.q[g][2 * i], w.q[g][2 * i + 1]);
    }
    static constexpr int BLOCK = 32, WBLOCK = 34;
    static __device__ __forceinline__ float weight(const uint8_t *blk, int e, int i) { return h2f(ld2(blk)) * (float)(int8_t)blk[2 + e + i]; }
};

/* One output term by term; a NaN stays one. */
template <class F>
__device__ __forceinline__ float exact_output(const uint8_t *w, const float *x, int K)
{
    float sum = 0.0f;
#pragma unroll 1
    for (int k = 0; k < K && sum == sum; k += 16) {
        const uint8_t *const blk = w + (u32)(k / F::BLOCK) * (u32)F::WBLOCK;
#pragma unroll
        for (int i = 0; i < 16; ++i) sum += F::weight(blk, k % F::BLOCK, i) * x[k + i];
    }
    return sum;
}

template <class F, int R>
__global__ void __launch_bounds__(64 * F32_WAVES, 2)
gemm_f32row_kernel(const float *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ bias, float *__restrict__ C,
                   int M, int N, int K, long wrow, long ldc, int ntg)
{
    /* a wave's activations of one step, token t at 256 t, chunk c in slot c ^ (t & 15); at the end the partial tiles */
    __shared__ __attribute__((aligned(16))) uint8_t xs_all[F32_WAVES][32 * 256];
    const int lane = threadIdx.x & 63, wave = wave_in_block();
    const int col = lane & 31, half = lane >> 5;
    const int t0 = (int)(blockIdx.x % (u32)ntg) * 32, n0 = (int)(blockIdx.x / (u32)ntg) * 32 * R;
    const int steps = (K + F::STEP - 1) / F::STEP, per = (steps + F32_WAVES - 1) / F32_WAVES;
    const int s0 = wave * per, s1 = min(steps, s0 + per);

    const float *xsrc[8];          /* row of the token this lane fetches in load instruction j */
#pragma unroll
    for (int j = 0; j < 8; ++j) xsrc[j] = A + (size_t)min(t0 + 4 * j + (lane >> 4), M - 1) * (size_t)K;
    const uint8_t *wr[R];
#pragma unroll
    for (int r = 0; r < R; ++r) wr[r] = B + (size_t)min(n0 + 32 * r + col, N - 1) * (size_t)wrow;

    ckq_v16f acc[R], zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = zero;

    uint8_t *const xs = xs_all[wave];
    typename F::Raw w[R], wn[R];
    ckq_v4i xn[8];
    auto fetch = [&](int s) {
#pragma unroll
        for (int j = 0; j < 8; ++j) xn[j] = *reinterpret_cast<const ckq_v4i *>(xsrc[j] + F::src_elem(s, lane & 15, K));
#pragma unroll
        for (int r = 0; r < R; ++r) F::load_row(wn[r], wr[r], s, half, K);
    };
    auto take = [&]() {
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int t = 4 * j + (lane >> 4);
            *reinterpret_cast<ckq_v4i *>(xs + 256 * t + 16 * ((lane & 15) ^ (t & 15))) = xn[j];
        }
#pragma unroll
        for (int r = 0; r < R; ++r) w[r] = wn[r];
    };
    auto compute = [&](int s) {
        typename F::Dec dec[R];
#pragma unroll
        for (int r = 0; r < R; ++r) F::decode(dec[r], w[r], s, K);
        /* two groups at a time: their two terms are added before they meet the sum so far */
#pragma unroll
        for (int g0 = 0; g0 < F::NG; g0 += 2) {
            Cut c[2][F::NK];
            ckq_v4i pa[2];
#pragma unroll
            for (int g = 0; g < 2; ++g) {
                float x[F::NK * 8];
#pragma unroll
                for (int i = 0; i < 2 * F::NK; ++i) {
                    const ckq_v4i v = *reinterpret_cast<const ckq_v4i *>(xs + 256 * col + 16 * (F::chunk(g0 + g, half, i) ^ (col & 15)));
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int e = v[j];
                        x[4 * i + j] = __builtin_bit_cast(float, e) * x_up(g);
                    }
                }
#pragma unroll
                for (int k = 0; k < F::NK; ++k) cut8(x + 8 * k, c[g][k]);
                if constexpr (F::MIN) {
                    /* this half's share of the group's sum of x, cut in three; against the cut rest of the min, the six
                     * products that matter in one MFMA, which also adds the halves */
                    const float p = ((x[0] + x[1]) + (x[2] + x[3])) + ((x[4] + x[5]) + (x[6] + x[7])) +
                                    (((x[8] + x[9]) + (x[10] + x[11])) + ((x[12] + x[13]) + (x[14] + x[15])));
                    const float m = p - top16(p), l = m - top16(m);
                    pa[g] = ckq_v4i{(int)pack_bf16(p, p), (int)pack_bf16(m, m), (int)pack_bf16(p, l), 0};
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                ckq_v16f two, sum;
                if constexpr (F::MIN) {
                    two = zero;
#pragma unroll
                    for (int g = 0; g < 2; ++g) {
                        const float h = dec[r].rest[g0 + g], m = h - top16(h), l = m - top16(m);
                        two = mfma_bf16(pa[g], ckq_v4i{(int)pack_bf16(h, m), (int)pack_bf16(h, m), (int)pack_bf16(l, h), 0}, two);
                    }
                }
#pragma unroll
                for (int g = 0; g < 2; ++g) {
                    sum = zero;
#pragma unroll
                    for (int k = 0; k < F::NK; ++k) {
                        const ckq_v4i b = F::operand(w[r], dec[r], g0 + g, k);
                        sum = mfma_bf16(c[g][k].lo, b, sum);
                        sum = mfma_bf16(c[g][k].mid, b, sum);
                        sum = mfma_bf16(c[g][k].hi, b, sum);
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        two[i] = F::MIN || g ? fmaf(dec[r].s[g0 + g], sum[i], F::MIN && !g ? -two[i] : two[i]) : dec[r].s[g0 + g] * sum[i];
                }
#pragma unroll
                for (int i = 0; i < 16; ++i) acc[r][i] += two[i];
            }
        }
    };
    if (s0 < s1) fetch(s0);
    for (int s = s0; s < s1; ++s) {
        take();
        if (s + 1 < s1) fetch(s + 1);
        __builtin_amdgcn_sched_barrier(0);
        compute(s);
        __builtin_amdgcn_sched_barrier(0);
    }

    constexpr int RP = R < 2 ? 1 : 2;
    float *const red = reinterpret_cast<float *>(&xs_all[0][0]);     /* [wave][RP * 16][64] */
    static_assert(F32_WAVES * RP * 16 * 64 * sizeof(float) <= sizeof(xs_all), "the partial tiles fit the activations' place");
    bool fix = false;
    __syncthreads();                         /* every wave is done with its activations */
    /* the eight partial tiles through LDS, two row tiles at a time; wave w finishes sixteenths 2 w .. of every lane */
#pragma unroll
    for (int q = 0; q < R; q += RP) {
        __syncthreads();                     /* every wave is done with the buffer (and its loads have landed) */
#pragma unroll
        for (int r = 0; r < RP; ++r)
#pragma unroll
            for (int i = 0; i < 16; ++i) red[(wave * RP * 16 + 16 * r + i) * 64 + lane] = acc[q + r][i];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2 * RP; ++j) {
            const int o = 2 * RP * wave + j, i = o & 15;
            float p[F32_WAVES];
#pragma unroll
            for (int k = 0; k < F32_WAVES; ++k) p[k] = red[(k * RP * 16 + o) * 64 + lane];
            const float v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            const int n = n0 + 32 * (q + (o >> 4)) + col, t = t0 + 8 * (i >> 2) + 4 * half + (i & 3);
            fix = fix || !(fabsf(v) < __builtin_inff());
            if (n < N && t < M) C[(size_t)t * ldc + n] = bias ? v + bias[n] : v;
        }
    }
    if (fix) {
#pragma unroll 1
        for (int j = 0; j < 2 * R; ++j) {
            const int o = 2 * RP * wave + j % (2 * RP), i = o & 15;
            const int n = n0 + 32 * (j / (2 * RP) * RP + (o >> 4)) + col, t = t0 + 8 * (i >> 2) + 4 * half + (i & 3);
            if (n >= N || t >= M) continue;
            float *const out = C + (size_t)t * ldc + n;
            if (fabsf(*out) < __builtin_inff()) continue;
            const float v = exact_output<F>(B + (size_t)n * (size_t)wrow, A + (size_t)t * (size_t)K, K);
            *out = bias ? v + bias[n] : v;
        }
    }
}

template <class F, int R, bool SHORT> constexpr bool f32_two_blocks = R == 1 && SHORT;

template <class F, int R, bool SHORT>
__global__ void __launch_bounds__(64 * F32_WAVES, (f32_two_blocks<F, R, SHORT> ? 4 : 2))
gemm_f32run_kernel(const float *__restrict__ A, const uint8_t *__restrict__ B, const float *__restrict__ bias, float *__restrict__ C,
                   int M, int N, int K, long wrow, long ldc, int ntg)
{
    constexpr int ROWS = 32 * R, RPI = 64 / F::LANES, NWL = (ROWS + RPI - 1) / RPI;      /* rows per load instruction, instructions per run */
    constexpr int WLDS = ROWS * F::PITCH, XLDS = 32 * 128, RED = F32_WAVES * (R < 2 ? 1 : 2) * 16 * 64 * 4;
    constexpr int RUNS = SHORT ? F::SHORT_RUNS : F32_WAVES, USED = RUNS * WLDS + F32_WAVES * XLDS;
    constexpr int AHEAD = SHORT || R == 1 || std::is_same<F, F32Q80>::value ? 2 : 1;      /* phases of activations on their way, as registers allow */
    /* weights of a run each wave, or (SHORT) of all runs; of each wave the activations of a phase, token t at 128 t, chunk c in slot
     * c ^ (t / 2 % 8); at the end the partial tiles */
    __shared__ __attribute__((aligned(16))) uint8_t smem[USED > RED ? USED : RED];
    const int lane = threadIdx.x & 63, wave = wave_in_block();
    const int col = lane & 31, half = lane >> 5;
    const int t0 = (int)(blockIdx.x % (u32)ntg) * 32, n0 = (int)(blockIdx.x / (u32)ntg) * ROWS;
    const int steps = (K + F::STEP - 1) / F::STEP, per = (steps + F32_WAVES - 1) / F32_WAVES;
    const int s0 = wave * per, s1 = min(steps, s0 + per);
    uint8_t *const wl = smem + wave * WLDS, *const xs = smem + RUNS * WLDS + wave * XLDS;

    /* weights: row and chunk of this lane in load instruction j */
    const int w_row = lane / F::LANES, w_chunk = lane % F::LANES;
    const uint8_t *const wbase = B + (size_t)n0 * (size_t)wrow;
    const int left = N - 1 - n0;
    const u32 row_bytes = (u32)wrow, par = (u32)(uintptr_t)wbase & 2u;
    ckq_v4i wn[NWL];
    auto run_bytes = [&](int run) { return min((u32)F::BYTES, row_bytes - (u32)run * (u32)F::BYTES); };
    auto w_src = [&](int j, int run) {
        int r = RPI * j + min(w_row, RPI - 1);
        asm volatile("" : "+v"(r));                          /* formed when it is needed, not kept for every j */
        return (size_t)min(r, left) * row_bytes + (u32)run * (u32)F::BYTES;
    };
    auto load_w = [&](int j, int run) {
        u32 t[4];
        if constexpr (F::SHIFT) {
            /* from the dword the block starts in; the last chunk from byte 196 of it, so that no load passes the dword the block ends in.  Of a
             * matrix that begins or ends within a dword the two bytes beside it are read too (no allocation ends within a dword) and shifted away */
            ld16<4>(t, wbase - par + (((w_src(j, run) + par) & ~(size_t)3) + (u32)(w_chunk < 13 ? 16 * w_chunk : 196)));
        } else ld16<2>(t, wbase + (w_src(j, run) + min(16u * (u32)w_chunk, run_bytes(run) - 16u)));
        return ckq_v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
    };
    auto put_w = [&](uint8_t *dst, int j, int run, ckq_v4i b) {
        const int row = RPI * j + w_row;
        uint8_t *const d = dst + row * F::PITCH;
        const bool on = w_row < RPI && row < ROWS;
        if constexpr (F::SHIFT) {
            const u32 sh = ((u32)w_src(j, run) + par) & 2u;
            u32 v[5];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = (u32)b[i];
            /* the neighbour's first dword; lane 13 holds dwords 49 .. 52 of the block's 53 */
            v[4] = (u32)dpp_get<0x101>((int)(w_chunk == 13 ? v[3] : v[0]));
            ckq_v4i o;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[i] = (int)__builtin_amdgcn_alignbyte(v[i + 1], v[i], sh);
            if (on && w_chunk < 13) *reinterpret_cast<ckq_v4i *>(d + 16 * w_chunk) = o;
            if (on && w_chunk == 13) *reinterpret_cast<u32 *>(d + 208) = v[3] >> (8 * sh);
        } else if (run_bytes(run) == (u32)F::BYTES) {
            if (on && 16 * w_chunk + 16 <= F::BYTES) *reinterpret_cast<ckq_v4i *>(d + 16 * w_chunk) = b;
            else if (on) *reinterpret_cast<int2 *>(d + 16 * w_chunk) = int2{b[2], b[3]};         /* the last 16 of 136 bytes */
        } else if (on) {
            uint16_t *const e = reinterpret_cast<uint16_t *>(d + min(16u * (u32)w_chunk, run_bytes(run) - 16u));
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                e[2 * i] = (uint16_t)((u32)b[i] & 0xffffu);
                e[2 * i + 1] = (uint16_t)((u32)b[i] >> 16);
            }
        }
    };
    auto fetch_w = [&](int run) {
#pragma unroll
        for (int j = 0; j < NWL; ++j) wn[j] = load_w(j, run);
    };
    auto take_w = [&](int run) {
#pragma unroll
        for (int j = 0; j < NWL; ++j) put_w(wl, j, run, wn[j]);
        __builtin_amdgcn_wave_barrier();                     /* the wave's own LDS accesses stay in this order */
    };

    /* row of the token this lane fetches in load instruction j */
    const float *const xbase = A + (size_t)t0 * (size_t)K;
    typename std::conditional<SHORT, u32, size_t>::type xsrc[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) xsrc[j] = (size_t)min(8 * j + (lane >> 3), M - 1 - t0) * (size_t)K;
    ckq_v4i xn[AHEAD][4];
    auto fetch_x = [&](int s, int p) {
#pragma unroll
        for (int j = 0; j < 4; ++j) xn[p % AHEAD][j] = *reinterpret_cast<const ckq_v4i *>(xbase + (xsrc[j] + F::src_elem(s, p, lane & 7, K)));
    };
    auto take_x = [&](int p) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int t = 8 * j + (lane >> 3);
            *reinterpret_cast<ckq_v4i *>(xs + 128 * t + 16 * ((lane & 7) ^ (t >> 1 & 7))) = xn[p % AHEAD][j];
        }
        __builtin_amdgcn_wave_barrier();
    };

    ckq_v16f acc[R], two[R], zero;
#pragma unroll
    for (int i = 0; i < 16; ++i) zero[i] = 0.0f;
#pragma unroll
    for (int r = 0; r < R; ++r) acc[r] = two[r] = zero;

    if (s0 < s1) {
        if constexpr (!SHORT) fetch_w(s0 / F::RUN);
        fetch_x(s0, 0);
        if constexpr (AHEAD == 2) fetch_x(s0, 1);
    }
    if constexpr (SHORT) {
        constexpr int SHARE = (RUNS * NWL + F32_WAVES - 1) / F32_WAVES;        /* load instructions of a wave, all under way together */
        const int n = (steps + F::RUN - 1) / F::RUN * NWL;
        ckq_v4i v[SHARE];
#pragma unroll
        for (int q = 0; q < SHARE; ++q) {
            const int i = wave + F32_WAVES * q;
            if (i < n) v[q] = load_w(i % NWL, i / NWL);
        }
#pragma unroll
        for (int q = 0; q < SHARE; ++q) {
            const int i = wave + F32_WAVES * q, run = i / NWL;
            if (i < n) put_w(smem + run * WLDS, i % NWL, run, v[q]);
        }
        __syncthreads();
    }
    for (int s = s0; s < s1; ++s) {
        if constexpr (!SHORT)
            if (s == s0 || s % F::RUN == 0) {
                take_w(s / F::RUN);
                if ((s / F::RUN + 1) * F::RUN < s1) fetch_w(s / F::RUN + 1);
            }
        typename F::Raw w[R];
        typename F::Dec dec[R];
        const uint8_t *const ws = SHORT ? smem + s / F::RUN * WLDS : wl;
#pragma unroll
        for (int r = 0; r < R; ++r) {
            F::load(w[r], ws + (32 * r + col) * F::PITCH, s, half);
            F::decode(dec[r], w[r], s, K);
        }
        /* two phases of 32 elements a token: a scale group each, or two groups of 16 */
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            constexpr int NG = F::NG / 2;                    /* groups of a phase */
            take_x(p);
            if (AHEAD == 1 && p == 0) fetch_x(s, 1);
            else if (s + 1 < s1) fetch_x(s + 1, AHEAD == 1 ? 0 : p);
            __builtin_amdgcn_sched_barrier(0);
            Cut c[NG][F::NK];
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                float x[F::NK * 8];
#pragma unroll
                for (int i = 0; i < 2 * F::NK; ++i) {
                    const int ch = NG == 1 ? 4 * half + i : 4 * g + 2 * half + i;
                    const ckq_v4i v = *reinterpret_cast<const ckq_v4i *>(xs + 128 * col + 16 * (ch ^ (col >> 1 & 7)));
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const int e = v[j];
                        x[4 * i + j] = __builtin_bit_cast(float, e) * x_up(NG == 1 ? p : g);
                    }
                }
#pragma unroll
                for (int k = 0; k < F::NK; ++k) cut8(x + 8 * k, c[g][k]);
            }
#pragma unroll
            for (int r = 0; r < R; ++r) {
                if constexpr (NG == 1) {
                    ckq_v16f sum = zero;
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const ckq_v4i b = F::operand(w[r], dec[r], p, k);
                        sum = mfma_bf16(c[0][k].lo, b, sum);
                        sum = mfma_bf16(c[0][k].mid, b, sum);
                        sum = mfma_bf16(c[0][k].hi, b, sum);
                    }
                    /* two groups are added before they meet the sum so far */
#pragma unroll
                    for (int i = 0; i < 16; ++i) two[r][i] = p ? fmaf(dec[r].s[p], sum[i], two[r][i]) : dec[r].s[p] * sum[i];
                    if (p) {
#pragma unroll
                        for (int i = 0; i < 16; ++i) acc[r][i] += two[r][i];
                    }
                } else {
#pragma unroll
                    for (int g = 0; g < NG; ++g) {
                        const ckq_v4i b = F::operand(w[r], dec[r], 2 * p + g, 0);
                        ckq_v16f sum = mfma_bf16(c[g][0].lo, b, zero);
                        sum = mfma_bf16(c[g][0].mid, b, sum);
                        sum = mfma_bf16(c[g][0].hi, b, sum);
#pragma unroll
                        for (int i = 0; i < 16; ++i) two[r][i] = g ? fmaf(dec[r].s[2 * p + g], sum[i], two[r][i]) : dec[r].s[2 * p + g] * sum[i];
                    }
#pragma unroll
                    for (int i = 0; i < 16; ++i) acc[r][i] += two[r][i];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        }
    }

    constexpr int RP = R < 2 ? 1 : 2;
    float *const red = reinterpret_cast<float *>(smem);      /* [wave][RP * 16][64] */
    bool fix = false;
    __syncthreads();                         /* every wave is done with its weights and activations */
    /* the eight partial tiles through LDS, two row tiles at a time; wave w finishes sixteenths 2 w .. of every lane */
#pragma unroll
    for (int q = 0; q < R; q += RP) {
        __syncthreads();                     /* every wave is done with the buffer (and its loads have landed) */
#pragma unroll
        for (int r = 0; r < RP; ++r)
#pragma unroll
            for (int i = 0; i < 16; ++i) red[(wave * RP * 16 + 16 * r + i) * 64 + lane] = acc[q + r][i];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < 2 * RP; ++j) {
            const int o = 2 * RP * wave + j, i = o & 15;
            float p[F32_WAVES];
#pragma unroll
            for (int k = 0; k < F32_WAVES; ++k) p[k] = red[(k * RP * 16 + o) * 64 + lane];
            const float v = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
            const int n = n0 + 32 * (q + (o >> 4)) + col, t = t0 + 8 * (i >> 2) + 4 * half + (i & 3);
            fix = fix || !(fabsf(v) < __builtin_inff());
            if (n < N && t < M) C[(size_t)t * ldc + n] = bias ? v + bias[n] : v;
        }
    }
    if (fix) {
#pragma unroll 1
        for (int j = 0; j < 2 * R; ++j) {
            const int o = 2 * RP * wave + j % (2 * RP), i = o & 15;
            const int n = n0 + 32 * (j / (2 * RP) * RP + (o >> 4)) + col, t = t0 + 8 * (i >> 2) + 4 * half + (i & 3);
            if (n >= N || t >= M) continue;
            float *const out = C + (size_t)t * ldc + n;
            if (fabsf(*out) < __builtin_inff()) continue;
            const float v = exact_output<F>(B + (size_t)n * (size_t)wrow, A + (size_t)t * (size_t)K, K);
            *out = bias ? v + bias[n] : v;
        }
    }
}

template <class F>
int launch_f32act(const float *A, const uint8_t *B, const float *bias, float *C, int M, int N, int K, long wrow, long ldc, hipStream_t s)
{
    const long long ntg = (M + 31) / 32, tiles = ntg * ((N + 31) / 32);
    /* Two row tiles per wave share the cut of x.  A round of 256 blocks, one on a CU, then takes about half as long again, so they pay where they
     * leave at most two thirds of the rounds.  Of 1585 launches of 2..256 tokens, 128..11008 rows and widths of 256..11008 the choice of all three
     * formats, forms below included, costs 0.1 (Q4_K), 0.5 (Q6_K) and 1.2 % (Q8_0) more than always taking the fastest, single ones up to 28 %;
     * from 192 blocks of two on, as it was, 2.0, 1.3 and 2.6 % and up to 48 (us, one tile -> two: Q4_K 31 x 8410 x 1280 15.0 -> 11.3, Q6_K 103 x 2275 x
     * 3584 36.7 -> 27.9, Q8_0 204 x 1431 x 6080 49.9 -> 37.6). */
    const long long rounds = (tiles + 255) / 256, rounds2 = (ntg * ((N + 63) / 64) + 255) / 256;
    int R = 2 * rounds >= 3 * rounds2 ? 2 : 1;
    auto kernel = R == 2 ? gemm_f32row_kernel<F, 2> : gemm_f32row_kernel<F, 1>;
    if constexpr (!std::is_same<F, F32Q4K>::value) {
        /* Same bits from all of them.
         *  - `once`, rows of up to SHORT_RUNS runs: weights loaded once a block, two blocks on a CU.  Where there is more than a block per CU
         *    1.02..1.31 (Q6_K, 75 x 7670 x 1024 20.9 -> 16.0 us) and 1.03..1.18 times (Q8_0) as fast as the row kernel; a block alone on its CU pays for
         *    the way through LDS and the barrier: Q6_K gains from two steps a wave on, Q8_0 never.
         *  - `runs`, weights in memory order.  Q6_K, whose row per lane is misaligned and takes the address path 160 cycles a load: always, as Q8_0 two bytes
         *    off a dword from nine steps a wave on (1.11..1.19; below, a wave loads runs that its neighbours load too: 0.94..0.99).  Q8_0 on a dword, whose
         *    rows a lane reads in whole dwords, gains where rows a multiple of 1024 elements apart fall on few cache sets (1.00..1.29), and else from ten
         *    steps on if the tokens fill the tile, since the way is as long for one as for 32 (6 and 16 tokens 0.92..1.00, from 28 on
         *    1.03..1.10), with two row tiles or not much more than half the CUs loading (179 to 194 blocks 0.95..1.05, 258 0.90..0.95). */
        const int per = ((K + F::STEP - 1) / F::STEP + F32_WAVES - 1) / F32_WAVES;
        const bool fits = K <= F::SHORT_RUNS * F::RUN * F::STEP;
        bool once, runs;
        if constexpr (std::is_same<F, F32Q6K>::value) {
            once = fits && (tiles > 256 || per > 1);
            runs = !fits;
        } else {
            once = fits && ntg * ((N + 32 * R - 1) / (32 * R)) > 256;
            runs = K % 64 ? per >= 9 : K % 1024 == 0 || (M >= 28 && per >= 10 && (R == 2 || tiles <= 160));
        }
        if (once) {
            R = 1;
            kernel = gemm_f32run_kernel<F, 1, true>;
        } else if (runs)
            kernel = R == 2 ? gemm_f32run_kernel<F, 2, false> : gemm_f32run_kernel<F, 1, false>;
    }
    const long long grid = ntg * ((N + 32 * R - 1) / (32 * R));
    if (grid > 0x7fffffffll) return CKQ_ESHAPE;
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(64 * F32_WAVES), 0, s, A, B, bias, C, M, N, K, wrow, ldc, (int)ntg);
    return (int)hipGetLastError();
}

} // namespace

int launch_gemm_f32act(int fmt, const float *A, const void *B, const float *bias, float *C, int M, int N, int K, long ldc, hipStream_t s)
{
    const uint8_t *W = (const uint8_t *)B;
    switch (fmt) {
    case CKQ_KERNEL_Q4K_F32: return launch_f32act<F32Q4K>(A, W, bias, C, M, N, K, (long)(K / 256) * 144, ldc, s);
    case CKQ_KERNEL_Q6K_F32: return launch_f32act<F32Q6K>(A, W, bias, C, M, N, K, (long)(K / 256) * 210, ldc, s);
    case CKQ_KERNEL_Q80_F32: return launch_f32act<F32Q80>(A, W, bias, C, M, N, K, (long)(K / 32) * 34, ldc, s);
    default: return CKQ_EFORMAT;
    }
}
