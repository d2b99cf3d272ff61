/*
 * ckq_gemm_rows16.hip - K-quant weights x Q8_K activations for a few to a few dozen tokens, on the gfx950 int8 matrix
 * cores, with the weights streamed from memory through LDS private to a wave.
 *
 * Where the tile kernels (ckq_gemm_q4k.hip and its siblings) move 128-row tiles through LDS and need hundreds of tokens
 * to pay for it, and the streaming kernel (ckq_gemv.hpp) spends one v_dot4 per four products and token, this kernel has
 * one WAVE multiply 16 weight rows with 16 tokens: the matrix instruction takes 16 tokens for the price of one, the
 * planes of a weight are formed once, and as in the streaming kernel the waves run on their own and nothing waits at
 * a barrier before the end.
 *
 * v_mfma_i32_16x16x64_i8: A = 16 tokens x 64 k, B = 64 k x 16 weight rows, D = 16 x 16 int32.  Lane l = 16 q + i holds
 * token / row i and the 16 k of quarter q; of D it holds row i and tokens 4 q .. 4 q + 3.  The 64 k of an instruction are
 * those a lane of the streaming kernel takes, ordered so that a lane's sixteen are one 16-byte run of the raw block's
 * quants (low or high nibbles) inside one scale; the activations are read in the same order.  Where several groups of tokens share them (but for Q5_K in the kernel of two groups), the planes are those of the tile kernels: Q4_K (sc >> 3) q and
 * (sc & 7) q, Q5_K / Q6_K the two bytes of the 16-bit product, each summed over the 256-block; the min term of Q4_K / Q5_K is
 * a bf16 MFMA of the mins and the bsum pairs split in two (ckq_gemm_q4k.hip).  All integers are exact.
 *
 * The integers being exact, only the order of the fp32 additions is left to choose, and it is that of the kernel the shape
 * would otherwise run on: the streaming kernel's term per 64 elements and tree (TREE), or the tile kernels' term per
 * 256-block and chains (GemmChains).  The terms meet in LDS; one thread per output adds them.
 *
 * Bound: for one token group nothing alone.  Vector instructions (110-260 per 256-block of 16 rows) issue in 36 to 51 % of the busy CUs' cycles, waves wait in
 * 35 to 45 %, and a block's loads, terms and sums add up; for several groups it is VALU issue (64 % at 93 tokens x 4864 x 1024).  Measured, weights from HBM, against the kernel that served the shape before (us): Q4_K 4096 x 4096 at 8 / 13 / 32
 * tokens 7.5 -> 6.1, 10.0 -> 6.5, 13.1 -> 8.1; 11008 x 4096 at 8 / 13: 14.7 -> 10.3, 15.6 -> 9.7; Q6_K 32000 x 4096 at
 * 8 / 13: 40.6 -> 27.1, 46.2 -> 28.3; 4096 x 11008 at 13: 20.7 -> 15.8; Q5_K 1024 x 4864 at 64: 16.8 -> 8.0.
 */
#include "ckq_formats.hpp"
#include "ckq_blocks.h"
#include "ckq_gemm_rows16.hpp"
#include "ckq_gemm_q4k.hpp"
#include <atomic>
#include <algorithm>
#include <type_traits>

namespace {

typedef float ckq_v4f __attribute__((ext_vector_type(4)));

/* What a lane keeps of its row's block header. */
struct Head {
    u32     sc[2];           /* Q4_K, Q5_K: scale of sub-block 2 g + q / 2 in byte 2 (g & 1) of [g / 2]; Q6_K: that of 16-run (n, q, odd) in byte odd of [n] */
    ckq_v4i mins;            /* bf16 m_2q, m_2q+1, m_2q, m_2q+1, 0... (Q4_K, Q5_K) */
    float   dw, dmin;
};

/* Header of a Q4_K / Q5_K block: the packed 6-bit scales and mins (layout: ckq_formats.hpp). */
__device__ __forceinline__ void head_k45(Head &p, const uint8_t *r, int q)
{
    const ckq_v4i hv = *reinterpret_cast<const ckq_v4i *>(r);
    const u32 h0 = (u32)hv[0], h1 = (u32)hv[1], h2 = (u32)hv[2], h3 = (u32)hv[3];
    const int s8 = 8 * (q >> 1), s16 = 16 * (q & 1);
    p.sc[0] = (h1 & 0x3f3f3f3fu) >> s8;
    p.sc[1] = ((h3 & 0x0f0f0f0fu) | ((h1 >> 2) & 0x30303030u)) >> s8;
    const u32 lo = (h2 >> s16) & 0x3f3fu, hi = ((h3 >> (s16 + 4)) & 0x0f0fu) | (((h2 >> s16) >> 2) & 0x3030u);
    const u32 mn = q < 2 ? lo : hi;
    const u32 pair = bf16_pair((float)(mn & 0xff), (float)((mn >> 8) & 0xff));
    p.mins = ckq_v4i{(int)pair, (int)pair, 0, 0};
    p.dw = h2f(h0 & 0xffff);
    p.dmin = h2f(h0 >> 16);
}

/* Four bytes times a 16-bit factor (+ add), split into the signed low and the high bytes of the products. */
__device__ __forceinline__ void byte_planes(u32 v, u32 sc2, u32 add2, int &lo, int &hi)
{
    const u32 e = __builtin_amdgcn_perm(0u, v, 0x0c020c00u), o = __builtin_amdgcn_perm(0u, v, 0x0c030c01u);
    const u32 te = pk_mad_u16(e, sc2, add2), to = pk_mad_u16(o, sc2, add2);      /* product + 128 */
    lo = (int)(__builtin_amdgcn_perm(to, te, 0x06020400u) ^ 0x80808080u);
    hi = (int)__builtin_amdgcn_perm(to, te, 0x07030501u);
}

__device__ __forceinline__ ckq_v4i lds16(const uint8_t *p) { return *reinterpret_cast<const ckq_v4i *>(p); }

/* One group of tokens: the quants as they are against one 32-run (slab) of the block at a time (v_mfma_i32_16x16x32_i8; lane quarter q has elements 32 s + 8 q ..
 * + 7 of slab s), the integers of a slab then times its scale, which a lane has for its row: four multiply-adds where forming planes and putting their sums
 * together costs more than the matrix instructions it saves (vector instructions of a 256-block in the first kernel, planes -> slabs: Q4_K 129 -> 110, in the streaming
 * kernel's order 215 -> 184, Q5_K 247 -> 140 and 333 -> 214, Q6_K 236 -> 186 and 292 -> 256; us, weights from the cache, tokens x rows x K: Q5_K 13 x 6144 x 4096 10.8 -> 9.3, 8 x 11008 x 4096 13.4 ->
 * 11.1, 6 x 4096 x 11008 12.5 -> 10.1; Q4_K 8 x 11008 x 4096 10.8 -> 10.2, 13 x 4096 x 11008 11.8 -> 11.4; Q6_K 13 x 4096 x 11008 14.0 -> 13.3, 16 x 3584 x 9728 13.2 -> 12.8;
 * Q6_K rows of two to four blocks lose up to 6 % where there are 8000 to 32000 of them, 8 x 15986 x 768 6.4 -> 6.7, 12 and 16 tokens the same, and gain 1 to 4 beyond).  Q6_K has a scale every 16: a second product with the first half of the tokens' run alone, times the
 * difference of the two scales.  raw(): the operands of SLABS slabs of the row at r, Q6_K 4 (q - 32); scales(): sc[s], or of Q6_K sc[2 s + half]. */
__device__ __forceinline__ long two_dwords(u32 lo, u32 hi) { return (long)((uint64_t)lo | ((uint64_t)hi << 32)); }
__device__ __forceinline__ void scales_k45(int (&sc)[16], const uint8_t *r)
{
    const ckq_v4i hv = *reinterpret_cast<const ckq_v4i *>(r);
    const u32 h1 = (u32)hv[1], h3 = (u32)hv[3], lo = h1 & 0x3f3f3f3fu, hi = (h3 & 0x0f0f0f0fu) | ((h1 >> 2) & 0x30303030u);
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        sc[k] = (int)((lo >> (8 * k)) & 0xffu);
        sc[4 + k] = (int)((hi >> (8 * k)) & 0xffu);
    }
}

/* Formats.  Position g of a 256-block: the 64 elements of one instruction, of which lane quarter q supplies the sixteen
 * from a_elem(g, q).  planes() forms them from the raw block of the lane's row at r (in LDS). */
struct R16Q4K {
    static constexpr int WBLOCK = 144, SHIFT = 3, CHUNKS = 9, PITCH = 144;
    static constexpr bool MIN = true, HALVES = false;
    static __device__ __forceinline__ u32 chunk_ofs(int c) { return 16u * (u32)c; }
    static __device__ __forceinline__ u32 a_elem(int g, int q) { return 64u * g + 16u * q; }
    static __device__ __forceinline__ void head(Head &p, const uint8_t *r, int q) { head_k45(p, r, q); }
    static __device__ __forceinline__ void planes(ckq_v4i &h, ckq_v4i &l, const Head &p, const uint8_t *r, int g, int q)
    {
        const ckq_v4i qs = lds16(r + 16 + 32 * g + 16 * (q & 1));
        auto pair_of_byte = [](u32 v, int k) { return __builtin_amdgcn_perm(0u, v, 0x0c000c00u | (u32)k | ((u32)k << 16)); };
        const u32 mh = pair_of_byte((p.sc[g >> 1] >> 3) & 0x07070707u, 2 * (g & 1)), ml = pair_of_byte(p.sc[g >> 1] & 0x07070707u, 2 * (g & 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32 n = ((u32)qs[i] >> (4 * (q >> 1))) & 0x0f0f0f0fu;
            h[i] = mul_bytes(n, mh);
            l[i] = mul_bytes(n, ml);
        }
    }
    static __device__ __forceinline__ void scales(int (&sc)[16], const uint8_t *r) { scales_k45(sc, r); }
    static constexpr int SLABS = 2;
    static __device__ __forceinline__ void raw(long (&b)[2], const uint8_t *r, int g, int q)
    {
        const uint2 v = *reinterpret_cast<const uint2 *>(r + 16 + 32 * g + 8 * q);
        b[0] = two_dwords(v.x & 0x0f0f0f0fu, v.y & 0x0f0f0f0fu);
        b[1] = two_dwords((v.x >> 4) & 0x0f0f0f0fu, (v.y >> 4) & 0x0f0f0f0fu);
    }
};

struct R16Q5K {
    static constexpr int WBLOCK = 176, SHIFT = 8, CHUNKS = 11, PITCH = 176;
    static constexpr bool MIN = true, HALVES = true;
    /* for the kernel of two groups: the quants of position g, and those of its first 32 elements alone (lane quarters 0 and 1) */
    static __device__ __forceinline__ void halves(ckq_v4i &all, ckq_v4i &first, const uint8_t *r, int g, int q)
    {
        const ckq_v4i qs = lds16(r + 48 + 32 * g + 16 * (q & 1)), qh = lds16(r + 16 + 16 * (q & 1));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32 n = ((u32)qs[i] >> (4 * (q >> 1))) & 0x0f0f0f0fu, v = n | ((((u32)qh[i] >> (2 * g + (q >> 1))) & 0x01010101u) << 4);
            all[i] = (int)v;
            first[i] = q < 2 ? (int)v : 0;
        }
    }
    static __device__ __forceinline__ u32 chunk_ofs(int c) { return 16u * (u32)c; }
    static __device__ __forceinline__ u32 a_elem(int g, int q) { return 64u * g + 16u * q; }
    static __device__ __forceinline__ void head(Head &p, const uint8_t *r, int q) { head_k45(p, r, q); }
    static __device__ __forceinline__ void planes(ckq_v4i &h, ckq_v4i &l, const Head &p, const uint8_t *r, int g, int q)
    {
        const ckq_v4i qs = lds16(r + 48 + 32 * g + 16 * (q & 1)), qh = lds16(r + 16 + 16 * (q & 1));
        const u32 sc2 = __builtin_amdgcn_perm(0u, p.sc[g >> 1], (g & 1) ? 0x0c020c02u : 0x0c000c00u);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32 n = ((u32)qs[i] >> (4 * (q >> 1))) & 0x0f0f0f0fu;
            const u32 hb = ((u32)qh[i] >> (2 * g + (q >> 1))) & 0x01010101u;              /* fifth bits of sub-block 2 g + q / 2 */
            int lo, hi;
            byte_planes(n | (hb << 4), sc2, 0x00800080u, lo, hi);
            h[i] = hi;
            l[i] = lo;
        }
    }
    static __device__ __forceinline__ void scales(int (&sc)[16], const uint8_t *r) { scales_k45(sc, r); }
    static constexpr int SLABS = 2;
    static __device__ __forceinline__ void raw(long (&b)[2], const uint8_t *r, int g, int q)
    {
        const uint2 f = *reinterpret_cast<const uint2 *>(r + 16 + 8 * q), v = *reinterpret_cast<const uint2 *>(r + 48 + 32 * g + 8 * q);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            auto five = [&](u32 n, u32 h) { return ((n >> (4 * k)) & 0x0f0f0f0fu) | (((h >> (2 * g + k)) & 0x01010101u) << 4); };
            b[k] = two_dwords(five(v.x, f.x), five(v.y, f.y));
        }
    }
};

struct R16Q6K {
    /* a 210-byte block as fourteen chunks, the last from byte 194 so that no load passes the block's end */
    static constexpr int WBLOCK = 210, SHIFT = 8, CHUNKS = 14, PITCH = 240;
    static constexpr bool MIN = false, HALVES = false;
    static __device__ __forceinline__ u32 chunk_ofs(int c) { return c < 13 ? 16u * (u32)c : 194u; }
    /* position g = 2 n + odd: the halves `odd` of the four 32-runs of 128-half n */
    static __device__ __forceinline__ u32 a_elem(int g, int q) { return 128u * (g >> 1) + 32u * q + 16u * (g & 1); }
    static __device__ __forceinline__ void head(Head &p, const uint8_t *r, int q)
    {
        const ckq_v4i sc = lds16(r + 192);
#pragma unroll
        for (int n = 0; n < 2; ++n) p.sc[n] = (u32)(q < 2 ? sc[2 * n] : sc[2 * n + 1]) >> (16 * (q & 1));
        p.dw = h2f(*reinterpret_cast<const uint16_t *>(r + 222));
        p.dmin = 0.0f;
    }
    static __device__ __forceinline__ void planes(ckq_v4i &h, ckq_v4i &l, const Head &p, const uint8_t *r, int g, int q)
    {
        const int n = g >> 1, odd = g & 1;
        const ckq_v4i ql = lds16(r + 64 * n + 32 * (q & 1) + 16 * odd), qh = lds16(r + 128 + 32 * n + 16 * odd);
        const int sc = __builtin_amdgcn_sbfe((int)p.sc[n], 8 * odd, 8);
        const u32 sc2 = __builtin_amdgcn_perm((u32)sc, (u32)sc, 0x05040504u);
        const u32 add = pk_mad_u16(sc2, 0xFFE0FFE0u, 0x00800080u);                   /* 128 - 32 sc */
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32 n4 = ((u32)ql[i] >> (4 * (q >> 1))) & 0x0f0f0f0fu, hb = (((u32)qh[i] >> (2 * q)) & 0x03030303u) << 4;
            int lo, hi;
            byte_planes(n4 | hb, sc2, add, lo, hi);
            h[i] = hi;
            l[i] = lo;
        }
    }
    static __device__ __forceinline__ void scales(int (&sc)[16], const uint8_t *r)
    {
        const ckq_v4i v = lds16(r + 192);
#pragma unroll
        for (int k = 0; k < 16; ++k) sc[k] = __builtin_amdgcn_sbfe(v[k >> 2], 8 * (k & 3), 8);
    }
    static constexpr int SLABS = 4;
    static __device__ __forceinline__ void raw(long (&b)[4], const uint8_t *r, int n, int q)
    {
        const uint2 l0 = *reinterpret_cast<const uint2 *>(r + 64 * n + 8 * q), l1 = *reinterpret_cast<const uint2 *>(r + 64 * n + 32 + 8 * q);
        const uint2 h = *reinterpret_cast<const uint2 *>(r + 128 + 32 * n + 8 * q);
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const uint2 l = t & 1 ? l1 : l0;
            /* 6-bit q in the upper bits of its byte, the top one turned: 4 (q - 32) */
            auto six = [&](u32 n4, u32 n2) {
                return ((t < 2 ? n4 << 2 : n4 >> 2) & 0x3c3c3c3cu) | (((n2 << (6 - 2 * t)) & 0xc0c0c0c0u) ^ 0x80808080u);
            };
            b[t] = two_dwords(six(l.x, h.x), six(l.y, h.y));
        }
    }
};
/* The sums of slab s: of the whole of it, and for Q6_K of its first half too; `I` += them times their scales. */
template <class F>
__device__ __forceinline__ void slab_sums(int (&I)[4], int s, long a, long ah, long b, const int (&sc)[16])
{
    const ckq_v4i zero = {0, 0, 0, 0};
    const ckq_v4i S = __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, zero, 0, 0, 0);
    if constexpr (F::MIN) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            I[r] += __mul24(S[r], sc[s]);
            asm("" : "+v"(I[r]));               /* one multiply-add, not two products and an addition of three */
        }
    } else {
        const ckq_v4i H = __builtin_amdgcn_mfma_i32_16x16x32_i8(ah, b, zero, 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            I[r] += __mul24(S[r], sc[2 * s + 1]);
            asm("" : "+v"(I[r]));
            I[r] += __mul24(H[r], sc[2 * s] - sc[2 * s + 1]);
            asm("" : "+v"(I[r]));
        }
    }
}
/* Q6_K, the two halves of slab s apart: ah, ao are the tokens' with the other half zero. */
__device__ __forceinline__ void slab_halves(int (&even)[4], int (&odd)[4], int s, long ah, long ao, long b, const int (&sc)[16])
{
    const ckq_v4i zero = {0, 0, 0, 0};
    const ckq_v4i H = __builtin_amdgcn_mfma_i32_16x16x32_i8(ah, b, zero, 0, 0, 0), O = __builtin_amdgcn_mfma_i32_16x16x32_i8(ao, b, zero, 0, 0, 0);
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        even[r] += __mul24(H[r], sc[2 * s]);
        odd[r] += __mul24(O[r], sc[2 * s + 1]);
        asm("" : "+v"(even[r]), "+v"(odd[r]));
    }
}
/* A position's integer from the sums over all of its 64 elements and over the first 32. */
__device__ __forceinline__ int halves_sum(int all, int first, int sc0, int sc1)
{
    int v = __mul24(first, sc0 - sc1);
    asm("" : "+v"(v));
    return v + __mul24(all, sc1);
}

/* Shape of a launch: what a block needs besides its problem. */
struct Rows16Shape { int M, nb; };

/* LDS of one wave: the 16 weight blocks of an item, the quants of NT tokens (256 bytes each, 16-byte chunk c in slot
 * c ^ token) and their bsums (32 bytes each). */
template <class F, int NT> constexpr int rows16_wave_lds() { return 16 * F::PITCH + NT * 288; }

/* One block computes a tile of 16 rows for NT (8 or 16) tokens.  Wave w takes the 256-blocks w, w + waves, ... of the
 * rows.  A block's bytes are loaded in memory order - 16 adjacent lanes read a token's 256 quants, 9 to 14 lanes a weight
 * block: a lane loading its own operand would touch a cache line of its own with every 16 bytes, and the address unit
 * would bound the launch (10.6 us instead of 9.4 at 11008 x 4096, 13 tokens, Q4_K; 44 instead of 27 at 32000 x 4096,
 * Q6_K) - and turned through LDS of the wave's own, the next block's loads in flight meanwhile.  A 256-block leaves
 * u = dw I1 - dmin I2 of its NT x 16 outputs in LDS; when all are done, one thread per output runs the chains of
 * multiply-adds over them in order, so that any wave may take any block whatever the chains.
 * More rows or more tokens (32, planes shared) per block were slower: fewer waves per CU fit the LDS. */
template <class F, int NT, bool TREE, bool GRP>
__global__ void __launch_bounds__(1024)
gemm_rows16_kernel(const uint8_t *W, const uint8_t *X, int N, Rows16Shape S, float *y, const float *bias, long ldy, GemmChains ch, Rows16Args grp)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, nthr = blockDim.x, nwave = nthr >> 6;
    const int lane = tid & 63, wave = wave_in_block();
    const int i16 = lane & 15, q = lane >> 4;
    const int M = S.M, nb = S.nb;
    int bid = (int)blockIdx.x;
    if constexpr (GRP) {
        if (bid >= grp.p[1].id0) {
            Rows16Problem p = grp.p[1];
            if (grp.n > 2 && bid >= grp.p[2].id0) p = grp.p[2];
            if (grp.n > 3 && bid >= grp.p[3].id0) p = grp.p[3];
            W = p.W; X = p.X; N = p.N; y = p.y; bias = p.bias; ldy = p.ldy; ch = p.ch;
            bid -= p.id0;
        }
    }
    const int n0 = bid * 16, t0 = (int)blockIdx.y * NT;
    const u32 xrow = (u32)nb * 292u, wpitch = (u32)nb * (u32)F::WBLOCK;
    uint8_t *const wl = smem + wave * rows16_wave_lds<F, NT>();           /* this wave's weights, quants, bsums */
    uint8_t *const al = wl + 16 * F::PITCH, *const bl = al + NT * 256;
    float *const us = reinterpret_cast<float *>(smem + nwave * rows16_wave_lds<F, NT>()), *const dxs = us + (TREE ? min(nb, 16) : nb) * (NT * 16);
    /* uniform bases, 32-bit lane offsets */
    const uint8_t *const wbase = W + (size_t)n0 * wpitch;
    const uint8_t *const xbase = X + (size_t)t0 * xrow;

    /* copy roles: weight chunk 64 j + lane -> (row, chunk), token chunk 64 j + lane -> (token, one of 16 of quants or, for a
     * min, 2 of bsums: without them Q6_K's are four loads instead of five, 4096 x 11008 at 13 tokens 16.5 -> 15.8 us, 7930 x 5376 at 15 19.9 -> 18.8) */
    constexpr int XC = F::MIN ? 18 : 16, NWL = (16 * F::CHUNKS + 63) / 64, NAL = (NT * XC + 63) / 64;
    u32 wsrc[NWL], wdst[NWL], asrc[NAL], adst[NAL];
#pragma unroll
    for (int j = 0; j < NWL; ++j) {
        const int e = min(64 * j + lane, 16 * F::CHUNKS - 1), r = e / F::CHUNKS, c = e % F::CHUNKS;
        wsrc[j] = (u32)min(r, N - 1 - n0) * wpitch + F::chunk_ofs(c);
        wdst[j] = (u32)(r * F::PITCH + 16 * c);
    }
#pragma unroll
    for (int j = 0; j < NAL; ++j) {
        const int e = min(64 * j + lane, NT * XC - 1), t = e / XC, c = e % XC;
        asrc[j] = (u32)min(t, M - 1 - t0) * xrow + 4u + 16u * (u32)c;
        adst[j] = (u32)(c < 16 ? 256 * t + 16 * (c ^ (t & 15)) : NT * 256 + 32 * t + 16 * (c - 16));
    }
    constexpr int QL = NT / 4;                       /* quarters of the result that hold tokens */
    const int ta = i16 & (NT - 1);
    const u32 abase = (u32)(256 * ta + 8 * (q & 1)), aslot = 16u * (u32)((q >> 1) ^ ta);        /* slab s: 16-byte chunk 2 s + q / 2 of the token, in slot (its number) ^ ta */
    const u32 first = q < 2 ? ~0u : 0u;
    auto slab_a = [&](int s, long &a, long &ah) {
        const uint2 v = *reinterpret_cast<const uint2 *>(al + abase + (aslot ^ (32u * (u32)s)));
        a = two_dwords(v.x, v.y);
        ah = two_dwords(v.x & first, v.y & first);
    };

    ckq_v4i wr[NWL], ar[NAL];
    auto fetch = [&](int b) {
        const uint8_t *wb = wbase + (size_t)((u32)b * (u32)F::WBLOCK), *xb = xbase + (size_t)((u32)b * 292u);
#pragma unroll
        for (int j = 0; j < NWL; ++j) {
            u32 t[4];
            ld16<F::WBLOCK % 4 == 0 ? 4 : 2>(t, wb + wsrc[j]);
            wr[j] = ckq_v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
        }
#pragma unroll
        for (int j = 0; j < NAL; ++j) {
            u32 t[4];
            ld16<4>(t, xb + asrc[j]);
            ar[j] = ckq_v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
        }
    };
    auto take = [&]() {
#pragma unroll
        for (int j = 0; j < NWL; ++j) *reinterpret_cast<ckq_v4i *>(wl + wdst[j]) = wr[j];
#pragma unroll
        for (int j = 0; j < NAL; ++j) *reinterpret_cast<ckq_v4i *>(al + adst[j]) = ar[j];
    };
    /* the two bsum pairs of position q */
    auto bsum_operand = [&]() {
        const int2 bs = *reinterpret_cast<const int2 *>(bl + 32 * ta + 8 * q);
        u32 lo, hi;
        min_operand(bs.x, bs.y, lo, hi);
        return ckq_v4i{(int)lo, (int)hi, 0, 0};
    };
    auto min_mfma = [&](const ckq_v4i &am, const ckq_v4i &mins) {
        const ckq_v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ckq_v8bf, am), __builtin_bit_cast(ckq_v8bf, mins), z, 0, 0, 0);
    };
    /* lane 16 q + i holds tokens 4 q .. 4 q + 3; of eight tokens the upper two quarters are copies */
    auto put = [&](int b, const float (&v)[4]) {
        float *u = us + b * (NT * 16) + lane;
#pragma unroll
        for (int r = 0; r < 4; ++r)
            if (NT > 8 || q < 2) u[r * (16 * QL)] = v[r];
    };
    const ckq_v4i zero = {0, 0, 0, 0};
    const uint8_t *const wrow = wl + i16 * F::PITCH;

    /* CHAIN: the integers of the whole 256-block, u = dw I1 - dmin I2 */
    auto block_term = [&](int b) {
        Head hd;
        F::head(hd, wrow, q);
        int sc[16], I[4] = {0, 0, 0, 0};
        F::scales(sc, wrow);
#pragma unroll
        for (int k = 0; k < 8 / F::SLABS; ++k) {
            long w[F::SLABS];
            F::raw(w, wrow, k, q);
#pragma unroll
            for (int j = 0; j < F::SLABS; ++j) {
                long a, ah;
                slab_a(F::SLABS * k + j, a, ah);
                slab_sums<F>(I, F::SLABS * k + j, a, ah, w[j], sc);
            }
        }
        float out[4];
        if constexpr (F::MIN) {
            const ckq_v4f i2 = min_mfma(bsum_operand(), hd.mins);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float f = (float)I[r];
                out[r] = hd.dw * f - hd.dmin * i2[r];
            }
        } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = hd.dw * (float)(I[r] >> 2);
        }
        put(b, out);
    };

    /* TREE: the fp32 terms of the four positions, added to the sums their lanes of the streaming kernel would hold */
    auto position_terms = [&](int b, float (&acc)[4][4]) {
        Head hd;
        F::head(hd, wrow, q);
        const ckq_v4i dxi = lds16(reinterpret_cast<const uint8_t *>(dxs + b * NT + 4 * (q & (QL - 1))));
        ckq_v4i am;
        if (F::MIN) am = bsum_operand();
        int sc[16];
        F::scales(sc, wrow);
        auto term = [&](int g, const int (&I)[4]) {
            ckq_v4f i2;
            if constexpr (F::MIN) i2 = min_mfma(am, q == g ? hd.mins : zero);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int di = dxi[r];
                const float dx = __builtin_bit_cast(float, di), f = (float)(F::MIN ? I[r] : I[r] >> 2);
                float v;
                if constexpr (F::MIN) v = (hd.dw * dx) * f - (hd.dmin * dx) * i2[r];
                else                  v = (hd.dw * dx) * f;
                asm volatile("" : "+v"(v));                  /* rounded before it is added, as there */
                acc[g][r] += v;
            }
        };
        if constexpr (F::MIN) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {                    /* slabs 2 g and 2 g + 1 */
                int I[4] = {0, 0, 0, 0};
                long w[F::SLABS];
                F::raw(w, wrow, g, q);
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    long a, ah;
                    slab_a(2 * g + j, a, ah);
                    slab_sums<F>(I, 2 * g + j, a, ah, w[j], sc);
                }
                term(g, I);
                __builtin_amdgcn_sched_barrier(0);
            }
        } else {
#pragma unroll
            for (int n = 0; n < 2; ++n) {                    /* position 2 n + odd: the halves `odd` of slabs 4 n .. 4 n + 3 */
                int even[4] = {0, 0, 0, 0}, odd[4] = {0, 0, 0, 0};
                long w[F::SLABS];
                F::raw(w, wrow, n, q);
#pragma unroll
                for (int s = 4 * n; s < 4 * n + 4; ++s) {
                    long a, ah;
                    slab_a(s, a, ah);
                    slab_halves(even, odd, s, ah, two_dwords((u32)a & ~first, (u32)((uint64_t)a >> 32) & ~first), w[s & 3], sc);
                }
                term(2 * n, even);
                term(2 * n + 1, odd);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
    };

    /* block scales of the tokens, [block][NT]: their loads go out first, so that waiting for them waits for nothing else */
    constexpr int ND = 2;
    const int nd = nb * NT;
    float dxv[ND];
    auto dx_load = [&](int e) {
        const int t = e % NT, b = e / NT;
        return __builtin_bit_cast(float, ld4<4>(xbase + (size_t)((u32)min(t, M - 1 - t0) * xrow + (u32)b * 292u)));
    };
#pragma unroll
    for (int k = 0; k < ND; ++k) dxv[k] = dx_load(min(tid + k * nthr, nd - 1));
    if (wave < nb) fetch(wave);
#pragma unroll
    for (int k = 0; k < ND; ++k)
        if (tid + k * nthr < nd) dxs[tid + k * nthr] = dxv[k];
    for (int e = tid + ND * nthr; e < nd; e += nthr) dxs[e] = dx_load(e);        /* long rows */
    if constexpr (TREE) {
        __syncthreads();                                                         /* for the scales only: the blocks' loads stay in flight */
        /* a lane of the streaming kernel holds positions l, l + 64, ...: blocks b, b + 16, ... meet in one sum per position */
        for (int b0 = wave; b0 < min(nb, 16); b0 += nwave) {
            float acc[4][4];
#pragma unroll
            for (int g = 0; g < 4; ++g)
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[g][r] = 0.0f;
            for (int b = b0; b < nb; b += 16) {
                take();
                const int next = b + 16 < nb ? b + 16 : b0 + nwave;
                if (next < nb && (b + 16 < nb || next < 16)) fetch(next);
                __builtin_amdgcn_sched_barrier(0);
                position_terms(b, acc);
                __builtin_amdgcn_sched_barrier(0);
            }
            float out[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
            put(b0, out);
        }
    } else {
        for (int b = wave; b < nb; b += nwave) {
            take();
            if (b + nwave < nb) fetch(b + nwave);
            __builtin_amdgcn_sched_barrier(0);
            block_term(b);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    __syncthreads();
    for (int e = tid; e < NT * 16; e += nthr) {
        const int l = e % (16 * QL), r = e / (16 * QL);
        const int tok = 4 * (l >> 4) + r;
        const float *u = us + r * (16 * QL) + l, *dx = dxs + tok;
        float v = 0.0f;
        if constexpr (TREE) {
            /* the streaming kernel's fixed tree over the lanes of a row, four of them per block */
            float t[16];
#pragma unroll
            for (int b = 0; b < 16; ++b) t[b] = b < nb ? u[b * (NT * 16)] : 0.0f;
#pragma unroll
            for (int w = 1; w < 16; w *= 2)
#pragma unroll
                for (int b = 0; b < 16; b += 2 * w) t[b] += t[b + w];
            v = t[0];
        } else {
            for (int sp = 0; sp < ch.splits; ++sp) {
                const int b0 = sp * ch.per, b1 = min(nb, b0 + ch.per);
                float c[2] = {0.0f, 0.0f};
                for (int b = b0; b < b1; b += 4) {
                    float uu[4], dd[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int bk = min(b + k, b1 - 1);
                        uu[k] = u[bk * (NT * 16)];
                        dd[k] = dx[bk * NT];
                    }
                    if (ch.kg == 2) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) c[k & 1] = b + k < b1 ? fmaf(dd[k], uu[k], c[k & 1]) : c[k & 1];
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k) c[0] = b + k < b1 ? fmaf(dd[k], uu[k], c[0]) : c[0];
                    }
                }
                if (ch.kg == 2) c[0] += c[1];
                v = sp ? v + c[0] : c[0];
            }
        }
        const int n = n0 + (l & 15), t = t0 + tok;
        if (n < N && t < M) y[(size_t)t * ldy + n] = bias ? v + bias[n] : v;
    }
}

/* Short rows, one group of tokens, many row tiles: the activations stay in registers.  Wave w of a block multiplies 256-block w of
 * every row tile the block goes through (nb of them, at most HOLD_NB), so the activations of that block are fetched once, in the
 * order of the instruction and never through LDS, and only weights stream: two blocks of a wave are on their way while one is worked on,
 * across tiles too, and the waves of a block read its rows as they lie in memory.  The terms of a round of `round` tiles gather in
 * LDS; then the waves meet at a barrier and four of them add up each tile.  The terms and their order are those of the kernel above.
 * Bound: HBM, and the vector operations of all waves at once when a tile arrives (11008 x 4096 twice, Q4_K: loads alone 10.2 us,
 * with the terms 14, with the sums and stores 16.8).  Against the kernel above, 13 tokens, weights from HBM (us): Q4_K 2 x 11008 x 4096
 * 20.5 -> 16.8, Q6_K 32000 x 4096 35.4 -> 29.2, Q5_K 2 x 11008 x 4096 23.5 -> 21.5, 151936 x 1024 39 -> 31.
 * Since then, slabs instead of planes (vector instructions a 256-block: Q4_K 126 -> 106, Q5_K 236 -> 128, Q6_K 241 -> 191), weights from the cache: 14.1 -> 13.8, 30.8 -> 29.6 (30000 x 3072 at
 * 16 tokens 24.8 -> 23.2), 19.4 -> 16.0, 34.1 -> 30.3.
 * A wave with a whole chain of blocks to itself, activations in LDS, was as fast on the first two (16.7, 29.2) and 26 on the third;
 * two blocks a wave (eight waves, two such blocks a CU) 20.5, 36.2 and 25.6. */
constexpr int HOLD_NB = 16;
template <class F, bool TREE, bool GRP>
__global__ void __launch_bounds__(64 * HOLD_NB)
gemm_rows16_hold_kernel(const uint8_t *W, const uint8_t *X, int N, int M, int nb, int tiles, int round, float *y, const float *bias, long ldy, GemmChains ch, Rows16Args grp)
{
    constexpr int NT = 16;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, nthr = blockDim.x, nwave = nthr >> 6;
    const int lane = tid & 63, wave = wave_in_block();
    const int i16 = lane & 15, q = lane >> 4;
    const u32 xrow = (u32)nb * 292u, wpitch = (u32)nb * (u32)F::WBLOCK;
    uint8_t *const wl = smem + wave * (16 * F::PITCH);                     /* this wave's weights */
    float *const dxs = reinterpret_cast<float *>(smem + nwave * (16 * F::PITCH)), *const us = dxs + HOLD_NB * NT;
    const uint8_t *const wrow = wl + i16 * F::PITCH;
    struct Tile { const uint8_t *w; float *y; const float *bias; long ldy; int n0, N, own; GemmChains ch; };
    auto tile_at = [&](int t) {
        Tile r = {W, y, bias, ldy, t, N, 0, ch};
        if constexpr (GRP) {
            if (t >= grp.p[1].id0) {
                Rows16Problem p = grp.p[1];
                if (grp.n > 2 && t >= grp.p[2].id0) p = grp.p[2];
                if (grp.n > 3 && t >= grp.p[3].id0) p = grp.p[3];
                r = {p.W, p.y, p.bias, p.ldy, t - p.id0, p.N, 0, p.ch};
            }
        }
        r.own = 16 * r.n0;
        r.n0 = min(r.own, r.N - 16);                /* the last tile starts early rather than end late; its rows before `own` are another's */
        r.w += (size_t)r.n0 * wpitch;
        return r;
    };

    constexpr int NWL = (16 * F::CHUNKS + 63) / 64;
    u32 wsrc[NWL];
#pragma unroll
    for (int j = 0; j < NWL; ++j) {
        const int e = min(64 * j + lane, 16 * F::CHUNKS - 1);
        wsrc[j] = (u32)(e / F::CHUNKS) * wpitch + F::chunk_ofs(e % F::CHUNKS);
    }
    auto fetch_w = [&](ckq_v4i (&v4)[NWL], int tile) {
        const uint8_t *wb = tile_at(tile).w + (u32)wave * (u32)F::WBLOCK;
#pragma unroll
        for (int j = 0; j < NWL; ++j) {
            u32 v[4];
            ld16<F::WBLOCK % 4 == 0 ? 4 : 2>(v, wb + wsrc[j]);
            v4[j] = ckq_v4i{(int)v[0], (int)v[1], (int)v[2], (int)v[3]};
        }
    };
    auto take = [&](const ckq_v4i (&v4)[NWL]) {
#pragma unroll
        for (int j = 0; j < NWL; ++j) {
            const int e = min(64 * j + lane, 16 * F::CHUNKS - 1);
            *reinterpret_cast<ckq_v4i *>(wl + (e / F::CHUNKS) * F::PITCH + 16 * (e % F::CHUNKS)) = v4[j];
        }
    };
    const u32 xlane = (u32)min(i16, M - 1) * xrow;
    auto fetch_a = [&](long (&a8)[8], int2 &bs) {
        const uint8_t *xb = X + (u32)wave * 292u;
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            u32 v[2];
            ld8<4>(v, xb + 4 + 32 * s + (xlane + 8u * (u32)q));
            a8[s] = two_dwords(v[0], v[1]);
        }
        if constexpr (F::MIN) {
            u32 v[2];
            ld8<4>(v, xb + 260 + (xlane + 8u * (u32)q));
            bs = int2{(int)v[0], (int)v[1]};
        }
    };
    auto bsum_operand = [&](const int2 &bs) {
        u32 lo, hi;
        min_operand(bs.x, bs.y, lo, hi);
        return int2{(int)lo, (int)hi};
    };
    auto min_mfma = [&](const int2 &am, const ckq_v4i &mins) {
        const ckq_v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
        const ckq_v4i a = {am.x, am.y, 0, 0};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ckq_v8bf, a), __builtin_bit_cast(ckq_v8bf, mins), z, 0, 0, 0);
    };
    const ckq_v4i zero = {0, 0, 0, 0};
    long a[8];                                     /* the activations of this wave's block, in the order of the instruction */
    const u32 first_half = q < 2 ? ~0u : 0u;
    int2 am = {};
    /* the terms of the block whose weights lie in wl */
    auto terms = [&](float *u) {
        Head hd;
        F::head(hd, wrow, q);
        u32 first = first_half;
        if (!F::MIN) asm volatile("" : "+v"(first));             /* Q6_K: the first halves of the slabs are formed for every tile; kept like the whole ones, they would spill */
        int sc[16];
        F::scales(sc, wrow);
        float out[4];
        if constexpr (TREE) {
            const ckq_v4i dxi = lds16(reinterpret_cast<const uint8_t *>(dxs + wave * NT + 4 * q));
            float acc[4][4];
            auto term = [&](int g, const int (&I)[4]) {
                ckq_v4f i2;
                if constexpr (F::MIN) i2 = min_mfma(am, q == g ? hd.mins : zero);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int di = dxi[r];
                    const float dx = __builtin_bit_cast(float, di), f = (float)(F::MIN ? I[r] : I[r] >> 2);
                    float v;
                    if constexpr (F::MIN) v = (hd.dw * dx) * f - (hd.dmin * dx) * i2[r];
                    else                  v = (hd.dw * dx) * f;
                    asm volatile("" : "+v"(v));                  /* rounded before it is added, as there */
                    acc[g][r] = 0.0f + v;
                }
                __builtin_amdgcn_sched_barrier(0);
            };
            if constexpr (F::MIN) {
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    int I[4] = {0, 0, 0, 0};
                    long w[F::SLABS];
                    F::raw(w, wrow, g, q);
#pragma unroll
                    for (int j = 0; j < 2; ++j) slab_sums<F>(I, 2 * g + j, a[2 * g + j], 0, w[j], sc);
                    term(g, I);
                }
            } else {
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    int even[4] = {0, 0, 0, 0}, odd[4] = {0, 0, 0, 0};
                    long w[F::SLABS];
                    F::raw(w, wrow, n, q);
#pragma unroll
                    for (int s = 4 * n; s < 4 * n + 4; ++s) slab_halves(even, odd, s, two_dwords((u32)a[s] & first, (u32)((uint64_t)a[s] >> 32) & first), two_dwords((u32)a[s] & ~first, (u32)((uint64_t)a[s] >> 32) & ~first), w[s & 3], sc);
                    term(2 * n, even);
                    term(2 * n + 1, odd);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = (acc[0][r] + acc[1][r]) + (acc[2][r] + acc[3][r]);
        } else {
            int I[4] = {0, 0, 0, 0};
#pragma unroll
            for (int k = 0; k < 8 / F::SLABS; ++k) {
                long w[F::SLABS];
                F::raw(w, wrow, k, q);
#pragma unroll
                for (int j = 0; j < F::SLABS; ++j) {
                    const long x = a[F::SLABS * k + j];
                    slab_sums<F>(I, F::SLABS * k + j, x, two_dwords((u32)x & first, (u32)((uint64_t)x >> 32) & first), w[j], sc);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (F::MIN) {
                const ckq_v4f i2 = min_mfma(am, hd.mins);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float f = (float)I[r];
                    out[r] = hd.dw * f - hd.dmin * i2[r];
                }
            } else {
#pragma unroll
                for (int r = 0; r < 4; ++r) out[r] = hd.dw * (float)(I[r] >> 2);
            }
        }
        *reinterpret_cast<float4 *>(u + wave * (NT * 16) + 4 * lane) = float4{out[0], out[1], out[2], out[3]};
    };
    /* the outputs of the tile whose terms lie at u: e is output e % 4 of lane e / 4 */
    auto finish = [&](const float *u, int tile, int first, int step) {
        const Tile tl = tile_at(tile);
        for (int e = first; e < NT * 16; e += step) {
            const int tok = 4 * (e >> 6) + (e & 3), n = tl.n0 + ((e >> 2) & 15);
            const float *ue = u + e;
            float v = 0.0f;
            if constexpr (TREE) {
                float x[16];
#pragma unroll
                for (int b = 0; b < 16; ++b) x[b] = b < nb ? ue[b * (NT * 16)] : 0.0f;
#pragma unroll
                for (int w = 1; w < 16; w *= 2)
#pragma unroll
                    for (int b = 0; b < 16; b += 2 * w) x[b] += x[b + w];
                v = x[0];
            } else {
                const float *dx = dxs + tok;
                for (int sp = 0; sp < tl.ch.splits; ++sp) {
                    const int b0 = sp * tl.ch.per, b1 = min(nb, b0 + tl.ch.per);
                    float c0 = 0.0f, c1 = 0.0f;
                    int b = b0;
                    for (; b + 8 <= b1; b += 8) {
                        float uu[8], dd[8];
#pragma unroll
                        for (int k = 0; k < 8; ++k) { uu[k] = ue[(b + k) * (NT * 16)]; dd[k] = dx[(b + k) * NT]; }
                        if (tl.ch.kg == 2) {
#pragma unroll
                            for (int k = 0; k < 8; k += 2) { c0 = fmaf(dd[k], uu[k], c0); c1 = fmaf(dd[k + 1], uu[k + 1], c1); }
                        } else {
#pragma unroll
                            for (int k = 0; k < 8; ++k) c0 = fmaf(dd[k], uu[k], c0);
                        }
                    }
                    for (; b < b1; ++b) {
                        const float uu = ue[b * (NT * 16)], dd = dx[b * NT];
                        if (tl.ch.kg == 2 && ((b - b0) & 1)) c1 = fmaf(dd, uu, c1);
                        else                                 c0 = fmaf(dd, uu, c0);
                    }
                    if (tl.ch.kg == 2) c0 += c1;
                    v = sp ? v + c0 : c0;
                }
            }
            if (tl.bias) v += tl.bias[n];          /* no load without a bias: waiting for it would wait for the stores before it */
            if (n >= tl.own && tok < M) tl.y[(size_t)tok * tl.ldy + n] = v;
        }
    };

    /* the tokens' block scales, [block][token]: the first loads go out before all others, so that waiting for them waits for nothing else */
    auto load_dx = [&](int e) {
        return __builtin_bit_cast(float, ld4<4>(X + (size_t)((u32)min(e & 15, M - 1) * xrow + (u32)(e >> 4) * 292u)));
    };
    const int ndx = nb * NT, tstep = (int)gridDim.x, tile0 = (int)blockIdx.x, mine = (tiles - tile0 + tstep - 1) / tstep;
    const float dx0 = load_dx(min(tid, ndx - 1));

    constexpr int D = 2;                           /* blocks of a wave on their way; with three 29.5 -> 31.8 us for the 32000 x 4096 above */
    ckq_v4i w[D][NWL];
    int left = mine, ft = tile0;                   /* tiles still to do; the next to fetch */
    auto fetch = [&](int r) {
        fetch_w(w[r], ft);
        ft += tstep;
    };
    fetch(0);
#pragma unroll
    for (int r = 1; r < D; ++r)
        if (left > r) fetch(r);
    fetch_a(a, am);
    if (tid < ndx) dxs[tid] = dx0;
    for (int e = tid + nthr; e < ndx; e += nthr) dxs[e] = load_dx(e);
    if (F::MIN) am = bsum_operand(am);
    if constexpr (TREE) __syncthreads();
    const int teams = max(nwave >> 2, 1), team = nwave >= 4 ? wave >> 2 : 0, usize = nb * (NT * 16);
    int i = 0, t = tile0;                          /* tiles of this round that are done; the current tile */
    auto step = [&](int r, auto more) {
        take(w[r]);
        if (more) fetch(r);
        __builtin_amdgcn_sched_barrier(0);
        terms(us + i * usize);
        __builtin_amdgcn_sched_barrier(0);
        ++i;
        const bool last = t + tstep >= tiles;
        if (i == round || last) {
            __syncthreads();
            if (team < teams)
                for (int j = team; j < i; j += teams) finish(us + j * usize, t - (i - 1 - j) * tstep, nwave >= 4 ? tid & 255 : tid, nwave >= 4 ? 256 : nthr);
            if (!last) __syncthreads();
            i = 0;
        }
        t += tstep;
    };
    for (; left >= 2 * D; left -= D) {
#pragma unroll
        for (int r = 0; r < D; ++r) step(r, std::true_type{});
    }
    for (; left > 0; left -= D) {
#pragma unroll
        for (int r = 0; r < D; ++r)
            if (left > r) step(r, left > r + D);
    }
}

/* Rows too long to keep their planes, several token groups: two groups of 16 tokens a block, so that the planes of a weight
 * block are formed once for both.  As in the first kernel wave w takes 256-blocks w, w + waves, ..., the next one's weights on their way;
 * a lane loads its own activations, in the order of the instruction.  Of TREE's terms, those of a position whose lane of the streaming
 * kernel has two blocks of the row (`wide` positions: blocks 0 .. wide - 1 and those from 16 on) go to LDS one by one, all others summed over their block.
 * Bound: VALU issue.  us against the first kernel: Q6_K 1024 x 4864 at 93 tokens 14.2 -> 9.0, Q5_K 11.4 -> 10.5, Q4_K 4096 x 4096 at 24 8.1 -> 7.0.
 * Q5_K's planes cost more than the 16-bit products they save (two scalings, a carry between the planes and a sum put together again), so its operands are
 * the quants themselves, once whole and once with the second scale's half zero: instructions of a pair and 256-block 286 -> 275 in the tile kernels' order, about
 * 420 -> 350 in TREE; us at 20 / 32 tokens: 2048 x 8192 10.7 -> 8.9, 1024 x 11008 13.0 -> 10.8, 2758 x 6400 at 22 14.2 -> 11.7, others 1.00-1.05.  Q4_K, whose planes are
 * two multiplications, would need more (TREE 0.99, tile kernels' order 168 -> 227), and the kernel that keeps its planes, which forms them once, gains nothing. */
template <class F, bool TREE, bool GRP>
__global__ void __launch_bounds__(768)
gemm_rows16_pair_kernel(const uint8_t *W, const uint8_t *X, int N, int M, int nb, float *y, const float *bias, long ldy, GemmChains ch, Rows16Args grp)
{
    constexpr int NT = 16, G = 2, OUT = G * NT * 16;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, nthr = blockDim.x, nwave = nthr >> 6;
    const int lane = tid & 63, wave = wave_in_block();
    const int i16 = lane & 15, q = lane >> 4;
    int bid = (int)blockIdx.x;
    if constexpr (GRP) {
        if (bid >= grp.p[1].id0) {
            Rows16Problem p = grp.p[1];
            if (grp.n > 2 && bid >= grp.p[2].id0) p = grp.p[2];
            if (grp.n > 3 && bid >= grp.p[3].id0) p = grp.p[3];
            W = p.W; X = p.X; N = p.N; y = p.y; bias = p.bias; ldy = p.ldy; ch = p.ch;
            bid -= p.id0;
        }
    }
    const int n0 = bid * 16, t0 = (int)blockIdx.y * (G * NT);
    const u32 xrow = (u32)nb * 292u, wpitch = (u32)nb * (u32)F::WBLOCK;
    uint8_t *const wl = smem + wave * (16 * F::PITCH);                     /* this wave's weights */
    float *const dxs = reinterpret_cast<float *>(smem + nwave * (16 * F::PITCH)), *const us = dxs + nb * (G * NT);
    const int wide = TREE ? max(nb - 16, 0) : 0;                           /* leaves of more than one block */
    /* terms: [block][output], or, of TREE, leaves wide .. 15 and then the four positions of the other leaves' blocks */
    float *const up = us + (min(nb, 16) - wide) * OUT;
    const uint8_t *const wbase = W + (size_t)n0 * wpitch;

    constexpr int NWL = (16 * F::CHUNKS + 63) / 64;
    u32 wsrc[NWL], wdst[NWL];
#pragma unroll
    for (int j = 0; j < NWL; ++j) {
        const int e = min(64 * j + lane, 16 * F::CHUNKS - 1), r = e / F::CHUNKS, c = e % F::CHUNKS;
        wsrc[j] = (u32)min(r, N - 1 - n0) * wpitch + F::chunk_ofs(c);
        wdst[j] = (u32)(r * F::PITCH + 16 * c);
    }
    ckq_v4i wr[NWL], a[G][4];
    u32 bs[G][2] = {}, xo[G];
#pragma unroll
    for (int k = 0; k < G; ++k) xo[k] = (u32)min(t0 + k * NT + i16, M - 1) * xrow;
    auto fetch_w = [&](int b) {
        const uint8_t *const wb = wbase + (size_t)((u32)b * (u32)F::WBLOCK);
#pragma unroll
        for (int j = 0; j < NWL; ++j) {
            u32 t[4];
            ld16<F::WBLOCK % 4 == 0 ? 4 : 2>(t, wb + wsrc[j]);
            wr[j] = ckq_v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
        }
    };
    auto fetch_a = [&](int b) {
        __builtin_amdgcn_sched_barrier(0);
        const uint8_t *const xb = X + (size_t)((u32)b * 292u);
#pragma unroll
        for (int k = 0; k < G; ++k) {
            if constexpr (F::MIN) ld8<4>(bs[k], xb + 260 + (xo[k] + 8u * (u32)q));
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                u32 t[4];
                ld16<4>(t, xb + 4 + F::a_elem(g, 0) + (xo[k] + F::a_elem(0, q)));
                a[k][g] = ckq_v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
            }
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    const int nd = nb * (G * NT);
    auto dx_load = [&](int e) {
        return __builtin_bit_cast(float, ld4<4>(X + (size_t)((u32)min(t0 + (e & (G * NT - 1)), M - 1) * xrow + (u32)(e / (G * NT)) * 292u)));
    };
    const float dx0 = dx_load(min(tid, nd - 1)), dx1 = dx_load(min(tid + nthr, nd - 1));
    if (wave < nb) { fetch_w(wave); fetch_a(wave); }
    if (tid < nd) dxs[tid] = dx0;
    if (tid + nthr < nd) dxs[tid + nthr] = dx1;
    for (int e = tid + 2 * nthr; e < nd; e += nthr) dxs[e] = dx_load(e);
    if constexpr (TREE) __syncthreads();

    const ckq_v4i zero = {0, 0, 0, 0};
    const uint8_t *const wrow = wl + i16 * F::PITCH;
    auto min_mfma = [&](const int2 &am, const ckq_v4i &mins) {
        const ckq_v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
        const ckq_v4i am4 = {am.x, am.y, 0, 0};
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ckq_v8bf, am4), __builtin_bit_cast(ckq_v8bf, mins), z, 0, 0, 0);
    };
    for (int b = wave; b < nb; b += nwave) {
#pragma unroll
        for (int j = 0; j < NWL; ++j) *reinterpret_cast<ckq_v4i *>(wl + wdst[j]) = wr[j];
        if (b + nwave < nb) fetch_w(b + nwave);
        __builtin_amdgcn_sched_barrier(0);
        Head hd;
        F::head(hd, wrow, q);
        int sc[16];
        if constexpr (F::HALVES) F::scales(sc, wrow);
        auto operands = [&](ckq_v4i &ph, ckq_v4i &pl, int g) {
            if constexpr (F::HALVES) F::halves(ph, pl, wrow, g, q);
            else F::planes(ph, pl, hd, wrow, g, q);
        };
        int2 am[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            am[k] = int2{};
            if constexpr (F::MIN) {
                u32 lo, hi;
                min_operand((int)bs[k][0], (int)bs[k][1], lo, hi);
                am[k] = int2{(int)lo, (int)hi};
            }
        }
        if constexpr (TREE) {
            const bool apart = b < wide || b >= 16;
            float *const u4 = up + (b < wide ? b : b - 16 + wide) * (4 * OUT) + 4 * lane;
            float t[G][4], s01[G][4];
            ckq_v4f dx[G];
#pragma unroll
            for (int k = 0; k < G; ++k) dx[k] = *reinterpret_cast<const ckq_v4f *>(dxs + b * (G * NT) + k * NT + 4 * q);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                ckq_v4i ph, pl;
                operands(ph, pl, g);
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    const ckq_v4i sh = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[k][g], ph, zero, 0, 0, 0);
                    const ckq_v4i sl = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[k][g], pl, zero, 0, 0, 0);
                    ckq_v4f i2;
                    if constexpr (F::MIN) i2 = min_mfma(am[k], q == g ? hd.mins : zero);
                    float v[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const float f = (float)(F::HALVES ? halves_sum(sh[r], sl[r], sc[2 * g], sc[2 * g + 1]) : (sh[r] << F::SHIFT) + sl[r]);
                        if constexpr (F::MIN) v[r] = (hd.dw * dx[k][r]) * f - (hd.dmin * dx[k][r]) * i2[r];
                        else                  v[r] = (hd.dw * dx[k][r]) * f;
                        asm volatile("" : "+v"(v[r]));              /* rounded before it is added, as in the streaming kernel */
                    }
                    if (apart) *reinterpret_cast<float4 *>(u4 + g * OUT + k * (NT * 16)) = float4{v[0], v[1], v[2], v[3]};
                    else {
#pragma unroll
                        for (int r = 0; r < 4; ++r) {
                            if (g == 0) t[k][r] = v[r];
                            if (g == 1) s01[k][r] = t[k][r] + v[r];
                            if (g == 2) t[k][r] = v[r];
                            if (g == 3) t[k][r] = s01[k][r] + (t[k][r] + v[r]);
                        }
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
            if (!apart) {
#pragma unroll
                for (int k = 0; k < G; ++k) *reinterpret_cast<float4 *>(us + (b - wide) * OUT + k * (NT * 16) + 4 * lane) = float4{t[k][0], t[k][1], t[k][2], t[k][3]};
            }
        } else {
            ckq_v4i sh[G], sl[G];
            int I[G][4] = {};
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                ckq_v4i ph, pl;
                operands(ph, pl, g);
#pragma unroll
                for (int k = 0; k < G; ++k) {
                    sh[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[k][g], ph, !F::HALVES && g ? sh[k] : zero, 0, 0, 0);
                    sl[k] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[k][g], pl, !F::HALVES && g ? sl[k] : zero, 0, 0, 0);
                    if constexpr (F::HALVES) {
#pragma unroll
                        for (int r = 0; r < 4; ++r) I[k][r] += halves_sum(sh[k][r], sl[k][r], sc[2 * g], sc[2 * g + 1]);
                    }
                }
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int k = 0; k < G; ++k) {
                ckq_v4f i2;
                if constexpr (F::MIN) i2 = min_mfma(am[k], hd.mins);
                float out[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const float f = (float)(F::HALVES ? I[k][r] : (sh[k][r] << F::SHIFT) + sl[k][r]);
                    if constexpr (F::MIN) out[r] = hd.dw * f - hd.dmin * i2[r];
                    else                  out[r] = hd.dw * f;
                }
                *reinterpret_cast<float4 *>(us + b * OUT + k * (NT * 16) + 4 * lane) = float4{out[0], out[1], out[2], out[3]};
            }
        }
        if (b + nwave < nb) fetch_a(b + nwave);
    }
    __syncthreads();
    for (int e = tid; e < OUT; e += nthr) {        /* output e % 4 of lane e / 4 of group e / 256 */
        const int tok = 16 * (e >> 8) + 4 * ((e >> 6) & 3) + (e & 3), n = n0 + ((e >> 2) & 15), t = t0 + tok;
        float v = 0.0f;
        if constexpr (TREE) {
            float x[16];
#pragma unroll
            for (int l = 0; l < 16; ++l) {
                if (l >= nb) x[l] = 0.0f;
                else if (l >= wide) x[l] = us[(l - wide) * OUT + e];
                else {
                    const float *const u0 = up + l * (4 * OUT) + e, *const u1 = u0 + wide * (4 * OUT);
                    float p[4];
#pragma unroll
                    for (int g = 0; g < 4; ++g) p[g] = u0[g * OUT] + u1[g * OUT];
                    x[l] = (p[0] + p[1]) + (p[2] + p[3]);
                }
            }
#pragma unroll
            for (int w = 1; w < 16; w *= 2)
#pragma unroll
                for (int l = 0; l < 16; l += 2 * w) x[l] += x[l + w];
            v = x[0] + 0.0f;                      /* the streaming kernel adds each term to a zero */
        } else {
            const float *ue = us + e, *dx = dxs + tok;
            for (int sp = 0; sp < ch.splits; ++sp) {
                const int b0 = sp * ch.per, b1 = min(nb, b0 + ch.per);
                float c[2] = {0.0f, 0.0f};
                for (int b = b0; b < b1; b += 4) {
                    float uu[4], dd[4];
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int bk = min(b + k, b1 - 1);
                        uu[k] = ue[bk * OUT];
                        dd[k] = dx[bk * (G * NT)];
                    }
                    if (ch.kg == 2) {
#pragma unroll
                        for (int k = 0; k < 4; ++k) c[k & 1] = b + k < b1 ? fmaf(dd[k], uu[k], c[k & 1]) : c[k & 1];
                    } else {
#pragma unroll
                        for (int k = 0; k < 4; ++k) c[0] = b + k < b1 ? fmaf(dd[k], uu[k], c[0]) : c[0];
                    }
                }
                if (ch.kg == 2) c[0] += c[1];
                v = sp ? v + c[0] : c[0];
            }
        }
        if (n < N && t < M) y[(size_t)t * ldy + n] = bias ? v + bias[n] : v;
    }
}

/* Short rows, several token groups: a block has a wave for every 256-block of its 16 rows (at most KEEP_NB of them) and goes
 * through `per` groups of 16 tokens, the planes and scales of its weights formed once and kept in registers.  The first kernel
 * forms them again for every group, and they are a good third of what bounds it there, VALU issue (Q5_K, 93 tokens: 480 vector
 * instructions a 256-block and group at 1024 x 4864, 64 % of the busy CUs' issue cycles).  The terms and their order are the same.
 * A group's quants and bsums are copied to LDS without passing through registers, as they lie in memory, as soon as the wave has read the group before: 240
 * instructions a 256-block and group where fetching them to registers and writing them took 301, and two thirds of the LDS instructions.  2 x 4864 x 1024
 * Q5_K at 93 tokens 20.9 us in the first kernel, 13.2 through registers, 11.2 now; over 400 launches of 17 to 256 tokens, 256 to 30000 rows, this against
 * through registers 1.06 on average (five 256-blocks a row, large 1.28-1.43; eight 1.03; all 0.86-1.59).  A lane loading its operands
 * itself needs no LDS and fewer instructions still, but its 64-byte pieces of sixteen tokens are twice the accesses of the L1, which bound
 * large launches (12.2; 64 x 11008 x 2048 Q6_K 17.8 -> 18.5). */
constexpr int KEEP_NB = 8, KEEP_WAVE_LDS = 16 * 288;            /* a group's quants and bsums; before them the 16 weight blocks */
template <class F, bool TREE, bool GRP>
__global__ void __launch_bounds__(64 * KEEP_NB)
gemm_rows16_keep_kernel(const uint8_t *W, const uint8_t *X, int N, int M, int parts, int per, float *y, const float *bias, long ldy, GemmChains ch, Rows16Args grp)
{
    constexpr int NT = 16;
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    const int tid = threadIdx.x, nthr = blockDim.x, nb = nthr >> 6;
    const int lane = tid & 63, wave = wave_in_block();
    const int i16 = lane & 15, q = lane >> 4;
    /* the `parts` blocks of a row tile follow one another on one XCD: blocks are dealt to the eight in turn */
    const int each = gridDim.x >> 3, odd = gridDim.x & 7, xcd = blockIdx.x & 7;
    const int id = xcd * each + min(xcd, odd) + (int)(blockIdx.x >> 3);
    int tile = id / parts;
    const int g0 = (id - tile * parts) * per, g1 = min(g0 + per, (M + NT - 1) / NT);
    if constexpr (GRP) {
        if (tile >= grp.p[1].id0) {
            Rows16Problem p = grp.p[1];
            if (grp.n > 2 && tile >= grp.p[2].id0) p = grp.p[2];
            if (grp.n > 3 && tile >= grp.p[3].id0) p = grp.p[3];
            W = p.W; X = p.X; N = p.N; y = p.y; bias = p.bias; ldy = p.ldy; ch = p.ch;
            tile -= p.id0;
        }
    }
    const int n0 = tile * 16;
    const u32 xrow = (u32)nb * 292u, wpitch = (u32)nb * (u32)F::WBLOCK;
    uint8_t *const al = smem + wave * KEEP_WAVE_LDS, *const bl = al + NT * 256;           /* this wave's weights first, then each group's quants and bsums */
    float *const us = reinterpret_cast<float *>(smem + nb * KEEP_WAVE_LDS);               /* two groups' terms: one written while the other is read */
    const int slots = nb <= 2 ? 2 : nb <= 4 ? 4 : 8;      /* of the tree; the last stay zero */
    float *const dxs = us + 2 * slots * (NT * 16);
    const uint8_t *const wbase = W + (size_t)n0 * wpitch + (u32)wave * (u32)F::WBLOCK;
    const uint8_t *const xbase = X + (u32)wave * 292u;

    /* 16-byte chunk c of token t goes to slot c ^ t; j = 4: the bsums */
    u32 asrc[5], dsrc;
    auto token_offsets = [&](int last) {
#pragma unroll
        for (int j = 0; j < 4; ++j) asrc[j] = (u32)min(4 * j + q, last) * xrow + 4u + 16u * (u32)(i16 ^ (4 * j + q));
        asrc[4] = (u32)min(lane >> 1, last) * xrow + 260u + 16u * (u32)(lane & 1);
        dsrc = (u32)min(i16, last) * xrow;
    };
    token_offsets(min(NT, M - g0 * NT) - 1);
    const ckq_v4i xsrd = {__builtin_amdgcn_readfirstlane((int)(u32)(uintptr_t)xbase), __builtin_amdgcn_readfirstlane((int)(u32)((uintptr_t)xbase >> 32)), 0x7fffffff, 0x00020000};
    const u32 adst = lds_address(al);
    u32 dr;
    auto fetch = [&](int gr) {
        const int k = gr * NT * (int)xrow;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int j = 0; j < 4; ++j) lds_copy16(xsrd, adst + 1024u * j, asrc[j], k);
        if (F::MIN && lane < 32) lds_copy16(xsrd, adst + 4096u, asrc[4], k);
        dr = ld4<4>(xbase + (size_t)(u32)k + dsrc);         /* last: once it is there, all are */
        __builtin_amdgcn_sched_barrier(0);
    };
    constexpr int NWL = (16 * F::CHUNKS + 63) / 64;
    ckq_v4i wr[NWL];
    u32 wdst[NWL];
#pragma unroll
    for (int j = 0; j < NWL; ++j) {
        const int e = min(64 * j + lane, 16 * F::CHUNKS - 1), r = e / F::CHUNKS, c = e % F::CHUNKS;
        u32 t[4];
        ld16<F::WBLOCK % 4 == 0 ? 4 : 2>(t, wbase + ((u32)min(r, N - 1 - n0) * wpitch + F::chunk_ofs(c)));
        wr[j] = ckq_v4i{(int)t[0], (int)t[1], (int)t[2], (int)t[3]};
        wdst[j] = (u32)(r * F::PITCH + 16 * c);
    }
#pragma unroll
    for (int j = 0; j < NWL; ++j) *reinterpret_cast<ckq_v4i *>(al + wdst[j]) = wr[j];
    __builtin_amdgcn_wave_barrier();
    Head hd;
    ckq_v4i ph[4], pl[4];
    const uint8_t *const wrow = al + i16 * F::PITCH;
    F::head(hd, wrow, q);
#pragma unroll
    for (int g = 0; g < 4; ++g) F::planes(ph[g], pl[g], hd, wrow, g, q);
    for (int e = tid; e < (slots - nb) * (NT * 16); e += nthr) us[nb * (NT * 16) + e] = us[(slots + nb) * (NT * 16) + e] = 0.0f;
    __builtin_amdgcn_s_waitcnt(0xc07f);           /* lgkmcnt(0): the weights have been read */
    asm volatile("" ::: "memory");
    fetch(g0);
    /* vmcnt(0): in the loop a group's loads are older than the stores of the group before, and only with nothing on its way here can
     * the compiler tell, and wait for the loads alone */
    __builtin_amdgcn_s_waitcnt(0x0f70);

    const ckq_v4i zero = {0, 0, 0, 0};
    for (int gr = g0, p = 0; gr < g1; ++gr, p ^= 1) {
        float *const u = us + p * slots * (NT * 16), *const dx = dxs + p * nb * NT;
        asm volatile("" : "+v"(dr));
        if (lane < NT) dx[wave * NT + lane] = __builtin_bit_cast(float, dr);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        int2 am = {};
        if constexpr (F::MIN) {
            const int2 b = *reinterpret_cast<const int2 *>(bl + 32 * i16 + 8 * q);
            u32 lo, hi;
            min_operand(b.x, b.y, lo, hi);
            am = int2{(int)lo, (int)hi};
        }
        ckq_v4i a[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) a[g] = lds16(al + 256 * i16 + 16 * ((int)(F::a_elem(g, q) >> 4) ^ i16));
        /* the next group comes where this one lay once it has been read: lgkmcnt(0) */
        __builtin_amdgcn_s_waitcnt(0xc07f);
        asm volatile("" : "+v"(a[0]), "+v"(a[1]), "+v"(a[2]), "+v"(a[3]), "+v"(am.x), "+v"(am.y) :: "memory");
        if (gr + 1 < g1) {
            if ((gr + 2) * NT > M) token_offsets(M - 1 - (gr + 1) * NT);
            fetch(gr + 1);
        }
        auto min_mfma = [&](const ckq_v4i &mins) {
            const ckq_v4f z = {0.0f, 0.0f, 0.0f, 0.0f};
            const ckq_v4i am4 = {am.x, am.y, 0, 0};
            return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ckq_v8bf, am4), __builtin_bit_cast(ckq_v8bf, mins), z, 0, 0, 0);
        };
        float out[4];
        if constexpr (TREE) {
            const ckq_v4i dxi = lds16(reinterpret_cast<const uint8_t *>(dx + wave * NT + 4 * q));
            float t[4][4];
            ckq_v4i sh[4], sl[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                sh[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[g], ph[g], zero, 0, 0, 0);
                sl[g] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[g], pl[g], zero, 0, 0, 0);
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                ckq_v4f i2;
                if constexpr (F::MIN) i2 = min_mfma(q == g ? hd.mins : zero);
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int di = dxi[r];
                    const float d = __builtin_bit_cast(float, di), f = (float)((sh[g][r] << F::SHIFT) + sl[g][r]);
                    float v;
                    if constexpr (F::MIN) v = (hd.dw * d) * f - (hd.dmin * d) * i2[r];
                    else                  v = (hd.dw * d) * f;
                    asm volatile("" : "+v"(v));              /* rounded before it is added, as in the streaming kernel */
                    t[g][r] = v;                             /* which adds it to a zero: made up for by the zero at the end */
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) out[r] = (t[0][r] + t[1][r]) + (t[2][r] + t[3][r]);
        } else {
            ckq_v4i sh, sl;
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                sh = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[g], ph[g], g ? sh : zero, 0, 0, 0);
                sl = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[g], pl[g], g ? sl : zero, 0, 0, 0);
            }
            ckq_v4f i2;
            if constexpr (F::MIN) i2 = min_mfma(hd.mins);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const float f = (float)((sh[r] << F::SHIFT) + sl[r]);
                if constexpr (F::MIN) out[r] = hd.dw * f - hd.dmin * i2[r];
                else                  out[r] = hd.dw * f;
            }
        }
        *reinterpret_cast<float4 *>(u + wave * (NT * 16) + 4 * lane) = float4{out[0], out[1], out[2], out[3]};
        /* one barrier a group: the terms of the group after next overwrite these, behind the next group's barrier */
        __syncthreads();
        const __amdgpu_buffer_rsrc_t yb = __builtin_amdgcn_make_buffer_rsrc(y + (size_t)(gr * NT) * ldy, 0, 0x7fffffff, 0x00020000);
        /* Four waves add the terms up, of eight the two fours in turn.  All store, the others past the buffer's end: a store that not every
         * way through the loop has would make the loads of the next group wait for it. */
        const bool mine = nthr <= NT * 16 || wave >> 2 == (nb == 8 ? gr & 1 : 0);
        int done = 0;
        do {
            const int e = min(done + (tid & (NT * 16 - 1)), NT * 16 - 1);          /* output e % 4 of lane e / 4 */
            const int tok = 4 * (e >> 6) + (e & 3), n = n0 + ((e >> 2) & 15);
            const bool live = mine && done + (tid & (NT * 16 - 1)) < NT * 16 && n < N && gr * NT + tok < M;
            const float *ue = u + e;
            float v = 0.0f;
            if (mine) {
                if constexpr (TREE) {
                    auto pair = [&](int b) { return ue[b * (NT * 16)] + ue[(b + 1) * (NT * 16)]; };
                    v = pair(0);
                    if (nb > 2) v += pair(2);
                    if (nb > 4) v += pair(4) + pair(6);
                    v += 0.0f;                    /* the rest of the tree, empty */
                } else {
                    for (int sp = 0; sp < ch.splits; ++sp) {
                        const int b0 = sp * ch.per, b1 = min(nb, b0 + ch.per);
                        float c[2] = {0.0f, 0.0f};
                        for (int b = b0; b < b1; ++b) {
                            const int k = ch.kg == 2 ? (b - b0) & 1 : 0;
                            const float uu = ue[b * (NT * 16)], dd = dx[b * NT + tok];
                            if (k) c[1] = fmaf(dd, uu, c[1]);
                            else   c[0] = fmaf(dd, uu, c[0]);
                        }
                        if (ch.kg == 2) c[0] += c[1];
                        v = sp ? v + c[0] : c[0];
                    }
                }
                if (bias) v += bias[min(n, N - 1)];
            }
            __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(u32, v), yb, live ? 4 * (tok * (int)ldy + n) : -4, 0, 0);
            done += nthr;
        } while (done < NT * 16);
    }
}

/* Waves per block: with two tiles per CU and more, blocks of four waves overlap each other's beginnings and ends
 * (32000 x 4096, 13 tokens: 27 us, with eight 41); with fewer, a tile's blocks spread over more waves.  A tile alone on its CU takes twelve
 * for rows of more than twelve 256-blocks: 44 launches of 64 to 256 tiles 1.02 on average, up to 1.11 (us, eight -> twelve: Q4_K 4096 x 4096 at 13
 * tokens 7.08 -> 6.81, Q5_K 3568 x 5888 10.2 -> 9.2, Q6_K 2048 x 5632 10.5 -> 9.3; sixteen 1.017; up to twelve blocks 0.98); but Q6_K rows of more than 32 in the
 * tile kernels' order, whose blocks come in more bytes, 0.986 over 100 launches (2048 x 8448 at 9 11.9 -> 12.6).  In the streaming kernel's order `nb` is
 * the sums that are dealt, sixteen at most, and twelve waves it is for Q6_K as well: 1.05 over 118 launches of 5 and 8 tokens, rows of 13 to 43 blocks (Q6_K of 33 1.06, of 43 1.01). */
int rows16_waves(int fmt, int tiles, int nb)
{
    int waves = tiles >= 512 ? 4 : tiles > 256 ? 8 : tiles > 64 ? (nb > 12 && (fmt != CKQ_FMT_Q6_K || nb <= 32) ? 12 : 8) : 16;
    while (waves > 4 && waves / 2 >= nb) waves /= 2;
    return waves;
}

template <class F, int NT, bool TREE>
int launch_rows16_nt(int fmt, Rows16Args &a, hipStream_t s)
{
    unsigned grid = 0;
    for (int i = 0; i < a.n; ++i) {
        a.p[i].id0 = (int)grid;
        grid += (unsigned)((a.p[i].N + 15) / 16);
    }
    const unsigned gy = (unsigned)((a.M + NT - 1) / NT);
    if (gy > 65535) return CKQ_ESHAPE;
    auto lds_bytes = [&](int w) { return (size_t)w * rows16_wave_lds<F, NT>() + (size_t)(TREE && a.nb > 16 ? 16 : a.nb) * (NT * 64) + (size_t)a.nb * (NT * 4); };
    int waves = rows16_waves(fmt, (int)(grid * gy), TREE ? (a.nb < 16 ? a.nb : 16) : a.nb);
    while (waves > 4 && lds_bytes(waves) > 160 * 1024) waves -= 4;
    const size_t lds = lds_bytes(waves);
    if (lds > 160 * 1024) return CKQ_ESHAPE;
    if (lds > 64 * 1024) {
        /* more than 64 KB of dynamic LDS is an opt-in per function and device; asked for once */
        static std::atomic<uint64_t> done[2];
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return (int)e;
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done[a.n > 1].load(std::memory_order_acquire) & bit)) {
            e = hipFuncSetAttribute(a.n > 1 ? (const void *)gemm_rows16_kernel<F, NT, TREE, true> : (const void *)gemm_rows16_kernel<F, NT, TREE, false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            done[a.n > 1].fetch_or(bit, std::memory_order_release);
        }
    }
    const Rows16Problem &p = a.p[0];
    const Rows16Shape S = {a.M, a.nb};
    if (a.n > 1)
        hipLaunchKernelGGL((gemm_rows16_kernel<F, NT, TREE, true>), dim3(grid, gy), dim3(64 * waves), lds, s, p.W, p.X, p.N, S, p.y, p.bias, p.ldy, p.ch, a);
    else
        hipLaunchKernelGGL((gemm_rows16_kernel<F, NT, TREE, false>), dim3(grid, gy), dim3(64 * waves), lds, s, p.W, p.X, p.N, S, p.y, p.bias, p.ldy, p.ch, a);
    return (int)hipGetLastError();
}

/* Blocks per row tile of the kernel that keeps its planes, 0: another kernel; its time in us.  With n blocks on the fullest CU, as many at once as sixteen waves
 * are, a block takes (its groups + per0) (a + short_row (1 / nb - 1/4) where nb < 4 + s waves a SIMD), what comes after the first round `later` of that, a launch t0 more; the
 * other kernels together 3.3..3.8 + ...: `other`, by nb and by thousands of tiles of 16 rows and tokens.  Fitted to 210 launches of 16 to 224 x 16 tokens and rows up to 14000, one to
 * eight blocks a row tile, in either order of the sums: 6 to 7 % rms (other: 7 to 11).  Over further launches the choice costs 0.2 to 0.5 % more than the best of all in
 * the streaming kernel's order, 0.9 to 2.6 in the tile kernels'; an older fit, to an older kernel and without rounds, cost 7.2 to 16.4 and 2.4 to 6.0, at most 75 (us: Q4_K 4630 x 512 at
 * 82 tokens 7.0 -> 5.1, Q5_K 993 x 256 at 194 6.0 -> 4.2, 2069 x 1280 at 219 9.7 -> 8.4). */
struct KeepFit { float t0, per0, a, s, short_row, later, other[4]; };
const KeepFit keep_fit[3][2] = {
    {{2.21f, 0.56f, 0.55f, 0.315f, 0.60f, 0.92f, {3.35f, -0.072f, 0.334f, 1.65f}}, {2.11f, 0.88f, 0.50f, 0.318f, 0.30f, 0.81f, {3.74f, 0.022f, 0.363f, 1.97f}}},
    {{1.84f, 1.65f, 0.64f, 0.246f, 0.41f, 0.72f, {3.27f, 0.115f, 0.571f, 1.22f}}, {1.66f, 2.00f, 0.57f, 0.230f, 0.26f, 0.68f, {3.82f, 0.088f, 0.706f, 1.49f}}},
    {{2.25f, 1.68f, 0.55f, 0.238f, 0.53f, 0.65f, {2.73f, 0.197f, 0.632f, 1.40f}}, {2.01f, 2.40f, 0.42f, 0.201f, 0.22f, 0.86f, {3.82f, 0.075f, 0.850f, 0.45f}}}};
int rows16_keep_parts(int fmt, bool tree, long tiles, int groups, int nb, float *time)
{
    if (nb > (fmt == CKQ_FMT_Q4_K ? 4 : KEEP_NB) || groups < 2 || tiles > 1 << 20 || groups > 1 << 10) return 0;
    const KeepFit &f = keep_fit[fmt == CKQ_FMT_Q4_K ? 0 : fmt == CKQ_FMT_Q5_K ? 1 : 2][tree];
    const int at_once = 16 / nb;
    const float block = f.a + (nb < 4 ? f.short_row * (1.0f / (float)nb - 0.25f) : 0.0f), wave = 0.25f * f.s * (float)nb;
    int best = 0;
    float least = 0.0f;
    for (int per = groups; per >= 1; --per) {
        const int parts = (groups + per - 1) / per;
        if (per > 1 && (groups + per - 2) / (per - 1) == parts) continue;          /* fewer groups a block in as many blocks */
        const long n = (tiles * parts + 255) / 256, full = n / at_once, rest = n % at_once;
        const float t = f.t0 + ((float)per + f.per0) * ((float)full * (block + wave * (float)at_once) + (rest ? (block + wave * (float)rest) * (full ? f.later : 1.0f) : 0.0f));
        if (!best || t < 1.02f * least) { least = best ? std::min(t, least) : t; best = parts; }       /* of two alike the shorter blocks */
    }
    const float n16 = 1e-3f * (float)(tiles * groups);
    if (least >= f.other[0] + f.other[1] * (float)nb + (f.other[2] * (float)nb + f.other[3]) * n16) return 0;
    if (time) *time = least;
    return best;
}

template <class F, bool TREE>
int launch_rows16_keep(Rows16Args &a, int parts, hipStream_t s)
{
    int tiles = 0;
    for (int i = 0; i < a.n; ++i) {
        a.p[i].id0 = tiles;
        tiles += (a.p[i].N + 15) / 16;
    }
    const int groups = (a.M + 15) / 16, per = (groups + parts - 1) / parts;
    const size_t lds = (size_t)a.nb * (KEEP_WAVE_LDS + 2 * 64) + (a.nb <= 2 ? 2 : a.nb <= 4 ? 4 : 8) * 2 * 1024;
    const Rows16Problem &p = a.p[0];
    const dim3 grid((unsigned)(tiles * parts)), block((unsigned)(64 * a.nb));
    if (a.n > 1)
        hipLaunchKernelGGL((gemm_rows16_keep_kernel<F, TREE, true>), grid, block, lds, s, p.W, p.X, p.N, a.M, parts, per, p.y, p.bias, p.ldy, p.ch, a);
    else
        hipLaunchKernelGGL((gemm_rows16_keep_kernel<F, TREE, false>), grid, block, lds, s, p.W, p.X, p.N, a.M, parts, per, p.y, p.bias, p.ldy, p.ch, a);
    return (int)hipGetLastError();
}

/* Blocks of a launch of the kernel that holds its activations, and their tiles a round; false: another kernel.  `tree` has four times the fp32 terms
 * and gains less.  Fitted to 200 launches of both kernels, 5 to 16 tokens, 1024 x 256 to 150000 x 1024 (time of the kernel above over this one's): up to
 * four 256-blocks a row and eight, which fill the 16 waves of a CU, 1.0-2.0 at any size (Q4_K 3328 x 1024 4.8 -> 4.1, Q6_K 79808 x 256 15.4 -> 8.3,
 * 39872 x 2048 23.8 -> 20.3), one or two blocks below a quarter of a round 0.95-1.0; five to seven 0.74-1.1 (they leave waves of the CU
 * idle); above eight from 1.7 rounds of the CUs on with the tile kernels' sums 1.0-1.47 where 14 to 16 waves are at work, from 4 on 1.04-1.26 with fewer;
 * with the streaming kernel's from 5 and 8, 0.99-1.09 (below: 0.88-1.03). */
template <class F>
bool rows16_hold(const Rows16Args &a, bool tree, int tiles, int *grid, int *round, size_t *lds)
{
    if (a.nb > HOLD_NB || a.M > 16) return false;
    for (int i = 0; i < a.n; ++i)
        if (a.p[i].X != a.p[0].X || a.p[i].N < 16) return false;
    const int occ = HOLD_NB / a.nb;                /* blocks on a CU */
    const float rounds = (float)tiles / (float)(256 * occ);
    float least = 0.0f;
    if (a.nb <= 2) least = 0.25f;
    else if (a.nb > 8) least = a.nb >= 14 ? (tree ? 5.0f : 1.7f) : (tree ? 8.0f : 4.0f);
    else if (a.nb > 4 && a.nb < 8) return false;
    if (rounds < least) return false;
    const size_t tile = (size_t)a.nb * 1024, fixed = (size_t)a.nb * (16 * F::PITCH) + HOLD_NB * 64;
    *grid = tiles < 256 * occ ? tiles : 256 * occ;
    const int most = (tiles + *grid - 1) / *grid, fit = (int)((160 * 1024 / occ - fixed) / tile), turns = (most + fit - 1) / fit;
    *round = (most + turns - 1) / turns;
    *lds = fixed + *round * tile;
    return true;
}

template <class F, bool TREE>
int launch_rows16_hold(Rows16Args &a, int tiles, int grid, int round, size_t lds, hipStream_t s)
{
    int id = 0;
    for (int i = 0; i < a.n; ++i) {
        a.p[i].id0 = id;
        id += (a.p[i].N + 15) / 16;
    }
    if (lds > 64 * 1024) {
        static std::atomic<uint64_t> done[2];      /* as in launch_rows16_nt */
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return (int)e;
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done[a.n > 1].load(std::memory_order_acquire) & bit)) {
            e = hipFuncSetAttribute(a.n > 1 ? (const void *)gemm_rows16_hold_kernel<F, TREE, true> : (const void *)gemm_rows16_hold_kernel<F, TREE, false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            done[a.n > 1].fetch_or(bit, std::memory_order_release);
        }
    }
    const Rows16Problem &p = a.p[0];
    if (a.n > 1)
        hipLaunchKernelGGL((gemm_rows16_hold_kernel<F, TREE, true>), dim3((unsigned)grid), dim3((unsigned)(64 * a.nb)), lds, s, p.W, p.X, p.N, a.M, a.nb, tiles, round, p.y, p.bias, p.ldy, p.ch, a);
    else
        hipLaunchKernelGGL((gemm_rows16_hold_kernel<F, TREE, false>), dim3((unsigned)grid), dim3((unsigned)(64 * a.nb)), lds, s, p.W, p.X, p.N, a.M, a.nb, tiles, round, p.y, p.bias, p.ldy, p.ch, a);
    return (int)hipGetLastError();
}

/* Waves and LDS of a launch of the kernel that takes groups in pairs; 0: another kernel.  From 420 launches of both, 17 to 130 tokens, rows of 9 to 43 blocks
 * (Q4_K 5): as long as a block for every group and row tile finds a CU of its own it loses (0.69-1.0, two groups in a row where there
 * could be two CUs), past that it wins while the pairs still do: Q4_K 1.01-1.36, Q5_K 1.12-1.45, Q6_K 1.22-1.67, in the streaming kernel's order 0.99-1.15 (there twelve waves
 * are 2-4 % ahead of eight).  With more pairs than CUs, eight waves: Q6_K 1.18-1.37 on average (0.94-1.61), Q5_K 1.07-1.16 but for three groups, 0.97;
 * Q4_K, whose planes are quickly formed, 0.92-1.09, and the streaming kernel's order 0.72-0.83.  Rows of which only one such block fits a CU lose too
 * (Q5_K 914 x 7168 at 175: tile kernel 18.6, this 23.2), and rows of up to four blocks, which have as many waves (Q4_K 2757 x 256 at 28: 5.1, planes kept 3.7). */
int rows16_pair_waves(int fmt, bool tree, long tiles, int groups, int nb, size_t *lds)
{
    const int wide = tree && nb > 16 ? nb - 16 : 0;
    const long pairs = tiles * ((groups + 1) / 2);
    if (nb < 5 || groups < 2 || groups > 1 << 10 || tiles * groups <= 256 || wide > 16) return 0;
    if (pairs > 256 && (tree || fmt == CKQ_FMT_Q4_K || (fmt == CKQ_FMT_Q5_K && groups == 3))) return 0;
    const int waves = std::min(pairs <= 256 ? 12 : 8, nb);
    const size_t pitch = fmt == CKQ_FMT_Q4_K ? R16Q4K::PITCH : fmt == CKQ_FMT_Q5_K ? R16Q5K::PITCH : R16Q6K::PITCH;
    const size_t terms = tree ? (size_t)(std::min(nb, 16) - wide) + 8 * wide : (size_t)nb;
    *lds = waves * (16 * pitch) + (size_t)nb * 128 + terms * 2048;
    return *lds > (pairs > 256 ? 80 : 160) * 1024 ? 0 : waves;
}

template <class F, bool TREE>
int launch_rows16_pair(Rows16Args &a, int waves, size_t lds, hipStream_t s)
{
    unsigned grid = 0;
    for (int i = 0; i < a.n; ++i) {
        a.p[i].id0 = (int)grid;
        grid += (unsigned)((a.p[i].N + 15) / 16);
    }
    const unsigned gy = (unsigned)((a.M + 31) / 32);
    if (lds > 64 * 1024) {
        static std::atomic<uint64_t> done[2];      /* as in launch_rows16_nt */
        int dev = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e != hipSuccess) return (int)e;
        const uint64_t bit = 1ull << (dev & 63);
        if (!(done[a.n > 1].load(std::memory_order_acquire) & bit)) {
            e = hipFuncSetAttribute(a.n > 1 ? (const void *)gemm_rows16_pair_kernel<F, TREE, true> : (const void *)gemm_rows16_pair_kernel<F, TREE, false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
            if (e != hipSuccess) return (int)e;
            done[a.n > 1].fetch_or(bit, std::memory_order_release);
        }
    }
    const Rows16Problem &p = a.p[0];
    if (a.n > 1)
        hipLaunchKernelGGL((gemm_rows16_pair_kernel<F, TREE, true>), dim3(grid, gy), dim3((unsigned)(64 * waves)), lds, s, p.W, p.X, p.N, a.M, a.nb, p.y, p.bias, p.ldy, p.ch, a);
    else
        hipLaunchKernelGGL((gemm_rows16_pair_kernel<F, TREE, false>), dim3(grid, gy), dim3((unsigned)(64 * waves)), lds, s, p.W, p.X, p.N, a.M, a.nb, p.y, p.bias, p.ldy, p.ch, a);
    return (int)hipGetLastError();
}

template <class F>
int launch_rows16(int fmt, Rows16Args &a, hipStream_t s)
{
    long tiles = 0;
    for (int i = 0; i < a.n; ++i) tiles += (a.p[i].N + 15) / 16;
    bool near = true;                              /* the kernel that keeps its planes has 32 bits for where a group's outputs lie */
    for (int i = 0; i < a.n; ++i) near = near && a.p[i].ldy < 1 << 25;
    const int parts = near ? rows16_keep_parts(fmt, a.tree, tiles, (a.M + 15) / 16, a.nb, nullptr) : 0;
    if (parts) return a.tree ? launch_rows16_keep<F, true>(a, parts, s) : launch_rows16_keep<F, false>(a, parts, s);
    int grid, round;
    size_t lds;
    if (tiles < 1 << 20 && rows16_hold<F>(a, a.tree, (int)tiles, &grid, &round, &lds))
        return a.tree ? launch_rows16_hold<F, true>(a, (int)tiles, grid, round, lds, s) : launch_rows16_hold<F, false>(a, (int)tiles, grid, round, lds, s);
    if (const int waves = rows16_pair_waves(fmt, a.tree, tiles, (a.M + 15) / 16, a.nb, &lds))
        return a.tree ? launch_rows16_pair<F, true>(a, waves, lds, s) : launch_rows16_pair<F, false>(a, waves, lds, s);
    if (a.tree) return a.M <= 8 ? launch_rows16_nt<F, 8, true>(fmt, a, s) : launch_rows16_nt<F, 16, true>(fmt, a, s);
    return launch_rows16_nt<F, 16, false>(fmt, a, s);           /* the tile kernels start above eight tokens */
}

} // namespace

float gemm_rows16_keep_time(int fmt, bool tree, size_t rows, int ntok, int nb)
{
    float t = 0.0f;
    return rows16_keep_parts(fmt, tree, (long)((rows + 15) / 16), (ntok + 15) / 16, nb, &t) ? t : 0.0f;
}

/* Fitted to the launches of the rule above in the tile kernels' order, 12-15 % rms. */
float gemm_rows16_pair_time(int fmt, size_t rows, int ntok, int nb)
{
    static const float fit[3][3] = {{3.2f, 0.04f, 0.27f}, {3.4f, 0.11f, 0.29f}, {2.6f, 0.09f, 0.30f}};
    size_t lds;
    const long tiles = (long)((rows + 15) / 16), groups = (ntok + 15) / 16;
    if (tiles > 1 << 20 || !rows16_pair_waves(fmt, false, tiles, (int)groups, nb, &lds)) return 0.0f;
    const float *f = fit[fmt == CKQ_FMT_Q4_K ? 0 : fmt == CKQ_FMT_Q5_K ? 1 : 2], on_cu = (float)(tiles * ((groups + 1) / 2)) / 256.0f;
    return f[0] + (f[1] + f[2] * fmaxf(on_cu, 1.0f)) * (float)nb;
}

int launch_gemm_rows16(int fmt, Rows16Args &a, hipStream_t s)
{
    switch (fmt) {
    case CKQ_FMT_Q4_K: return launch_rows16<R16Q4K>(fmt, a, s);
    case CKQ_FMT_Q5_K: return launch_rows16<R16Q5K>(fmt, a, s);
    case CKQ_FMT_Q6_K: return launch_rows16<R16Q6K>(fmt, a, s);
    default: return CKQ_EFORMAT;
    }
}
