/*
 * ckq_gemm_q80_dw.hip - prefill GEMM, Q8_0 weights x Q8_0 activations, on the gfx950 int8 matrix cores, for rows that start on
 * dwords and hold an even number of blocks (K a multiple of 64); ckq_gemm_q80.hip takes the others.
 *
 *   C[t][n] = sum_j dx(t,j) * (dw(n,j) * S(t,n,j))   (+ bias[n]),   S = the integer dot of 32-block j
 *
 * What bounds it: the scaling of the integers, which cannot be summed over blocks before it, once the copies are out of the way:
 * - Fetched block by block from 2-byte aligned addresses, as the other kernel has to, every lane of a copy is a memory access of
 *   its own and the requests bound the launch.  Here rows travel as they lie in memory, in dword-aligned 16-byte chunks, and are
 *   read where they are (image below).
 * - v_mfma_i32_16x16x32_i8, K = 32 being one block, starts from the accumulator 0x4B400000, so that its result read as fp32 is
 *   exactly M + S (M = 1.5 * 2^23, |S| < 2^20).  t = fma(dw, M + S, -dw M) is dw S rounded once (dw M has 13 bits), and acc =
 *   fma(dx, t, acc): two plain fp32 operations per output and block, against the other kernel's convert, product and
 *   multiply-add with a lane broadcast.
 *   A row whose fp16 scale is infinite gives NaN that way; such outputs are summed again term by term at the end.
 * - Tokens are the A operand, weight rows the B operand: lane 16 q + i holds ONE weight row and tokens 4 q .. 4 q + 3 of a
 *   16 x 16 result.  LDS row 64 h + 16 g + i is weight row 64 h + 4 i + g, so a lane ends with four adjacent rows.
 * - K advances 128 (four blocks) per iteration, two stages.  Of the eight waves, four take two of the blocks and four the
 *   other two, each 64 rows x 32 tokens; the partial tiles are added through LDS at the end.  That gives a tile alone on its
 *   CU two waves per SIMD and two tiles four.
 *
 * Measured, us, the other kernel (weights two bytes off) -> this one: 333 tokens x 4864 x 4096 51.3 -> 37.8, 512 x 9728 x 896
 * 34.7 -> 25.5, 2048 x 11008 x 4096 426 -> 322, 464 x 37134 x 2048 218 -> 154, 24 x 4864 x 4096 15.7 -> 13.9.  At 2048 tokens a block's
 * iteration takes 1970 cycles of its CU, of which the vector instructions issue 1260 and the matrix instructions 510 (counters).
 *
 * Block = 8 waves = 64 tokens x 128 weight rows.
 */
#include "ckq_gemm_common.hpp"

constexpr int GEMM8_BM = 64, GEMM8_BN = 128, GEMM8_KB = 4;   /* tokens, rows, 32-blocks per iteration */
constexpr int GEMM8_THREADS = 512;
constexpr int GEMM8_PITCH = 144;                 /* bytes of an operand row's image in LDS: see below */
constexpr int GEMM8_REGION = 24 * GEMM8_PITCH;   /* the rows a wave brings in: sixteen weight rows, eight tokens */
typedef float ckq_v4f __attribute__((ext_vector_type(4)));

/* Output (weight row w, activation row x) over blocks [j0, j1), one term at a time. */
__device__ __forceinline__ float q80_output(const uint8_t *w, const uint8_t *x, int j0, int j1)
{
    float acc = 0.0f;
    for (int j = j0; j < j1; ++j) {
        int s = 0;
        for (int i = 0; i < 8; ++i) s = dot4((int)ld4<2>(w + 34 * j + 2 + 4 * i), (int)ld4<2>(x + 34 * j + 2 + 4 * i), s);
        acc = __builtin_fmaf(h2f(ld2(w + 34 * j)), h2f(ld2(x + 34 * j)) * (float)s, acc);
    }
    return acc;
}

/* Global -> LDS, 16 bytes per lane from rs + ofs + k to dst + 16 lane.  Written out because the compiler, which cannot know which
 * bytes of an LDS object a copy in flight still has to write, waits for all of them before the next read of that object; the
 * one wait there has to be is the loop's. */
__device__ __forceinline__ void lds_copy16(const ckq_v4i &rs, u32 dst, u32 ofs, int k)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(dst), "v"(ofs), "s"(rs), "s"(k) : "memory");
}
__device__ __forceinline__ u32 lds_address(const void *p) { return (u32)(uintptr_t)(__attribute__((address_space(3))) const void *)p; }

/*
 * LDS image of an operand row, 144 bytes for the four blocks of an iteration: the 136 bytes as they are in memory, 34 dwords, in
 * nine 16-byte chunks (adjacent lanes of a copy fetch adjacent chunks, all from dword-aligned addresses).  Chunk 8 holds the last
 * sixteen, so dwords 30 to 33 of the run lie at 32 to 35.  A pair of blocks is 17 dwords: [d0 q0q1] seven of quants [q30q31 d1]
 * eight of quants.  Once a row has landed, the lane in charge makes [q0q1 q30q31] of the first and the ninth - the order of
 * the 32 products of a block is free as long as both operands have the same - and leaves the scales as fp32 in dwords nobody
 * reads (slot).  Lane quarter q takes dwords q and q + 4 of a block: with rows 36 dwords apart every bank then serves two lanes.
 */
template <bool DUMP>
__global__ void __launch_bounds__(GEMM8_THREADS, DUMP ? 2 : 4) gemm_q80_dw_kernel(GemmArgs a)
{
    constexpr int BM = GEMM8_BM, BN = GEMM8_BN, KB = GEMM8_KB, PITCH = GEMM8_PITCH, MAGIC = 0x4B400000;
    __shared__ __attribute__((aligned(16))) uint8_t stage[2][8 * GEMM8_REGION];

    const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_block();
    const int i16 = lane & 15, q = lane >> 4;
    const int kh = wave >> 2, rh = (wave >> 1) & 1, th = wave & 1;

    /* token tiles fastest inside an XCD, so each XCD's L2 sees a weight tile once */
    const GemmWork work = gemm_work(a, (a.nb + KB - 1) / KB);
    const int id = work.id, xcd = id & 7, seq = id >> 3;
    const int tt = seq % a.ntt;
    const int nt = (seq / a.ntt) * 8 + xcd;
    if (nt >= work.nnt) return;
    const int t0 = tt * BM, n0 = nt * BN;
    const int nblk = a.nb;                                  /* 32-blocks per row */
    const u32 stride = (u32)nblk * 34u;                     /* bytes per weight row and per activation row */
    const int it0 = work.k0, niter = work.k1;               /* this block runs iterations [it0, niter) */
    const uint8_t *wbase = work.B + (size_t)n0 * stride;    /* uniform */
    const uint8_t *xbase = a.A + (size_t)t0 * stride;       /* uniform */
    auto buffer = [](const uint8_t *p) {
        const uint64_t b = (uint64_t)p;
        return ckq_v4i{__builtin_amdgcn_readfirstlane((int)(u32)b), __builtin_amdgcn_readfirstlane((int)(u32)(b >> 32)), 0x7fffffff, 0x00020000};
    };
    const ckq_v4i bw = buffer(wbase), bx = buffer(xbase);
    auto w_row = [&](int l) { return (u32)min(64 * (l >> 6) + 4 * (l & 15) + ((l >> 4) & 3), work.N - 1 - n0) * stride; };
    auto x_row = [&](int t) { return (u32)min(t, a.M - 1 - t0) * stride; };

    /* A wave copies sixteen weight rows (144 chunks, three instructions) and eight tokens (72 chunks, two) into its region of a
     * stage, and finishes the same rows when they have landed. */
    u32 c_src[5];
    bool c_on[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) {
        const int ci = 64 * (i < 3 ? i : i - 3) + lane, r = ci / 9, c = ci % 9;
        c_on[i] = ci < (i < 3 ? 144 : 72);
        c_src[i] = (i < 3 ? w_row(16 * wave + min(r, 15)) : x_row(8 * wave + min(r, 7))) + (u32)min(16 * c, 120);
    }
    auto copy = [&](int it, uint8_t *sg) {
        const u32 dst = lds_address(sg + GEMM8_REGION * wave);
#pragma unroll
        for (int i = 0; i < 5; ++i)
            if (c_on[i]) lds_copy16(i < 3 ? bw : bx, dst + (u32)(i < 3 ? 1024 * i : 16 * PITCH + 1024 * (i - 3)), c_src[i], it * (KB * 34));
    };
    /* K ends after 17 dwords of the iteration: fetched one by one, a 16-byte chunk could pass the end of the matrix */
    auto copy_tail = [&](int it, uint8_t *sg) {
        for (int e = lane; e < 24 * 17; e += 64) {
            const int r = e / 17, d = e % 17;
            const uint8_t *const src = r < 16 ? wbase + w_row(16 * wave + r) : xbase + x_row(8 * wave + r - 16);
            *reinterpret_cast<u32 *>(sg + GEMM8_REGION * wave + PITCH * r + 4 * d) = ld4<4>(src + (u32)it * (KB * 34u) + 4u * (u32)d);
        }
    };
    /* the dword with the scale of block 2 p + o of a row whose number has bit 3 = s: rows 8 apart start on the same bank */
    auto slot = [](int p, int o_xor_s) { return p ? 30 + o_xor_s : o_xor_s ? 25 : 8; };
    /* two lanes per row, one for each pair of blocks */
    const int f_row = lane >> 1, f_p = lane & 1, f_s = f_row < 16 ? f_row >> 3 : wave & 1;
    auto finish = [&](int it, uint8_t *sg) {
        if (f_row >= 24) return;
        u32 *const d = reinterpret_cast<u32 *>(sg + GEMM8_REGION * wave + PITCH * f_row);
        const bool live = 2 * f_p < nblk - it * KB;
        const u32 d0 = d[17 * f_p], d8 = d[17 * f_p + 8];
        d[17 * f_p] = __builtin_amdgcn_alignbyte(d8, d0, 2);
        d[slot(f_p, f_s)] = live ? __builtin_bit_cast(u32, h2f(d0 & 0xffff)) : 0u;
        d[slot(f_p, 1 ^ f_s)] = live ? __builtin_bit_cast(u32, h2f(d8 >> 16)) : 0u;
    };

    ckq_v4f acc[2][4];                                      /* [token group][row group] */
#pragma unroll
    for (int tg = 0; tg < 2; ++tg)
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[tg][g] = ckq_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    ckq_v4i magic = {MAGIC, MAGIC, MAGIC, MAGIC};
    asm volatile("" : "+v"(magic));                         /* kept in registers: as a constant it is copied before every use */

    /* this lane's operands of the wave's two blocks, and where their scales are */
    const int opd = 17 * kh + q, opd_hi = opd + 9 + (kh ? 6 : 4);       /* block 3 ends in the last chunk */
    auto operand = [](const uint8_t *p, int lo, int hi) {
        const u32 *const d = reinterpret_cast<const u32 *>(p);
        return (long)((uint64_t)d[lo] | ((uint64_t)d[hi] << 32));
    };
    auto compute = [&](const uint8_t *sg, int it) {
        const uint8_t *const wl = sg + 4 * rh * GEMM8_REGION + i16 * PITCH;
        const uint8_t *const xl = sg + (4 * th + (i16 >> 3)) * GEMM8_REGION + (16 + (i16 & 7)) * PITCH;
        const uint8_t *const xs = sg + (4 * th + (q >> 1)) * GEMM8_REGION + (16 + 4 * (q & 1)) * PITCH;
#pragma unroll
        for (int jj = 0; jj < 2; ++jj) {
            const int lo = jj ? opd + 9 : opd, hi = jj ? opd_hi : opd + 4;
            long w[4], x[2];
            u32 dwb[4], dxb[2][4];                          
#pragma unroll
            for (int tg = 0; tg < 2; ++tg) x[tg] = operand(xl + 2 * GEMM8_REGION * tg, lo, hi);
#pragma unroll
            for (int g = 0; g < 4; ++g) w[g] = operand(wl + GEMM8_REGION * g, lo, hi);
#pragma unroll
            for (int g = 0; g < 4; ++g) dwb[g] = reinterpret_cast<const u32 *>(wl + GEMM8_REGION * g)[slot(kh, jj ^ (i16 >> 3))];
#pragma unroll
            for (int tg = 0; tg < 2; ++tg)
#pragma unroll
                for (int r = 0; r < 4; ++r) dxb[tg][r] = reinterpret_cast<const u32 *>(xs + 2 * GEMM8_REGION * tg + PITCH * r)[slot(kh, jj ^ (q >> 1))];
            float dwm[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) dwm[g] = __builtin_bit_cast(float, dwb[g]) * -12582912.0f;
#pragma unroll
            for (int tg = 0; tg < 2; ++tg) {
                ckq_v4i d[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) d[g] = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[tg], w[g], magic, 0, 0, 0);
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float t[4];
#pragma unroll
                    for (int r = 0; r < 4; ++r) {
                        const int di = d[g][r];
                        t[r] = __builtin_fmaf(__builtin_bit_cast(float, dwb[g]), __builtin_bit_cast(float, di), dwm[g]);
                        if constexpr (DUMP) {
                            int tr = t0 + 32 * th + 16 * tg + 4 * q + r;
                            asm volatile("" : "+v"(tr));   /* store addresses formed here, not kept in registers */
                            const int n = n0 + 64 * rh + 4 * i16 + g, b = it * KB + 2 * kh + jj;
                            if (tr < a.M && n < work.N && b < nblk) a.dump[((size_t)tr * work.N + n) * nblk + (size_t)b] = di - MAGIC;
                        }
                    }
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[tg][g][r] = __builtin_fmaf(__builtin_bit_cast(float, dxb[tg][r]), t[r], acc[tg][g][r]);
                }
            }
            /* block by block: scheduled together, the two would need more registers than four waves per SIMD have */
            asm volatile("" : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[0][2]), "+v"(acc[0][3]),
                              "+v"(acc[1][0]), "+v"(acc[1][1]), "+v"(acc[1][2]), "+v"(acc[1][3]) :: "memory");
        }
    };

    const int nfull = min(niter, nblk / KB);
    if (it0 < nfull) {
        auto landed = [] {                                  /* vmcnt(0) lgkmcnt(0) */
            __builtin_amdgcn_s_waitcnt(0x0070);
            asm volatile("" ::: "memory");
        };
        auto meet = [] {                                    /* lgkmcnt(0) */
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        copy(it0, stage[0]);
        landed();
        finish(it0, stage[0]);
        meet();
        auto step = [&](int it, uint8_t *cur, uint8_t *next) {
            copy(min(it + 1, nfull - 1), next);
            __builtin_amdgcn_sched_barrier(0);
            compute(cur, it);
            __builtin_amdgcn_sched_barrier(0);
            landed();
            finish(min(it + 1, nfull - 1), next);
            meet();
        };
        if constexpr (DUMP) {                               /* one copy of the stores */
            for (int it = it0; it < nfull; ++it) step(it, stage[(it - it0) & 1], stage[(it - it0 + 1) & 1]);
        } else for (int it = it0; it < nfull; it += 2) {
            step(it, stage[0], stage[1]);
            if (it + 1 < nfull) step(it + 1, stage[1], stage[0]);
        }
    }
    if (nfull < niter) {
        copy_tail(nfull, stage[0]);
        finish(nfull, stage[0]);
        __syncthreads();
        compute(stage[0], nfull);
        __syncthreads();
    }

    /* the two halves of K: waves kh keep token group kh and hand the other one over */
    ckq_v4f *const give = reinterpret_cast<ckq_v4f *>(kh ? stage[1] : stage[0]) + (wave & 3) * 256 + lane;
    const ckq_v4f *const take = reinterpret_cast<const ckq_v4f *>(kh ? stage[0] : stage[1]) + (wave & 3) * 256 + lane;
#pragma unroll
    for (int g = 0; g < 4; ++g) give[64 * g] = kh ? acc[0][g] : acc[1][g];
    __syncthreads();
    ckq_v4f o4[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) o4[g] = (kh ? acc[1][g] : acc[0][g]) + take[64 * g];

    /* lane: rows n .. n + 3, tokens t .. t + 3 */
    const GemmOut o = work.out;
    const bool vec_ok = (o.ldc % 4 == 0) && (((uintptr_t)o.C) % 16 == 0) && (n0 + BN <= work.N);
    const int n = n0 + 64 * rh + 4 * i16, t = t0 + 32 * th + 16 * kh + 4 * q;
    float bv[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) bv[g] = o.bias && n + g < work.N ? o.bias[n + g] : 0.0f;
    bool fix = false;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
        if (t + r >= a.M) continue;
        float *dst = o.C + (size_t)(t + r) * o.ldc + n;
        float v[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            fix = fix || o4[g][r] != o4[g][r];
            v[g] = o4[g][r] + bv[g];
        }
        if (vec_ok) *reinterpret_cast<float4 *>(dst) = make_float4(v[0], v[1], v[2], v[3]);
        else {
#pragma unroll
            for (int g = 0; g < 4; ++g) if (n + g < work.N) dst[g] = v[g];
        }
    }
    if (fix) {
        for (int e = 0; e < 16; ++e) {
            const int tr = t + (e >> 2), nr = n + (e & 3);
            if (tr >= a.M || nr >= work.N) continue;
            float *dst = o.C + (size_t)tr * o.ldc + nr;
            if (*dst == *dst) continue;
            *dst = q80_output(work.B + (size_t)nr * stride, a.A + (size_t)tr * stride, it0 * KB, min(nblk, niter * KB)) +
                   (o.bias ? o.bias[nr] : 0.0f);
        }
    }
}

/* g: operands, sizes, ntt and nnt set by the caller (ckq_gemm_q80.hip). */
int gemm_q80_dw_launch(GemmArgs &g, hipStream_t s)
{
    const unsigned grid = (unsigned)(g.ntt * ((g.nnt + 7) / 8 * 8));
    const int steps = (g.nb + GEMM8_KB - 1) / GEMM8_KB;
#if CKQ_WITH_DUMP
    if (g.dump) return gemm_launch_split(gemm_q80_dw_kernel<true>, g, grid, steps, s, GEMM8_THREADS);
#endif
    return gemm_launch_split(gemm_q80_dw_kernel<false>, g, grid, steps, s, GEMM8_THREADS);
}
int gemm_q80_dw_launch_group(GemmArgs &g, const GemmGroupIn &in, hipStream_t s)
{
    return gemm_launch_grouped(gemm_q80_dw_kernel<false>, g, in, s, GEMM8_THREADS);
}
