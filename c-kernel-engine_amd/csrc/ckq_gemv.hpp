/*
 * ckq_gemv.hpp - the weight-streaming dequant-dot kernel (decode GEMV and token
 * tiles of up to eight activation rows) and its launch-shape selection, as
 * templates over the per-format traits of ckq_formats.hpp.  Each format is
 * instantiated in a translation unit of its own (ckq_gemv_<fmt>.hip).
 */
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "ckq_blocks.h"
#include "ckq_formats.hpp"
#include "ckq_producers.hpp"
#include "ckq_launch.h"

constexpr int CKQ_GROUP_MAX = 4;   /* independent matmuls of one shape in one launch */

struct GemvArgs {
    float         *y;
    const uint8_t *W;
    const uint8_t *X;
    const float   *bias;
    int32_t       *sub;
    int  nrows, npos, ntok, row0, row1, nsub_row;
    long wrow, xrow, ldy;
};

/* Problems 1..3 of a grouped launch (blockIdx.z = g > 0); problem 0 is in GemvArgs. */
struct GemvGroup {
    float         *y[CKQ_GROUP_MAX - 1];
    const uint8_t *W[CKQ_GROUP_MAX - 1];
    const uint8_t *X[CKQ_GROUP_MAX - 1];
    const float   *bias[CKQ_GROUP_MAX - 1];
    int nrows[CKQ_GROUP_MAX - 1];           /* rows of each further problem (the grid covers the largest) */
    int ldy[CKQ_GROUP_MAX - 1];             /* and its output row stride */
    int n;                                  /* problems in the launch, 1 = not grouped */
};


/* The producer step of a launch that has one (gemv_pro_kernel): RMSNorm (gamma non-null) or the quantizer, rows of x stride
 * floats apart -> Q8_K blocks, in LDS for the launch's own matmuls and at out. */
struct GemvPro { const float *x, *gamma; uint8_t *out; long stride; float eps; };
__host__ __device__ __forceinline__ constexpr size_t pro_image_bytes(size_t tile_bytes) { return (tile_bytes + 15) & ~(size_t)15; }

/*
 * Tiled kernel (token tiles MT >= 1; DUMP: the same instantiation also stores
 * the raw integer sub-block dots of every (token, row), for the exactness tests).  One wave
 * handles (64/LPR)*RPI weight rows: LPR lanes share a row, lane l of the group
 * owns positions l, l+LPR, ... (PPL of them per pass).  All weight and
 * activation loads of a pass are issued before anything is decoded.  There is
 * no loop over rows: the grid supplies the parallelism.  The fp32 partials are
 * summed over the LPR lanes with a fixed DPP tree; the last lane of the group
 * stores.
 */
template <class F, int LPR, int PPL, int MT, int RPI, bool DUMP, int WPB, bool LDSX, bool GRP, bool PRO>
__device__ __forceinline__ void gemv_body(const uint8_t *W, const uint8_t *X, long wrow, long xrow, int row0, int row1, int npos, int ntok,
                                          float *y, const float *bias, long ldy, int32_t *sub, int nsub_row, int nrows, const GemvGroup &grp,
                                          const GemvPro &pro)
{
    /* The arguments are scalars, those the first loads need in front: the
     * first fourteen registers' worth arrive preloaded with the wave (build
     * flag -amdgpu-kernarg-preload-count) instead of through a scalar load
     * that every wave waits for before it can issue its first weight load. */
    const int g = GRP ? (int)blockIdx.z : 0;
    const int row1g = GRP && g ? grp.nrows[g - 1] : row1;    /* problems of a group may differ in their row count */
    const long ldyg = GRP && g ? (long)grp.ldy[g - 1] : ldy;
    const GemvArgs a = {y, W, X, bias, sub, nrows, npos, ntok, row0, row1g, nsub_row, wrow, xrow, ldyg};
    constexpr int SLOTS = 64 / LPR;
    extern __shared__ __attribute__((aligned(16))) uint8_t xs[];   /* LDSX: the MT activation rows */
    /* grouped launch: blockIdx.z picks the problem (a separate instantiation: the extra
     * argument loads lengthen the start of every wave, which a bandwidth-bound launch
     * of a few microseconds feels) */
    float *const         gy    = g == 0 ? a.y    : grp.y[g - 1];
    const uint8_t *const gW    = g == 0 ? a.W    : grp.W[g - 1];
    const uint8_t *const gX    = g == 0 ? a.X    : grp.X[g - 1];
    const float *const   gbias = g == 0 ? a.bias : grp.bias[g - 1];
    const int lane = threadIdx.x & 63, wave = wave_in_block();
    const int slot = lane / LPR, l = lane % LPR;
    const int wave_row = a.row0 + (blockIdx.x * WPB + wave) * (SLOTS * RPI);   /* uniform */
    const bool live = wave_row < a.row1;
    if (!LDSX && !live) return;
    if (GRP && a.row0 + (int)blockIdx.x * (WPB * SLOTS * RPI) >= a.row1) return;      /* all of the block: a narrower problem of the group */
    const int wrow_c = min(wave_row, a.row1 - 1);
    const int rbase = wave_row + slot * RPI;
    const int t0 = blockIdx.y * MT;
    /* dump layout: [problem of the group][token][row of nrows][sub-block] */
    const size_t dump_base = DUMP && GRP ? (size_t)g * a.ntok * a.nrows * a.nsub_row : 0;
    const uint8_t *wbase = gW + (size_t)wrow_c * a.wrow;                      /* uniform */

    /* Every wave of the block reads the same activation rows: they are staged
     * once in LDS instead of once per wave through the vector cache.  Their
     * loads go out first, all at once (one round trip, they hit in L2), the
     * weight loads follow, and only then are the staged values written. */
    constexpr int XNT = 64 * WPB, XU = MT == 1 ? 2 : 4;
    const int mt_live = min(MT, a.ntok - t0);
    const uint8_t *xsrc = gX + (size_t)t0 * (size_t)a.xrow;
    const int xbytes = (int)((long)mt_live * a.xrow), xn = xbytes / F::XS_SRC;   /* staging units */
    const u32 xcap = (u32)((long)MT * a.xrow / F::XS_SRC);                                     /* units of a full tile */
    u32 xv[XU][F::XS_REGS];
    /* PRO: wave w turns 256-blocks w, w + WPB, ... of the tile's rows into Q8_K, block column by block column */
    constexpr int XC = PRO ? (LPR / 4 + WPB - 1) / WPB : 1;
    float4 px[XC][MT], pg[XC];
    const int pnb = a.npos / 4;
    if constexpr (PRO) {
#pragma unroll
        for (int c = 0; c < XC; ++c)
#pragma unroll
            for (int t = 0; t < MT; ++t)
                px[c][t] = reinterpret_cast<const float4 *>(pro.x + (size_t)(t0 + min(t, mt_live - 1)) * (size_t)pro.stride + 256 * min(wave + WPB * c, pnb - 1))[lane];
        if (pro.gamma) {
#pragma unroll
            for (int c = 0; c < XC; ++c) pg[c] = reinterpret_cast<const float4 *>(pro.gamma + 256 * min(wave + WPB * c, pnb - 1))[lane];
        }
    }
    if (LDSX && !PRO) {
#pragma unroll
        for (int u = 0; u < XU; ++u) {
            const int i = u * XNT + (int)threadIdx.x;                 /* units past the tile re-read its last one */
            F::xs_ld(xv[u], xsrc + (u32)F::XS_SRC * (u32)min(i, xn - 1));
        }
    }

    float acc[RPI][MT];
#pragma unroll
    for (int r = 0; r < RPI; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) acc[r][t] = 0.0f;

    u32 rowoff[RPI];   /* byte offset of the lane's r-th row from wbase, clamped to the last row */
#pragma unroll
    for (int r = 0; r < RPI; ++r) rowoff[r] = (u32)(min(rbase + r, a.row1 - 1) - wrow_c) * (u32)a.wrow;

    for (int p0 = 0; p0 < a.npos; p0 += LPR * PPL) {
        typename F::Wt  w[RPI][PPL];
        typename F::Act act[MT >= 4 ? 1 : MT][PPL];   /* wide tiles stream their activations instead */
#pragma unroll
        for (int p = 0; p < PPL; ++p) {
            const int pos = min(p0 + p * LPR + l, a.npos - 1);
            const typename F::Off o = F::w_off(pos);
#pragma unroll
            for (int r = 0; r < RPI; ++r) {
                typename F::Off orow = o;
                F::off_shift(orow, rowoff[r]);
                F::load_w(w[r][p], wbase, orow);
            }
        }
        if constexpr (PRO) {
            float *const rows = reinterpret_cast<float *>(xs + pro_image_bytes((size_t)MT * (size_t)a.xrow));
            const int D = 64 * a.npos, rfl = (int)(rms_lds_bytes((size_t)D) / 4);
#pragma unroll
            for (int c = 0; c < XC; ++c)
#pragma unroll
                for (int t = 0; t < MT; ++t)
                    if (t < mt_live && wave + WPB * c < pnb) rms_stage(rows + t * rfl, D, wave + WPB * c, lane, px[c][t]);
            if (pro.gamma) {
                __syncthreads();
                const int ct = wave + WPB * (lane >> 3);              /* eight lanes walk a token's eight chains */
                if (ct < mt_live) rms_chain(rows + ct * rfl, D, lane & 7);
                __syncthreads();
            }
            /* the rows come back from LDS: held in registers beside the weights they would not fit */
#pragma unroll 1
            for (int t = 0; t < mt_live; ++t) {
                const float rstd = pro.gamma ? rms_rstd(rows + t * rfl, D, pro.eps) : 0.0f;
#pragma unroll
                for (int c = 0; c < XC; ++c) {
                    const int b = wave + WPB * c;
                    if (b >= pnb) continue;
                    const float4 v = rms_unstage(rows + t * rfl, D, b, lane);
                    uint8_t *const out = xs + (u32)t * (u32)a.xrow + 292u * (u32)b;
                    if (pro.gamma) rms_quant_block(v, pg[c], rstd, lane, out);
                    else {
                        const float e[4] = {v.x, v.y, v.z, v.w};
                        q8k_quantize_block(e, lane, out);
                    }
                }
            }
            __syncthreads();
            if (blockIdx.x == 0 && (!GRP || g == 0)) {                /* the step's own result */
                u32 *const out = reinterpret_cast<u32 *>(pro.out + (size_t)t0 * (size_t)a.xrow);
                for (int i = threadIdx.x; i < xbytes / 4; i += XNT) out[i] = reinterpret_cast<const u32 *>(xs)[i];
            }
        } else if (LDSX && p0 == 0) {
            /* the staged activations' loads are older than the weight loads
             * just issued, so waiting for them does not wait for the weights */
#pragma unroll
            for (int u = 0; u < XU; ++u) {
                const int i = u * XNT + (int)threadIdx.x;
                if (i < xn) F::xs_st(xs, xv[u], (u32)i, xcap);
            }
            for (int i = XNT * XU + (int)threadIdx.x; i < xn; i += XNT) {       /* long token tiles */
                u32 v[F::XS_REGS];
                F::xs_ld(v, xsrc + (u32)F::XS_SRC * (u32)i);
                F::xs_st(xs, v, (u32)i, xcap);
            }
            if (F::XS_SRC == 16) {
                const int tail = (xbytes & 15) >> 1;  /* plain-copy images: rows are a whole number of 2-byte units */
                if ((int)threadIdx.x < tail) {
                    const u32 o = 16u * (u32)xn + 2u * threadIdx.x;
                    *reinterpret_cast<uint16_t *>(xs + o) = (uint16_t)ld2(xsrc + o);
                }
            }
            __syncthreads();
        }
        if constexpr (MT >= 4) {
            /* wide token tiles: the weights of a position are decoded once, then
             * the tokens' activations stream through from LDS one at a time
             * (holding all of them in registers would leave two waves per SIMD) */
#pragma unroll
            for (int p = 0; p < PPL; ++p) {
                const int  upos  = p0 + p * LPR + l;
                const bool valid = upos < a.npos;
                const int  pos   = min(upos, a.npos - 1);
                typename F::Dec dec[RPI];
#pragma unroll
                for (int r = 0; r < RPI; ++r) F::decode(dec[r], w[r][p], pos);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    typename F::Act at;
                    if (LDSX) {
                        const int tl = min(t, a.ntok - t0 - 1);                    /* uniform */
                        F::load_act_lds(at, xs, tl, pos, (u32)a.xrow, a.npos, xcap);
                    } else {
                        const int tok = min(t0 + t, a.ntok - 1);                   /* uniform */
                        F::load_act(at, gX + (size_t)tok * a.xrow, pos);
                    }
#pragma unroll
                    for (int r = 0; r < RPI; ++r) {
                        int sub[F::NSUB];
                        const float v = F::dot(dec[r], at, sub);
                        acc[r][t] += valid ? v : 0.0f;
                        if (DUMP && valid && rbase + r < a.row1 && t0 + t < a.ntok) {
#pragma unroll
                            for (int i = 0; i < F::NSUB; ++i)
                                a.sub[dump_base + ((size_t)(t0 + t) * a.nrows + (rbase + r)) * a.nsub_row + F::sub_index(pos, i)] = sub[i];
                        }
                    }
                }
            }
        } else {
#pragma unroll
        for (int p = 0; p < PPL; ++p) {
            const int pos = min(p0 + p * LPR + l, a.npos - 1);
#pragma unroll
            for (int t = 0; t < MT; ++t) {
                if (LDSX) {
                    const int tl = min(t, a.ntok - t0 - 1);                    /* uniform */
                    F::load_act_lds(act[t][p], xs, tl, pos, (u32)a.xrow, a.npos, xcap);
                } else {
                    const int tok = min(t0 + t, a.ntok - 1);                   /* uniform */
                    F::load_act(act[t][p], gX + (size_t)tok * a.xrow, pos);
                }
            }
        }
#pragma unroll
        for (int p = 0; p < PPL; ++p) {
            const int  upos  = p0 + p * LPR + l;
            const bool valid = upos < a.npos;
            const int  pos   = min(upos, a.npos - 1);
#pragma unroll
            for (int r = 0; r < RPI; ++r) {
                typename F::Dec dec;
                F::decode(dec, w[r][p], pos);
#pragma unroll
                for (int t = 0; t < MT; ++t) {
                    int sub[F::NSUB];
                    const float v = F::dot(dec, act[t][p], sub);
                    acc[r][t] += valid ? v : 0.0f;
                    if (DUMP && valid && rbase + r < a.row1 && t0 + t < a.ntok) {
#pragma unroll
                        for (int i = 0; i < F::NSUB; ++i)
                            a.sub[dump_base + ((size_t)(t0 + t) * a.nrows + (rbase + r)) * a.nsub_row + F::sub_index(pos, i)] = sub[i];
                    }
                }
            }
        }
        }
    }

#pragma unroll
    for (int r = 0; r < RPI; ++r)
#pragma unroll
        for (int t = 0; t < MT; ++t) {
            const float s = group_sum<LPR>(acc[r][t]);
            const int row = rbase + r, tok = t0 + t;
            if (!DUMP && l == LPR - 1 && row < a.row1 && tok < a.ntok)
                gy[(size_t)tok * a.ldy + row] = gbias ? s + gbias[row] : s;
        }
}

template <class F, int LPR, int PPL, int MT, int RPI, bool DUMP, int WPB, bool LDSX, bool GRP = false>
__global__ void __launch_bounds__(64 * WPB) __attribute__((amdgpu_waves_per_eu(DUMP ? 1 : MT == 1 && PPL == 1 && RPI == 1 ? F::OCC1 : MT == 1 && PPL == 1 && RPI == 2 && LPR == 64 ? F::OCC2 : MT >= 4 && PPL == 1 ? 4 : 1)))
gemv_kernel(const uint8_t *W, const uint8_t *X, long wrow, long xrow, int row0, int row1, int npos, int ntok,
            float *y, const float *bias, long ldy, int32_t *sub, int nsub_row, int nrows, GemvGroup grp)
{
    gemv_body<F, LPR, PPL, MT, RPI, DUMP, WPB, LDSX, GRP, false>(W, X, wrow, xrow, row0, row1, npos, ntok, y, bias, ldy, sub, nsub_row, nrows, grp, GemvPro{});
}

/* A producer step and the matmuls that read its result in one launch. */
template <class F, int LPR, int MT, int RPI>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(MT >= 4 || RPI == 2 ? 3 : 4)))
gemv_pro_kernel(const uint8_t *W, long wrow, long xrow, int row1, int npos, int ntok, GemvPro pro,
                float *y, const float *bias, long ldy, int nrows, GemvGroup grp)
{
    gemv_body<F, LPR, 1, MT, RPI, false, 4, true, true, true>(W, nullptr, wrow, xrow, 0, row1, npos, ntok, y, bias, ldy, nullptr, 0, nrows, grp, pro);
}

/* Rows the grid has to cover: the computed range, or the largest problem of a group. */
static int launch_rows(const GemvArgs &a, const GemvGroup &grp) { return grp.n > 1 ? a.nrows : a.row1 - a.row0; }

/* Token tiles a launch can carry in gridDim.y; longer token lists go out as
 * several launches over consecutive token ranges (ckq_grid_chunk). */
constexpr int CKQ_GRID_Y_MAX = 65535;

template <class F, int LPR, int PPL, int MT, int RPI, bool DUMP, int WPB, bool LDSX>
static int launch_one(const GemvArgs &a0, const GemvGroup &grp, hipStream_t s)
{
    constexpr int rows_per_block = WPB * (64 / LPR) * RPI;
    const int nr = launch_rows(a0, grp);
    const size_t lds = LDSX ? F::xs_lds_bytes((size_t)MT * (size_t)a0.xrow) : 0;
    if (grp.n > 1) {
        if constexpr (LDSX) {                            /* grouped launches stage their activations in LDS */
            dim3 grid((nr + rows_per_block - 1) / rows_per_block, (a0.ntok + MT - 1) / MT, (unsigned)grp.n);
            hipLaunchKernelGGL((gemv_kernel<F, LPR, PPL, MT, RPI, DUMP, WPB, LDSX, true>), grid, dim3(64 * WPB), lds, s,
                               a0.W, a0.X, a0.wrow, a0.xrow, a0.row0, a0.row1, a0.npos, a0.ntok, a0.y, a0.bias, a0.ldy, a0.sub,
                               a0.nsub_row, a0.nrows, grp);
            return (int)hipGetLastError();
        }
        return CKQ_EINVAL;
    }
    const long per = (long)MT * CKQ_GRID_Y_MAX;
    if (a0.sub && a0.ntok > per) return CKQ_EINVAL;      /* the dump is indexed by the token of the whole call */
    for (long c = 0; c * per < a0.ntok; ++c) {
        long first, count;
        ckq_grid_chunk(a0.ntok, per, c, &first, &count);
        GemvArgs a = a0;
        a.X = a0.X + (size_t)first * (size_t)a0.xrow;
        a.y = a0.y ? a0.y + (size_t)first * (size_t)a0.ldy : nullptr;
        a.ntok = (int)count;
        dim3 grid((nr + rows_per_block - 1) / rows_per_block, (a.ntok + MT - 1) / MT, 1);
        hipLaunchKernelGGL((gemv_kernel<F, LPR, PPL, MT, RPI, DUMP, WPB, LDSX, false>), grid, dim3(64 * WPB), lds, s,
                           a.W, a.X, a.wrow, a.xrow, a.row0, a.row1, a.npos, a.ntok, a.y, a.bias, a.ldy, a.sub,
                           a.nsub_row, a.nrows, grp);
        const int rc = (int)hipGetLastError();
        if (rc) return rc;
    }
    return 0;
}

/* Activation rows are staged in LDS when the token tile fits in 64 KB.  The
 * dump build of an instantiation exists for the staged form only. */
template <class F, int LPR, int PPL, int MT, int RPI, int WPB>
static int launch_tile(const GemvArgs &a, const GemvGroup &grp, hipStream_t s)
{
    const bool fits = F::xs_lds_bytes((size_t)MT * (size_t)a.xrow) <= 65536;
    if (a.sub) {
#if CKQ_WITH_DUMP
        if constexpr (F::TOKEN_TILES) {
            if (fits) return launch_one<F, LPR, PPL, MT, RPI, true, WPB, true>(a, grp, s);
            if (MT == 1 && grp.n == 1) return launch_one<F, LPR, PPL, 1, 1, true, 4, false>(a, grp, s);
        }
        return CKQ_EINVAL;
#else
        return CKQ_ENODUMP;      /* the dump builds live in libckernel_quant_hip_dump.so */
#endif
    }
    if (fits) return launch_one<F, LPR, PPL, MT, RPI, false, WPB, true>(a, grp, s);
    return launch_one<F, LPR, PPL, MT, RPI, false, WPB, false>(a, grp, s);
}

/* Two rows per slot serve the staged tokens twice, but leave CUs without a block where the matrix is small: then one row
 * per slot, and smaller token tiles while that too leaves some.  Measured (us; 2, 4 and 7 tokens): Q5_K 1024 x 4864
 * 3.9 -> 3.2, 5.2 -> 3.9, 7.5 -> 5.2; 4096 x 1024 at 4 and 7 3.5 -> 2.8, 4.5 -> 3.3; Q6_K 1024 x 11008 at 2 and 4 6.5 -> 5.2,
 * 9.0 -> 7.3; Q4_K 2048 x 2048 at 7 4.5 -> 3.2; 12000 x 1024 at 4 4.4 -> 4.1, Q8_0 at 7 6.7 -> 5.8.  Rows that take a wave
 * each lose from 256 blocks of two rows per slot on (2048 x 8192, Q6_K at 4: 7.4 -> 8.2), shorter ones from 512. */
static void gemv_token_tile(int lpr, int rows, int n, int ntok, int *mt, int *rpi)
{
    const long few = lpr < 64 ? 512 : 256;
    const long slots = ((long)rows * lpr + 255) / 256 * (long)n;      /* blocks of one row per slot and a token tile */
    *mt = ntok == 2 ? 2 : ntok <= 4 ? 4 : 8;
    *rpi = 2;                        /* the staged tile serves twice the weights */
    if (slots >= 2 * few) return;
    *rpi = 1;
    while (*mt > 2 && slots * ((ntok + *mt - 1) / *mt) <= 256) *mt /= 2;
}

/* Rows per wave-slot and waves per block for each token tile: one row per
 * slot in 256-thread blocks for the bandwidth-bound single-token case (as many
 * of the matrix's loads in flight as the CUs can hold, small barrier groups),
 * fewer rows in flight as the tile grows. */
template <class F, int LPR, int PPL>
static int launch_mt(const GemvArgs &a, const GemvGroup &grp, int max_mt, hipStream_t s)
{
    if (a.ntok == 1 || max_mt == 1) {
        /* 256-thread blocks; a second row per slot once the matrix needs more
         * than two rounds of resident waves anyway (halves the activation
         * staging per weight byte) */
        const long waves = ((long)launch_rows(a, grp) * LPR + 63) / 64;
        if (PPL == 1 && waves > 16384) return launch_tile<F, LPR, PPL, 1, 2, 4>(a, grp, s);
        /* rows longer than one pass: each staged activation row is shared
         * between eight weight rows, as 512-thread blocks (a whole number of
         * blocks per CU on the usual projection shapes) or, for the largest
         * matrices, two rows per slot */
        if (PPL > 1 && launch_rows(a, grp) >= 8192) return launch_tile<F, LPR, PPL, 1, 2, 4>(a, grp, s);
        if (PPL > 1 && launch_rows(a, grp) >= 2048) return launch_tile<F, LPR, PPL, 1, 1, 8>(a, grp, s);
        return launch_tile<F, LPR, PPL, 1, 1, 4>(a, grp, s);
    }
    if constexpr (F::TOKEN_TILES) {
        int mt, rpi;
        gemv_token_tile(LPR, launch_rows(a, grp), grp.n, a.ntok, &mt, &rpi);
        /* a tile that LDS does not hold is read from memory again by every wave, position by position: a smaller one that it does hold is up to
         * three times as fast although the weights are read more often (us: Q8_0 11 x 16532 x 7296 174 -> 69, 8 x 4096 x 7296 25.2 -> 14.3, 5 x 1500 x 11008
         * 30.9 -> 11.4, Q5_0 8 x 11000 x 8192 62.1 -> 33.8, Q5_K 8 x 1500 x 8192 10.9 -> 8.0; Q5_0 12 x 1500 x 11008 23.8 -> 24.4); the bits of a token are the same */
        while (mt > 2 && F::xs_lds_bytes((size_t)mt * (size_t)a.xrow) > 65536) mt /= 2;
        if (rpi == 1) {
            if (mt == 2) return launch_tile<F, LPR, PPL, 2, 1, 4>(a, grp, s);
            if (mt == 4) return launch_tile<F, LPR, PPL, 4, 1, 4>(a, grp, s);
            return launch_tile<F, LPR, PPL, 8, 1, 4>(a, grp, s);
        }
        if (mt == 2) return launch_tile<F, LPR, PPL, 2, 2, 4>(a, grp, s);
        if (mt == 4) return launch_tile<F, LPR, PPL, 4, 2, 4>(a, grp, s);
        return launch_tile<F, LPR, PPL, 8, 2, 4>(a, grp, s);
    }
    return CKQ_EINVAL;   /* formats without token tiles are always launched with max_mt == 1 */
}

/* Entry of a format's translation unit: picks the lane mapping from the row
 * length.  a.sub non-NULL selects the dump build of the same instantiation. */
template <class F>
static int launch_fmt(const GemvArgs &a, const GemvGroup &grp, int max_mt, hipStream_t s)
{
    const int np = a.npos;
    if (np <= 8)  return launch_mt<F, 8, 1>(a, grp, max_mt, s);
    if (np <= 16) return launch_mt<F, 16, 1>(a, grp, max_mt, s);
    if (np <= 32) return launch_mt<F, 32, 1>(a, grp, max_mt, s);
    if (np <= 64) return launch_mt<F, 64, 1>(a, grp, max_mt, s);
    if (np <= 128) return launch_mt<F, 64, 2>(a, grp, max_mt, s);
    if (np <= 192) return launch_mt<F, 64, 3>(a, grp, max_mt, s);
    return launch_mt<F, 64, 4>(a, grp, max_mt, s);   /* longer rows loop in passes of 256 positions */
}

/*
 * Producer step and matmuls in one launch: rows of up to 32 positions (K of up to 2048).  Where a step is a few microseconds, half
 * of which are a launch's beginning and end, every block makes the quantized rows for itself, in LDS, while its weights are on their way;
 * the first block of a token tile stores them as the step's own result.  The arithmetic is that of the producer kernels, so every
 * buffer keeps its bits.  It pays while the fullest CU makes no more than PRO_UNITS 256-blocks that way (blocks on it x tokens of a tile x
 * 256-blocks of a row).  Measured, us per layer of a decode chain (RMSNorm, Q/K/V, quantizer, O, RMSNorm, gate and up, SwiGLU, down; K and V narrow),
 * separate -> joined: one token, 768 wide 20.0 -> 14.8, 1024 wide 20.4 -> 16.6, 2048 wide 24.4 -> 23.6; four tokens, 1024 wide 25.0 -> 23.4
 * without gate and up (48 units), 25.9 with them; 2048 wide 31.4, with RMSNorm and Q/K/V joined (64 units) 35.7.
 */
constexpr int PRO_UNITS = 16;
template <class F, int LPR, int MT, int RPI>
static int launch_pro_one(const GemvArgs &a, const GemvGroup &grp, const GemvPro &pro, hipStream_t s)
{
    constexpr int rows_per_block = 4 * (64 / LPR) * RPI;
    const size_t lds = pro_image_bytes((size_t)MT * (size_t)a.xrow) + MT * rms_lds_bytes((size_t)a.npos * 64);
    if (lds > 65536) return CKQ_ENOGROUP;
    long blocks = (a.row1 + rows_per_block - 1) / rows_per_block;
    for (int i = 0; i + 1 < grp.n; ++i) blocks += (grp.nrows[i] + rows_per_block - 1) / rows_per_block;
    blocks *= (a.ntok + MT - 1) / MT;
    if ((blocks + 255) / 256 * MT * (a.npos / 4) > PRO_UNITS) return CKQ_ENOGROUP;
    const dim3 grid((a.nrows + rows_per_block - 1) / rows_per_block, (a.ntok + MT - 1) / MT, (unsigned)grp.n);
    hipLaunchKernelGGL((gemv_pro_kernel<F, LPR, MT, RPI>), grid, dim3(256), lds, s, a.W, a.wrow, a.xrow, a.row1, a.npos, a.ntok, pro, a.y, a.bias, a.ldy, a.nrows, grp);
    return (int)hipGetLastError();
}
template <class F, int LPR>
static int launch_pro_lpr(const GemvArgs &a, const GemvGroup &grp, const GemvPro &pro, hipStream_t s)
{
    int mt = 1, rpi = 1;
    if (a.ntok > 1) gemv_token_tile(LPR, a.nrows, grp.n, a.ntok, &mt, &rpi);
    if (mt == 1) return launch_pro_one<F, LPR, 1, 1>(a, grp, pro, s);
    if (mt == 2) return rpi == 2 ? launch_pro_one<F, LPR, 2, 2>(a, grp, pro, s) : launch_pro_one<F, LPR, 2, 1>(a, grp, pro, s);
    /* tiles of four at most: eight tokens' rows beside the weights would not fit the registers.  Rows of 32 lanes, five 256-blocks and more, are past
     * PRO_UNITS in such a tile whatever the grid */
    if constexpr (LPR == 32) return CKQ_ENOGROUP;
    else return rpi == 2 ? launch_pro_one<F, LPR, 4, 2>(a, grp, pro, s) : launch_pro_one<F, LPR, 4, 1>(a, grp, pro, s);
}
static_assert(PRO_UNITS < 4 * 5, "rows of 32 lanes and a tile of four tokens: launch_pro_lpr");
template <class F>
static int launch_pro(const GemvArgs &a, const GemvGroup &grp, const GemvPro &pro, hipStream_t s)
{
    if (a.npos > 32) return CKQ_ENOGROUP;
    return a.npos <= 8 ? launch_pro_lpr<F, 8>(a, grp, pro, s) : a.npos <= 16 ? launch_pro_lpr<F, 16>(a, grp, pro, s) : launch_pro_lpr<F, 32>(a, grp, pro, s);
}

/* One function per trait, each defined in its own translation unit. */
int ckq_gemv_launch_q4k(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q5k(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q6k(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q80(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q80p(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q50(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q80_f32(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q4k_f32(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_launch_q6k_f32(const GemvArgs &a, const GemvGroup &grp, hipStream_t s);
int ckq_gemv_pro_launch_q4k(const GemvArgs &a, const GemvGroup &grp, const GemvPro &pro, hipStream_t s);
int ckq_gemv_pro_launch_q5k(const GemvArgs &a, const GemvGroup &grp, const GemvPro &pro, hipStream_t s);
int ckq_gemv_pro_launch_q6k(const GemvArgs &a, const GemvGroup &grp, const GemvPro &pro, hipStream_t s);
