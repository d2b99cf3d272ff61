/*
 * ckq_gemm_common.hpp - what the four matrix-core GEMM kernels share: operand
 * vector types, the launch arguments, the K-split bookkeeping and the entry
 * points of each kernel's translation unit.
 */
#pragma once
#include <mutex>
#include "ckq_device.hpp"
#include "ckq_launch.h"

typedef int   ckq_v4i  __attribute__((ext_vector_type(4)));
typedef int   ckq_v16i __attribute__((ext_vector_type(16)));
typedef float ckq_v16f __attribute__((ext_vector_type(16)));
typedef __bf16 ckq_v8bf __attribute__((ext_vector_type(8)));
typedef unsigned short ckq_v2u16 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) void ckq_lds_void;
typedef const __attribute__((address_space(1))) void ckq_glb_void;

/* One weight matrix of a grouped launch: several matrices that multiply the same activations (Q/K/V,
 * gate/up) share a grid.  id0 is where a matrix begins: among the tiles of all matrices, which are dealt as one (GemmArgs::units; gemm_launch_grouped); among the tiles of
 * weight rows (ckq_gemm_q4k_t96.hip); or its first block id, of gemm_blocks(ntt, nnt), where every matrix is dealt by itself (units = 0; gemm_deal_ragged_last). */
constexpr int GEMM_GROUP_MAX = 4;
struct GemmProblem {
    const uint8_t *B;
    const float   *bias;
    float         *C;
    long           ldc;
    int            N, nnt, id0;
    int            tt0, ntt;   /* its token tiles: all of the matrix, or the whole ones, or the ragged one (gemm_deal_ragged_last) */
};

struct GemmArgs {
    const uint8_t *A;     /* Q8_K activations, M rows of nb blocks */
    const uint8_t *B;     /* Q4_K weights, N rows of nb blocks */
    const float   *bias;  /* N or null */
    float         *C;     /* M x ldc */
    int  M, N, nb;
    long ldc;
    int  ntt, nnt;        /* token tiles, weight-row tiles */
    /* grouped launch: ngroup > 1 matrices, never split along K; B, bias, C, N, ldc, nnt above are those of grp[0] */
    int  ngroup;
    GemmProblem grp[GEMM_GROUP_MAX];
    /* what is dealt to the XCDs as one (gemm_work): the tiles of all matrices, times the splits; 0: every matrix by itself, from its id0 on */
    int    units;
    /* split K: piece s handles K-steps [s * k_per, min(k_steps, (s + 1) * k_per)) and
     * writes its partial tile, without bias, to part + s * M * N (row pitch N) */
    int    splits, k_per;
    float *part;
    float *ext_part;       /* caller-provided scratch for `part` (launch options), or null */
    size_t ext_part_bytes;
    /* dump builds only: the exact integer block sums behind every output,
     * dump[((t * N + n) * nblk + b) * per + i] (per = 2: I1, I2 for Q4_K and
     * Q5_K; per = 1 for Q6_K and, with nblk = K / 32, for Q8_0) */
    int32_t *dump;
};

/* Where a lane of a dump build stores the sums of output (token offset `tok`
 * from the lane's first token, its row): nothing for rows or tokens outside
 * the matrix. */
/* A uniform value the compiler must take as new each time: keeps the 64 store
 * addresses of a dump from being hoisted out of the K loop into registers. */
__device__ __forceinline__ size_t gemm_opaque(size_t v)
{
    asm volatile("" : "+s"(v));
    return v;
}

struct GemmDumpLane {
    int32_t *p;          /* &dump[((t_first * N + n) * nblk + b) * per] */
    size_t   tok_stride; /* N * nblk * per */
    int      tok_left;   /* tokens from t_first to the end of the matrix */
    bool     row_ok;
    __device__ __forceinline__ void put(int tok, int i, int v) const
    {
        if (row_ok && tok < tok_left) p[(size_t)tok * tok_stride + i] = v;
    }
};

/* Launch options of the four GEMMs: `sums` non-NULL runs the dump build
 * (GemmArgs::dump); `scratch` non-NULL is caller-provided device memory of
 * scratch_bytes for the partial tiles of a K-split launch, used instead of the
 * library's grow-only workspace (nothing is allocated then; a split that needs
 * more returns CKQ_ESCRATCH). */
struct GemmOpts {
    int32_t *sums;
    float   *scratch;
    size_t   scratch_bytes;
};

/* Of `total` things the one that block `id` takes, -1: none: eight equal runs, one for each XCD (blocks go round the XCDs in turn). */
__host__ __device__ __forceinline__ int gemm_deal(int id, int total)
{
    const int xcd = id & 7, seq = id >> 3;
    return seq < (total >> 3) + (xcd < (total & 7) ? 1 : 0) ? xcd * (total >> 3) + (xcd < (total & 7) ? xcd : total & 7) + seq : -1;
}

/* The tiles of a launch, ntt token tiles of nnt tiles of weight rows, token tiles fastest so that neighbours share weights, are dealt
 * to the XCDs in eight equal runs (blocks go round the XCDs in turn, and each has an L2 of its own): whole rows of
 * tiles per XCD leave some with a row more, and with few rows CUs there with two or three tiles beside others with one (us, rows of
 * tiles -> runs: Q6_K 680 tokens x 2111 rows x 4352 57.8 -> 32.6, Q5_K 67 x 1509 x 10240 32.6 -> 21.3, Q4_K 339 x 1432 x 6656 33.0 -> 20.8;
 * 60 random sizes 0.5 to 5 % on average, the same bits).  gemm_blocks: block ids to launch; false: no tile. */
__host__ __device__ __forceinline__ bool gemm_tile(int id, int ntt, int nnt, int &nt, int &tt)
{
    const int t = gemm_deal(id, ntt * nnt);
    nt = t / ntt;
    tt = t - nt * ntt;
    return t >= 0;
}
__host__ __device__ __forceinline__ constexpr int gemm_blocks(int ntt, int nnt) { return (ntt * nnt + 7) & ~7; }

/* What one block of a GEMM launch does: which tile (weight-row tile nt, token tile tt; -1: none), which K-steps, where it
 * writes and whether it adds the bias. */
struct GemmOut { float *C; long ldc; const float *bias; };
struct GemmWork { int tile, k0, k1; GemmOut out; const uint8_t *B; int N, nnt, tt0, ntt; };
/* A launch of pieces of K is as wide as the chip (gemm_choose_splits), and takes as long as its fullest XCD: 84 tiles in three pieces, 252 blocks, were 33 for
 * the 32 CUs of four XCDs, and so two rounds, as long as each piece's tiles were dealt by themselves (three matrices of 84 tiles were 33 where 32 do).  All pieces of all tiles
 * are dealt as one, piece by piece, so that an XCD has one or two pieces of K of many tiles, which share activations as well as weights.  us, tokens x
 * rows x K: Q6_K 384 x 1792 x 6400 43.3 -> 30.5, Q5_K 150 x 3584 x 9984 60.7 -> 36.2, Q4_K 379 x 768 x 7168 25.8 -> 21.5, Q8_0 321 x 1792 x 4864 32.3 -> 25.9; 49
 * sizes of that kind 1.29 on average (1.02 to 1.68), 60 others 1.00.  The sums and their order are the same. */
__device__ __forceinline__ GemmWork gemm_work(const GemmArgs &a, int k_steps)
{
    const int id = blockIdx.x;
    int u = a.units ? gemm_deal(id, a.units) : id;
    if (a.ngroup > 1) {
        /* uniform selects, no indexing: the argument block stays in scalar registers */
        GemmProblem g = a.grp[0];
        if (u >= a.grp[1].id0) g = a.grp[1];
        if (a.ngroup > 2 && u >= a.grp[2].id0) g = a.grp[2];
        if (a.ngroup > 3 && u >= a.grp[3].id0) g = a.grp[3];
        u = a.units ? (u < 0 ? -1 : u - g.id0) : gemm_deal(id - g.id0, g.ntt * g.nnt);
        return {u, 0, k_steps, {g.C, g.ldc, g.bias}, g.B, g.N, g.nnt, g.tt0, g.ntt};
    }
    if (a.splits <= 1) return {u, 0, k_steps, {a.C, a.ldc, a.bias}, a.B, a.N, a.nnt, 0, a.ntt};
    const int tiles = a.ntt * a.nnt, sp = u < 0 ? 0 : u / tiles, k0 = sp * a.k_per;
    return {u - sp * tiles, k0, min(k_steps, k0 + a.k_per),
            {a.part + (size_t)sp * (size_t)a.M * (size_t)a.N, (long)a.N, nullptr}, a.B, a.N, a.nnt, 0, a.ntt};
}
/* Its tile; false: it has none. */
__device__ __forceinline__ bool gemm_tile(const GemmWork &w, int &nt, int &tt)
{
    nt = w.tile / w.ntt;
    tt = w.tile - nt * w.ntt + w.tt0;
    return w.tile >= 0;
}

/* Split K when the tile grid leaves most of the chip idle: `tiles` blocks of
 * `k_steps` loop iterations each.  Returns the number of splits (1 = none) so
 * that tiles * splits approaches the CU count while every split keeps at
 * least four iterations. */
static int gemm_choose_splits(int tiles, int k_steps)
{
    if (tiles >= 160 || k_steps < 8) return 1;
    int s = 256 / tiles;
    if (s > k_steps / 4) s = k_steps / 4;
    if (s > 16) s = 16;
    return s < 2 ? 1 : s;
}

/* Global -> LDS, 16 bytes per lane from rs + ofs + k to dst + 16 lane.  Written out because the compiler, which cannot know which
 * bytes of an LDS object a copy in flight still has to write, waits for all of them before the next read of that object; the
 * one wait there has to be is the loop's. */
__device__ __forceinline__ void lds_copy16(const ckq_v4i &rs, u32 dst, u32 ofs, int k)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(dst), "v"(ofs), "s"(rs), "s"(k) : "memory");
}
/* The source of such copies: a uniform address. */
__device__ __forceinline__ ckq_v4i gemm_buffer(const uint8_t *p)
{
    return ckq_v4i{__builtin_amdgcn_readfirstlane((int)(u32)(uintptr_t)p), __builtin_amdgcn_readfirstlane((int)(u32)((uintptr_t)p >> 32)), 0x7fffffff, 0x00020000};
}
/* The same, four bytes per lane to dst + 4 lane. */
__device__ __forceinline__ void lds_copy4(const ckq_v4i &rs, u32 dst, u32 ofs, int k)
{
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds" ::"s"(dst), "v"(ofs), "s"(rs), "s"(k) : "memory");
}
__device__ __forceinline__ u32 lds_address(const void *p) { return (u32)(uintptr_t)(__attribute__((address_space(3))) const void *)p; }

constexpr int GEMM_TILE_ROWS = 128;    /* weight rows per tile, all four kernels */

/* Scratch for the partial tiles of K-split launches (kind 0) and for weights
 * rewritten for another kernel (kind 1): one grow-only device buffer per
 * stream and kind (work on one stream is ordered, so consecutive launches may
 * share it).  Growing it allocates and therefore synchronises.  The caller
 * holds gemm_split_mutex() from here until its last kernel is enqueued, so two
 * host threads launching on one stream cannot interleave their kernel pairs.
 * Defined in ckq_kernels.hip. */
std::recursive_mutex &gemm_split_mutex();
int gemm_workspace(int kind, hipStream_t s, size_t bytes, float **out);
/* C = bias + partial 0 + partial 1 + ... in that order (ckq_kernels.hip). */
int gemm_launch_reduce(float *C, long ldc, const float *part, const float *bias, int M, int N, int splits, hipStream_t s);

/* Common launch tail: sets up the split, launches `kernel` on all pieces of all tiles
 * and, when split, the ordered reduction. */
template <class Kernel>
static int gemm_launch_split(Kernel kernel, GemmArgs &g, int k_steps, hipStream_t s, unsigned threads = 256)
{
    g.splits = gemm_choose_splits(g.ntt * g.nnt, k_steps);
    g.k_per = (k_steps + g.splits - 1) / g.splits;
    g.splits = (k_steps + g.k_per - 1) / g.k_per;          /* no empty split */
    g.units = g.ntt * g.nnt * g.splits;
    g.part = nullptr;
    const dim3 grid((unsigned)gemm_blocks(g.units, 1));
    if (g.splits <= 1) {
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, s, g);
        return (int)hipGetLastError();
    }
    const size_t need = (size_t)g.splits * (size_t)g.M * (size_t)g.N * sizeof(float);
    if (g.ext_part) {
        /* caller-provided scratch: nothing is allocated and nothing is locked
         * (calls that share the scratch must not overlap).  Every partial
         * entry the reduction reads is written by the split kernel first, so
         * the scratch needs no clearing. */
        if (need > g.ext_part_bytes) return CKQ_ESCRATCH;
        g.part = g.ext_part;
        hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, s, g);
        const int rc = (int)hipGetLastError();
        if (rc) return rc;
        return gemm_launch_reduce(g.C, g.ldc, g.part, g.bias, g.M, g.N, g.splits, s);
    }
    std::lock_guard<std::recursive_mutex> lock(gemm_split_mutex());
    int rc = gemm_workspace(0, s, need, &g.part);
    if (rc) return rc;
    hipLaunchKernelGGL(kernel, grid, dim3(threads), 0, s, g);
    rc = (int)hipGetLastError();
    if (rc) return rc;
    return gemm_launch_reduce(g.C, g.ldc, g.part, g.bias, g.M, g.N, g.splits, s);
}


/* packed u16x2 multiply-add, lane-wise (v_pk_mad_u16) */
__device__ __forceinline__ u32 pk_mad_u16(u32 a, u32 b, u32 c)
{
    const ckq_v2u16 x = __builtin_bit_cast(ckq_v2u16, a), y = __builtin_bit_cast(ckq_v2u16, b),
                    z = __builtin_bit_cast(ckq_v2u16, c);
    return __builtin_bit_cast(u32, (ckq_v2u16)(x * y + z));
}

/* acc += u * (lane 16*(l/16) + R of x): the multiply-add takes its first factor
 * from lane R of the caller's 16-lane row (DPP row_newbcast), so sixteen values
 * held one per lane serve sixteen instructions without being spread out first.
 * x must come from memory (LDS), not from a VALU instruction right before. */
__device__ __forceinline__ float fmac_row_lane(float acc, float x, float u, int r)
{
#define CKQ_BC(R) case R: asm("v_fmac_f32_dpp %0, %1, %2 row_newbcast:" #R " row_mask:0xf bank_mask:0xf" : "+v"(acc) : "v"(x), "v"(u)); break;
    switch (r) {
        CKQ_BC(0) CKQ_BC(1) CKQ_BC(2) CKQ_BC(3) CKQ_BC(4) CKQ_BC(5) CKQ_BC(6) CKQ_BC(7)
        CKQ_BC(8) CKQ_BC(9) CKQ_BC(10) CKQ_BC(11) CKQ_BC(12) CKQ_BC(13) CKQ_BC(14) CKQ_BC(15)
    }
#undef CKQ_BC
    return acc;
}

/* A value that a VALU instruction computed, made safe as the x of fmac_row_lane: a DPP
 * instruction must not read a register a VALU instruction wrote in the two issue slots before it. */
__device__ __forceinline__ float dpp_source(float x)
{
    asm volatile("s_nop 1" : "+v"(x));
    return x;
}

/* Which token of its 32-token group output r = (lane & 15) of a lane is (the 32x32 MFMA result layout:
 * register r of lane l is row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32). */
__device__ __forceinline__ int mfma32_row_of_lane(int lane)
{
    return 8 * ((lane & 15) >> 2) + 4 * (lane >> 5) + (lane & 3);
}

/* A result leaves the chip once: the K-quant kernels store theirs non-temporally (whole 128-byte runs per wave
 * instruction; a tile's results are not read again by the launch that writes them, and the next launch runs on other
 * XCDs' L2s anyway): 1-2 % per launch.  The Q8_0 kernel, whose lanes store 16 bytes each to different rows, is 5-14 %
 * slower that way and keeps plain stores. */
#ifndef CKQ_GEMM_NT_STORE
#define CKQ_GEMM_NT_STORE 1
#endif
__device__ __forceinline__ void gemm_store(float *p, float v)
{
#if CKQ_GEMM_NT_STORE
    __builtin_nontemporal_store(v, p);
#else
    *p = v;
#endif
}

/* K split in SPLITS pieces by the waves of a block (gemm_q4k_ksplit_kernel and its siblings): the pieces of a tile of 64 tokens x 32 rows meet in LDS, which
 * the block has done with but for its own wave's part at red + wave * part, and are added in the order of the splits. */
template <int SPLITS>
__device__ __forceinline__ void gemm_ksplit_store(const GemmArgs &a, float *red, int part, const ckq_v16f (&acc)[2], int t0, int n0, int wave, int lane)
{
#pragma unroll
    for (int i = 0; i < 32; ++i) red[wave * part + 64 * i + lane] = acc[i >> 4][i & 15];
    __syncthreads();
    const int n = n0 + (lane & 31);
    if (n >= a.N) return;
    const float bias = a.bias ? a.bias[n] : 0.0f;
    for (int i = wave; i < 32; i += SPLITS) {
        float v = red[64 * i + lane];
#pragma unroll
        for (int sp = 1; sp < SPLITS; ++sp) v += red[sp * part + 64 * i + lane];
        const int r = i & 15, t = t0 + 32 * (i >> 4) + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (t < a.M) gemm_store(&a.C[(size_t)t * a.ldc + n], a.bias ? v + bias : v);
    }
}

/* The pieces of such a launch in place of one of tiles of 64 tokens x 128 rows, up to max_per 256-blocks a piece, 0: no.  Four waves
 * fill a CU's LDS, so every block gets a place at once: a second round would cost more than the second launch it saves (Q4_K, 300 tokens x 3840 x
 * 2000: 320 blocks of three waves). */
constexpr int GEMM_KSPLIT_Q4K = 7, GEMM_KSPLIT_Q5K = 9, GEMM_KSPLIT_Q6K = 7;       /* measured at the kernels */
static int gemm_ksplit_pieces(int M, long N, int nb, int max_per)
{
    const long ntt = (M + 63) / 64, tiles = ntt * ((N + GEMM_TILE_ROWS - 1) / GEMM_TILE_ROWS);
    if (tiles >= 160) return 0;
    const int s = gemm_choose_splits((int)tiles, nb), per = (nb + s - 1) / s, k = (nb + per - 1) / per;
    return k >= 2 && k <= 4 && per <= max_per && ntt * ((N + 31) / 32) <= (k == 2 ? 512 : 256) ? k : 0;
}
template <class Kernel>
static int gemm_launch_ksplit(Kernel k2, Kernel k3, Kernel k4, GemmArgs &g, int k, hipStream_t s)
{
    g.k_per = (g.nb + k - 1) / k;
    /* refused as a split among blocks is where its partial tiles have no room, though none are written here: what a size is answered does not hang on the kernel */
    if (g.ext_part && (size_t)k * (size_t)g.M * (size_t)g.N * sizeof(float) > g.ext_part_bytes) return CKQ_ESCRATCH;
    g.nnt = (g.N + 31) / 32;
    hipLaunchKernelGGL(k == 2 ? k2 : k == 3 ? k3 : k4, dim3((unsigned)gemm_blocks(g.ntt, g.nnt)), dim3((unsigned)(64 * k)), 0, s, g);
    return (int)hipGetLastError();
}

/* Grouped launch: the matrices of `in` against the same M x K activations, as one grid (no K split; the
 * callers group only what fills the chip without one). */
struct GemmGroupIn {
    int          n;
    const void  *B[GEMM_GROUP_MAX];
    const float *bias[GEMM_GROUP_MAX];
    float       *C[GEMM_GROUP_MAX];
    int          N[GEMM_GROUP_MAX];
    long         ldc[GEMM_GROUP_MAX];
};
/* Below this many tiles a single matrix is split along K instead (gemm_choose_splits); a group is not. */
constexpr int GEMM_GROUP_MIN_TILES = 160;
static int gemm_group_tiles(const GemmGroupIn &in, int M, int tokens_per_tile, int rows_per_tile = GEMM_TILE_ROWS)
{
    int tiles = 0;
    for (int p = 0; p < in.n; ++p)
        tiles += ((M + tokens_per_tile - 1) / tokens_per_tile) * ((in.N[p] + rows_per_tile - 1) / rows_per_tile);
    return tiles;
}
template <class Kernel>
static int gemm_launch_grouped(Kernel kernel, GemmArgs &g, const GemmGroupIn &in, hipStream_t s, unsigned threads = 256)
{
    unsigned grid = 0;
    g.ngroup = in.n;
    for (int p = 0; p < in.n; ++p) {
        const int nnt = (in.N[p] + GEMM_TILE_ROWS - 1) / GEMM_TILE_ROWS;
        g.grp[p] = {(const uint8_t *)in.B[p], in.bias[p], in.C[p], in.ldc[p], in.N[p], nnt, (int)grid, 0, g.ntt};
        grid += (unsigned)(g.ntt * nnt);
    }
    g.units = (int)grid;
    grid = (grid + 7) & ~7u;
    g.B = g.grp[0].B; g.bias = g.grp[0].bias; g.C = g.grp[0].C; g.N = g.grp[0].N; g.ldc = g.grp[0].ldc; g.nnt = g.grp[0].nnt;
    g.splits = 1; g.k_per = 0; g.part = nullptr;
    hipLaunchKernelGGL(kernel, dim3(grid, 1u), dim3(threads), 0, s, g);
    return (int)hipGetLastError();
}

/* Kernels with two blocks on a CU: whether the ragged token tiles (a matrix' last, of M % bm tokens, at most half a tile: less of everything
 * but the arithmetic) belong behind the whole ones of all matrices.  They do where the whole tiles of an XCD just fill its 32 CUs, or
 * once or twice its 64 slots, and the ragged ones are too many: what is left over is then short blocks alone.  us, in turn with the
 * ragged ones | last: Q5_K 405 tokens x 2 x 11008 rows x 2816 97.6 | 93.1, 276 x 2 x 7680 x 2048 47.1 | 43.0, 139 x 2 x 5888 x 1536 24.6 | 22.6;
 * Q4_K 405 x 2 x 11008 x 4096 109.9 | 106.0.  Where a few whole ones are left over as well those come late (Q5_K 341 x 2 x 6912 x 2048, 68 of an XCD,
 * 44.9 | 47.6; after two rounds blocks are out of step and four more do no harm), and so do tiles of more than half (227 x 2 x 8960 x 2816
 * 59.0 | 63.6); beyond that there is nothing to gain (Q5_K, 37 launches that the rule takes: 1.05 on average, 0.99 and more; 73 others 1.00, 0.92 to 1.09). */
static bool gemm_ragged_last(const GemmGroupIn &in, int M, int bm)
{
    if (M < bm || M % bm == 0 || M % bm > bm / 2 || 2 * in.n > GEMM_GROUP_MAX) return false;
    int whole = 0, all = 0;                    /* tiles of the fullest XCD */
    for (int p = 0; p < in.n; ++p) {
        const int nnt = (in.N[p] + GEMM_TILE_ROWS - 1) / GEMM_TILE_ROWS;
        whole += gemm_blocks(M / bm, nnt) / 8;
        all += (M / bm + 1) * nnt;
    }
    all = (all + 7) / 8;                       /* all tiles of all matrices are dealt as one (gemm_work) */
    return (whole <= 32 && all > 32) || (whole <= 64 && all > 64) || (whole <= 132 && all > 128);
}

/* One matrix or a group with the ragged token tiles as problems of their own behind the whole ones; returns the blocks to launch. */
static int gemm_deal_ragged_last(GemmArgs &g, const GemmGroupIn &in, int bm)
{
    const int nfull = g.M / bm;
    int grid = 0;
    g.ngroup = 0;
    for (int ragged = 0; ragged < 2; ++ragged)
        for (int p = 0; p < in.n; ++p) {
            const int nnt = (in.N[p] + GEMM_TILE_ROWS - 1) / GEMM_TILE_ROWS, ntt = ragged ? 1 : nfull;
            g.grp[g.ngroup++] = {(const uint8_t *)in.B[p], in.bias[p], in.C[p], in.ldc[p], in.N[p], nnt, grid, ragged ? nfull : 0, ntt};
            grid += gemm_blocks(ntt, nnt);
        }
    g.units = 0; g.splits = 1; g.k_per = 0; g.part = nullptr;
    return grid;
}
template <class Kernel>
static int gemm_launch_ragged_last(Kernel kernel, GemmArgs &g, const GemmGroupIn &in, int bm, hipStream_t s)
{
    const int grid = gemm_deal_ragged_last(g, in, bm);
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid, 1u), dim3(256u), 0, s, g);
    return (int)hipGetLastError();
}

/* The four kernels, one translation unit each: C[m*ldc + n] = dot(B row n, A row m) (+ bias[n]).
 * See GemmOpts for the options.  The _group forms return CKQ_ENOGROUP when the matrices are better
 * launched one by one (too few tiles to fill the chip without a K split). */
int launch_gemm_q4k_mfma_group(const void *A, const GemmGroupIn &in, int M, int K, hipStream_t s);
int launch_gemm_q5k_mfma_group(const void *A, const GemmGroupIn &in, int M, int K, hipStream_t s);
int launch_gemm_q6k_mfma_group(const void *A, const GemmGroupIn &in, int M, int K, hipStream_t s);
int launch_gemm_q80_mfma_group(const void *A, const GemmGroupIn &in, int M, int K, hipStream_t s);
/* Q8_0 operands that start on dwords: ckq_gemm_q80_dw.hip */
static inline bool gemm_q80_on_dwords(const void *A, const void *B) { return ((uintptr_t)A | (uintptr_t)B) % 4 == 0; }
int gemm_q80_dw_launch(GemmArgs &g, hipStream_t s);
int gemm_q80_dw_launch_group(GemmArgs &g, const GemmGroupIn &in, hipStream_t s);
int launch_gemm_q4k_mfma(const void *A, const void *B, const float *bias, float *C, int M, int N, int K, long ldc, const GemmOpts &opts, hipStream_t s);
int launch_gemm_q5k_mfma(const void *A, const void *B, const float *bias, float *C, int M, int N, int K, long ldc, const GemmOpts &opts, hipStream_t s);
int launch_gemm_q6k_mfma(const void *A, const void *B, const float *bias, float *C, int M, int N, int K, long ldc, const GemmOpts &opts, hipStream_t s);
int launch_gemm_q80_mfma(const void *A, const void *B, const float *bias, float *C, int M, int N, int K, long ldc, const GemmOpts &opts, hipStream_t s);
