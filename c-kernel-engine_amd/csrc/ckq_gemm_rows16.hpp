/*
 * ckq_gemm_rows16.hpp - matmuls of a few to a few dozen tokens on the int8 matrix cores, one wave per
 * 256-block of 16 rows: launch interface of ckq_gemm_rows16.hip.
 */
#pragma once
#include "ckq_gemm_common.hpp"

/* The kernel stands in for two others and gives the bits of the one it replaces.  TREE: the streaming kernel's order, one
 * fp32 term per 64 elements and a fixed tree over them.  Otherwise the tile kernels': one term per 256-block, run through
 * chains of multiply-adds in ascending block order, the chains added split by split, the two wave groups of a split
 * first. */
struct GemmChains { int splits, per, kg; };

/* The chains gemm_launch_split gives `tiles` tiles of `steps` steps. */
static inline GemmChains gemm_chains_split(int tiles, int steps)
{
    const int s = gemm_choose_splits(tiles, steps), per = (steps + s - 1) / s;
    return {(steps + per - 1) / per, per, 1};
}
/* The chains of the tile kernel that launch_gemm_*_mfma would run. */
GemmChains gemm_q4k_chains(int M, int N, int K);
GemmChains gemm_q5k_chains(int M, int N, int K);
GemmChains gemm_q6k_chains(int M, int N, int K);
/* Has the caller asked for one of the tile kernels (ckq_set_prefill_variant)? */
bool gemm_q4k_forced();
bool gemm_q5k_forced();
bool gemm_q6k_forced();
/* Those of a shared launch of several matrices; false: launch_gemm_*_mfma_group would not take it. */
bool gemm_q4k_group_chains(const GemmGroupIn &in, int M, int K, GemmChains *ch);
bool gemm_q5k_group_chains(const GemmGroupIn &in, int M, int K, GemmChains *ch);
bool gemm_q6k_group_chains(const GemmGroupIn &in, int M, int K, GemmChains *ch);

struct Rows16Problem {
    const uint8_t *W, *X;
    float         *y;
    const float   *bias;
    long           ldy;
    int            N, id0;           /* rows; first block id */
    GemmChains     ch;
};
struct Rows16Args {
    int M, nb, n;
    bool tree;                       /* for all problems of the launch */
    Rows16Problem p[GEMM_GROUP_MAX];
};
/* Estimated time in us of such a launch where its kernel for short rows and several token groups runs, else 0. */
float gemm_rows16_keep_time(int fmt, bool tree, size_t rows, int ntok, int nb);
/* The same for its kernel that takes token groups in pairs, in the order of the tile kernels. */
float gemm_rows16_pair_time(int fmt, size_t rows, int ntok, int nb);
/* One launch over a.n problems of one format, width and token count (id0 is filled in). */
int launch_gemm_rows16(int fmt, Rows16Args &a, hipStream_t s);
constexpr int ROWS16_MAX_K = 64 * 256;      /* the terms of a longer row would not fit the LDS */
