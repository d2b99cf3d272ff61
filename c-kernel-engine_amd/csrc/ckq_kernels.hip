/*
 * ckq_kernels.hip - gfx950 kernels of the quantized dequant-dot path and their
 * C launchers.
 *
 *   gemv_kernel<F,...>      weight rows x up to 8 activation rows (decode and
 *                           small-batch prefill); weights are streamed once
 *                           with 128-bit loads, unpacked in registers, dotted
 *                           with v_dot4_i32_i8, reduced with DPP.
 *   quantize_q8_k_kernel    fp32 -> Q8_K, bit-exact with the reference; also SiLU(gate)*up -> Q8_K
 *   quantize_q8_0_kernel    fp32 -> Q8_0, bit-exact with the reference
 *   rmsnorm_q8_k_fused_kernel  RMSNorm -> Q8_K in one pass, bit-exact with the reference's FMA build
 *   dequant_rows_kernel     row dequantizers / quantized embedding lookup, bit-exact
 *   copy_kernel             plain streaming copy (counter calibration)
 *   read_kernel             plain streaming read (launch-floor calibration)
 *
 * wave64 only; every kernel is launched with 256-thread blocks.
 */
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include "ckq_blocks.h"
#include "ckq_formats.hpp"
#include "ckq_producers.hpp"
#include "ckq_launch.h"
#include "ckq_pure.h"

/* ========================================================================= */
/* GEMV                                                                       */
/* ========================================================================= */

/* Which kernel serves a matmul of `ntok` tokens.  The weight-streaming dot4
 * kernel takes up to eight tokens per pass over the weights; the matrix-core
 * GEMMs read the weights once for any token count but have a floor of 13-19 us
 * (their K loop waits on global->LDS copies of ~1.5 us latency with only two or
 * three stages to cover it).  Measured crossover: one pass always streams;
 * beyond that the streaming kernel stays ahead while (passes x weight bytes,
 * at least 3 MB each) fits the budget - 20 MB, 40 MB for the Q5_K GEMM whose
 * floor is higher.  Examples at 9-16 tokens: Q4_K 4096x4096 (9.4 MB) streams
 * (12 us against 14), 11008x4096 (25 MB) goes to the matrix cores (19 us
 * against 25-28), the Q8_0 LM head 151936x896 likewise (67 us against 89-102);
 * Q8_0 4864x896 streams up to 32 tokens. */
constexpr int CKQ_STREAM_TOKENS = 8;
#include <atomic>
#include <type_traits>
static std::atomic<int> g_gemm_policy{0};      /* 0 automatic, 1 matrix cores above one pass, 2 always stream */

extern "C" void ckq_launch_set_gemm_policy(int policy) { g_gemm_policy.store(policy < 0 || policy > 2 ? 0 : policy); }

/* Q8_0 has its own estimate (us, weight bytes in MB): streaming 4.8 + passes * MB / 5.0 (MB / 3.6 for rows it must read with
 * 2-byte-aligned loads), matrix cores max(14, 9 + MB / 2.5), measured with ckq_gemm_q80.hip.  LM head 151936x896 (145 MB):
 * 9-16 tokens stream, 17 and more go to the matrix cores; 4864x896 (4.6 MB) streams up to 72 tokens.  Rows on dwords run the
 * faster ckq_gemm_q80_dw.hip since, which is ahead earlier (two passes over large matrices: 16 tokens, 32000x4096 60 against 28; the
 * second kernel's 8 to 14 us for small ones), but the line also says which order of sums a size has, whether it may be split along K and
 * so needs scratch, and stays where it is at every K (rows of an odd number of blocks, which it serves too, included): the tile kernel's one chain of additions over a row is less exact than the streaming
 * kernel's terms per lane and tree (rms error of the rms result at K = 7296: 1.9e-7, with two teams 1.4e-7, against 0.8e-7). */
static bool gemm_q80_on_matrix_cores(int ntok, size_t weight_bytes, bool aligned_rows)
{
    const int policy = g_gemm_policy.load(std::memory_order_relaxed);
    if (ntok <= CKQ_STREAM_TOKENS || policy == 2) return false;
    if (policy == 1) return true;
    const float passes = (float)((ntok + CKQ_STREAM_TOKENS - 1) / CKQ_STREAM_TOKENS), mb = (float)weight_bytes * 1e-6f;
    return 4.8f + passes * mb / (aligned_rows ? 5.0f : 3.6f) > fmaxf(14.0f, 9.0f + mb / 2.5f);
}

static bool gemm_on_matrix_cores(int ntok, size_t weight_bytes, size_t budget_mb)
{
    const int policy = g_gemm_policy.load(std::memory_order_relaxed);
    if (ntok <= CKQ_STREAM_TOKENS || policy == 2) return false;
    if (policy == 1) return true;
    const size_t passes = (size_t)(ntok + CKQ_STREAM_TOKENS - 1) / CKQ_STREAM_TOKENS;
    const size_t per = weight_bytes > ((size_t)3 << 20) ? weight_bytes : ((size_t)3 << 20);
    return passes * per > (budget_mb << 20);
}

/* fp32 activations.  The streaming kernel decodes the weights again for every token; the matrix-core kernel
 * (ckq_gemm_f32act.hip) decodes them once per 32 tokens.  Fitted to launches of both over 141..11008 rows, widths
 * of 512..8192 and 1..200 tokens (us): streaming 4 + 0.125 / 0.18 / 0.16 (Q4_K / Q6_K / Q8_0) per million products; matrix cores
 * 6 + 0.020 / 0.024 / 0.024 per million products of the tokens rounded up to 32, but never less than 5 + 1.35 (Q4_K 1.5) for every
 * 64 elements a wave walks through (an eighth of K).  4096 x 4096 Q6_K: 4 tokens 14.5 against 19 (streams), 8 tokens 26 against
 * 19, 96 tokens 270 against 31; 141 x 8192 streams up to 96 tokens. */
static bool f32act_on_matrix_cores(int fmt, int ntok, int nrows, int K)
{
    const int policy = g_gemm_policy.load(std::memory_order_relaxed);
    if (ntok < 2 || policy == 2) return false;
    if (policy == 1) return true;
    const float per = fmt == CKQ_KERNEL_Q4K_F32 ? 0.125f : fmt == CKQ_KERNEL_Q6K_F32 ? 0.18f : 0.16f;
    const float per_matrix = fmt == CKQ_KERNEL_Q4K_F32 ? 0.020f : 0.024f, per_step = fmt == CKQ_KERNEL_Q4K_F32 ? 1.5f : 1.35f;
    const float mw = (float)nrows * (float)K * 1e-6f;
    const float t_stream = 4.0f + per * mw * (float)ntok;
    const float t_matrix = fmaxf(5.0f + per_step * (float)((K + 511) / 512), 6.0f + per_matrix * mw * (float)((ntok + 31) / 32 * 32));
    return t_stream > t_matrix;
}

#include "ckq_gemv.hpp"
#include "ckq_gemm_common.hpp"
#include "ckq_gemm_f32act.hpp"
#include "ckq_gemm_rows16.hpp"

/* C = bias + partial 0 + partial 1 + ... in that order: the result does not
 * depend on which block finished first.  A thread adds V (4 or 1) adjacent
 * outputs.  The loads of eight, four or two partials go out together; one by
 * one, each was a trip to memory of its own (whole launches, us: Q4_K 20 x 512 x 8192
 * 13.5 -> 11.7, Q5_K 200 x 1024 x 8192 20.1 -> 17.9, Q4_K 225 x 3072 x 3072 17.8 -> 17.0). */
template <int V>
__global__ void __launch_bounds__(256) gemm_splitk_reduce_kernel(float *__restrict__ C, long ldc, const float *__restrict__ part,
                                                                 const float *__restrict__ bias, int M, int N, int splits)
{
    typedef float vec __attribute__((ext_vector_type(V)));
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V, mn = (size_t)M * (size_t)N;
    if (i >= mn) return;
    const int t = (int)(i / (size_t)N), n = (int)(i % (size_t)N);
    vec v = {}, b = {};
    if (bias) b = *reinterpret_cast<const vec *>(bias + n);
    auto add = [&](auto group, int s) {
        constexpr int G = decltype(group)::value;
        vec p[G];
#pragma unroll
        for (int k = 0; k < G; ++k) p[k] = *reinterpret_cast<const vec *>(part + (size_t)(s + k) * mn + i);
#pragma unroll
        for (int k = 0; k < G; ++k) v = s + k ? v + p[k] : p[k];
    };
    int s = 0;
    for (; s + 8 <= splits; s += 8) add(std::integral_constant<int, 8>{}, s);
    if (s + 4 <= splits) { add(std::integral_constant<int, 4>{}, s); s += 4; }
    if (s + 2 <= splits) { add(std::integral_constant<int, 2>{}, s); s += 2; }
    if (s < splits) add(std::integral_constant<int, 1>{}, s);
    *reinterpret_cast<vec *>(C + (size_t)t * ldc + n) = bias ? v + b : v;
}


static std::recursive_mutex g_split_mu;
std::recursive_mutex &gemm_split_mutex() { return g_split_mu; }

/* Grow-only device scratch per (device, stream, kind); see ckq_gemm_common.hpp.
 * kind 0: partial tiles of a K split; kind 1: weights rewritten for another kernel.
 * When all slots are taken the least recently used one is recycled: the device is
 * synchronised (its stream may no longer exist), its buffer freed.  A destroyed
 * stream whose handle value is given out again finds the old stream's slot: harmless,
 * that stream's work has ended and the buffer is still this device's memory.
 * ckq_launch_release_stream gives a stream's slots back explicitly. */
namespace {
constexpr int WS_SLOTS = 32;
struct WsSlot { hipStream_t s; int kind, dev; void *p; size_t cap; unsigned epoch; };
WsSlot   g_ws[WS_SLOTS];
uint64_t g_ws_key[WS_SLOTS], g_ws_use[WS_SLOTS], g_ws_clock = 0;
uint64_t ws_key(int dev, hipStream_t s, int kind)
{
    /* lossless for user-space handles (below 2^56), 32 devices and four kinds; never 0 */
    return (1ull << 63) | ((uint64_t)(kind & 3) << 61) | ((uint64_t)(dev & 31) << 56) | ((uint64_t)(uintptr_t)s & ((1ull << 56) - 1));
}
}

static int workspace_slot(int kind, hipStream_t s, size_t bytes, WsSlot **out, bool *fresh);

int gemm_workspace(int kind, hipStream_t s, size_t bytes, float **out)
{
    WsSlot *sl = nullptr;
    const int rc = workspace_slot(kind, s, bytes, &sl, nullptr);
    if (rc == 0) *out = (float *)sl->p;
    return rc;
}

static int workspace_slot(int kind, hipStream_t s, size_t bytes, WsSlot **out, bool *fresh)
{
    std::lock_guard<std::recursive_mutex> lock(g_split_mu);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    const uint64_t key = ws_key(dev, s, kind);
    int i = ckq_workspace_pick(g_ws_key, g_ws_use, WS_SLOTS, key);
    WsSlot *sl = &g_ws[i];
    if (g_ws_key[i] != key) {
        if (g_ws_key[i] != 0 && sl->p) {                 /* recycle */
            int cur = dev;
            if (sl->dev != cur) (void)hipSetDevice(sl->dev);
            e = hipDeviceSynchronize();
            if (e == hipSuccess) e = hipFree(sl->p);
            if (sl->dev != cur) (void)hipSetDevice(cur);
            if (e != hipSuccess) return (int)e;
        }
        g_ws_key[i] = key;
        *sl = {s, kind, dev, nullptr, 0, 0u};
    }
    g_ws_use[i] = ++g_ws_clock;
    if (fresh) *fresh = sl->cap < bytes;
    if (sl->cap < bytes) {
        if (sl->p) {
            e = hipStreamSynchronize(s);
            if (e != hipSuccess) return (int)e;
            (void)hipFree(sl->p);
            sl->p = nullptr; sl->cap = 0;
        }
        const size_t cap = bytes + bytes / 2;
        e = hipMalloc(&sl->p, cap);
        if (e != hipSuccess) return (int)e;
        sl->cap = cap;
    }
    *out = sl;
    return 0;
}

/* Frees the scratch held for `stream` on the current device (call before the
 * stream is destroyed, after its work has been synchronised). */
extern "C" int ckq_launch_release_stream(void *stream)
{
    std::lock_guard<std::recursive_mutex> lock(g_split_mu);
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    for (int i = 0; i < WS_SLOTS; ++i) {
        if (g_ws_key[i] == 0 || g_ws[i].s != (hipStream_t)stream || g_ws[i].dev != dev) continue;
        if (g_ws[i].p) {
            e = hipStreamSynchronize((hipStream_t)stream);
            if (e != hipSuccess) return (int)e;
            (void)hipFree(g_ws[i].p);
        }
        g_ws_key[i] = 0;
        g_ws_use[i] = 0;
        g_ws[i] = {};
    }
    return 0;
}


int gemm_launch_reduce(float *C, long ldc, const float *part, const float *bias, int M, int N, int splits, hipStream_t s)
{
    const size_t mn = (size_t)M * (size_t)N;
    if (N % 4 == 0 && ldc % 4 == 0 && ((uintptr_t)C | (uintptr_t)part | (uintptr_t)bias) % 16 == 0)
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel<4>, dim3((unsigned)((mn / 4 + 255) / 256)), dim3(256), 0, s, C, ldc, part, bias, M, N, splits);
    else
        hipLaunchKernelGGL(gemm_splitk_reduce_kernel<1>, dim3((unsigned)((mn + 255) / 256)), dim3(256), 0, s, C, ldc, part, bias, M, N, splits);
    return (int)hipGetLastError();
}



/* Q5_0 block -> Q8_0 block: the scale is kept, the 32 values become int8
 * q - 16.  One thread per block. */
__device__ __forceinline__ void q5_0_to_q8_0_block(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, size_t i)
{
    FmtQ50::Wt w;
    FmtQ50::Off o;
    o.blk = 0;
    FmtQ50::load_w(w, src + i * 22, o);
    FmtQ50::Dec d;
    FmtQ50::decode(d, w, 0);
    uint8_t *out = dst + i * 34;
    *reinterpret_cast<uint16_t *>(out) = (uint16_t)w.d;
#pragma unroll
    for (int k = 0; k < 8; ++k) {             /* 34-byte blocks: 2-byte aligned stores */
        reinterpret_cast<uint16_t *>(out + 2)[2 * k] = (uint16_t)((u32)d.q[k] & 0xffffu);
        reinterpret_cast<uint16_t *>(out + 2)[2 * k + 1] = (uint16_t)((u32)d.q[k] >> 16);
    }
}
__global__ void __launch_bounds__(256) q5_0_to_q8_0_kernel(const uint8_t *__restrict__ src, uint8_t *__restrict__ dst, size_t nblocks)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < nblocks) q5_0_to_q8_0_block(src, dst, i);
}

static int launch_gemm_q50_via_q80(const void *A, const void *B, const float *bias, float *C,
                                   int M, int N, int K, long ldc, hipStream_t s)
{
    const size_t nblocks = (size_t)N * (size_t)(K / 32);
    std::lock_guard<std::recursive_mutex> lock(g_split_mu);   /* the scratch is shared by launches on this stream */
    float *tmp = nullptr;
    int rc = gemm_workspace(1, s, nblocks * 34, &tmp);
    if (rc) return rc;
    hipLaunchKernelGGL(q5_0_to_q8_0_kernel, dim3((unsigned)((nblocks + 255) / 256)), dim3(256), 0, s,
                       (const uint8_t *)B, (uint8_t *)tmp, nblocks);
    rc = (int)hipGetLastError();
    if (rc) return rc;
    return launch_gemm_q80_mfma(A, tmp, bias, C, M, N, K, ldc, GemmOpts{}, s);
}

static bool weights_dword_aligned(const GemvArgs &a, const GemvGroup &grp)
{
    uintptr_t bits = reinterpret_cast<uintptr_t>(a.W);
    for (int i = 0; i + 1 < grp.n; ++i) bits |= reinterpret_cast<uintptr_t>(grp.W[i]);
    return (bits & 3) == 0;
}

/* Whether the matrix-core kernel on 16-row tiles (ckq_gemm_rows16.hip) takes a matmul of `rows` rows (all matrices of a
 * launch) that would otherwise go to the tile kernels (`tiles`) or to the streaming kernel.  The results are the same bits
 * either way, so only time decides.  Fitted to launches of all three over 128..16000 rows, widths of 256..11008 and 3..400
 * tokens (us; nb: 256-blocks of a row, mb: megabytes of weights, n16: thousands of 256-blocks of 16 rows times groups of 16
 * tokens); the rule's choices cost 0.3 % (against streaming) and 1.3 % (against the tiles) more than always taking the faster, single
 * shapes up to a third (Q6_K 14911 x 1536 at 75 tokens: 22, tiles 17; Q4_K 4556 x 9984 at 30: 22, tiles 18):
 *   rows16     3.6 + 0.12 nb + (Q4_K 0.36, Q5_K 0.65, Q6_K 0.71) n16; up to 256 tokens of short rows gemm_rows16_keep_time
 *              (Q5_K 4864 x 1024 at 192 tokens: 10.3, tiles 13.7; 4096 x 2048 at 256: 17.2, tiles 19.5); groups of tokens in pairs gemm_rows16_pair_time
 *   tiles      11 + 0.2 mb + 0.0015 tokens mb, an under-estimate almost everywhere; against groups in pairs Q5_K 13.3 + 0.164 mb + 0.0048 tokens mb and
 *              Q6_K 13.8 + 0.083 mb + 0.0044 tokens mb (11 % rms over 207 launches of 9 to 200 tokens, where the first cost 4.1 and 7.3 % more than the
 *              faster kernel and these cost 1.5 and 0.6; Q4_K's own fit would cost 5.2 instead of 1.0)
 *   K split    where the pieces of K are waves of a block (gemm_ksplit_pieces), fitted to 450 launches of 17 to 700 tokens, 5 to 11 % rms: 4.1 + 1.44 per + 0.16 mb + 3.3 out
 *              (per: 256-blocks of a piece, out: millions of outputs; Q5_K 3.7, 1.83, 0.12, 2.8, Q6_K 3.75, 1.73, 0.18, 3.7), and rows16 there 3.4 + 0.11 nb +
 *              0.6 n16 (2.8, 0.154, 0.85; 2.8, 0.26, 0.22 and with more than one block a CU 1.7, 0.43, 0.70: 7 % rms over 22 launches, where the former made
 *              half of 46 us, and the choice cost up to 113 % instead of none: 111 tokens x 6912 x 3759 46.4 -> 22.8, 29 x 6912 x 7371 30.0 -> 23.4),
 *              groups in pairs 3.7 + (0.135 + 0.135 blocks on a CU) nb (3.4, 0.09, 0.32; 4.6, -0.024, 0.344).  By the estimates above the choice cost 5.6, 7.1 and 4.5 % more than the faster kernel, single sizes 48; by these 0.4 (us: Q4_K 172 tokens x 2560 x 3385
 *              18.8 -> 13.5, Q5_K 146 x 3840 x 2084 18.7 -> 13.7, Q6_K 329 x 3328 x 1257 20.2 -> 13.7).  Not for calls that bring their scratch
 *              (`own_scratch`): a 16-row kernel needs none, and what goes to a split of K is refused where the partial tiles would be more than that scratch,
 *              so these calls keep the estimates above, by which none is refused that a 16-row kernel took before there were splits among waves (the
 *              groups in pairs take many of Q5_K and Q6_K that were).
 *   short rows, up to 256 tokens of two groups and more (t_keep), against the tiles: 6.2 + (0.26 + 0.41 rounds + 0.62 CU) nb + 0.88 out (rounds: of 256 tiles of 64 tokens x 128 rows, CU:
 *              tiles a CU, one at least, since some kernels have two blocks on a CU; Q5_K 6.6, 0.32, 0.70, 0.78, 1.04, Q6_K 7.3, 0, 1.11, 0.45, 0.77; 4 to 5 % rms over 1146 launches of
 *              17 to 256 tokens, 200 to 32000 rows, where the line above has 20 to 28) and gemm_rows16_keep_time once more, with the outputs and rows of three blocks, which leave
 *              a wave's place idle: 0.66 + 0.82 t + 0.97 out + 0.09 t where nb = 3 (0.14, 0.98, 0.47, 0.04; 0.21, 0.985, 0.43, 0.08).  The choice costs 0.2 to 0.3 % more
 *              than the faster kernel, by the line above 0.8 to 1.5, at most 53 (us: Q4_K 120 tokens x 256 x 27284 13.4 -> 10.1, Q5_K 117 x 256 x 26823 14.5 -> 11.2, 185 x 1792 x
 *              3199 19.5 -> 15.0).
 *   streaming  above eight tokens the larger of 2.9 and 2.2 + 0.0075 lanes + (23.5, 23.5, 29) million lanes of all rows and passes,
 *              a row's 64-element positions being dealt to 8, 16, 32 or 64 lanes or to 2 to 4 passes of 64 (stream_lanes): small
 *              matrices stream at up to some 60 tokens (Q5_K 290 x 1792 at 25: 3.0, here 4.6; Q6_K 435 x 1536 at 13 3.0, here 4.8);
 *              several matrices take a launch each; against short rows' t_keep 2.4 + 14.9 w + 2.7 sqrt w (w: those lanes; Q5_K 2.2, 10.4, 6.0, Q6_K 2.15, 9.2, 8.65; 5.5 to 11 % rms
 *              over 900 launches of 17 to 120 tokens) and 1.17 t - 0.8 (1.32 t - 1.6; 1.4 t - 1.95): costs 0.1 to 0.25 % more than the faster kernel instead of 0.6 to 1.9, at most
 *              27 instead of 60 (us: Q6_K 47 tokens x 2048 x 368 7.0 -> 4.4, Q5_K 64 x 256 x 1141 4.9 -> 3.9)
 *   5 to 8 tokens, one to three matrices in a launch, weights from HBM: 2.64 + 0.0043 lanes + 7.6 million lanes of all rows + 0.237 mb + 0.022 lanes where the grid (the largest
 *              matrix's for each) is more than a block a CU, 65536 lanes (Q5_K 2.71, 0.006, 8.0, 0.206, 0.0254; Q6_K 2.88, 0.0085, 11.7, 0.182, 0.0348: 10 to 11 % rms), against the 16-row
 *              tiles' larger of 3.38 + 0.116 nb and 3.71 + 0.327 mb (3.45, 0.133, 3.83, 0.296; 3.39, 0.181, 3.76, 0.291: 7 % rms): 4692 launches of 64 to 40000 rows, widths of 256 to
 *              16384. The choice costs 0.2 to 0.3 % more than the faster kernel; by a line without lanes, each matrix of a group for itself, it cost 7 to 8, at most 130 (us:
 *              Q6_K 6 tokens x (4352, 1088, 1088) x 4352 25.5 -> 11.1, Q5_K 8 x (4352, 1088, 1088) x 4352 21.0 -> 10.1, Q4_K 8 x (5120, 1280, 1280) x 5120 21.1 -> 10.3, 8 x 2304 x 2304 6.7 -> 5.2)
 *   3 and 4 tokens, one pass of half the width: 2.48 + 0.0008 lanes + 4.36 million lanes (1.15 times that for rows above 6144) + 0.141 mb + 0.0129 lanes where the grid is more than two blocks a CU
 *              (2.62, 0.0004, 6.04, 0.098, 0.0148; 2.70, 0.0043, 7.19, 0.103, 0.0189) against 1.1 times the larger of 3.04 + 0.142 nb and 3.73 + 0.311 mb (3.15, 0.151, 3.88, 0.279; 3.27,
 *              0.188, 3.86, 0.288): 6 to 8 % rms over 2100 launches. By the rule before, for large Q6_K matrices alone, the choice cost 2.7 % more than the faster kernel, by this 0.8: 332
 *              launches by more than 5 % faster, 8 by more than 3 % slower (us: Q5_K 4 x 11264 x 2560 13.0 -> 9.8, Q6_K 4 x (4352, 2176, 2176) x 4352 18.3 -> 14.5; not moved, Q5_K 4 x 4096 x 8192 7.6 against 9.5).
 * Two tokens never move.  The forced policies keep their kernels: 1 the tile kernels, 2 the
 * streaming kernel at any number of tokens; and so does a tile kernel that the caller asked for.  Forced itself
 * (ckq_launch_set_rows16) it goes before all of them, in the order of the kernel that the policy asks for. */
static int stream_lanes(int positions)
{
    for (int n : {8, 16, 32, 64, 128, 192})
        if (positions <= n) return n;
    return (positions + 255) / 256 * 256;
}
static std::atomic<int> g_rows16_forced{0};           /* bit per format tag */
extern "C" void ckq_launch_set_rows16(int fmt, int on)
{
    if (fmt < 0 || fmt > 31) return;
    if (on) g_rows16_forced.fetch_or(1 << fmt);
    else g_rows16_forced.fetch_and(~(1 << fmt));
}
/* gemm_rows16_keep_time as it was fitted before, for calls that bring their scratch: rows of eight blocks are the only ones that this kernel and a split of K
 * both take, and no call is to be refused for want of scratch because an estimate of time was fitted again. */
static float keep_time_own_scratch(int f, size_t rows, int ntok)
{
    const long tiles = (long)((rows + 15) / 16), groups = (ntok + 15) / 16;
    if (f == 0 || groups < 2 || tiles > 1 << 20) return 0.0f;
    float least = 0.0f;
    for (long parts = 1; (groups + parts - 1) / parts >= 2; ++parts) {
        const float t = 2.5f + (1.5f + (float)((groups + parts - 1) / parts)) * (0.45f + 0.54f * (float)((tiles * parts + 255) / 256));
        if (parts == 1 || t <= least) least = t;
    }
    return least < 4.4f + 1e-3f * (f == 1 ? 4.98f : 5.82f) * (float)(tiles * groups) ? least : 0.0f;
}
static float rows16_q4k_time(float nb, size_t rows, int ntok) { return 3.6f + 0.12f * nb + 0.58e-3f * nb * (float)((rows + 15) / 16) * (float)((ntok + 15) / 16); }
/* A matrix of fewer than 160 tiles on its own: split along K or not, or by the 16-row kernel (Q5_K, Q6_K: fitted to 631 launches of whichever the rule takes, 17 to 130 tokens, 12 % rms; Q4_K rows of
 * less than eight blocks, never split, by their length alone: one round of tiles). */
static float single_time(int f, float nb, size_t rows, int ntok)
{
    static const float c[2][6] = {{2.09f, 0.224f, 0.218f, 13.8f, 0.50f, 176e-6f}, {2.13f, 0.232f, 0.127f, 15.0f, 0.565f, 210e-6f}};
    const float out = 1e-6f * (float)ntok * (float)rows;
    if (f) return c[f - 1][0] + c[f - 1][1] * nb + c[f - 1][2] * c[f - 1][5] * nb * (float)rows + (c[f - 1][3] + c[f - 1][4] * nb) * out;
    return fminf(nb < 8.0f ? 5.5f + 1.2f * nb : 7.2f + 0.22f * nb + 0.22f * 144e-6f * nb * (float)rows, rows16_q4k_time(nb, rows, ntok));
}
/* Three to eight tokens, `rows` rows in one launch of either kernel; the streaming kernel's grid follows the largest of its matrices: `grid_rows`, their number times its
 * rows. The figures are described above; at three and four tokens the 16-row tiles have to be ahead by a tenth, as the times lie closer than
 * the fits do there. */
static float rows16_one_pass_time(int f, int ntok, size_t rows, int K, bool alone = true)
{
    static const float c[2][3][4] = {{{3.04f, 0.142f, 3.73f, 0.311f}, {3.15f, 0.151f, 3.88f, 0.279f}, {3.27f, 0.188f, 3.86f, 0.288f}},
                                     {{3.38f, 0.116f, 3.71f, 0.327f}, {3.45f, 0.133f, 3.83f, 0.296f}, {3.39f, 0.181f, 3.76f, 0.291f}}}, block[3] = {144e-6f, 176e-6f, 210e-6f};
    const float nb = (float)(K / 256), *t = c[ntok > 4][f];
    /* Q4_K, five to eight tokens, rows of up to four blocks: by the fit alone they streamed where the 16-row tiles are the faster ones and had been taken (us, streaming | 16-row tiles: 8 x 8695 x 1024
     * 5.55 | 4.77, 5 x 7256 x 1024 4.62 | 4.31; 242 such launches: the choice costs 0.9 % more than the faster kernel, 3.4 without).  Not against a launch that has the producer too (`alone`): 5 x 13113 x 256
     * 5.7 in one, 7.2 in two */
    const float short_rows = alone && f == 0 && ntok > 4 && nb <= 4.0f ? 0.93f : 1.0f;
    return (ntok > 4 ? short_rows : 1.1f) * fmaxf(t[0] + t[1] * nb, t[2] + t[3] * nb * (float)rows * block[f]);
}
static float stream_one_pass_time(int f, int ntok, size_t rows, size_t grid_rows, int K)
{
    static const float c[2][3][5] = {{{2.48f, 0.0008f, 4.36f, 0.141f, 0.0129f}, {2.62f, 0.0004f, 6.04f, 0.098f, 0.0148f}, {2.70f, 0.0043f, 7.19f, 0.103f, 0.0189f}},
                                     {{2.64f, 0.0043f, 7.6f, 0.237f, 0.0220f}, {2.71f, 0.0060f, 8.0f, 0.206f, 0.0254f}, {2.88f, 0.0085f, 11.7f, 0.182f, 0.0348f}}}, block[3] = {144e-6f, 176e-6f, 210e-6f};
    const int lanes = stream_lanes(K / 64);
    const bool second_round = grid_rows * (size_t)(lanes < 16 ? 16 : lanes > 64 ? 64 : lanes) > (ntok > 4 ? 65536 : 131072);
    const float *t = c[ntok > 4][f], few_blocks = ntok <= 4 && K > 6144 ? 1.15f : 1.0f;       /* four long tokens fill the LDS of a CU with few blocks */
    return t[0] + t[1] * (float)lanes + few_blocks * t[2] * 1e-6f * (float)rows * (float)lanes + t[3] * (float)(K / 256) * (float)rows * block[f] + (second_round ? t[4] * (float)lanes : 0.0f);
}
/* Q6_K at three and four tokens, rows of more than 4096, 20 MB of weights and more, a tenth of the streaming kernel's lanes idle: the passes over a row with few blocks on a CU, whose LDS the four
 * tokens fill, take up to 1.7 times the estimate below, and by it the 16-row tiles lost what they had had (180 such launches of one to three matrices, weights from HBM: streaming / 16-row tiles 1.37
 * in the middle, 1.77 at most, one 0.94 and two 0.99; us: 4 x 3 x 3831 x 11008 45.6 | 29.3, 3 x 2 x 7984 x 10496 54.7 | 35.2, 4 x (8517, 4258, 4258) x 6912 34.4 | 29.4). */
static bool q6k_long_rows_of_few_tokens(int f, int ntok, size_t rows, int K)
{
    return f == 2 && ntok <= 4 && K > 4096 && (float)rows * (float)(K / 256) * 210e-6f >= 20.0f && 10 * stream_lanes(K / 64) >= 11 * (K / 64);
}
/* Several matrices of three to eight tokens, which have one order of their sums in either kernel: all of them to the 16-row tiles, or none (a choice by matrix sent Q and K/V of
 * one group to two launches, or all to a streaming launch that each alone was too small to be faster than). */
static bool rows16_as_one(int fmt, int ntok, int K)
{
    return ntok > 2 && ntok <= CKQ_STREAM_TOKENS && K <= ROWS16_MAX_K && g_gemm_policy.load(std::memory_order_relaxed) != 2 && !(g_rows16_forced.load(std::memory_order_relaxed) >> fmt & 1);
}
static bool group_takes_rows16(int fmt, int ntok, int n, const int *rows, int K, bool streams_as_one, bool alone = true)
{
    const int f = fmt == CKQ_FMT_Q4_K ? 0 : fmt == CKQ_FMT_Q5_K ? 1 : 2;
    size_t all = 0, largest = 0;
    float apart = 0.0f;
    for (int i = 0; i < n; ++i) {
        const size_t r = (size_t)rows[i];
        all += r;
        if (r > largest) largest = r;
        apart += fminf(rows16_one_pass_time(f, ntok, r, K), stream_one_pass_time(f, ntok, r, r, K));
    }
    return q6k_long_rows_of_few_tokens(f, ntok, all, K) || rows16_one_pass_time(f, ntok, all, K, alone) < (streams_as_one ? stream_one_pass_time(f, ntok, all, largest * (size_t)n, K) : apart);
}
static bool take_rows16(int fmt, int ntok, size_t rows, int K, bool tiles, int launches = 1, bool own_scratch = false, size_t shared_tiles = 0, float t_singles = 0.0f)
{
    if (ntok < 2 || K > ROWS16_MAX_K) return false;
    if (g_rows16_forced.load(std::memory_order_relaxed) >> fmt & 1) return true;
    const int policy = g_gemm_policy.load(std::memory_order_relaxed);
    const int f = fmt == CKQ_FMT_Q4_K ? 0 : fmt == CKQ_FMT_Q5_K ? 1 : 2;
    const bool tile_forced = f == 0 ? gemm_q4k_forced() : f == 1 ? gemm_q5k_forced() : gemm_q6k_forced();
    if (ntok < 3 || policy == 2 || (tiles && (policy == 1 || tile_forced))) return false;
    static const float per_block[3] = {0.36f, 0.65f, 0.71f}, per_lane[3] = {23.5f, 23.5f, 29.0f};
    const float nb = (float)(K / 256), mb = (float)rows * nb * (f == 0 ? 144e-6f : f == 1 ? 176e-6f : 210e-6f);
    const int lanes = stream_lanes(K / 64);
    if (ntok <= CKQ_STREAM_TOKENS) return q6k_long_rows_of_few_tokens(f, ntok, rows, K) || rows16_one_pass_time(f, ntok, rows, K) < stream_one_pass_time(f, ntok, rows, rows, K);
    const float t_keep = ntok > 256 ? 0.0f : own_scratch && tiles && K == 2048 ? keep_time_own_scratch(f, rows, ntok) : gemm_rows16_keep_time(fmt, !tiles, rows, ntok, K / 256);
    const float t_pair = tiles && t_keep <= 0.0f ? gemm_rows16_pair_time(fmt, rows, ntok, K / 256) : 0.0f;
    const float t_rows = t_keep > 0.0f ? t_keep : t_pair > 0.0f ? t_pair : 3.6f + 0.12f * nb + per_block[f] * 1e-3f * nb * (float)((rows + 15) / 16) * (float)((ntok + 15) / 16);
    float t_else;
    /* Q5_K and Q6_K, several matrices that together are too few tiles for a shared launch: the tile kernels would take one or two launches for EACH, and what the estimates below know is one for all.
     * Where the 16-row tiles are ahead by a tenth they have it (fitted to 699 groups of 17 to 130 tokens, 13 % rms). 529 further groups of up to 400 tokens: 3.2 % faster on average, 54 by more than 5 %,
     * none by more than 4 % slower (us, one by one -> 16-row tiles in one launch: Q5_K 105 x 3 x 2304 x 2304 30.0 -> 20.5, 98 x (3072, 1536, 1536) x 3072 31.1 -> 21.8, Q6_K 64 x (5120, 1280, 1280) x
     * 5120 41.8 -> 28.6; left, 34 x (8704, 1088, 1088) x 8704 52.3 | 63.4). */
    if (f > 0 && tiles && ntok > 16 && launches > 1 && shared_tiles == 0 && !own_scratch) {
        static const float group[2][3] = {{2.85f, 0.303f, 0.583e-3f}, {2.97f, 0.282f, 0.575e-3f}};
        if (1.1f * (group[f - 1][0] + group[f - 1][1] * nb + group[f - 1][2] * nb * (float)((rows + 15) / 16) * (float)((ntok + 15) / 16)) < t_singles) return true;
    }
    if (const int pieces = tiles && launches == 1 && !own_scratch && rows < 1 << 24
                               ? gemm_ksplit_pieces(ntok, (long)rows, K / 256, f == 0 ? GEMM_KSPLIT_Q4K : f == 1 ? GEMM_KSPLIT_Q5K : GEMM_KSPLIT_Q6K) : 0) {
        static const float split[3][4] = {{4.1f, 1.44f, 0.16f, 3.3f}, {3.7f, 1.83f, 0.12f, 2.8f}, {3.75f, 1.73f, 0.18f, 3.7f}},
                           single[4][3] = {{3.4f, 0.11f, 0.6f}, {2.8f, 0.154f, 0.85f}, {2.8f, 0.26f, 0.22f}, {1.7f, 0.43f, 0.7f}},
                           pair[3][3] = {{3.7f, 0.135f, 0.135f}, {3.4f, 0.09f, 0.32f}, {4.6f, -0.024f, 0.344f}};
        const float r16 = (float)((rows + 15) / 16), groups = (float)((ntok + 15) / 16), per = (float)((K / 256 + pieces - 1) / pieces);
        const float t = split[f][0] + split[f][1] * per + split[f][2] * mb + split[f][3] * 1e-6f * (float)ntok * (float)rows;
        if (t_keep > 0.0f) return t_keep < t;
        if (t_pair > 0.0f) return pair[f][0] + (pair[f][1] + pair[f][2] * fmaxf(r16 * (float)((ntok + 31) / 32) / 256.0f, 1.0f)) * nb < t;
        const float *one = single[f == 2 && r16 * groups > 256.0f ? 3 : f];
        return one[0] + one[1] * nb + one[2] * 1e-3f * nb * r16 * groups < t;
    }
    const float out = 1e-6f * (float)ntok * (float)rows;
    if (tiles && t_keep > 0.0f && !(own_scratch && K == 2048)) {
        static const float tile[3][5] = {{6.18f, 0.26f, 0.41f, 0.62f, 0.88f}, {6.57f, 0.32f, 0.70f, 0.78f, 1.04f}, {7.28f, -0.02f, 1.11f, 0.45f, 0.77f}},
                           keep[3][4] = {{0.66f, 0.82f, 0.97f, 0.09f}, {0.14f, 0.98f, 0.47f, 0.04f}, {0.21f, 0.985f, 0.43f, 0.08f}};
        const float on_cu = (float)((rows + 127) / 128) * (float)((ntok + 63) / 64) / 256.0f;
        return keep[f][0] + (keep[f][1] + (nb == 3.0f ? keep[f][3] : 0.0f)) * t_keep + keep[f][2] * out <
               tile[f][0] + (tile[f][1] + tile[f][2] * ceilf(on_cu) + tile[f][3] * fmaxf(on_cu, 1.0f)) * nb + tile[f][4] * out;
    }
    /* Q4_K, several groups, against ONE launch of unsplit tiles (a single matrix of 160 tiles and more, or several of so many together): the 16-row kernel takes
     * 0.58 ns a 256-block of 16 rows and 16 tokens there, its blocks all over each other, and not the 0.36 of a few blocks a CU, and the tiles' time goes by rounds of their blocks. 60 launches of
     * 17 to 300 tokens, rows of 5 to 16 blocks, us, 16-row kernel | tiles: 65 x 2 x 6912 x 1536 19.0 | 14.3, 133 x 2 x 3840 x 1280 17.9 | 12.6, 32 x 2 x 11008 x 3840 28.2 | 22.1,
     * 257 x 2 x 3584 x 768 16.5 | 11.0; and 32 x 2 x 10240 x 1280 stays (11.6 | 13.0). Where several matrices are fewer tiles than that they go out one by one, and the estimates of those add up:
     * 98 x (2816, 1408, 1408) x 2816 27.5 one by one, 20.1 together. */
    const size_t unsplit = launches == 1 ? (rows + 127) / 128 * (size_t)((ntok + 63) / 64) : shared_tiles;
    if (f == 0 && tiles && !own_scratch && ntok > 16 && t_keep <= 0.0f && t_pair <= 0.0f && (unsplit >= 160 || (launches > 1 && unsplit == 0))) {
        const float t_tiles = !unsplit ? t_singles : unsplit <= 256 ? (nb < 8.0f ? 6.2f + 1.35f * nb : 8.5f + 0.95f * nb) : unsplit <= 512 ? 6.1f + 2.2f * nb : unsplit <= 768 ? 9.2f + 3.3f * nb : 11.0f + 4.6f * nb;
        return rows16_q4k_time(nb, rows, ntok) < t_tiles;
    }
    if (tiles) t_else = f == 0 || t_pair <= 0.0f ? 11.0f + (0.2f + 0.0015f * (float)ntok) * mb : f == 1 ? 13.3f + (0.164f + 0.0048f * (float)ntok) * mb : 13.8f + (0.083f + 0.0044f * (float)ntok) * mb;
    else {
        const float t_launch = 2.2f + 0.0075f * (float)lanes, w = 1e-6f * (float)rows * (float)lanes * (float)((ntok + 7) / 8);
        if (t_keep > 0.0f) {
            static const float stream[3][3] = {{2.39f, 14.9f, 2.69f}, {2.2f, 10.4f, 6.0f}, {2.15f, 9.2f, 8.65f}}, keep[3][2] = {{-0.78f, 1.17f}, {-1.56f, 1.32f}, {-1.95f, 1.4f}};
            return keep[f][0] + keep[f][1] * t_keep < stream[f][0] + stream[f][1] * w + stream[f][2] * sqrtf(w) + (float)(launches - 1) * t_launch;
        }
        t_else = fmaxf(2.9f, t_launch + per_lane[f] * w) + (float)(launches - 1) * t_launch;
    }
    return t_rows < t_else;
}

/* K-quants: does a matmul of this size go to the tile kernels (or, at their sizes, to the 16-row tiles)? */
static bool kquant_on_matrix_cores(int fmt, int ntok, size_t rows, int K)
{
    return gemm_on_matrix_cores(ntok, rows * (size_t)(K / 256) * (fmt == CKQ_FMT_Q4_K ? 144 : fmt == CKQ_FMT_Q5_K ? 176 : 210), fmt == CKQ_FMT_Q5_K ? 40 : 20);
}

/* Where a matmul of a whole matrix goes. */
static int launch_route(int fmt, int nrows, int K, int ntok, int aligned, bool own_scratch)
{
    bool tiles;
    switch (fmt) {
    case CKQ_FMT_Q4_K: case CKQ_FMT_Q5_K: case CKQ_FMT_Q6_K:
        tiles = kquant_on_matrix_cores(fmt, ntok, (size_t)nrows, K);
        if (take_rows16(fmt, ntok, (size_t)nrows, K, tiles, 1, own_scratch)) return tiles ? CKQ_ROUTE_ROWS16_TILES : CKQ_ROUTE_ROWS16_STREAM;
        break;
    case CKQ_FMT_Q8_0: tiles = gemm_q80_on_matrix_cores(ntok, (size_t)nrows * (K / 32) * 34, K % 64 == 0 && aligned); break;
    case CKQ_FMT_Q5_0: tiles = gemm_on_matrix_cores(ntok, (size_t)nrows * (K / 32) * 22, 20); break;
    case CKQ_KERNEL_Q80_F32: case CKQ_KERNEL_Q4K_F32: case CKQ_KERNEL_Q6K_F32: tiles = f32act_on_matrix_cores(fmt, ntok, nrows, K); break;
    default: return CKQ_EFORMAT;
    }
    return tiles ? CKQ_ROUTE_TILES : CKQ_ROUTE_STREAM;
}

extern "C" int ckq_launch_route(int fmt, int nrows, int K, int ntok, int aligned) { return launch_route(fmt, nrows, K, ntok, aligned, false); }

/* The chains of multiply-adds of such a launch: those of the tile kernel where it stands in for one, so that the result
 * has the tile kernel's bits. */
static GemmChains rows16_chains(int fmt, int ntok, int nrows, int K, bool tiles)
{
    if (!tiles) return {1, K / 256, 1};
    return fmt == CKQ_FMT_Q4_K ? gemm_q4k_chains(ntok, nrows, K) : fmt == CKQ_FMT_Q5_K ? gemm_q5k_chains(ntok, nrows, K) : gemm_q6k_chains(ntok, nrows, K);
}

/* LDS bytes of the staged token tile of a grouped launch against the 64 KB a
 * block may use: MT rows of activations, MT = token count rounded up to the
 * tile sizes launch_mt knows (1, 2, 4, 8); Q8_0 activations are re-laid out to
 * 36 bytes per block. */
static bool group_tile_fits_lds(int fmt, int K, int ntok)
{
    const size_t mt = ntok <= 1 ? 1 : ntok == 2 ? 2 : ntok <= 4 ? 4 : 8;
    size_t bytes;
    switch (fmt) {
    case CKQ_FMT_Q4_K: case CKQ_FMT_Q5_K: case CKQ_FMT_Q6_K: bytes = FmtQ4K::xs_lds_bytes(mt * (size_t)(K / 256) * 292); break;
    case CKQ_FMT_Q8_0: case CKQ_FMT_Q5_0:                     bytes = FmtQ80::xs_lds_bytes(mt * (size_t)(K / 32) * 34); break;
    default: return false;
    }
    return bytes <= 65536;
}

/* Where several K-quant matrices against the same `ntok` tokens go.  Up to eight tokens: the 16-row tiles (all of them) or the streaming kernel.  Beyond: the 16-row tiles in the
 * order of either (one order a launch), in place of the tile kernels' shared launch where they would take it, else of the single launches and with the bits of either; the tile kernels'
 * shared launch; or CKQ_ENOGROUP, one by one.  *grouped: whether the shared launch would be taken, whose chains *shared then are. */
static int kquant_group_route(int fmt, const GemmGroupIn &in, int M, int K, bool *grouped, GemmChains *shared)
{
    const int f = fmt == CKQ_FMT_Q4_K ? 0 : fmt == CKQ_FMT_Q5_K ? 1 : 2;
    size_t rows = 0;
    for (int p = 0; p < in.n; ++p) rows += (size_t)in.N[p];
    *grouped = kquant_on_matrix_cores(fmt, M, rows, K) &&
               (f == 0 ? gemm_q4k_group_chains(in, M, K, shared) : f == 1 ? gemm_q5k_group_chains(in, M, K, shared) : gemm_q6k_group_chains(in, M, K, shared));
    bool tiles[GEMM_GROUP_MAX], alike = true;
    float t_singles = 0.0f;
    for (int p = 0; p < in.n; ++p) {
        tiles[p] = *grouped || kquant_on_matrix_cores(fmt, M, (size_t)in.N[p], K);
        alike = alike && tiles[p] == tiles[0];
        t_singles += single_time(f, (float)(K / 256), (size_t)in.N[p], M);
    }
    if (alike && take_rows16(fmt, M, rows, K, tiles[0], in.n, false, *grouped ? (size_t)gemm_group_tiles(in, M, 64) : 0, t_singles)) return tiles[0] ? CKQ_ROUTE_ROWS16_TILES : CKQ_ROUTE_ROWS16_STREAM;
    return *grouped ? CKQ_ROUTE_TILES : CKQ_ENOGROUP;
}
static int group_route(int fmt, int n, const int *rows, int K, int ntok)
{
    if (ntok <= CKQ_STREAM_TOKENS) {
        /* two tokens, and the policies that ask for a kernel, have one answer for all sizes */
        const bool rows16 = rows16_as_one(fmt, ntok, K) ? group_takes_rows16(fmt, ntok, n, rows, K, group_tile_fits_lds(fmt, K, ntok)) : take_rows16(fmt, ntok, (size_t)rows[0], K, false);
        return rows16 ? CKQ_ROUTE_ROWS16_STREAM : CKQ_ROUTE_STREAM;
    }
    GemmGroupIn in = {};
    in.n = n;
    for (int p = 0; p < n; ++p) in.N[p] = rows[p];
    bool grouped;
    GemmChains shared = {};
    return kquant_group_route(fmt, in, ntok, K, &grouped, &shared);
}
extern "C" int ckq_launch_group_route(int fmt, int n, const int *rows, int K, int ntok)
{
    if (n < 2 || n > CKQ_GROUP_MAX || K < 256 || K % 256 || ntok < 1 || (fmt != CKQ_FMT_Q4_K && fmt != CKQ_FMT_Q5_K && fmt != CKQ_FMT_Q6_K)) return CKQ_EINVAL;
    return group_route(fmt, n, rows, K, ntok);
}

static int launch_rows16_one(int fmt, const GemvArgs &a, bool tiles, int K, hipStream_t s)
{
    Rows16Args r = {};
    r.tree = !tiles;
    r.M = a.ntok; r.nb = K / 256; r.n = 1;
    r.p[0] = {a.W, a.X, a.y, a.bias, a.ldy, a.nrows, 0, rows16_chains(fmt, a.ntok, a.nrows, K, tiles)};
    return launch_gemm_rows16(fmt, r, s);
}

static const GemvGroup k_no_group = {{}, {}, {}, {}, {}, {}, 1};

static int launch_gemv_args(int fmt, GemvArgs &a, const GemvGroup &grp, int K, void *stream, const GemmOpts &opts = GemmOpts{});

/* `subdots`, when non-NULL, selects the dump build of the streaming kernel's
 * instantiation for these sizes: out[(t * nrows + row) * nsub + i], nothing
 * is written to y. */
extern "C" int ckq_launch_gemv(int fmt, float *y, const void *W, const void *X, const float *bias,
                               int nrows, int K, int ntok, long ldy, int row0, int row1,
                               int32_t *subdots, void *stream)
{
    if ((!y && !subdots) || !W || !X || nrows <= 0 || K <= 0 || ntok <= 0) return CKQ_EINVAL;
    if (row0 < 0) row0 = 0;
    if (row1 > nrows) row1 = nrows;
    if (row0 >= row1) return 0;
    if (subdots && ntok > CKQ_STREAM_TOKENS) return CKQ_EINVAL;
    GemvArgs a = {};
    a.y = y; a.W = (const uint8_t *)W; a.X = (const uint8_t *)X; a.bias = bias; a.sub = subdots;
    a.nrows = nrows; a.ntok = ntok; a.row0 = row0; a.row1 = row1; a.ldy = ldy;
    return launch_gemv_args(fmt, a, k_no_group, K, stream);
}

/* `n` (2..CKQ_GROUP_MAX) independent matmuls of one format and input width,
 * each with its own number of rows - the Q/K/V (grouped-query attention makes
 * K and V narrower than Q) or the gate/up projections of a token - as one
 * launch of the streaming kernel: the launches' fixed start-up cost is paid
 * once and the chip holds n times the loads in flight.  Up to eight tokens; a
 * token tile too large for LDS is issued as separate launches.  `subdots`,
 * when non-NULL, runs the dump build of the grouped instantiation instead:
 * out[((g * ntok + t) * max_rows + row) * nsub + i]. */
extern "C" int ckq_launch_gemv_group(int fmt, int n, float *const *y, const void *const *W, const void *const *X,
                                     const float *const *bias, const int *rows, const long *ldys, int K, int ntok,
                                     int32_t *subdots, void *stream)
{
    if (n < 1 || n > CKQ_GROUP_MAX || !W || !X || !rows || K <= 0 || ntok < 1 || ntok > CKQ_STREAM_TOKENS)
        return CKQ_EINVAL;
    if (!subdots && (!y || !ldys)) return CKQ_EINVAL;
    int nrows = 0;                                  /* the grid and the launch shape follow the largest problem */
    for (int i = 0; i < n; ++i) {
        if (rows[i] <= 0) return CKQ_EINVAL;
        if (rows[i] > nrows) nrows = rows[i];
    }
    for (int i = 0; i < n && !subdots; ++i)
        if (ldys[i] < rows[i] || ldys[i] > 0x7fffffff || !y[i]) return CKQ_EINVAL;
    for (int i = 0; i < n; ++i)
        if (!W[i] || !X[i]) return CKQ_EINVAL;
    /* K-quants: one choice for all matrices */
    const bool kquant = !subdots && (fmt == CKQ_FMT_Q4_K || fmt == CKQ_FMT_Q5_K || fmt == CKQ_FMT_Q6_K) && K % 256 == 0;
    if (kquant && n > 1 && group_route(fmt, n, rows, K, ntok) == CKQ_ROUTE_ROWS16_STREAM) {
        Rows16Args r = {};
        r.M = ntok; r.nb = K / 256; r.tree = true; r.n = n;
        for (int i = 0; i < n; ++i) r.p[i] = {(const uint8_t *)W[i], (const uint8_t *)X[i], y[i], bias ? bias[i] : nullptr, ldys[i], rows[i], 0, {}};
        return launch_gemm_rows16(fmt, r, (hipStream_t)stream);
    }
    /* Every grouped kernel stages its token tile in LDS.  A tile that does not
     * fit (the tile is the token count rounded up to 1, 2, 4 or 8 rows of
     * activations) goes out as n separate launches, which stream it instead. */
    if (n == 1 || !group_tile_fits_lds(fmt, K, ntok)) {
        if (subdots) return CKQ_EINVAL;
        for (int i = 0; i < n; ++i) {
            const int rc = ckq_launch_gemv(fmt, y[i], W[i], X[i], bias ? bias[i] : nullptr, rows[i], K, ntok, ldys[i], 0,
                                           rows[i], nullptr, stream);
            if (rc) return rc;
        }
        return 0;
    }
    auto launch_some = [&](const int *which, int count) {
        float *sy[CKQ_GROUP_MAX];
        const void *sW[CKQ_GROUP_MAX], *sX[CKQ_GROUP_MAX];
        const float *sb[CKQ_GROUP_MAX];
        int srows[CKQ_GROUP_MAX];
        long sld[CKQ_GROUP_MAX];
        for (int i = 0; i < count; ++i) {
            const int k = which[i];
            sy[i] = y[k]; sW[i] = W[k]; sX[i] = X[k]; sb[i] = bias ? bias[k] : nullptr; srows[i] = rows[k]; sld[i] = ldys[k];
        }
        return ckq_launch_gemv_group(fmt, count, sy, sW, sX, sb, srows, sld, K, ntok, nullptr, stream);
    };
    /* Q8_0 rows of an even number of blocks: matrices that start on a dword and ones that do not run different kernels */
    if (!subdots && fmt == CKQ_FMT_Q8_0 && K % 64 == 0) {
        int on[CKQ_GROUP_MAX], off[CKQ_GROUP_MAX], non = 0, noff = 0;
        for (int i = 0; i < n; ++i) {
            if ((uintptr_t)W[i] % 4 == 0) on[non++] = i;
            else off[noff++] = i;
        }
        if (non && noff) {
            const int rc = launch_some(on, non);
            return rc ? rc : launch_some(off, noff);
        }
    }
    GemvArgs a = {};
    GemvGroup grp = k_no_group;
    a.y = subdots ? nullptr : y[0]; a.W = (const uint8_t *)W[0]; a.X = (const uint8_t *)X[0];
    a.bias = bias && !subdots ? bias[0] : nullptr; a.sub = subdots;
    a.nrows = nrows; a.ntok = ntok; a.row0 = 0; a.row1 = rows[0]; a.ldy = subdots ? nrows : ldys[0];
    for (int i = 1; i < n; ++i) {
        grp.y[i - 1] = subdots ? nullptr : y[i]; grp.W[i - 1] = (const uint8_t *)W[i]; grp.X[i - 1] = (const uint8_t *)X[i];
        grp.bias[i - 1] = bias && !subdots ? bias[i] : nullptr;
        grp.nrows[i - 1] = rows[i];
        grp.ldy[i - 1] = subdots ? nrows : (int)ldys[i];
    }
    grp.n = n;
    return launch_gemv_args(fmt, a, grp, K, stream);
}

extern "C" int ckq_launch_gemv_pro(int fmt, int n, float *const *y, const void *const *W, const float *const *bias, const int *rows, const long *ldys,
                                   int K, int ntok, const float *x, const float *gamma, float eps, long stride, void *xq, void *stream)
{
    if (n < 1 || n > CKQ_GROUP_MAX || ntok < 1 || ntok > CKQ_STREAM_TOKENS || K < 256 || K > 2048 || K % 256 || stride < K || stride % 4) return CKQ_ENOGROUP;
    const size_t wblock = fmt == CKQ_FMT_Q4_K ? 144 : fmt == CKQ_FMT_Q5_K ? 176 : fmt == CKQ_FMT_Q6_K ? 210 : 0;
    if (!wblock || !x || !xq) return CKQ_ENOGROUP;
    /* The 16-row tiles want quantized activations: the producer's launch and theirs.  At five to eight tokens this kernel streams the weights for two tiles of tokens, and where they beat ONE
     * streaming launch they are no slower with the producer: of 867 launches of 256 to 2048 columns that could be joined 7 yield, in two launches 0.74 to 1.00 of the joined time.  (40 more would be 3 to
     * 24 % faster in two, most of them rows of one block; longer rows of the same models are past PRO_UNITS.)  Whole layers of 512 to 2048 columns, 5 to 8 tokens, against a choice by matrix: 0.945 on
     * average, the slowest two of 300 1.02 and 1.01. */
    const bool as_one = rows16_as_one(fmt, ntok, K);
    if (as_one && ntok > 4 && group_takes_rows16(fmt, ntok, n, rows, K, true, false)) return CKQ_ENOGROUP;
    const size_t xbytes = ((size_t)(ntok - 1) * (size_t)stride + (size_t)K) * 4, qbytes = (size_t)ntok * (size_t)(K / 256) * 292;
    if (ckq_ranges_overlap(xq, qbytes, x, xbytes) || (gamma && ckq_ranges_overlap(xq, qbytes, gamma, (size_t)K * 4))) return CKQ_ENOGROUP;
    GemvArgs a = {};
    GemvGroup grp = k_no_group;
    for (int i = 0; i < n; ++i) {
        if (!y[i] || !W[i] || rows[i] <= 0 || ldys[i] < rows[i] || ldys[i] > 0x7fffffff || (!as_one && take_rows16(fmt, ntok, (size_t)rows[i], K, false))) return CKQ_ENOGROUP;
        /* every block reads x: nothing it is made of may be written by the launch before the last has, nor xq read */
        const size_t ybytes = ((size_t)(ntok - 1) * (size_t)ldys[i] + (size_t)rows[i]) * 4;
        if (ckq_ranges_overlap(y[i], ybytes, x, xbytes) || (gamma && ckq_ranges_overlap(y[i], ybytes, gamma, (size_t)K * 4)) || ckq_ranges_overlap(y[i], ybytes, xq, qbytes) ||
            ckq_ranges_overlap(xq, qbytes, W[i], (size_t)rows[i] * (size_t)(K / 256) * wblock) || (bias[i] && ckq_ranges_overlap(xq, qbytes, bias[i], (size_t)rows[i] * 4)))
            return CKQ_ENOGROUP;
        if (rows[i] > a.nrows) a.nrows = rows[i];
        if (i) {
            grp.y[i - 1] = y[i]; grp.W[i - 1] = (const uint8_t *)W[i]; grp.bias[i - 1] = bias[i]; grp.nrows[i - 1] = rows[i]; grp.ldy[i - 1] = (int)ldys[i];
        }
    }
    grp.n = n;
    a.y = y[0]; a.W = (const uint8_t *)W[0]; a.bias = bias[0]; a.ntok = ntok; a.row1 = rows[0]; a.ldy = ldys[0];
    a.npos = K / 64; a.wrow = (long)((size_t)(K / 256) * wblock); a.xrow = (long)(K / 256) * 292;
    const GemvPro pro = {x, gamma, (uint8_t *)xq, stride, eps};
    return fmt == CKQ_FMT_Q4_K ? ckq_gemv_pro_launch_q4k(a, grp, pro, (hipStream_t)stream) : fmt == CKQ_FMT_Q5_K ? ckq_gemv_pro_launch_q5k(a, grp, pro, (hipStream_t)stream)
         : ckq_gemv_pro_launch_q6k(a, grp, pro, (hipStream_t)stream);
}

static int launch_gemv_args(int fmt_flags, GemvArgs &a, const GemvGroup &grp, int K, void *stream, const GemmOpts &opts)
{
    int fmt = fmt_flags;
    float *const y = a.y;
    const void *const W = a.W, *const X = a.X;
    const float *const bias = a.bias;
    const int nrows = a.nrows, ntok = a.ntok, row0 = a.row0, row1 = a.row1;
    const long ldy = a.ldy;
    hipStream_t s = (hipStream_t)stream;
    const bool dump = a.sub != nullptr;
    const bool whole = !dump && grp.n == 1 && row0 == 0 && row1 == nrows;   /* what a matrix-core GEMM can take */
    const bool aligned = weights_dword_aligned(a, grp);
    const int route = whole ? launch_route(fmt, nrows, K, ntok, aligned, opts.scratch != nullptr) : CKQ_ROUTE_STREAM;
    switch (fmt) {
    case CKQ_FMT_Q4_K:
        if (K % 256) return CKQ_ESHAPE;
        if (route == CKQ_ROUTE_ROWS16_STREAM || route == CKQ_ROUTE_ROWS16_TILES) return launch_rows16_one(fmt, a, route == CKQ_ROUTE_ROWS16_TILES, K, s);
        if (route == CKQ_ROUTE_TILES) return launch_gemm_q4k_mfma(X, W, bias, y, ntok, nrows, K, ldy, opts, s);
        a.npos = K / 64; a.wrow = (long)(K / 256) * 144; a.xrow = (long)(K / 256) * 292; a.nsub_row = K / 32;
        return ckq_gemv_launch_q4k(a, grp, s);
    case CKQ_FMT_Q5_K:
        if (K % 256) return CKQ_ESHAPE;
        if (route == CKQ_ROUTE_ROWS16_STREAM || route == CKQ_ROUTE_ROWS16_TILES) return launch_rows16_one(fmt, a, route == CKQ_ROUTE_ROWS16_TILES, K, s);
        if (route == CKQ_ROUTE_TILES) return launch_gemm_q5k_mfma(X, W, bias, y, ntok, nrows, K, ldy, opts, s);
        a.npos = K / 64; a.wrow = (long)(K / 256) * 176; a.xrow = (long)(K / 256) * 292; a.nsub_row = K / 32;
        return ckq_gemv_launch_q5k(a, grp, s);
    case CKQ_FMT_Q6_K:
        if (K % 256) return CKQ_ESHAPE;
        if (route == CKQ_ROUTE_ROWS16_STREAM || route == CKQ_ROUTE_ROWS16_TILES) return launch_rows16_one(fmt, a, route == CKQ_ROUTE_ROWS16_TILES, K, s);
        if (route == CKQ_ROUTE_TILES) return launch_gemm_q6k_mfma(X, W, bias, y, ntok, nrows, K, ldy, opts, s);
        a.npos = K / 64; a.wrow = (long)(K / 256) * 210; a.xrow = (long)(K / 256) * 292; a.nsub_row = K / 16;
        return ckq_gemv_launch_q6k(a, grp, s);
    case CKQ_FMT_Q8_0:
        if (K % 32) return CKQ_ESHAPE;
        if (route == CKQ_ROUTE_TILES) return launch_gemm_q80_mfma(X, W, bias, y, ntok, nrows, K, ldy, opts, s);
        a.wrow = (long)(K / 32) * 34; a.xrow = (long)(K / 32) * 34; a.nsub_row = K / 32;
        /* rows of an even number of blocks at dword-aligned addresses: two blocks per position, aligned loads */
        if (K % 64 == 0 && aligned) {
            a.npos = K / 64;
            return ckq_gemv_launch_q80p(a, grp, s);
        }
        a.npos = K / 32;
        return ckq_gemv_launch_q80(a, grp, s);
    case CKQ_FMT_Q5_0:
        if (K % 32) return CKQ_ESHAPE;
        /* prefill: the blocks are rewritten as Q8_0 blocks (same scale, values
         * q - 16: every dot product is unchanged) and go to the Q8_0 GEMM */
        if (route == CKQ_ROUTE_TILES) {
            if (opts.scratch) return CKQ_ESCRATCH;       /* the rewritten weights would need an allocation */
            return launch_gemm_q50_via_q80(X, W, bias, y, ntok, nrows, K, ldy, s);
        }
        a.npos = K / 32; a.wrow = (long)(K / 32) * 22; a.xrow = (long)(K / 32) * 34; a.nsub_row = K / 32;
        return ckq_gemv_launch_q50(a, grp, s);
    case CKQ_KERNEL_Q80_F32:
        if (K % 32) return CKQ_ESHAPE;
        if (dump || grp.n > 1) return CKQ_EINVAL;
        if (route == CKQ_ROUTE_TILES) return launch_gemm_f32act(fmt, (const float *)X, W, bias, y, ntok, nrows, K, ldy, s);
        a.npos = K / 32; a.wrow = (long)(K / 32) * 34; a.xrow = (long)K * 4; a.nsub_row = K / 32;
        return ckq_gemv_launch_q80_f32(a, grp, s);
    case CKQ_KERNEL_Q4K_F32:
        if (K % 256) return CKQ_ESHAPE;
        if (dump || grp.n > 1) return CKQ_EINVAL;
        if (route == CKQ_ROUTE_TILES) return launch_gemm_f32act(fmt, (const float *)X, W, bias, y, ntok, nrows, K, ldy, s);
        a.npos = K / 64; a.wrow = (long)(K / 256) * 144; a.xrow = (long)K * 4; a.nsub_row = K / 64;
        return ckq_gemv_launch_q4k_f32(a, grp, s);
    case CKQ_KERNEL_Q6K_F32:
        if (K % 256) return CKQ_ESHAPE;
        if (dump || grp.n > 1) return CKQ_EINVAL;
        if (route == CKQ_ROUTE_TILES) return launch_gemm_f32act(fmt, (const float *)X, W, bias, y, ntok, nrows, K, ldy, s);
        a.npos = K / 64; a.wrow = (long)(K / 256) * 210; a.xrow = (long)K * 4; a.nsub_row = K / 64;
        return ckq_gemv_launch_q6k_f32(a, grp, s);
    default:
        return CKQ_EFORMAT;
    }
}

/* Several weight matrices of one format against the same quantized activations (Q/K/V, gate/up at
 * prefill sizes) as ONE matrix-core launch: the tiles of all matrices share a grid, so the narrow ones
 * (K and V under grouped-query attention) fill the chip together with the wide one instead of each
 * taking a K-split launch of its own, and one launch boundary replaces n.  Every tile is computed
 * exactly as the single-matrix launch without a K split computes it.  CKQ_ENOGROUP: not taken (the
 * streaming kernel would serve these sizes, or the tiles of all matrices together still leave most of
 * the chip idle); the caller then issues the matrices one by one. */
extern "C" int ckq_launch_gemm_group(int fmt, int n, float *const *C, const void *const *B, const void *A,
                                     const float *const *bias, const int *N, const long *ldc, int K, int M, void *stream)
{
    if (n < 2 || n > GEMM_GROUP_MAX || M <= CKQ_STREAM_TOKENS || !A || K <= 0) return CKQ_ENOGROUP;
    GemmGroupIn in = {};
    in.n = n;
    size_t rows = 0;
    bool aligned = true;
    for (int p = 0; p < n; ++p) {
        if (!C[p] || !B[p] || N[p] <= 0 || ldc[p] < N[p]) return CKQ_EINVAL;
        in.B[p] = B[p]; in.bias[p] = bias ? bias[p] : nullptr; in.C[p] = C[p]; in.N[p] = N[p]; in.ldc[p] = ldc[p];
        rows += (size_t)N[p];
        aligned = aligned && ((uintptr_t)B[p] % 4 == 0);
    }
    hipStream_t s = (hipStream_t)stream;
    if ((fmt == CKQ_FMT_Q4_K || fmt == CKQ_FMT_Q5_K || fmt == CKQ_FMT_Q6_K) && K % 256 == 0) {
        GemmChains shared = {};
        bool grouped;
        const int route = kquant_group_route(fmt, in, M, K, &grouped, &shared);
        if (route == CKQ_ROUTE_ROWS16_TILES || route == CKQ_ROUTE_ROWS16_STREAM) {
            const bool tiles = route == CKQ_ROUTE_ROWS16_TILES;
            Rows16Args r = {};
            r.M = M; r.nb = K / 256; r.n = n; r.tree = !tiles;
            for (int p = 0; p < n; ++p)
                r.p[p] = {(const uint8_t *)B[p], (const uint8_t *)A, C[p], bias ? bias[p] : nullptr, ldc[p], N[p], 0,
                          grouped ? shared : rows16_chains(fmt, M, N[p], K, tiles)};
            return launch_gemm_rows16(fmt, r, s);
        }
        if (route == CKQ_ENOGROUP) return CKQ_ENOGROUP;
    }
    switch (fmt) {
    case CKQ_FMT_Q4_K:
        if (K % 256) return CKQ_ESHAPE;
        return launch_gemm_q4k_mfma_group(A, in, M, K, s);
    case CKQ_FMT_Q5_K:
        if (K % 256) return CKQ_ESHAPE;
        return launch_gemm_q5k_mfma_group(A, in, M, K, s);
    case CKQ_FMT_Q6_K:
        if (K % 256) return CKQ_ESHAPE;
        return launch_gemm_q6k_mfma_group(A, in, M, K, s);
    case CKQ_FMT_Q8_0:
        if (K % 32) return CKQ_ESHAPE;
        if (!gemm_q80_on_matrix_cores(M, rows * (K / 32) * 34, K % 64 == 0 && aligned)) return CKQ_ENOGROUP;
        return launch_gemm_q80_mfma_group(A, in, M, K, s);
    default:
        return CKQ_ENOGROUP;
    }
}

/* ---- the entry point that allocates nothing ---------------------------------
 * Scratch for the partial tiles of a K-split GEMM, held in the code object:
 * every device the library runs on holds its own copy, at its own address,
 * until the process ends.  Host code never uses the array's name as an
 * address: the per-device address comes from hipGetSymbolAddress, once per
 * device, with that device current.  The array keeps the last call's
 * contents; nothing in it has to start at zero (the split kernel writes every
 * partial entry the reduction reads).  Calls that overlap on one GPU race. */
static __device__ __align__(256) unsigned char scratch[CKQ_NOALLOC_SCRATCH_BYTES];
constexpr int CKQ_MAX_DEVICES = 64;
static std::atomic<void *> g_scratch_ptr[CKQ_MAX_DEVICES];

static int noalloc_scratch(void **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return (int)e;
    if (dev < 0 || dev >= CKQ_MAX_DEVICES) return (int)hipErrorInvalidDevice;
    void *p = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return (int)e;
        if (!p) return (int)hipErrorInvalidSymbol;
        g_scratch_ptr[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return 0;
}

extern "C" int ckq_launch_noalloc_setup(void)
{
    void *p;
    return noalloc_scratch(&p);
}

extern "C" int ckq_launch_gemv_noalloc(int fmt, float *y, const void *W, const void *X, const float *bias,
                                       int nrows, int K, int ntok, long ldy, void *stream)
{
    if (fmt != CKQ_FMT_Q4_K && fmt != CKQ_FMT_Q5_K && fmt != CKQ_FMT_Q6_K && fmt != CKQ_FMT_Q8_0) return CKQ_EFORMAT;
    if (!y || !W || !X || nrows <= 0 || K <= 0 || ntok <= 0 || ldy < nrows) return CKQ_EINVAL;
    void *p = nullptr;
    {
        /* The scratch address of this device is normally resolved by ckq_init().  Resolving it
         * here, on a first call, may load the code object, which is not legal while the stream
         * is being captured: such a call is refused instead. */
        int dev = 0;
        if (hipGetDevice(&dev) == hipSuccess && dev >= 0 && dev < CKQ_MAX_DEVICES &&
            !g_scratch_ptr[dev].load(std::memory_order_acquire)) {
            hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
            if (hipStreamIsCapturing((hipStream_t)stream, &st) == hipSuccess && st != hipStreamCaptureStatusNone)
                return (int)hipErrorStreamCaptureUnsupported;
            (void)hipGetLastError();
        }
    }
    const int rc = noalloc_scratch(&p);
    if (rc) return rc;
    GemvArgs a = {};
    a.y = y; a.W = (const uint8_t *)W; a.X = (const uint8_t *)X; a.bias = bias; a.sub = nullptr;
    a.nrows = nrows; a.ntok = ntok; a.row0 = 0; a.row1 = nrows; a.ldy = ldy;
    return launch_gemv_args(fmt, a, k_no_group, K, stream, GemmOpts{nullptr, (float *)p, CKQ_NOALLOC_SCRATCH_BYTES});
}

/* The matrix-core GEMM of `fmt`, whatever the token count, with its integer
 * block sums stored next to the result: sums[((t * N + n) * nblk + b) * per + i],
 * nblk = K / 256 and per = 2 (I1, I2) for Q4_K and Q5_K, per = 1 (I) for Q6_K,
 * nblk = K / 32 and per = 1 (the block dot) for Q8_0.  For the exactness tests. */
extern "C" int ckq_launch_gemm_block_sums(int fmt, const void *A, const void *B, const float *bias, float *C, int32_t *sums,
                                          int M, int N, int K, long ldc, void *stream)
{
    if (!A || !B || !C || !sums || M <= 0 || N <= 0 || K <= 0 || ldc < N) return CKQ_EINVAL;
    hipStream_t s = (hipStream_t)stream;
    switch (fmt) {
    case CKQ_FMT_Q4_K: return K % 256 ? CKQ_ESHAPE : launch_gemm_q4k_mfma(A, B, bias, C, M, N, K, ldc, GemmOpts{sums, nullptr, 0}, s);
    case CKQ_FMT_Q5_K: return K % 256 ? CKQ_ESHAPE : launch_gemm_q5k_mfma(A, B, bias, C, M, N, K, ldc, GemmOpts{sums, nullptr, 0}, s);
    case CKQ_FMT_Q6_K: return K % 256 ? CKQ_ESHAPE : launch_gemm_q6k_mfma(A, B, bias, C, M, N, K, ldc, GemmOpts{sums, nullptr, 0}, s);
    case CKQ_FMT_Q8_0: return K % 32 ? CKQ_ESHAPE : launch_gemm_q80_mfma(A, B, bias, C, M, N, K, ldc, GemmOpts{sums, nullptr, 0}, s);
    default: return CKQ_EFORMAT;
    }
}

/* ========================================================================= */
/* Activation quantizers                                                      */
/* ========================================================================= */

/* fp32 -> Q8_K, one wave per 256-element block, lane l owns elements 4l..4l+3
 * (q8k_quantize_block holds the reference's rules).  SWIGLU: the quantizer's
 * input is SiLU(x) * up instead of x.  Rows of the input are ldx floats apart,
 * bpr blocks of 256 per row.  Bound: memory once rows are many (us, inputs not in the L2: 2048 x 4096 11.1 -> 9.7, SwiGLU 512 x 4864 8.0 -> 7.4,
 * 512 x 11008 13.3 -> 12.2, 2048 x 11008 47.0 -> 43.7 = 4.8 TB/s, when a value's rounding went from six operations to two and
 * block numbers from 64 bits to 32: 219 -> 93 and 366 -> 243 vector instructions), launch and latency below.  Four blocks a wave, sixteen lanes
 * each, their divisions and maxima shared: 9.8, 7.2, 12.7, 40.6, and 3.2 -> 3.7 for SwiGLU 93 x 4864. */
template <bool SWIGLU>
__global__ void __launch_bounds__(256) quantize_q8_k_kernel(const float *__restrict__ x, const float *__restrict__ up,
                                                            uint8_t *__restrict__ y, u32 nblocks, u32 bpr, long ldx)
{
    const u32 blk = blockIdx.x * 4 + (u32)wave_in_block();
    if (blk >= nblocks) return;
    pro_quantize_block<SWIGLU>(x, up, y, blk, bpr, ldx, threadIdx.x & 63);
}

template <bool SWIGLU>
static int launch_quantize_q8_k(const float *x, const float *up, void *y, long nblocks, int bpr, long ldx, hipStream_t s)
{
    if (nblocks > 0x7fffffffl) return CKQ_ESHAPE;
    hipLaunchKernelGGL(quantize_q8_k_kernel<SWIGLU>, dim3((unsigned)((nblocks + 3) / 4)), dim3(256), 0, s, x, up, (uint8_t *)y, (u32)nblocks, (u32)bpr, ldx);
    return (int)hipGetLastError();
}

/*
 * fp32 -> Q8_0, eight lanes per 32-element block (reference:
 * gemm_kernels_q8_0.c:70-146).  d = amax/127 stored as fp16 (RNE);
 * id = amax ? 127/amax : 0; q = RNE(x*id) saturated.
 */
__device__ __forceinline__ void quantize_q8_0_blocks(const float *__restrict__ x, uint8_t *__restrict__ y, long nblocks, u32 block)
{
    const long t = (long)block * 256 + threadIdx.x;
    const long blk = t >> 3;
    const int  j = (int)(t & 7);
    const bool live = blk < nblocks;
    const long b = live ? blk : nblocks - 1;
    const float4 v = reinterpret_cast<const float4 *>(x + b * 32)[j];
    const float e[4] = {v.x, v.y, v.z, v.w};
    float amax = fmaxf(fmaxf(fabsf(e[0]), fabsf(e[1])), fmaxf(fabsf(e[2]), fabsf(e[3])));
    amax = fmaxf(amax, dpp_get<0xB1>(amax));                 /* eight lanes: quad_perm twice, row_half_mirror */
    amax = fmaxf(amax, dpp_get<0x4E>(amax));
    amax = fmaxf(amax, dpp_get<0x141>(amax));
    const float d  = amax / 127.0f;
    const float id = amax != 0.0f ? 127.0f / amax : 0.0f;
    u32 packed[1];
    q8_round(e, id, packed);
    if (!live) return;
    uint8_t *out = y + b * 34;
    uint16_t *o16 = reinterpret_cast<uint16_t *>(out + 2 + 4 * j);   /* 2-byte aligned */
    o16[0] = (uint16_t)packed[0];
    o16[1] = (uint16_t)(packed[0] >> 16);
    if (j == 0) *reinterpret_cast<uint16_t *>(out) = __builtin_bit_cast(uint16_t, (_Float16)d);
}

__global__ void __launch_bounds__(256) quantize_q8_0_kernel(const float *__restrict__ x, uint8_t *__restrict__ y, long nblocks)
{
    quantize_q8_0_blocks(x, y, nblocks, blockIdx.x);
}

/* Both of what a Q5_0 matmul on the matrix cores waits for: weights rewritten as Q8_0 blocks (the first `wgrid` blocks, the longer part) and
 * activations quantized.  Neither fills the chip, and neither needs the other: two launches of 5.4 and 2.9 us in one of about 6 (512 tokens, 9728 x 896). */
__global__ void __launch_bounds__(256) q5_0_operands_kernel(const uint8_t *__restrict__ W, uint8_t *__restrict__ W8, size_t wblocks, u32 wgrid,
                                                            const float *__restrict__ x, uint8_t *__restrict__ xq, long xblocks)
{
    if (blockIdx.x < wgrid) {
        const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
        if (i < wblocks) q5_0_to_q8_0_block(W, W8, i);
    } else
        quantize_q8_0_blocks(x, xq, xblocks, blockIdx.x - wgrid);
}

extern "C" int ckq_launch_quantize_q8_k(const float *x, void *y, int rows, int k, void *stream)
{
    if (!x || !y || rows <= 0 || k <= 0) return CKQ_EINVAL;
    if (k % 256) return CKQ_ESHAPE;
    const long nblocks = (long)rows * (k / 256);
    return launch_quantize_q8_k<false>(x, nullptr, y, nblocks, k / 256, (long)k, (hipStream_t)stream);
}

/* y[row] = Q8_K(SiLU(gate[row]) * up[row]), rows of gate and up ld floats apart. */
extern "C" int ckq_launch_swiglu_q8_k(const float *gate, const float *up, void *y, int rows, int k, long ld, void *stream)
{
    if (!gate || !up || !y || rows <= 0 || k <= 0 || ld < k) return CKQ_EINVAL;
    if (k % 256 || ld % 4 || ((uintptr_t)gate | (uintptr_t)up) % 16) return CKQ_ESHAPE;
    const long nblocks = (long)rows * (k / 256);
    return launch_quantize_q8_k<true>(gate, up, y, nblocks, k / 256, ld, (hipStream_t)stream);
}

extern "C" int ckq_launch_quantize_q8_0(const float *x, void *y, int rows, int k, void *stream)
{
    if (!x || !y || rows <= 0 || k <= 0) return CKQ_EINVAL;
    if (k % 32) return CKQ_ESHAPE;
    const long nblocks = (long)rows * (k / 32);
    hipLaunchKernelGGL(quantize_q8_0_kernel, dim3((unsigned)((nblocks * 8 + 255) / 256)), dim3(256), 0,
                       (hipStream_t)stream, x, (uint8_t *)y, nblocks);
    return (int)hipGetLastError();
}

/* y = x W^T with x quantized to Q8_0 at xq on the way, as ckq_launch_quantize_q8_0 and ckq_launch_gemv one after the other give it. */
extern "C" int ckq_launch_quantize_gemv_q8_0(int fmt, const float *x, void *xq, float *y, const void *W, const float *bias, int nrows, int K, int ntok, long ldy, void *stream)
{
    const size_t wblocks = (size_t)nrows * (size_t)(K / 32);
    const long xblocks = (long)ntok * (K / 32);
    const unsigned wgrid = (unsigned)((wblocks + 255) / 256), xgrid = (unsigned)((xblocks * 8 + 255) / 256);
    if (fmt != CKQ_FMT_Q5_0 || !x || !xq || !y || !W || nrows <= 0 || K <= 0 || K % 32 || ntok <= 0 || (wblocks + 255) / 256 + (size_t)xgrid > 0x7fffffffu ||
        ckq_launch_route(fmt, nrows, K, ntok, 1) != CKQ_ROUTE_TILES) {
        const int rc = ckq_launch_quantize_q8_0(x, xq, ntok, K, stream);
        return rc ? rc : ckq_launch_gemv(fmt, y, W, xq, bias, nrows, K, ntok, ldy, 0, nrows, nullptr, stream);
    }
    hipStream_t const s = (hipStream_t)stream;
    std::lock_guard<std::recursive_mutex> lock(g_split_mu);   /* the scratch is shared by launches on this stream */
    float *tmp = nullptr;
    int rc = gemm_workspace(1, s, wblocks * 34, &tmp);
    if (rc) return rc;
    hipLaunchKernelGGL(q5_0_operands_kernel, dim3(wgrid + xgrid), dim3(256), 0, s, (const uint8_t *)W, (uint8_t *)tmp, wblocks, wgrid, x, (uint8_t *)xq, xblocks);
    rc = (int)hipGetLastError();
    return rc ? rc : launch_gemm_q80_mfma(xq, tmp, bias, y, ntok, nrows, K, ldy, GemmOpts{}, s);
}

/*
 * Fused producer RMSNorm -> Q8_K, one block per token (the arithmetic is rms_row's, ckq_producers.hpp).  A single row is
 * a chain of latencies: its load, the serial sum of squares, the block maximum.  The sum reads 16 bytes at a time, the
 * maximum goes through DPP, and x stays in registers: 4096 wide, one row 5.1 -> 4.2 us, 512 rows 7.1 -> 6.0,
 * 2048 rows 23.3 -> 12.1.
 */
template <int GREG, bool AHEAD>
__global__ void __launch_bounds__(1024) rmsnorm_q8_k_fused_kernel(const float *__restrict__ input, const float *__restrict__ gamma,
                                                                  uint8_t *__restrict__ y, int d_model, long in_stride, float eps)
{
    extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
    rms_row<GREG, AHEAD>(input + (size_t)blockIdx.x * in_stride, gamma, y + (size_t)blockIdx.x * (d_model / 256) * 292,
                  d_model, eps, reinterpret_cast<float *>(smem));
}

template <int GREG, bool AHEAD>
static int launch_rms_form(const float *input, const float *gamma, uint8_t *y, int tokens, int d_model, long stride, float eps, int waves, hipStream_t s)
{
    const size_t lds = rms_lds_bytes((size_t)d_model);
    if (lds > 64 * 1024) {
        /* more than 64 KB of dynamic LDS is an opt-in per function and per device: set on every
         * such call for the device that is current (rows this long are rare; the call is cheap) */
        hipError_t e = hipFuncSetAttribute((const void *)rmsnorm_q8_k_fused_kernel<GREG, AHEAD>,
                                           hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return (int)e;
    }
    hipLaunchKernelGGL((rmsnorm_q8_k_fused_kernel<GREG, AHEAD>), dim3((unsigned)tokens), dim3(64 * waves), lds, s, input, gamma, y, d_model, stride, eps);
    return (int)hipGetLastError();
}
template <int GREG>
static int launch_rms(const float *input, const float *gamma, uint8_t *y, int tokens, int d_model, long stride, float eps, int waves, hipStream_t s)
{
    return tokens <= 512 ? launch_rms_form<GREG, true>(input, gamma, y, tokens, d_model, stride, eps, waves, s)
                         : launch_rms_form<GREG, false>(input, gamma, y, tokens, d_model, stride, eps, waves, s);
}

extern "C" int ckq_launch_rmsnorm_q8_k_fused(const float *input, const float *gamma, void *y, int tokens, int d_model,
                                             int aligned_embed_dim, float eps, void *stream)
{
    if (!input || !gamma || !y || tokens <= 0 || d_model <= 0 || aligned_embed_dim < d_model) return CKQ_EINVAL;
    if (d_model % 256 || aligned_embed_dim % 4) return CKQ_ESHAPE;
    if (rms_lds_bytes((size_t)d_model) > 160 * 1024) return CKQ_ESHAPE;        /* the row is staged in LDS */
    /* A wave for every 256-block of the row, up to sixteen while a row has a CU to itself, up to eight for two and four rows on a CU, whose chains
     * then run side by side.  More rows take four waves each, so that more of them fit, unless their image in LDS leaves room for four anyway (8192 and wider).  The
     * chains read ahead up to two rows a CU.  us, up to 512 rows sixteen waves without reading ahead -> eight with it: 4096 wide 300 rows 6.6 -> 6.2,
     * 512 rows 7.1 -> 6.5, 8192 wide 512 rows 11.8 -> 11.1, 2048 wide 4.4 -> 4.2; beyond, four -> eight: 700 rows, 4096 wide 7.9 -> 7.6, 8192 wide
     * 15.7 -> 13.1, 2048 rows of 8192 32.2 -> 28.1 (eight: of 4096 13.7 -> 15.0, 1500 rows of 6144 17.0 -> 17.8). */
    const int nb = d_model / 256, most = tokens <= 256 ? 16 : tokens <= 1024 || nb >= 32 ? 8 : 4, waves = nb < most ? nb : most, per = (nb + waves - 1) / waves;
    uint8_t *const out = (uint8_t *)y;
    hipStream_t const s = (hipStream_t)stream;
    if (per == 1) return launch_rms<1>(input, gamma, out, tokens, d_model, (long)aligned_embed_dim, eps, waves, s);
    if (per == 2) return launch_rms<2>(input, gamma, out, tokens, d_model, (long)aligned_embed_dim, eps, waves, s);
    return launch_rms<4>(input, gamma, out, tokens, d_model, (long)aligned_embed_dim, eps, waves, s);
}

/* ========================================================================= */
/* Row dequantizers and quantized embedding lookup                            */
/* ========================================================================= */

/* Elements of a quantized row with the reference's operation order; products and differences are rounded one by one
 * (reference: dequant_kernels.c:276-296 Q8_0, :336-385 Q4_K, :396-430 Q6_K).  A thread takes unit `u` of the row, RUNS runs of
 * four elements: run i is elements at(u, i) .. + 3. */
template <int FMT, int RUNS> struct DequantUnit;

template <> struct DequantUnit<CKQ_FMT_Q8_0, 1> {
    static __device__ __forceinline__ u32 at(u32 u, int) { return 4 * u; }
    static __device__ __forceinline__ void get(float4 (&v)[1], const uint8_t *row, u32 u)
    {
#pragma clang fp contract(off)
        const uint8_t *blk = row + (u >> 3) * 34u;
        const float d = h2f(ld2(blk));
        const u32 q = ld4<2>(blk + 2 + 4 * (u & 7));
        v[0] = make_float4(d * (float)sbyte(q, 0), d * (float)sbyte(q, 1), d * (float)sbyte(q, 2), d * (float)sbyte(q, 3));
    }
};

template <> struct DequantUnit<CKQ_FMT_Q4_K, 1> {
    static __device__ __forceinline__ u32 at(u32 u, int) { return 4 * u; }
    static __device__ __forceinline__ void get(float4 (&v)[1], const uint8_t *row, u32 u)
    {
#pragma clang fp contract(off)
        const uint8_t *blk = row + (u >> 6) * 144u;
        const u32 j = (u >> 3) & 7, l = 4 * (u & 7);         /* sub-block j, element l of it */
        const u32 hdr0 = ld4<4>(blk);
        u32 sc2, mn2;
        k4_scale_pair(ld4<4>(blk + 4), ld4<4>(blk + 8), ld4<4>(blk + 12), (int)(j >> 1), &sc2, &mn2);
        const u32 sc = (sc2 >> (8 * (j & 1))) & 0xff, mn = (mn2 >> (8 * (j & 1))) & 0xff;
        const float dj = h2f(hdr0 & 0xffff) * (float)sc, mj = h2f(hdr0 >> 16) * (float)mn;
        const u32 qs = ld4<4>(blk + 16 + 32 * (j >> 1) + l);
        const u32 nib = (j & 1) ? (qs >> 4) & 0x0f0f0f0fu : qs & 0x0f0f0f0fu;
        v[0] = make_float4(dj * (float)(nib & 0xff) - mj, dj * (float)((nib >> 8) & 0xff) - mj, dj * (float)((nib >> 16) & 0xff) - mj, dj * (float)(nib >> 24) - mj);
    }
};

template <> struct DequantUnit<CKQ_FMT_Q6_K, 1> {
    static __device__ __forceinline__ u32 at(u32 u, int) { return 4 * u; }
    static __device__ __forceinline__ void get(float4 (&v)[1], const uint8_t *row, u32 u)
    {
#pragma clang fp contract(off)
        const uint8_t *blk = row + (u >> 6) * 210u;
        const u32 n = (u >> 5) & 1, r = (u >> 3) & 3, l = 4 * (u & 7);       /* half n, run r, element l */
        const u32 lo = ld4<2>(blk + 64 * n + l + 32 * (r & 1)), hi = ld4<2>(blk + 128 + 32 * n + l);
        const u32 q = ((r >> 1) ? (lo >> 4) & 0x0f0f0f0fu : lo & 0x0f0f0f0fu) | (((hi >> (2 * r)) & 0x03030303u) << 4);
        const float ds = h2f(ld2(blk + 208)) * (float)(int8_t)blk[192 + 8 * n + 2 * r + (l >> 4)];
        v[0] = make_float4(ds * (float)((int)(q & 0xff) - 32), ds * (float)((int)((q >> 8) & 0xff) - 32),
                           ds * (float)((int)((q >> 16) & 0xff) - 32), ds * (float)((int)(q >> 24) - 32));
    }
};

/* Eight bytes of a 64-element group: their low nibbles are in one sub-block, their high ones in the next. */
template <> struct DequantUnit<CKQ_FMT_Q4_K, 4> {
    static __device__ __forceinline__ u32 at(u32 u, int i) { return 64 * (u >> 2) + 32 * (i >> 1) + 8 * (u & 3) + 4 * (i & 1); }
    static __device__ __forceinline__ void get(float4 (&v)[4], const uint8_t *row, u32 u)
    {
#pragma clang fp contract(off)
        const uint8_t *blk = row + (u >> 4) * 144u;
        const u32 g = (u >> 2) & 3;
        u32 h[4], qs[2], sc2, mn2;
        ld16<4>(h, blk);
        ld8<4>(qs, blk + 16 + 32 * g + 8 * (u & 3));
        k4_scale_pair(h[1], h[2], h[3], (int)g, &sc2, &mn2);
        const float d = h2f(h[0] & 0xffff), dmin = h2f(h[0] >> 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int odd = i >> 1;
            const float dj = d * (float)((sc2 >> (8 * odd)) & 0xff), mj = dmin * (float)((mn2 >> (8 * odd)) & 0xff);
            const u32 nib = (qs[i & 1] >> (4 * odd)) & 0x0f0f0f0fu;
            v[i] = make_float4(dj * (float)(nib & 0xff) - mj, dj * (float)((nib >> 8) & 0xff) - mj, dj * (float)((nib >> 16) & 0xff) - mj, dj * (float)(nib >> 24) - mj);
        }
    }
};

/* Four bytes of the high bits of a 128-element half and what belongs to them: one run in each of its four runs of 32. */
template <> struct DequantUnit<CKQ_FMT_Q6_K, 4> {
    static __device__ __forceinline__ u32 at(u32 u, int i) { return 128 * (u >> 3) + 32 * i + 4 * (u & 7); }
    static __device__ __forceinline__ void get(float4 (&v)[4], const uint8_t *row, u32 u)
    {
#pragma clang fp contract(off)
        const uint8_t *blk = row + (u >> 4) * 210u;
        const u32 n = (u >> 3) & 1, l = 4 * (u & 7);
        const u32 lo[2] = {ld4<2>(blk + 64 * n + l), ld4<2>(blk + 64 * n + l + 32)}, hi = ld4<2>(blk + 128 + 32 * n + l);
        u32 sc[2];
        ld8<2>(sc, blk + 192 + 8 * n);
        const float d = h2f(ld2(blk + 208));
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const u32 q = ((lo[r & 1] >> (4 * (r >> 1))) & 0x0f0f0f0fu) | (((hi >> (2 * r)) & 0x03030303u) << 4);
            const float ds = d * (float)(int)__builtin_amdgcn_sbfe((int)sc[r >> 1], 16 * (r & 1) + 8 * (l >> 4), 8);
            v[r] = make_float4(ds * (float)((int)(q & 0xff) - 32), ds * (float)((int)((q >> 8) & 0xff) - 32),
                               ds * (float)((int)((q >> 16) & 0xff) - 32), ds * (float)((int)(q >> 24) - 32));
        }
    }
};

/*
 * out[t][0..n_row) for t < n_out_rows: rows t < tokens hold the dequantized
 * source row (ids ? clamp(ids[t]) : t), plus pos[t] where asked, zero from
 * n_valid on; rows from `tokens` on are zero (reference:
 * src/kernels/embedding_kernels.c:76-196).  Bound: two latencies, the id's and its row's, and the stores.
 */
template <int FMT, int RUNS>
__global__ void __launch_bounds__(256) dequant_rows_kernel(const uint8_t *__restrict__ table, const int32_t *__restrict__ ids,
                                                           const float *__restrict__ pos, float *__restrict__ out, int vocab,
                                                           int n_valid, int n_row, u32 row_bytes, int tokens, int n_out_rows, u32 col_blocks, u32 width)
{
    typedef DequantUnit<FMT, RUNS> Unit;
    /* The output row rides in blockIdx.x with the column block (gridDim.y stops at 65 535 rows).  All blocks of row t go to XCD t % 8, blocks going round
     * the XCDs in turn, as block t of a launch with a block a row does: the norm that reads the rows finds them in its L2 (lookup and norm on an idle GPU,
     * us with the host's part, blocks in order -> so: Q6_K 512 rows of 4096 24.8 -> 22.4, 256 of 8192 26.4 -> 23.9). */
    const u32 seq = blockIdx.x >> 3;
    const int t = (int)(8 * (seq / col_blocks) + (blockIdx.x & 7));
    const u32 u = (seq % col_blocks) * width + threadIdx.x;
    if (t >= n_out_rows || u >= (u32)n_row / (4 * RUNS)) return;
    float4 v[RUNS];
#pragma unroll
    for (int i = 0; i < RUNS; ++i) v[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t < tokens) {
        int src = t;
        if (ids) {
            const int id = ids[t];
            src = (id < 0 || id >= vocab) ? 0 : id;
        }
        Unit::get(v, table + (size_t)src * row_bytes, u);
#pragma unroll
        for (int i = 0; i < RUNS; ++i) {
            const u32 e = Unit::at(u, i);
            if (pos) {
                const float4 p = *reinterpret_cast<const float4 *>(pos + (size_t)t * n_row + e);
                v[i].x += p.x; v[i].y += p.y; v[i].z += p.z; v[i].w += p.w;
            }
            if (e + 0 >= (u32)n_valid) v[i].x = 0.f;
            if (e + 1 >= (u32)n_valid) v[i].y = 0.f;
            if (e + 2 >= (u32)n_valid) v[i].z = 0.f;
            if (e + 3 >= (u32)n_valid) v[i].w = 0.f;
        }
    }
#pragma unroll
    for (int i = 0; i < RUNS; ++i) *reinterpret_cast<float4 *>(out + (size_t)t * n_row + Unit::at(u, i)) = v[i];
}

/* Elements a thread takes, and the threads of a block: as many as an equal share of the row needs, whole waves.
 * Sixteen elements a thread need a third of the loads but leave a quarter of the threads: they win once a launch of four each, 1024 to a block, has
 * more blocks than the chip holds at once (2048; Q4_K, whose loads are wider as it is, twice that), while a narrow row's sixteens leave lanes of its last wave without work,
 * all but sixteen of a row of 256.  From 130 launches a format of 1 to 40000 rows, 256 to 8192 wide, random ids (us, four -> sixteen): Q6_K 1024 rows of 4096 7.6 -> 6.3,
 * 2048 of 8192 24.3 -> 19.0, 1024 of 2048 4.2 -> 4.3, 3000 of 256 3.1 -> 3.5; Q4_K 1500 of 4096 10.0 -> 9.6, 2048 of 8192 23.5 -> 19.7, 384 of 5120 4.0 -> 4.7, 2048
 * of 1024 4.2 -> 4.7.  The rule's choices are within 1.5 % of the faster form, but for Q4_K 3000 of 1280 (7.2 -> 7.7) and 1024 of 5120 (9.0 -> 9.3).
 * Blocks of 256 threads whatever the row: four a thread 4096 of 256 3.4 -> 3.8, sixteen a thread 1024 of 5120 Q6_K 7.6 -> 9.5. */
extern "C" int ckq_launch_dequant_form(int fmt, int n_row, int n_out_rows, int *width)
{
    const bool q4 = fmt == CKQ_FMT_Q4_K;
    const long long most = n_row <= (q4 ? 1024 : 512) ? 8ll << 20 : q4 ? 4ll << 20 : 2ll << 20;
    const int e = fmt != CKQ_FMT_Q8_0 && n_row >= 512 && (long long)n_row * n_out_rows > most ? 16 : 4;
    const int units = n_row / e, col_blocks = (units + 255) / 256;
    *width = ((units + col_blocks - 1) / col_blocks + 63) & ~63;
    return e;
}

extern "C" int ckq_launch_dequant_rows(int fmt, const void *table, const int32_t *ids, int vocab, const float *pos,
                                       float *out, int n_valid, int n_row, int tokens, int n_out_rows, void *stream)
{
    if (!table || !out || n_row <= 0 || n_out_rows <= 0 || tokens < 0 || n_valid < 0) return CKQ_EINVAL;
    if (fmt != CKQ_FMT_Q4_K && fmt != CKQ_FMT_Q6_K && fmt != CKQ_FMT_Q8_0) return CKQ_EFORMAT;
    if (n_row % (fmt == CKQ_FMT_Q8_0 ? 32 : 256)) return CKQ_ESHAPE;
    if (tokens > n_out_rows) tokens = n_out_rows;
    if (n_valid > n_row) n_valid = n_row;
    const u32 rb = (u32)ckq_row_bytes(fmt, n_row);
    int width;
    const bool wide = ckq_launch_dequant_form(fmt, n_row, n_out_rows, &width) == 16;
    const int col_blocks = (n_row / (wide ? 16 : 4) + 255) / 256;
    const long long blocks = ((long long)n_out_rows + 7) / 8 * 8 * col_blocks;
    if (blocks > 0x7fffffffll) return CKQ_ESHAPE;
    const dim3 grid((unsigned)blocks), block((unsigned)width);
    hipStream_t s = (hipStream_t)stream;
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, block, 0, s, (const uint8_t *)table, ids, pos, out, vocab, n_valid, n_row, rb, tokens, n_out_rows, (u32)col_blocks, (u32)width);
    };
    switch (fmt) {
    case CKQ_FMT_Q4_K: launch(wide ? dequant_rows_kernel<CKQ_FMT_Q4_K, 4> : dequant_rows_kernel<CKQ_FMT_Q4_K, 1>); break;
    case CKQ_FMT_Q6_K: launch(wide ? dequant_rows_kernel<CKQ_FMT_Q6_K, 4> : dequant_rows_kernel<CKQ_FMT_Q6_K, 1>); break;
    default:           launch(dequant_rows_kernel<CKQ_FMT_Q8_0, 1>); break;
    }
    return (int)hipGetLastError();
}

/* ========================================================================= */
/* Streaming copy                                                             */
/* ========================================================================= */
__global__ void __launch_bounds__(256) copy_kernel(uint4 *__restrict__ dst, const uint4 *__restrict__ src, size_t n16)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n16) dst[i] = src[i];
}

/* Reads `n16` 16-byte units and keeps nothing: what one launch costs when it
 * only has to pull that many bytes out of HBM (the floor for a GEMV whose
 * weights are that large). */
typedef unsigned ckq_v4u __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) read_kernel(const ckq_v4u *__restrict__ src, size_t n16, unsigned *sink)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n16) return;
    const ckq_v4u v = __builtin_nontemporal_load(src + i);
    if ((v[0] ^ v[1] ^ v[2] ^ v[3]) == 0x9e3779b9u && v[0] == 0x7f4a7c15u) *sink = v[0];   /* never true in practice */
}

/* The same read as a tuned streaming kernel: a grid sized to what the chip
 * holds at once (`blocks` blocks of 256 threads), every lane keeping U
 * independent 16-byte loads in flight per trip and striding through the buffer,
 * so that neither block dispatch nor a one-load-per-lane dependency limits the
 * rate.  The fastest (blocks, U) the benchmark finds is the launch floor it
 * prices the GEMV against. */
template <int U>
__global__ void __launch_bounds__(256) read_stream_kernel(const ckq_v4u *__restrict__ src, size_t n16, unsigned *sink)
{
    const size_t stride = (size_t)gridDim.x * 256;
    size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    ckq_v4u acc = {0u, 0u, 0u, 0u};
    for (; i + (U - 1) * stride < n16; i += U * stride) {
        ckq_v4u v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = src[i + u * stride];
#pragma unroll
        for (int u = 0; u < U; ++u) acc ^= v[u];
    }
    for (; i < n16; i += stride) acc ^= src[i];
    if ((acc[0] ^ acc[1] ^ acc[2] ^ acc[3]) == 0x9e3779b9u && acc[0] == 0x7f4a7c15u) *sink = acc[0];   /* never true in practice */
}

extern "C" int ckq_launch_read_tuned(const void *src, size_t bytes, void *sink, int blocks, int unroll, void *stream)
{
    if (!src || !sink || bytes < 16 || blocks <= 0) return CKQ_EINVAL;
    const size_t n16 = bytes / 16;
    const dim3 grid((unsigned)blocks), block(256);
    hipStream_t s = (hipStream_t)stream;
    switch (unroll) {
    case 1: hipLaunchKernelGGL(read_stream_kernel<1>, grid, block, 0, s, (const ckq_v4u *)src, n16, (unsigned *)sink); break;
    case 2: hipLaunchKernelGGL(read_stream_kernel<2>, grid, block, 0, s, (const ckq_v4u *)src, n16, (unsigned *)sink); break;
    case 4: hipLaunchKernelGGL(read_stream_kernel<4>, grid, block, 0, s, (const ckq_v4u *)src, n16, (unsigned *)sink); break;
    case 8: hipLaunchKernelGGL(read_stream_kernel<8>, grid, block, 0, s, (const ckq_v4u *)src, n16, (unsigned *)sink); break;
    default: return CKQ_EINVAL;
    }
    return (int)hipGetLastError();
}

extern "C" int ckq_launch_read(const void *src, size_t bytes, void *sink, void *stream)
{
    if (!src || !sink || bytes < 16) return CKQ_EINVAL;
    const size_t n16 = bytes / 16;
    hipLaunchKernelGGL(read_kernel, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (const ckq_v4u *)src, n16, (unsigned *)sink);
    return (int)hipGetLastError();
}

extern "C" int ckq_launch_copy(void *dst, const void *src, size_t bytes, void *stream)
{
    if (!dst || !src || bytes == 0 || (bytes & 15)) return CKQ_EINVAL;
    const size_t n16 = bytes / 16;
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)((n16 + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                       (uint4 *)dst, (const uint4 *)src, n16);
    return (int)hipGetLastError();
}
