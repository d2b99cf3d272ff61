/*
 * ckq_gemm_q80_dw.hip - prefill GEMM, Q8_0 weights x Q8_0 activations, on the gfx950 int8 matrix cores, for operands that start on
 * dwords; ckq_gemm_q80.hip takes the others.
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
 *   A row whose fp16 scale is infinite gives NaN that way; such outputs are summed again term by term at the end.  That is for broken inputs only:
 *   where every output is NaN, a launch takes up to 50 times as long (397 x 3 x 2458 x 1696 2030 us).
 * - Tokens are the A operand, weight rows the B operand: lane 16 q + i holds ONE weight row and tokens 4 q .. 4 q + 3 of a
 *   16 x 16 result.  LDS row 64 h + 16 g + i is weight row 64 h + 4 i + g, so a lane ends with four adjacent rows.
 * - K advances 128 (four blocks) per iteration, two stages.  Of the eight waves, four take two of the blocks and four the
 *   other two, each 64 rows x 16 TG tokens; the partial tiles are added through LDS at the end.  That gives a tile alone on its
 *   CU two waves per SIMD and two tiles four.
 * - The scales, as fp32, lie beside the rows as [block][row] and [block][token], so that a lane's four rows or tokens are one
 *   16-byte read.
 *
 * Tile = 32 TG tokens x 128 weight rows.  With two tiles on a CU vector instructions issue in 83 % of its cycles (2048 x 11008 x 4096, 96 tokens; matrix
 * instructions 32 %, LDS bank conflicts 23 %); with one of two teams in 66 % (333 x 4864 x 4096; 23 and 22 %), with one of one team in 52.  What
 * counts is how many operations, copies (a run of a row costs the address path its five cycles whatever the run's length) and LDS reads there are per product, and
 * whether a CU has another tile's to fill in:
 * - 96 tokens save weights copied and read per product and, for some sizes, a round of tiles: 2048 x 11008 x 4096 (tokens,
 *   rows, K) 321 -> 290 us against 64 tokens, 464 x 37134 x 2048 161 -> 131, 512 x 9728 x 896 26.2 -> 22.6.
 * - 32 tokens do half the work where no more tokens are there: 32 x 37134 x 2048 33.8 -> 24.9.
 * - Two TEAMS of eight waves, each with one half of K and its own stages, where a tile would be alone on its CU anyway: 333 x 4864 x 4096
 *   42.5 -> 34.6, 70 x 11008 x 4096 42.4 -> 32.0, 256 x 4096 x 4096 29.1 -> 24.6.  The second team runs half an iteration behind the
 *   first (one barrier more before, one less after), so that one computes while the other waits for its copies and
 *   finishes them; in step they gain half of that (36.9 for the first).
 * Against ckq_gemm_q80.hip (weights two bytes off): 333 x 4864 x 4096 51.3, 512 x 9728 x 896 34.7, 2048 x 11008 x 4096 426.
 *
 * Rows of an odd number of blocks (K = 32 mod 64) start on a dword and two bytes behind one in turn.  A wave's sixteen rows of one operand are
 * therefore all even or all odd ones: of those the quants of one block in two lie on dwords and of the other two bytes off, which costs two more LDS reads
 * and two byte alignments an operand and block.  With their quantizer, against ckq_gemm_q80.hip: 133 x 5950 x 10272 112.6 -> 71.0, 1628 x 5551 x 6752 336 ->
 * 251, 512 x 4096 x 8224 103.5 -> 79.8 (K = 8192: 67.5), 118 x 13225 x 4960 61 -> 48; 31 sizes 1.18 on average (1.05 to 1.58).  rms error 0.54 to 0.84 of that kernel's.
 * A last iteration of fewer blocks is copied like the others while the one before it is multiplied, and reaches into what follows the row: fetched apart,
 * dword by dword and at the end, it was a round trip to memory that nothing hid (1040 x 672 x 8640 56.1 -> 54.0, odd 487 x 17537 x 1248 88.2 -> 81.5).
 */
#include "ckq_gemm_common.hpp"

constexpr int GEMM8_BN = 128, GEMM8_KB = 4;      /* rows, 32-blocks per iteration */
constexpr int GEMM8_THREADS = 512;               /* of a team */
enum { DW_WHOLE, DW_EVEN, DW_ODD };              /* 32-blocks per row: a multiple of GEMM8_KB, another even number, an odd one */
constexpr int GEMM8_PITCH = 144;                 /* bytes of an operand row's image in LDS: see below */
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

/*
 * LDS image of an operand row, 144 bytes for the four blocks of an iteration: the 136 bytes as they are in memory, 34 dwords, in
 * nine 16-byte chunks (adjacent lanes of a copy fetch adjacent chunks, all from dword-aligned addresses).  Chunk 8 holds the last
 * sixteen, so dwords 30 to 33 of the run lie at 32 to 35 (of an odd number of blocks, whose run may start two bytes early, dwords 31 to 34).  A pair of blocks is 17 dwords: [d0 q0q1] seven of quants [q30q31 d1]
 * eight of quants.  Once a row has landed, the lane in charge makes [q0q1 q30q31] of the first and the ninth - the order of
 * the 32 products of a block is free as long as both operands have the same - and leaves the scales as fp32.  Lane quarter q takes
 * dwords q and q + 4 of a block: a dword at a time, with rows 36 dwords apart and the waves' regions a multiple of four rows, every bank would serve one lane.
 * But the two are one instruction (ds_read2_b32), and two dwords for each of 32 lanes fall on half of the banks twice: sixteen rows lie on those of one residue modulo 4,
 * and q and q + 4 have the same one.  Conflicts are 17 to 23 % of the busy cycles by the counters, other kernels here have 0 to 6; two dwords in a row are not tried.
 */
template <int TG, int TEAMS, int ROWS, bool DUMP>
__global__ void __launch_bounds__(GEMM8_THREADS * TEAMS, DUMP ? 2 : 4) gemm_q80_dw_kernel(GemmArgs a)
{
    constexpr bool ODD = ROWS == DW_ODD, PART = ROWS != DW_WHOLE;
    constexpr int BM = 32 * TG, BN = GEMM8_BN, KB = GEMM8_KB, PITCH = GEMM8_PITCH, MAGIC = 0x4B400000;
    constexpr int XR = 4 * TG, REGION = (16 + XR) * PITCH;  /* a wave brings in sixteen weight rows and XR tokens */
    constexpr int WSCALES = 8 * REGION, XSCALES = WSCALES + KB * BN * 4, STAGE = XSCALES + KB * BM * 4;     /* fp32 scales, [block][row], [block][token] */
    __shared__ __attribute__((aligned(16))) uint8_t stages[TEAMS][2][STAGE];

    const int tid = threadIdx.x, lane = tid & 63, wave = wave_in_block() & 7, team = TEAMS == 1 ? 0 : wave_in_block() >> 3;
    uint8_t (*const stage)[STAGE] = stages[team];
    const int i16 = lane & 15, q = lane >> 4;
    const int kh = wave >> 2, rh = (wave >> 1) & 1, th = wave & 1;

    /* token tiles fastest inside an XCD, so each XCD's L2 sees a weight tile once */
    const GemmWork work = gemm_work(a, (a.nb + KB - 1) / KB);
    int nt, tt;
    if (!gemm_tile(work, nt, tt)) return;
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
    /* token slot l of the tile: of an odd number of blocks, sixteen even tokens and sixteen odd ones in turn */
    auto token_at = [](int l) { return ODD ? (l & ~31) + 2 * (l & 15) + ((l >> 4) & 1) : l; };
    /* rows that are not there: the last one that is, of the same parity if there is one (other bytes would be taken for its scales) */
    auto clamped = [](int r, int last) {
        const int c = min(r, last);
        return (u32)(ODD && c > 0 ? c - ((c ^ r) & 1) : c);
    };
    auto w_row = [&](int l) { return clamped(64 * (l >> 6) + 4 * (l & 15) + ((l >> 4) & 3), work.N - 1 - n0) * stride; };
    auto x_row = [&](int l) { return clamped(token_at(l), a.M - 1 - t0) * stride; };

    /* A wave copies sixteen weight rows (144 chunks, three instructions) and XR tokens (36 chunks for four, one instruction;
     * 72 and 108, two) into its region of a stage, and finishes the same rows when they have landed. */
    constexpr int NC = 3 + (9 * XR + 63) / 64, LAST_CHUNK = ODD ? 124 : 120;
    u32 c_src[NC];
    bool c_on[NC];
#pragma unroll
    for (int i = 0; i < NC; ++i) {
        const int ci = 64 * (i < 3 ? i : i - 3) + lane, r = ci / 9, c = ci % 9;
        c_on[i] = ci < (i < 3 ? 144 : 9 * XR);
        c_src[i] = ((i < 3 ? w_row(16 * wave + min(r, 15)) : x_row(XR * wave + min(r, XR - 1))) & ~3u) + (u32)min(16 * c, LAST_CHUNK);
    }
    /* The last iteration may hold fewer blocks.  Its chunks then reach into the rows behind, but not past the end of the operand: those that
     * would start 16 bytes before it instead, and what its last row needs of them, one dword or two, is fetched when the rest has landed. */
    const int w_last = work.N - 1 - n0, x_last = a.M - 1 - t0;
    auto last_chunk_of = [&](int rows) {
        const size_t bytes = (size_t)rows * stride;
        return (u32)min((bytes & ~(size_t)3) - 16, (size_t)0x7fffffe0);
    };
    const u32 w_end = last_chunk_of(w_last + 1), x_end = last_chunk_of(x_last + 1);
    auto copy = [&](int it, uint8_t *sg) {
        const u32 dst = lds_address(sg + REGION * wave);
        auto all = [&](auto src, int k) __attribute__((always_inline)) {
#pragma unroll
            for (int i = 0; i < NC; ++i)
                if (c_on[i]) lds_copy16(i < 3 ? bw : bx, dst + (u32)(i < 3 ? 1024 * i : 16 * PITCH + 1024 * (i - 3)), src(i), k);
        };
        const int k = __builtin_amdgcn_readfirstlane(it * (KB * 34));
        if (!PART || it * KB + KB <= nblk) all([&](int i) { return c_src[i]; }, k);
        else all([&](int i) { return i < 3 ? min(c_src[i] + (u32)k, w_end) : min(c_src[i] + (u32)k, x_end); }, __builtin_amdgcn_readfirstlane(k & 0));
    };
    /* two lanes per row, one for each pair of blocks */
    const int f_row = lane >> 1, f_p = lane & 1;
    const int f_w = f_row < 16 ? WSCALES + 4 * (64 * (wave >> 2) + 4 * f_row + (wave & 3)) : XSCALES + 4 * (XR * wave + f_row - 16);
    const int f_pitch = f_row < 16 ? 4 * BN : 4 * BM;
    auto finish = [&](int it, uint8_t *sg) {
        if (f_row >= 16 + XR) return;
        u32 *const d = reinterpret_cast<u32 *>(sg + REGION * wave + PITCH * f_row);
        if constexpr (ODD) {
            const int p = f_row < 16 ? wave & 1 : (XR * wave + f_row - 16) >> 4 & 1, left = nblk - it * KB - 2 * f_p;
            const u32 e0 = d[17 * f_p], e1 = d[17 * f_p + 8 + p];
            float *const sc = reinterpret_cast<float *>(sg + f_w + 2 * f_p * f_pitch);
            *sc = left > 0 ? h2f(e0 >> (16 * p) & 0xffff) : 0.0f;
            *reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(sc) + f_pitch) = left > 1 ? h2f(e1 >> (16 - 16 * p) & 0xffff) : 0.0f;
            return;
        }
        const bool live = 2 * f_p < nblk - it * KB;
        const u32 d0 = d[17 * f_p], d8 = d[17 * f_p + 8];
        d[17 * f_p] = __builtin_amdgcn_alignbyte(d8, d0, 2);
        float *const sc = reinterpret_cast<float *>(sg + f_w + 2 * f_p * f_pitch);
        *sc = live ? h2f(d0 & 0xffff) : 0.0f;
        *reinterpret_cast<float *>(reinterpret_cast<uint8_t *>(sc) + f_pitch) = live ? h2f(d8 >> 16) : 0.0f;
    };

    auto mend = [&](int it, uint8_t *sg) {
        const int r = lane, slot = r < 16 ? 16 * wave + r : XR * wave + r - 16, row = r < 16 ? 64 * (slot >> 6) + 4 * (slot & 15) + ((slot >> 4) & 3) : token_at(slot);
        if (r >= 16 + XR || row != (r < 16 ? w_last : x_last)) return;
        /* 34 bytes a block, from a dword or from two bytes behind one: dwords 8, 16 or 24 and 25, the last of which may be half of one */
        const int left = nblk - it * KB;
        const u32 ofs = (u32)row * stride;
        const u32 at = (ofs & ~3u) + (u32)it * (KB * 34u) + 32u * (u32)left;
        const uint8_t *const src = r < 16 ? wbase + at : xbase + at;
        u32 *const d = reinterpret_cast<u32 *>(sg + REGION * wave + PITCH * r) + 8 * left;
        d[0] = left == 1 && !(ofs & 2) ? ld2(src) : ld4<4>(src);
        if (left == 3) d[1] = !(ofs & 2) ? ld2(src + 4) : ld4<4>(src + 4);
    };

    ckq_v4f acc[TG][4];                                     /* [token group][row group] */
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[tg][g] = ckq_v4f{0.0f, 0.0f, 0.0f, 0.0f};
    ckq_v4i magic = {MAGIC, MAGIC, MAGIC, MAGIC};
    asm volatile("" : "+v"(magic));                         /* kept in registers: as a constant it is copied before every use */

    /* this lane's operands of the wave's two blocks, and where their scales are */
    const int opd = 17 * kh + q, opd_hi = ODD ? opd + 13 + (kh && q ? 1 : 0) : opd + 9 + (kh ? 6 : 4);       /* block 3 ends in the last chunk */
    auto operand = [](const uint8_t *p, int lo, int hi) {
        const u32 *const d = reinterpret_cast<const u32 *>(p);
        return (long)((uint64_t)d[lo] | ((uint64_t)d[hi] << 32));
    };
    /* ODD: of rows of parity p the quants of block jj start on a dword (jj != p) or two bytes behind one */
    auto odd_operand = [&](const uint8_t *r, int jj, int p) __attribute__((always_inline)) {
        const u32 *const d = reinterpret_cast<const u32 *>(r);
        const int lo = jj ? opd + 9 : opd + p, hi = jj ? opd_hi : lo + 4;
        if (__builtin_constant_p(p) && jj != p) return (long)((uint64_t)d[lo] | ((uint64_t)d[hi] << 32));
        const u32 sh = jj != p ? 0 : 2;
        return (long)((uint64_t)__builtin_amdgcn_alignbyte(d[lo + 1], d[lo], sh) | ((uint64_t)__builtin_amdgcn_alignbyte(d[hi + 1], d[hi], sh) << 32));
    };
    auto compute_block = [&](const uint8_t *sg, int it, int jj) __attribute__((always_inline)) {
        const uint8_t *const wl = sg + 4 * rh * REGION + i16 * PITCH;
        /* token t of the tile is row 16 + t % XR of wave t / XR */
        auto token = [&](int t) { return sg + (t / XR) * REGION + (16 + t % XR) * PITCH; };
        const int tw = 16 * TG * th;
        const int lo = jj ? opd + 9 : opd, hi = jj ? opd_hi : opd + 4;
        long w[4], x[TG];
        auto take_x = [&](int tg) __attribute__((always_inline)) {
            const uint8_t *const r = token(tw + 16 * tg + i16);
            x[tg] = !ODD ? operand(r, lo, hi) : TG % 2 ? odd_operand(r, jj, (th + tg) & 1) : odd_operand(r, jj, tg & 1);
        };
        constexpr int AHEAD = ODD && TG == 3 ? 1 : TG;          /* three groups' operands and their pieces do not fit the registers of four waves per SIMD */
#pragma unroll
        for (int tg = 0; tg < AHEAD; ++tg) take_x(tg);
#pragma unroll
        for (int g = 0; g < 4; ++g) w[g] = ODD ? odd_operand(wl + REGION * g, jj, g & 1) : operand(wl + REGION * g, lo, hi);
        const ckq_v4f dwb = *reinterpret_cast<const ckq_v4f *>(sg + WSCALES + 4 * ((2 * kh + jj) * BN + 64 * rh + 4 * i16));
        float dwm[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) dwm[g] = dwb[g] * -12582912.0f;
#pragma unroll
        for (int tg = 0; tg < TG; ++tg) {
            if (tg >= AHEAD) {
                asm volatile("" ::: "memory");
                take_x(tg);
            }
            const ckq_v4f dxb = *reinterpret_cast<const ckq_v4f *>(sg + XSCALES + 4 * ((2 * kh + jj) * BM + tw + 16 * tg + 4 * q));
            ckq_v4i d[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) d[g] = __builtin_amdgcn_mfma_i32_16x16x32_i8(x[tg], w[g], magic, 0, 0, 0);
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                float t[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int di = d[g][r];
                    t[r] = __builtin_fmaf(dwb[g], __builtin_bit_cast(float, di), dwm[g]);
                    if constexpr (DUMP) {
                        int tr = t0 + token_at(tw + 16 * tg + 4 * q + r);
                        asm volatile("" : "+v"(tr));   /* store addresses formed here, not kept in registers */
                        const int n = n0 + 64 * rh + 4 * i16 + g, b = it * KB + 2 * kh + jj;
                        if (tr < a.M && n < work.N && b < nblk) a.dump[((size_t)tr * work.N + n) * nblk + (size_t)b] = di - MAGIC;
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) acc[tg][g][r] = __builtin_fmaf(dxb[r], t[r], acc[tg][g][r]);
            }
        }
        /* block by block: scheduled together, the two would need more registers than four waves per SIMD have */
#pragma unroll
        for (int tg = 0; tg < TG; ++tg) asm volatile("" : "+v"(acc[tg][0]), "+v"(acc[tg][1]), "+v"(acc[tg][2]), "+v"(acc[tg][3]) :: "memory");
    };

    /* the iterations in TEAMS runs, the whole ones in equal parts and one with fewer blocks to the last team; a team that has one less still comes to the barriers */
    const int nrun = (max(min(niter, nblk / KB) - it0, 0) + TEAMS - 1) / TEAMS, nstep = TEAMS == 1 ? niter - it0 : max(nrun, niter - it0 - nrun);
    const int run0 = it0 + team * nrun, run1 = TEAMS == 1 || team ? niter : run0 + nrun;
    {
        auto landed = [] {                                  /* vmcnt(0) lgkmcnt(0) */
            __builtin_amdgcn_s_waitcnt(0x0070);
            asm volatile("" ::: "memory");
        };
        auto meet = [] {                                    /* lgkmcnt(0) */
            __builtin_amdgcn_s_waitcnt(0xc07f);
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        };
        auto at = [&](int it) { return min(it, niter - 1); };
        copy(at(run0), stage[0]);
        landed();
        finish(at(run0), stage[0]);
        meet();
        if (TEAMS == 2 && team) __builtin_amdgcn_s_barrier();
        auto step = [&](int it, uint8_t *cur, uint8_t *next) {
            copy(at(it + 1), next);
            __builtin_amdgcn_sched_barrier(0);
            if (TEAMS == 1 || it < run1) compute_block(cur, it, 0);
            if (TEAMS == 2) __builtin_amdgcn_s_barrier();
            if (TEAMS == 1 || it < run1) compute_block(cur, it, 1);
            __builtin_amdgcn_sched_barrier(0);
            landed();
            finish(at(it + 1), next);
            meet();
        };
        /* rows of whole iterations go on copying to the end, a step more of one kind: the last step apart costs short rows 1 % (512 x 9728 x 896) */
        const int nloop = PART ? nstep - 1 : nstep;
        if constexpr (DUMP || (ODD && TG == 3)) {           /* one copy of the stores; of three groups and an odd number of blocks two spill a register */
            for (int k = 0; k < nloop; ++k) step(run0 + k, stage[k & 1], stage[(k + 1) & 1]);
        } else for (int k = 0; k < nloop; k += 2) {
            step(run0 + k, stage[0], stage[1]);
            if (k + 1 < nloop) step(run0 + k + 1, stage[1], stage[0]);
        }
        if constexpr (PART) {
            const int it = run0 + nstep - 1;
            uint8_t *const cur = stage[(nstep - 1) & 1];
            if (niter * KB > nblk && (w_last < BN || x_last < BM)) {
                if (it == niter - 1) mend(it, cur);
                meet();
            }
            if (TEAMS == 1 || it < run1) compute_block(cur, it, 0);
            if (TEAMS == 2) __builtin_amdgcn_s_barrier();
            if (TEAMS == 1 || it < run1) compute_block(cur, it, 1);
        }
        if (TEAMS == 2 && !team) __builtin_amdgcn_s_barrier();
        if (PART) __syncthreads();                          /* the stages have been read */
    }

    /* the parts of K: of the 2 TEAMS waves of a sub-tile, wave `part` keeps token groups tg with tg % (2 TEAMS) == part and hands
     * the others over */
    constexpr int PARTS = 2 * TEAMS;
    const int part = 2 * team + kh;
    ckq_v4f *const meet_at = reinterpret_cast<ckq_v4f *>(stages[0][0]) + (wave & 3) * 256 + lane;     /* [token group][part but the keeper][wave of the part][row group][lane] */
    static_assert(TG * (PARTS - 1) * 16384 <= (int)sizeof(stages), "");
    auto place = [&](int tg, int p) { return meet_at + 1024 * ((PARTS - 1) * tg + p - (p > tg % PARTS ? 1 : 0)); };
#pragma unroll
    for (int tg = 0; tg < TG; ++tg)
        if (tg % PARTS != part) {
#pragma unroll
            for (int g = 0; g < 4; ++g) place(tg, part)[64 * g] = acc[tg][g];
        }
    __syncthreads();

    /* lane: rows n .. n + 3, tokens t .. t + 3 */
    const GemmOut o = work.out;
    const bool vec_ok = (o.ldc % 4 == 0) && (((uintptr_t)o.C) % 16 == 0) && (n0 + BN <= work.N);
    const int n = n0 + 64 * rh + 4 * i16;
    float bv[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) bv[g] = o.bias && n + g < work.N ? o.bias[n + g] : 0.0f;
#pragma unroll
    for (int tg = 0; tg < TG; ++tg) {
        if (tg % PARTS != part) continue;
        constexpr int TSTEP = ODD ? 2 : 1;
        const int t = t0 + token_at(16 * (TG * th + tg) + 4 * q);
        ckq_v4f o4[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            ckq_v4f v[PARTS];
#pragma unroll
            for (int p = 0; p < PARTS; ++p) v[p] = p == tg % PARTS ? acc[tg][g] : place(tg, p)[64 * g];
            o4[g] = v[0] + v[1];
            if constexpr (TEAMS == 2) o4[g] += v[2] + v[3];
        }
        bool fix = false;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            if (t + TSTEP * r >= a.M) continue;
            float *dst = o.C + (size_t)(t + TSTEP * r) * o.ldc + n;
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
                const int tr = t + TSTEP * (e >> 2), nr = n + (e & 3);
                if (tr >= a.M || nr >= work.N) continue;
                float *dst = o.C + (size_t)tr * o.ldc + nr;
                if (*dst == *dst) continue;
                *dst = q80_output(work.B + (size_t)nr * stride, a.A + (size_t)tr * stride, it0 * KB, min(nblk, niter * KB)) +
                       (o.bias ? o.bias[nr] : 0.0f);
            }
        }
    }
}

/* The forms of the kernel: token groups of 16 per wave, teams; blocks of it that fit a CU; and what a launch takes, in us:
 * launch + iterations of a team x (wait x rounds of the fullest CU + work x blocks on it) + round x rounds, 1.45 per million
 * floats written and read again, 2.4 for the launch that adds a K split.  Fitted to 110 launches of all five (9 to 1500 tokens, 300 to
 * 152000 rows, K of 256 to 8192; 9 to 12 % rms): the choice is 2 % slower than the best form of each on average, and
 * 12 % faster than 64 tokens and one team throughout. */
struct DwForm { int tg, teams, fit; float launch, wait, work, round; };
static const DwForm dw_forms[5] = {{1, 1, 3, 4.0f, 0.40f, 0.39f, 0.0f}, {2, 1, 2, 4.7f, 0.45f, 0.575f, 0.0f}, {3, 1, 2, 5.3f, 0.74f, 0.58f, 0.0f},
                                   {1, 2, 1, 3.1f, 1.18f, 0.0f, 1.9f}, {2, 2, 1, 3.2f, 1.6f, 0.0f, 2.5f}};

/* The form for `row_tiles` tiles of weight rows in all; single: one matrix, which may be split along K.  64 tokens and one team
 * are always possible; another form only if its chains of multiply-adds are no longer (fewer splits of K would make them so, and the
 * error larger) and, if it is split, with no more scratch than that form or the entry point that allocates nothing has; rows of an odd number of
 * blocks, which were another kernel's, never with more than that form.  Their 32-token tiles of two teams take 1.5 us an iteration where the others take 1.18 (four
 * more LDS reads in a step that waits for itself): 1040 x 672 x 8608 64.5 with them, 57.7 with 64 tokens, one team and a split. */
static int dw_form(int M, int nb, long rows, long row_tiles, bool single)
{
    const int steps = (nb + GEMM8_KB - 1) / GEMM8_KB;
    const float out = 1e-6f * (float)M * (float)rows;
    int best = 0, chain = 0;
    float least = 0.0f;
    size_t scratch = 0;
    for (int k : {1, 0, 2, 3, 4}) {
        const DwForm &f = dw_forms[k];
        const long tiles = (long)((M + 32 * f.tg - 1) / (32 * f.tg)) * row_tiles;
        int s = single && tiles < 160 ? gemm_choose_splits((int)tiles, steps) : 1;
        const int per = (steps + s - 1) / s, iters = (per + f.teams - 1) / f.teams;
        s = (steps + per - 1) / per;
        const size_t need = s > 1 ? (size_t)s * (size_t)M * (size_t)rows * 4 : 0;
        if (k == 1) {
            chain = iters;
            scratch = nb % 2 || need > CKQ_NOALLOC_SCRATCH_BYTES ? need : CKQ_NOALLOC_SCRATCH_BYTES;
        } else if (iters > chain || need > scratch || (f.teams > 1 && (s > 1 || !single))) continue;
        const long on_cu = (tiles * s + 255) / 256, rounds = (on_cu + f.fit - 1) / f.fit;
        const float wait = nb % 2 && k == 3 ? 1.5f : f.wait;       /* 32 tokens, two teams, rows of an odd number of blocks */
        const float t = f.launch + (float)iters * (wait * (float)rounds + f.work * (float)on_cu) + f.round * (float)rounds +
                        1.45f * out * (float)(s > 1 ? 1 + 2 * s : 1) + (s > 1 ? 2.4f : 0.0f);
        if (k == 1 || t < least) { least = t; best = k; }
    }
    return best;
}

/* g: operands, sizes, nnt set by the caller (ckq_gemm_q80.hip). */
template <int TG, int TEAMS, int ROWS>
static int dw_launch_rows(GemmArgs &g, hipStream_t s)
{
    g.ntt = (g.M + 32 * TG - 1) / (32 * TG);
    const int steps = (g.nb + GEMM8_KB - 1) / GEMM8_KB;
#if CKQ_WITH_DUMP
    if (g.dump) return gemm_launch_split(gemm_q80_dw_kernel<TG, TEAMS, ROWS, true>, g, steps, s, GEMM8_THREADS * TEAMS);
#endif
    return gemm_launch_split(gemm_q80_dw_kernel<TG, TEAMS, ROWS, false>, g, steps, s, GEMM8_THREADS * TEAMS);
}
template <int TG, int TEAMS>
static int dw_launch(GemmArgs &g, hipStream_t s)
{
    if (g.nb % 2) return dw_launch_rows<TG, TEAMS, DW_ODD>(g, s);
    return g.nb % GEMM8_KB ? dw_launch_rows<TG, TEAMS, DW_EVEN>(g, s) : dw_launch_rows<TG, TEAMS, DW_WHOLE>(g, s);
}
int gemm_q80_dw_launch(GemmArgs &g, hipStream_t s)
{
    if (g.nb % 2 && g.ext_part) {
        /* what a size is answered does not hang on the form: refused where the split of 64-token tiles has no room */
        const int steps = (g.nb + GEMM8_KB - 1) / GEMM8_KB, sp = gemm_choose_splits((g.M + 63) / 64 * g.nnt, steps), per = (steps + sp - 1) / sp, k = (steps + per - 1) / per;
        if (k > 1 && (size_t)k * (size_t)g.M * (size_t)g.N * sizeof(float) > g.ext_part_bytes) return CKQ_ESCRATCH;
    }
    switch (dw_form(g.M, g.nb, g.N, g.nnt, true)) {
    case 0: return dw_launch<1, 1>(g, s);
    case 1: return dw_launch<2, 1>(g, s);
    case 2: return dw_launch<3, 1>(g, s);
    case 3: return dw_launch<1, 2>(g, s);
    default: return dw_launch<2, 2>(g, s);
    }
}
template <int TG>
static int dw_launch_group(GemmArgs &g, const GemmGroupIn &in, hipStream_t s)
{
    g.ntt = (g.M + 32 * TG - 1) / (32 * TG);
    if (g.nb % 2) return gemm_launch_grouped(gemm_q80_dw_kernel<TG, 1, DW_ODD, false>, g, in, s, GEMM8_THREADS);
    if (g.nb % GEMM8_KB) return gemm_launch_grouped(gemm_q80_dw_kernel<TG, 1, DW_EVEN, false>, g, in, s, GEMM8_THREADS);
    return gemm_launch_grouped(gemm_q80_dw_kernel<TG, 1, DW_WHOLE, false>, g, in, s, GEMM8_THREADS);
}
int gemm_q80_dw_launch_group(GemmArgs &g, const GemmGroupIn &in, hipStream_t s)
{
    long rows = 0, tiles = 0;
    for (int p = 0; p < in.n; ++p) {
        rows += in.N[p];
        tiles += (in.N[p] + GEMM8_BN - 1) / GEMM8_BN;
    }
    switch (dw_form(g.M, g.nb, rows, tiles, false)) {
    case 0: return dw_launch_group<1>(g, in, s);
    case 1: return dw_launch_group<2>(g, in, s);
    default: return dw_launch_group<3>(g, in, s);
    }
}
