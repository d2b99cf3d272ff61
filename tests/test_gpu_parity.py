"""GPU parity tests: the HIP path, called through the C ABI, against the CPU
oracle on the same seeded inputs and against the golden fixtures.

Bars: quantizer outputs and integer sub-block dots bit-exact; fp32 outputs
within 1e-4 of the oracle, normalised by max|y_ref| (pointwise relative error
is not meaningful here: the reference's own builds differ from each other by
1e-3 pointwise on cancelling rows while agreeing to 1e-6 of max|y|)."""
import ctypes
import importlib
import sys

import numpy as np
import pytest

import ckq_testlib as T

pytestmark = pytest.mark.gpu

ckq = importlib.import_module("c-kernel-engine_amd")
P = ckq.parity
TOL = 1e-4
FMTS = ["q4_k", "q5_k", "q6_k", "q8_0"]


def say(*a):
    print(*a)
    sys.stdout.flush()


@pytest.fixture(scope="module", autouse=True)
def _lib():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a device"
    L = ckq.lib()          # raises if the HIP library is not built: no fallback
    assert L.ckq_init() == 0
    yield L
    L.ckq_weights_clear()


MATRIX_CORE_TESTS = ("mfma", "split_k", "q5_0_row_and_token")


@pytest.fixture(autouse=True)
def _gemm_policy(request, _lib):
    """Tests aimed at the matrix-core GEMMs force them for every token count
    above eight (the automatic choice would send their small shapes to the
    streaming kernel); everything else runs with the automatic choice."""
    forced = any(k in request.node.name for k in MATRIX_CORE_TESTS)
    _lib.ckq_set_gemm_policy(1 if forced else 0)
    yield
    _lib.ckq_set_gemm_policy(0)


def make_case(fmt, rows, K, kind, seed, tokens=1):
    if kind == "rand":
        W = T.random_blocks(fmt, rows * (K // T.ELEMS[fmt]), seed)
    else:
        W = T.synth_weights(fmt, rows, K, seed)
    xf = T.normal(tokens * K, 0.0, 1.0, seed + 1000)
    xq = T.oracle_quantize(xf, T.act_fmt(fmt), rows=tokens)
    return W, xf, xq


# ---- quantizers: bit-exact ------------------------------------------------------

def test_quantize_q8_k_golden_host_and_device():
    import torch
    G = T.golden()
    x, want = G["q8k_in"], G["q8k_out"]
    say("quantize_row_q8_k host path, n =", len(x))
    got = P.quantize(x, "q8_k")
    assert np.array_equal(got, want)
    say("ckq_quantize_q8_k_dev")
    got = P.dev_quantize(P.to_device(x), "q8_k").cpu().numpy()
    assert np.array_equal(got, want)
    # ck_test_ wrapper
    out = np.zeros_like(want)
    ckq.lib().ck_test_quantize_q8_k(T.ptr(x), T.ptr(out), len(x))
    assert np.array_equal(out, want)


def test_quantize_q8_0_golden_host_and_device():
    G = T.golden()
    x, want = G["q80_in"], G["q80_out"]
    say("quantize_row_q8_0 host path, n =", len(x))
    assert np.array_equal(P.quantize(x, "q8_0"), want)
    assert np.array_equal(P.dev_quantize(P.to_device(x), "q8_0").cpu().numpy(), want)


@pytest.mark.parametrize("std,seed", [(1.0, 1), (0.02, 2), (37.0, 3), (1e-6, 4)])
def test_quantize_bit_exact_vs_oracle_large(std, seed):
    rows, k = 96, 4096
    x = T.normal(rows * k, 0.0, std, seed)
    # plant ties and zero blocks
    x[0:256] = 0.0
    x[256 + 5] = 9.0 * std
    x[256 + 99] = -9.0 * std
    say("quantize q8_k / q8_0 rows=%d k=%d std=%g" % (rows, k, std))
    xd = P.to_device(x)
    for fmt in ("q8_k", "q8_0"):
        want = T.oracle_quantize(x, fmt, rows=rows)
        got = P.dev_quantize(xd, fmt, rows=rows).cpu().numpy()
        assert np.array_equal(got, want), fmt


@pytest.mark.parametrize("fmt", ["q8_k", "q8_0"])
def test_quantizers_round_blocks_of_one_wave_the_short_and_the_long_way(fmt):
    """Blocks whose values round by one addition beside blocks that need the saturating conversion: values half way between two
    quants (the largest 127 makes the scale 1), an infinity, a block whose inverse scale is infinite, the smallest whose
    is not, the largest finite values, and (Q8_K, whose rule for them is the order of comparisons) NaNs, alone and beside zeros only."""
    k = 4096
    x = T.normal(64 * k, 0.0, 1.0, seed=77).reshape(-1, 256)
    x[1] = np.arange(256) % 127 + 0.5
    x[1, ::2] *= -1
    x[1, 31::32] = 127.0
    x[3, 40], x[5, 200] = np.inf, -np.inf
    x[7] *= np.float32(1e-38)
    x[9] = np.where(np.arange(256) % 3 == 0, np.float32(3.8e-37), np.float32(-1.3e-37))
    x[11] *= np.float32(3e38) / np.abs(x[11]).max()
    if fmt == "q8_k":
        x[13, 17] = np.nan
        x[14] = 0.0
        x[14, 3] = np.nan
    x = np.ascontiguousarray(x.reshape(-1))
    say("quantizers, short and long rounding", fmt)
    got, want = P.dev_quantize(P.to_device(x), fmt, rows=64).cpu().numpy(), T.oracle_quantize(x, fmt, rows=64)
    assert np.array_equal(got, want), np.nonzero(got != want)[0][:8]


def test_quantize_batch_equals_rows_host():
    x = T.normal(7 * 768, seed=12)
    whole = P.quantize(x, "q8_k", rows=7)
    rows = np.concatenate([P.quantize(x[r * 768:(r + 1) * 768], "q8_k") for r in range(7)])
    assert np.array_equal(whole, rows)


# ---- integer sub-block dots: bit-exact -----------------------------------------

# K values chosen to hit every lane mapping of the kernel: 4..32 positions per
# row (sub-wave rows), 64, 2-4 positions per lane, and the multi-pass loop.
K_SWEEP = {"q4_k": [256, 512, 1024, 2048, 4096, 4864, 11008, 16384, 20480],
           "q5_k": [256, 1024, 4864, 11008],
           "q6_k": [256, 512, 1024, 2048, 4096, 11008, 16384, 20480],
           "q8_0": [32, 128, 512, 896, 1024, 2048, 4096, 8192, 10240]}


@pytest.mark.parametrize("fmt", FMTS)
def test_subblock_dots_bit_exact(fmt):
    rows = 37
    for K in K_SWEEP[fmt]:
        W, _, xq = make_case(fmt, rows, K, "rand", 40 + K)
        say("subblock dots", fmt, "rows", rows, "K", K)
        got = P.dev_subblock_dots(fmt, P.to_device(W), P.to_device(xq), rows, K).cpu().numpy()
        want = T.oracle_subdots(fmt, W, xq, rows, K)
        assert np.array_equal(got, want), (fmt, K)


# ---- GEMV fp32 --------------------------------------------------------------------

@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("kind", ["rand", "enc"])
def test_gemv_golden_fixture(fmt, kind):
    G = T.golden()
    M, K, _ = (int(v) for v in G["shape"])
    W = G["w_%s_%s" % (fmt, kind)]
    xq = G["act_q80" if fmt == "q8_0" else "act_q8k"]
    say("gemv golden", fmt, kind)
    y = P.gemv(fmt, W, xq, M, K)
    for build in ("avx2", "avx512"):
        assert T.norm_err(y, G["y_%s_%s_%s" % (fmt, kind, build)]) <= TOL
    c = P.gemm_nt(fmt, xq, W, G["bias"], 3, M, K)
    assert T.norm_err(c, G["c_%s_%s_avx2" % (fmt, kind)]) <= TOL


@pytest.mark.parametrize("fmt", FMTS)
def test_gemv_vs_oracle_k_sweep(fmt):
    rows = 53
    for K in K_SWEEP[fmt]:
        for kind in ("rand", "enc"):
            W, _, xq = make_case(fmt, rows, K, kind, 90 + K)
            say("gemv dev", fmt, kind, "rows", rows, "K", K)
            y = P.dev_gemm_nt(fmt, P.to_device(xq), P.to_device(W), None, 1, rows, K).cpu().numpy().reshape(-1)
            ref = T.oracle_gemv(fmt, W, xq, rows, K)
            assert T.norm_err(y, ref) <= TOL, (fmt, K, kind)
            exact = T.oracle_exact(fmt, W, xq, rows, K)
            assert T.norm_err(y, exact) <= TOL


@pytest.mark.parametrize("fmt", FMTS)
def test_gemv_row_counts(fmt):
    """Row counts around the wave/block tiling, including a single row."""
    K = 1024 if fmt != "q8_0" else 896
    for rows in (1, 2, 3, 15, 16, 17, 63, 64, 65, 127, 257):
        W, _, xq = make_case(fmt, rows, K, "rand", 7 * rows)
        say("gemv rows", fmt, rows)
        y = P.gemv(fmt, W, xq, rows, K)
        assert T.norm_err(y, T.oracle_gemv(fmt, W, xq, rows, K)) <= TOL, rows


def test_stored_bsums_semantics():
    """Q4_K/Q5_K consume the activation's STORED bsums; Q6_K never reads them
    (reference unittest/test_parallel_gemv.py:66-85 feeds zeroed bsums)."""
    G = T.golden()
    M, K, _ = (int(v) for v in G["shape"])
    xz = G["act_q8k_zero_bsums"]
    for fmt in ("q4_k", "q5_k", "q6_k"):
        for kind in ("rand", "enc"):
            say("zero bsums", fmt, kind)
            y = P.gemv(fmt, G["w_%s_%s" % (fmt, kind)], xz, M, K)
            assert T.norm_err(y, G["y_%s_%s_zero_bsums" % (fmt, kind)]) <= TOL


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k", "q8_0"])
def test_parallel_union_equals_serial(fmt):
    """Calling the thread-split entry point for every ith reproduces the serial
    result (reference unittest/test_parallel_gemv.py:112-170)."""
    rows, K = 301, 1024
    W, _, xq = make_case(fmt, rows, K, "rand", 5)
    serial = P.gemv(fmt, W, xq, rows, K)
    # default ("rows", the reference's semantics): every call computes exactly its own range
    ckq.lib().ckq_set_parallel_whole(-1)
    for nth in (1, 3, 8, 64):
        for simd in (False, True):
            say("parallel", fmt, "nth", nth, "simd", simd)
            y = P.gemv_parallel(fmt, W, xq, rows, K, nth, simd)
            assert np.array_equal(y, serial)
    # a single ith touches only its own rows
    y = np.full(rows, -5.0, np.float32)
    ckq.lib().gemv_q4_k_q8_k_parallel(T.ptr(y), T.ptr(W), T.ptr(xq), rows, K, 1, 4) if fmt == "q4_k" else None
    if fmt == "q4_k":
        dr = (rows + 3) // 4
        assert np.all(y[:dr] == -5.0) and np.all(y[2 * dr:] == -5.0)
        assert np.array_equal(y[dr:2 * dr], serial[dr:2 * dr])
    # "whole" mode: ith 0 computes everything, the rest return; the union is still the serial result
    ckq.lib().ckq_set_parallel_whole(1)
    try:
        assert np.array_equal(P.gemv_parallel(fmt, W, xq, rows, K, 8, True), serial)
        y = np.zeros(rows, np.float32)
        fn = getattr(ckq.lib(), P._GEMV[fmt] + "_parallel_simd")
        fn(T.ptr(y), T.ptr(W), T.ptr(xq), rows, K, 0, 8)
        assert np.array_equal(y, serial)
        y = np.full(rows, -5.0, np.float32)
        fn(T.ptr(y), T.ptr(W), T.ptr(xq), rows, K, 3, 8)     # another ith: returns at once
        assert np.all(y == -5.0)
    finally:
        ckq.lib().ckq_set_parallel_whole(-1)


# ---- batched decode / small GEMM -------------------------------------------------------

@pytest.mark.parametrize("fmt", FMTS)
def test_gemm_nt_token_counts(fmt):
    N, K = 77, 1024
    bias = T.normal(N, 0.0, 0.5, seed=8)
    for M in (1, 2, 3, 4, 5, 8, 9, 17):
        W, _, xq = make_case(fmt, N, K, "enc", 300 + M, tokens=M)
        say("gemm_nt", fmt, "tokens", M)
        ref = T.oracle_gemm_nt(fmt, xq, W, bias, M, N, K)
        c = P.gemm_nt(fmt, xq, W, bias, M, N, K)
        assert T.norm_err(c, ref) <= TOL, M
        cd = P.dev_gemm_nt(fmt, P.to_device(xq), P.to_device(W), P.to_device(bias), M, N, K).cpu().numpy()
        assert np.array_equal(cd, c)       # host and device paths run the same kernel
        # each row of a batch equals the single-token GEMV of that token
        ab = T.row_bytes(T.act_fmt(fmt), K)
        y0 = P.gemv(fmt, W, xq[(M - 1) * ab:M * ab].copy(), N, K)
        assert T.norm_err(c[M - 1] - bias, y0) <= 1e-6


def test_gemm_layouts_and_wrappers():
    """gemm_* writes Y[n*M + row]; ck_test_* quantize internally; fp32 adapters."""
    rows, K, tok = 40, 1024, 3
    L = ckq.lib()
    for fmt, gemm in (("q4_k", "gemm_q4_k_q8_k"), ("q6_k", "gemm_q6_k_q8_k")):
        W, xf, xq = make_case(fmt, rows, K, "enc", 17, tokens=tok)
        say("gemm layout", fmt)
        Y = np.zeros(tok * rows, np.float32)
        getattr(L, gemm)(T.ptr(Y), T.ptr(W), T.ptr(xq), rows, tok, K)
        ref = T.oracle_gemm_nt(fmt, xq, W, None, tok, rows, K)
        assert T.norm_err(Y.reshape(tok, rows), ref) <= TOL
        out = np.zeros(tok * rows, np.float32)
        getattr(L, "ck_test_gemm_" + fmt)(T.ptr(W), T.ptr(xf), T.ptr(out), rows, K, tok)
        assert T.norm_err(out.reshape(tok, rows), ref) <= TOL
        one = np.zeros(1, np.float32)
        getattr(L, "ck_test_gemv_" + fmt)(T.ptr(W), T.ptr(xf), T.ptr(one), K)
        assert abs(one[0] - ref[0, 0]) <= TOL * np.max(np.abs(ref))
    # Q5_K fp32 adapters
    W, xf, xq = make_case("q5_k", rows, K, "enc", 19, tokens=tok)
    y = np.zeros(rows, np.float32)
    L.gemv_q5_k(T.ptr(y), T.ptr(W), T.ptr(xf), rows, K)
    assert T.norm_err(y, T.oracle_gemv("q5_k", W, xq, rows, K)) <= TOL
    bias = T.normal(rows, seed=3)
    c = np.zeros(tok * rows, np.float32)
    L.gemm_nt_q5_k(T.ptr(xf), T.ptr(W), T.ptr(bias), T.ptr(c), tok, rows, K)
    assert T.norm_err(c.reshape(tok, rows), T.oracle_gemm_nt("q5_k", xq, W, bias, tok, rows, K)) <= TOL
    # Q8_0: vec_dot, fp32-activation GEMV, ck_test wrappers
    W, xf, xq = make_case("q8_0", rows, K, "enc", 23, tokens=tok)
    s = np.zeros(1, np.float32)
    L.vec_dot_q8_0_q8_0(K, T.ptr(s), T.ptr(W), T.ptr(xq))
    ref = T.oracle_gemv("q8_0", W, xq, rows, K)
    assert abs(s[0] - ref[0]) <= TOL * np.max(np.abs(ref))
    y = np.zeros(rows, np.float32)
    L.gemv_q8_0(T.ptr(y), T.ptr(W), T.ptr(xf), rows, K)
    want = np.zeros(rows, np.float32)
    T.oracle().orc_gemv_q8_0(T.ptr(want), T.ptr(W), T.ptr(xf), rows, K)
    assert T.norm_err(y, want) <= TOL
    out = np.zeros(rows, np.float32)
    L.ck_test_gemv_q8_0(T.ptr(W), T.ptr(xf), T.ptr(out), rows, K)
    assert T.norm_err(out, ref) <= TOL
    W6, _, xq6 = make_case("q6_k", 1, K, "rand", 29)
    s = np.zeros(1, np.float32)
    L.vec_dot_q6_k_q8_k(K, T.ptr(s), T.ptr(W6), T.ptr(xq6))
    assert abs(s[0] - T.oracle_gemv("q6_k", W6, xq6, 1, K)[0]) <= TOL * abs(s[0]) + 1e-6


def test_weight_cache_follows_content():
    """Same host address, new bytes: the resident copy is refreshed."""
    rows, K = 32, 1024
    W, _, xq = make_case("q4_k", rows, K, "rand", 61)
    y1 = P.gemv("q4_k", W, xq, rows, K)
    W2, _, _ = make_case("q4_k", rows, K, "rand", 62)
    W[:] = W2
    y2 = P.gemv("q4_k", W, xq, rows, K)
    assert T.norm_err(y2, T.oracle_gemv("q4_k", W2, xq, rows, K)) <= TOL
    assert T.norm_err(y1, y2) > 1e-3


# ---- full benchmark shapes ----------------------------------------------------------------

FULL = [("q4_k", 4096, 4096), ("q4_k", 11008, 4096), ("q6_k", 32000, 4096), ("q6_k", 4096, 11008),
        ("q5_k", 4864, 1024), ("q5_k", 896, 4864), ("q8_0", 151936, 896)]


@pytest.mark.parametrize("fmt,rows,K", FULL)
def test_full_size_shapes(fmt, rows, K):
    import torch
    W = T.synth_weights(fmt, rows, K, seed=rows + K)
    xf = T.normal(K, 0.0, 1.0, seed=K)
    say("full size", fmt, rows, K)
    xd = P.to_device(xf)
    xq_d = P.dev_quantize(xd, T.act_fmt(fmt))
    xq = xq_d.cpu().numpy()
    assert np.array_equal(xq, T.oracle_quantize(xf, T.act_fmt(fmt)))
    Wd = P.to_device(W)
    y = P.dev_gemm_nt(fmt, xq_d, Wd, None, 1, rows, K).cpu().numpy().reshape(-1)
    ref = T.oracle_gemv(fmt, W, xq, rows, K)
    assert T.norm_err(y, ref) <= TOL
    # size-independent properties: determinism, and linearity in the rows
    y2 = P.dev_gemm_nt(fmt, xq_d, Wd, None, 1, rows, K).cpu().numpy().reshape(-1)
    assert np.array_equal(y, y2)
    rb = T.row_bytes(fmt, K)
    perm = np.random.default_rng(1).permutation(rows)
    Wp = np.ascontiguousarray(W.reshape(rows, rb)[perm]).reshape(-1)
    yp = P.dev_gemm_nt(fmt, xq_d, P.to_device(Wp), None, 1, rows, K).cpu().numpy().reshape(-1)
    assert np.array_equal(yp, y[perm])     # a row's result does not depend on where the row sits
    torch.cuda.synchronize()


@pytest.mark.parametrize("M", [2, 4, 8])
def test_batched_decode_small_model_shapes(M):
    """Qwen2-0.5B-like shapes, M tokens (hidden 896 zero-padded to K=1024)."""
    for fmt, rows, K in (("q5_k", 896, 1024), ("q5_k", 128, 1024), ("q5_k", 4864, 1024), ("q5_k", 896, 4864),
                         ("q8_0", 4096, 896)):
        W, _, xq = make_case(fmt, rows, K, "enc", rows + M, tokens=M)
        say("batched decode", fmt, rows, K, "M", M)
        c = P.dev_gemm_nt(fmt, P.to_device(xq), P.to_device(W), None, M, rows, K).cpu().numpy()
        assert T.norm_err(c, T.oracle_gemm_nt(fmt, xq, W, None, M, rows, K)) <= TOL

# ---- fp32 activations, no activation quantization -------------------------------------------

F32_FMTS = ["q4_k", "q6_k", "q8_0"]


@pytest.mark.parametrize("fmt", F32_FMTS)
@pytest.mark.parametrize("kind", ["rand", "enc"])
def test_f32act_golden_fixture(fmt, kind):
    """gemv_q4_k / gemv_q6_k / gemm_nt_q4_k / _q6_k / _q8_0 through the drop-in
    symbols (host pointers) against the reference builds' own outputs."""
    G = T.golden()
    M, K, TOK = (int(v) for v in G["shape"])
    W, xf, bias = G["w_%s_%s" % (fmt, kind)], G["act_f32"], G["bias"]
    say("f32act golden", fmt, kind)
    c = P.gemm_nt_f32act(fmt, xf, W, bias, TOK, M, K)
    for build in ("avx2", "avx512"):
        assert T.norm_err(c.reshape(-1), G["c_%s_%s_f32w_%s" % (fmt, kind, build)]) <= TOL
    if fmt != "q8_0":
        y = P.gemv_f32act(fmt, W, xf, M, K)
        assert T.norm_err(y, G["y_%s_%s_f32w_avx2" % (fmt, kind)]) <= TOL
        assert ckq.lib().dot_q4_k is not None
    Y = P.gemm_f32act(fmt, W, xf, M, TOK, K)                   # Y[n*M + row]
    assert T.norm_err(Y, T.oracle_gemm_nt_f32act(fmt, xf, W, None, TOK, M, K)) <= TOL
    if fmt == "q4_k":
        import ctypes as C
        r = ckq.lib().dot_q4_k(C.c_void_p(W.ctypes.data), C.c_void_p(xf.ctypes.data), K)
        assert abs(r - y[0]) <= TOL * max(1.0, np.abs(y).max())


@pytest.mark.parametrize("fmt", F32_FMTS)
def test_f32act_vs_oracle_shapes(fmt):
    """Ragged row counts, short and long rows, several tokens, device pointers."""
    blk = 32 if fmt == "q8_0" else 256
    for rows, K, M in ((1, blk, 1), (7, 2 * blk, 3), (130, 1024, 2), (257, 4096, 1), (33, 11008 if fmt != "q8_0" else 896, 5)):
        W, xf, _ = make_case(fmt, rows, K, "rand" if rows % 2 else "enc", rows + K, tokens=M)
        bias = T.normal(rows, 0.0, 0.5, seed=rows)
        say("f32act", fmt, rows, K, "M", M)
        c = P.dev_gemm_nt_f32act(fmt, P.to_device(xf), P.to_device(W), P.to_device(bias), M, rows, K).cpu().numpy()
        assert T.norm_err(c.reshape(M, rows), T.oracle_gemm_nt_f32act(fmt, xf, W, bias, M, rows, K)) <= TOL
        # K not a multiple of the block size: nothing is written
    out = np.full(4, 7.0, np.float32)
    getattr(ckq.lib(), "gemv_" + fmt)(P._p(out), P._p(np.zeros(4096, np.uint8)), P._p(np.zeros(100, np.float32)), 4, 100)
    assert np.all(out == 7.0)


def test_f32act_full_size():
    """11008 x 4096 Q4_K with fp32 activations against dequantize-then-matmul in fp64."""
    rows, K = 11008, 4096
    W, xf, _ = make_case("q4_k", rows, K, "enc", 77)
    say("f32act full size")
    y = P.dev_gemm_nt_f32act("q4_k", P.to_device(xf), P.to_device(W), None, 1, rows, K).cpu().numpy().reshape(-1)
    want = T.np_dequant("q4_k", W).reshape(rows, K).astype(np.float64) @ xf.astype(np.float64)
    assert T.norm_err(y, want) <= TOL

# ---- fused producer: rmsnorm -> Q8_K, bit-exact -----------------------------------------------

def test_rmsnorm_q8_k_fused_golden_host_and_device():
    G = T.golden()
    TF, DF, AF = (int(v) for v in G["rms_shape"])
    x, g, eps = G["rms_in"], G["rms_gamma"], float(G["rms_eps"][0])
    say("rmsnorm_q8_k_fused golden")
    assert np.array_equal(P.rmsnorm_q8_k_fused(x, g, TF, DF, AF, eps), G["rms_out"])
    out = P.dev_rmsnorm_q8_k_fused(P.to_device(x), P.to_device(g), TF, DF, AF, eps).cpu().numpy()
    assert np.array_equal(out, G["rms_out"])


@pytest.mark.parametrize("tokens,D,stride", [(513, 256, 256), (513, 1024, 1028), (520, 4096, 4096), (513, 4352, 4352), (2, 4352, 4352),
                                             (3, 8192, 8200), (512, 768, 768), (1, 40704, 40704)])
def test_rmsnorm_q8_k_fused_launch_shapes_bit_exact(tokens, D, stride):
    """Both sides of the token count that takes four waves a row, one to many 256-blocks a wave, rows that no wave count
    divides, padded rows, the longest row that fits."""
    x = T.normal(tokens * stride, 0.0, 3.0, 60 + D)
    x.reshape(tokens, stride)[-1, :256] = 0.0
    g = T.normal(D, 1.0, 0.3, 61 + D)
    say("rmsnorm_q8_k_fused", tokens, D, stride)
    ref = np.zeros(tokens * (D // 256) * 292, np.uint8)
    T.oracle().orc_rmsnorm_q8_k_fused(T.ptr(x), T.ptr(g), T.ptr(ref), tokens, D, stride, ctypes.c_float(1e-6))
    out = P.dev_rmsnorm_q8_k_fused(P.to_device(x), P.to_device(g), tokens, D, stride, 1e-6).cpu().numpy()
    assert np.array_equal(out, ref)


@pytest.mark.parametrize("where", [(0, 3), (3, 252), (17, 18), (62, 255), (31, 32), (0, 255)])
def test_q8_k_scale_is_the_first_of_the_largest(where):
    """Two elements of the largest magnitude and opposite signs: the scale's sign is the first one's, in whichever lanes they are."""
    x = np.clip(T.normal(512, 0.0, 1.0, 71), -3.0, 3.0)
    x[where[0]], x[where[1]] = -7.0, 7.0
    x[256 + where[0]], x[256 + where[1]] = 7.0, -7.0
    assert np.array_equal(P.dev_quantize(P.to_device(x), "q8_k").cpu().numpy(), T.oracle_quantize(x, "q8_k"))


@pytest.mark.parametrize("tokens,D,std,seed", [(1, 256, 1.0, 1), (5, 4096, 1.0, 2), (64, 1024, 30.0, 3),
                                                (3, 11008 // 256 * 256, 1e-3, 4), (512, 4096, 2.0, 5)])
def test_rmsnorm_q8_k_fused_bit_exact_vs_oracle(tokens, D, std, seed):
    x = T.normal(tokens * D, 0.0, std, seed)
    g = T.normal(D, 1.0, 0.3, seed + 50)
    say("rmsnorm_q8_k_fused", tokens, D, std)
    ref = np.zeros(tokens * (D // 256) * 292, np.uint8)
    T.oracle().orc_rmsnorm_q8_k_fused(T.ptr(x), T.ptr(g), T.ptr(ref), tokens, D, D, ctypes.c_float(1e-6))
    out = P.dev_rmsnorm_q8_k_fused(P.to_device(x), P.to_device(g), tokens, D).cpu().numpy()
    assert np.array_equal(out, ref)
    if tokens <= 8:
        # feeding the GEMV: same result as quantized-activation GEMV on the oracle's blocks
        W = T.synth_weights("q4_k", 64, D, seed + 9)
        y = P.dev_gemm_nt("q4_k", P.to_device(out), P.to_device(W), None, tokens, 64, D).cpu().numpy()
        assert T.norm_err(y, T.oracle_gemm_nt("q4_k", ref, W, None, tokens, 64, D)) <= TOL

@pytest.mark.parametrize("tokens,D", [(1, 256), (2, 512), (5, 768), (256, 1280), (257, 1280), (3, 4096), (256, 4352), (1, 16640)])
def test_rmsnorm_q8_k_fused_rows_alone_on_their_cu_bit_exact(tokens, D):
    """Rows that have a CU to themselves read their chains further ahead: one, two, an odd and an even number of runs of 32
    values, the last number of tokens that does so and the first that does not."""
    x, g = T.normal(tokens * D, 0.1, 1.0, seed=D), T.normal(D, 1.0, 0.3, seed=D + 1)
    say("rmsnorm_q8_k_fused, rows alone", tokens, D)
    ref = np.zeros(tokens * (D // 256) * 292, np.uint8)
    T.oracle().orc_rmsnorm_q8_k_fused(T.ptr(x), T.ptr(g), T.ptr(ref), tokens, D, D, ctypes.c_float(1e-6))
    assert np.array_equal(P.dev_rmsnorm_q8_k_fused(P.to_device(x), P.to_device(g), tokens, D).cpu().numpy(), ref)


@pytest.mark.parametrize("tokens,D", [(257, 256), (512, 2304), (512, 4096), (513, 2048), (513, 4352), (700, 8192), (1024, 4096), (1025, 2304), (1025, 8192), (300, 16640)])
def test_rmsnorm_q8_k_fused_rows_that_share_a_cu_bit_exact(tokens, D):
    """More rows than CUs: eight waves a row and four, with and without reading ahead, rows of fewer blocks than waves, of a multiple and of some
    more, rows whose LDS image leaves room for four of them, and one that takes the CU for itself."""
    x, g = T.normal(tokens * D, 0.1, 1.0, seed=D), T.normal(D, 1.0, 0.3, seed=D + 1)
    say("rmsnorm_q8_k_fused, rows that share a CU", tokens, D)
    ref = np.zeros(tokens * (D // 256) * 292, np.uint8)
    T.oracle().orc_rmsnorm_q8_k_fused(T.ptr(x), T.ptr(g), T.ptr(ref), tokens, D, D, ctypes.c_float(1e-6))
    assert np.array_equal(P.dev_rmsnorm_q8_k_fused(P.to_device(x), P.to_device(g), tokens, D).cpu().numpy(), ref)


# ---- row dequantizers and quantized embedding lookup, bit-exact -----------------------------

@pytest.mark.parametrize("fmt", ["q4_k", "q6_k", "q8_0"])
def test_dequant_rows_bit_exact(fmt):
    G = T.golden()
    w, want = G["deq_%s_w" % fmt], G["deq_%s_out" % fmt]
    say("dequant row golden", fmt)
    assert np.array_equal(P.dequant_row(fmt, w, len(want)).view(np.uint32), want.view(np.uint32))
    if fmt != "q8_0":
        # the parity scripts' name for the same routine (reference src/ck_parity_api.c:189-197)
        out = np.zeros(len(want), np.float32)
        getattr(ckq.lib(), "ck_test_dequant_" + fmt)(T.ptr(w), T.ptr(out), len(want))
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
    # larger, against the oracle
    n = 64 * 1024
    W = T.random_blocks(fmt, n // T.ELEMS[fmt], 91)
    ref = np.zeros(n, np.float32)
    getattr(T.oracle(), "orc_dequant_%s_row" % fmt)(T.ptr(W), T.ptr(ref), ctypes.c_size_t(n))
    got = P.dev_dequant_rows(fmt, P.to_device(W), None, 0, None, n, n, 1, 1).cpu().numpy().reshape(-1)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("add_pos", [0, 1])
def test_embedding_forward_golden_and_oracle(fmt, add_pos):
    G = T.golden()
    VOC, ED, AED, CTX, NTOK = (int(v) for v in G["emb_shape"])
    ids, pos, tab = G["emb_ids"], G["emb_pos"], G["emb_table_" + fmt]
    say("embedding golden", fmt, add_pos)
    out = P.embedding_forward(fmt, ids, NTOK, VOC, tab, pos, ED, AED, CTX, add_pos, fill=9.0)
    assert np.array_equal(out.reshape(-1).view(np.uint32), G["emb_out_%s_pos%d" % (fmt, add_pos)].view(np.uint32))
    # a model-sized lookup on the device: 64 tokens of a 32000 x 4096 table (Q8_0: 151936 x 896)
    voc, dim = (151936, 896) if fmt == "q8_0" else (32000, 4096)
    tabL = T.random_blocks(fmt, voc * (dim // T.ELEMS[fmt]), 92)
    idsL = np.random.default_rng(5).integers(-3, voc + 3, size=64).astype(np.int32)
    posL = T.normal(80 * dim, 0.0, 0.1, seed=93)
    ref = np.full(80 * dim, 9.0, np.float32)
    T.oracle().orc_embedding_forward(T.FMT[fmt], T.ptr(idsL), 64, voc, T.ptr(tabL), T.ptr(posL), T.ptr(ref), dim - 8, dim, 80, add_pos)
    got = P.dev_dequant_rows(fmt, P.to_device(tabL), P.to_device(idsL), voc, P.to_device(posL) if add_pos else None,
                             dim - 8, dim, 64, 80).cpu().numpy().reshape(-1)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k", "q8_0"])
@pytest.mark.parametrize("n_row,n_valid", [(256, 256), (512, 511), (768, 2), (4096, 4093), (4352, 4352), (8448, 8447)])
def test_dequant_rows_at_the_edges_of_their_units(fmt, n_row, n_valid):
    """Rows of one block, of a whole number of thread blocks and of some threads more; zeros from an element on that is inside a run of four; rows
    behind the last token; ids outside the vocabulary; positions."""
    voc, rows, tokens = 40, 7, 5
    tab = T.random_blocks(fmt, voc * (n_row // T.ELEMS[fmt]), n_row)
    ids = np.array([0, voc - 1, voc, -1, 17], np.int32)
    pos = T.normal(rows * n_row, 0.0, 0.1, seed=n_row)
    for add_pos in (0, 1):
        ref = np.full(rows * n_row, 9.0, np.float32)
        T.oracle().orc_embedding_forward(T.FMT[fmt], T.ptr(ids), tokens, voc, T.ptr(tab), T.ptr(pos), T.ptr(ref), n_valid, n_row, rows, add_pos)
        say("dequant rows", fmt, n_row, n_valid, add_pos)
        got = P.dev_dequant_rows(fmt, P.to_device(tab), P.to_device(ids), voc, P.to_device(pos) if add_pos else None, n_valid, n_row, tokens, rows)
        assert np.array_equal(got.cpu().numpy().reshape(-1).view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("fmt,n_row,rows", [("q4_k", 512, 16400), ("q4_k", 1280, 3300), ("q4_k", 5376, 800), ("q6_k", 512, 16400), ("q6_k", 768, 2800),
                                            ("q6_k", 5376, 400), ("q8_0", 96, 9), ("q8_0", 1312, 9)])
def test_dequant_rows_of_large_launches_and_uneven_blocks(fmt, n_row, rows):
    """Launches large enough for sixteen elements a thread, and blocks of fewer threads than 256: rows of one block and of two with a last wave that is part
    empty; zeros from an element on that is inside a run of four, rows behind the last token, ids outside the vocabulary, positions."""
    voc, tokens, n_valid = 300, rows - 3, n_row - 5
    width = ctypes.c_int()
    assert ckq.lib().ckq_launch_dequant_form(P.FMT[fmt], n_row, rows, ctypes.byref(width)) == (4 if fmt == "q8_0" else 16)
    assert width.value < 256
    tab = T.random_blocks(fmt, voc * (n_row // T.ELEMS[fmt]), n_row)
    ids = np.random.default_rng(n_row).integers(-2, voc + 2, size=tokens).astype(np.int32)
    pos = T.normal(rows * n_row, 0.0, 0.1, seed=n_row)
    for add_pos in (0, 1):
        ref = np.full(rows * n_row, 9.0, np.float32)
        T.oracle().orc_embedding_forward(T.FMT[fmt], T.ptr(ids), tokens, voc, T.ptr(tab), T.ptr(pos), T.ptr(ref), n_valid, n_row, rows, add_pos)
        say("dequant rows, large launches", fmt, n_row, rows, add_pos)
        got = P.dev_dequant_rows(fmt, P.to_device(tab), P.to_device(ids), voc, P.to_device(pos) if add_pos else None, n_valid, n_row, tokens, rows)
        assert np.array_equal(got.cpu().numpy().reshape(-1).view(np.uint32), ref.view(np.uint32))


# ---- prefill GEMM on the matrix cores (Q4_K, token counts above 16) -------------------------

@pytest.mark.parametrize("M,N,K", [(17, 128, 256), (33, 200, 1024), (64, 96, 512), (100, 333, 2048),
                                   (128, 1, 256), (65, 129, 4096)])
def test_gemm_mfma_q4_k_vs_oracle(M, N, K):
    bias = T.normal(N, 0.0, 0.5, seed=N)
    for kind in ("rand", "enc"):
        W, _, xq = make_case("q4_k", N, K, kind, 700 + M + N, tokens=M)
        say("gemm mfma q4_k", kind, "M", M, "N", N, "K", K)
        ref = T.oracle_gemm_nt("q4_k", xq, W, bias, M, N, K)
        c = P.dev_gemm_nt("q4_k", P.to_device(xq), P.to_device(W), P.to_device(bias), M, N, K).cpu().numpy()
        assert T.norm_err(c, ref) <= TOL, (M, N, K, kind)
        # the matrix-core path and the dot4 path agree token by token
        ab = T.row_bytes("q8_k", K)
        y = P.gemv("q4_k", W, xq[(M - 1) * ab:M * ab].copy(), N, K)
        assert T.norm_err(c[M - 1] - bias, y) <= 2e-6
        ch = P.gemm_nt("q4_k", xq, W, bias, M, N, K)      # host-pointer entry point, same kernel
        assert np.array_equal(ch, c)


def test_gemm_mfma_stored_bsums_and_extremes():
    """Stored bsums are consumed (zeroed bsums drop the min term), and the
    extreme quant values (nibble 15, scale 63, q8 = -128/127) stay exact."""
    M, N, K = 64, 64, 512
    W, _, xq = make_case("q4_k", N, K, "rand", 911, tokens=M)
    xz = xq.copy().reshape(-1, 292)
    xz[:, 260:292] = 0
    xz = xz.reshape(-1)
    ref = T.oracle_gemm_nt("q4_k", xz, W, None, M, N, K)
    c = P.dev_gemm_nt("q4_k", P.to_device(xz), P.to_device(W), None, M, N, K).cpu().numpy()
    assert T.norm_err(c, ref) <= TOL
    # extremes: all nibbles 15, all scales/mins 63, activations alternating -128 / 127
    Wb = W.copy().reshape(-1, 144)
    Wb[:, 4:16] = 0xFF
    Wb[:, 16:] = 0xFF
    Wb = Wb.reshape(-1)
    xb = xq.copy().reshape(-1, 292)
    q = np.where(np.arange(256) % 2 == 0, -128, 127).astype(np.int8)
    xb[:, 4:260] = q.view(np.uint8)
    xb[:, 260:292] = np.tile(np.array([-8] * 16, np.int16).view(np.uint8), 1)
    xb = xb.reshape(-1)
    ref = T.oracle_gemm_nt("q4_k", xb, Wb, None, M, N, K)
    c = P.dev_gemm_nt("q4_k", P.to_device(xb), P.to_device(Wb), None, M, N, K).cpu().numpy()
    assert T.norm_err(c, ref) <= TOL
    # largest positive dot: activations all 127
    xb = xb.reshape(-1, 292)
    xb[:, 4:260] = 127
    xb[:, 260:292] = np.array([127 * 16] * 16, np.int16).view(np.uint8)
    xb = xb.reshape(-1)
    ref = T.oracle_gemm_nt("q4_k", xb, Wb, None, M, N, K)
    c = P.dev_gemm_nt("q4_k", P.to_device(xb), P.to_device(Wb), None, M, N, K).cpu().numpy()
    assert T.norm_err(c, ref) <= TOL


def test_gemm_mfma_full_prefill_shape():
    """M=512, N=11008, K=4096.  The oracle is evaluated on a sample of weight
    rows (the whole product would take minutes on the CPU); every token is
    checked for those rows, and the GEMM is checked against the GEMV kernel on
    whole rows of C for a few tokens."""
    M, N, K = 512, 11008, 4096
    W = T.synth_weights("q4_k", N, K, seed=5150)
    xf = T.normal(M * K, 0.0, 1.0, seed=5151)
    bias = T.normal(N, 0.0, 0.5, seed=5152)
    say("gemm mfma full prefill shape")
    xq_d = P.dev_quantize(P.to_device(xf), "q8_k", rows=M)
    xq = xq_d.cpu().numpy()
    Wd, bd = P.to_device(W), P.to_device(bias)
    c = P.dev_gemm_nt("q4_k", xq_d, Wd, bd, M, N, K).cpu().numpy()
    rb = T.row_bytes("q4_k", K)
    rows = np.array([0, 1, 31, 32, 127, 128, 5000, 5503, 5504, 8191, 8192, 9000, 11006, 11007])
    Wsub = np.ascontiguousarray(W.reshape(N, rb)[rows]).reshape(-1)
    ref = T.oracle_gemm_nt("q4_k", xq, Wsub, np.ascontiguousarray(bias[rows]), M, len(rows), K)
    assert T.norm_err(c[:, rows], ref) <= TOL
    ab = T.row_bytes("q8_k", K)
    for t in (0, 63, 64, 300, 511):
        y = P.dev_gemm_nt("q4_k", P.to_device(xq[t * ab:(t + 1) * ab].copy()), Wd, bd, 1, N, K).cpu().numpy().reshape(-1)
        assert T.norm_err(c[t], y) <= 2e-6, t
    assert np.array_equal(P.dev_gemm_nt("q4_k", xq_d, Wd, bd, M, N, K).cpu().numpy(), c)


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
def test_gemm_mfma_more_tiles_than_block_slots(fmt):
    """A ragged grid larger than the chip holds at once (549 tiles of 64 tokens
    x 128 rows for Q4_K, nine K-blocks), with a bias: blocks of a second round
    start while others still run.  Oracle on weight rows spread over the row
    tiles for every token, whole rows against the GEMV kernel for a few tokens,
    same bits on a second run."""
    M, N, K = 520, 7700, 2304
    W = T.synth_weights(fmt, N, K, seed=5350)
    xf = T.normal(M * K, 0.0, 1.0, seed=5351)
    bias = T.normal(N, 0.0, 0.5, seed=5352)
    say("gemm mfma more tiles than slots", fmt)
    af = P.act_format(fmt)
    xq_d = P.dev_quantize(P.to_device(xf), af, rows=M)
    xq = xq_d.cpu().numpy()
    Wd, bd = P.to_device(W), P.to_device(bias)
    c = P.dev_gemm_nt(fmt, xq_d, Wd, bd, M, N, K).cpu().numpy()
    rb = T.row_bytes(fmt, K)
    rows = np.array([0, 127, 128, 3583, 3584, 7039, 7040, 7167, 7168, 7169, 7423, 7424, 7679, 7680, 7698, 7699])
    Wsub = np.ascontiguousarray(W.reshape(N, rb)[rows]).reshape(-1)
    ref = T.oracle_gemm_nt(fmt, xq, Wsub, np.ascontiguousarray(bias[rows]), M, len(rows), K)
    assert T.norm_err(c[:, rows], ref) <= TOL
    ab = T.row_bytes(af, K)
    for t in (0, 63, 64, 300, 511, 512, 519):
        y = P.dev_gemm_nt(fmt, P.to_device(xq[t * ab:(t + 1) * ab].copy()), Wd, bd, 1, N, K).cpu().numpy().reshape(-1)
        assert T.norm_err(c[t], y) <= 2e-6, t
    assert np.array_equal(P.dev_gemm_nt(fmt, xq_d, Wd, bd, M, N, K).cpu().numpy(), c)


# ---- prefill GEMM on the matrix cores, Q6_K (token counts above 16) --------------------------

@pytest.mark.parametrize("M,N,K", [(17, 128, 256), (33, 200, 1024), (64, 96, 512), (100, 333, 2048),
                                   (128, 1, 256), (65, 129, 4096),
                                   (130, 8320, 256), (512, 4224, 512)])    # the last two use 128-token tiles
def test_gemm_mfma_q6_k_vs_oracle(M, N, K):
    bias = T.normal(N, 0.0, 0.5, seed=N)
    for kind in ("rand", "enc"):
        W, _, xq = make_case("q6_k", N, K, kind, 900 + M + N, tokens=M)
        say("gemm mfma q6_k", kind, "M", M, "N", N, "K", K)
        ref = T.oracle_gemm_nt("q6_k", xq, W, bias, M, N, K)
        c = P.dev_gemm_nt("q6_k", P.to_device(xq), P.to_device(W), P.to_device(bias), M, N, K).cpu().numpy()
        assert T.norm_err(c, ref) <= TOL, (M, N, K, kind)
        # the matrix-core path and the dot4 path agree token by token
        ab = T.row_bytes("q8_k", K)
        for t in (0, M - 1):
            y = P.gemv("q6_k", W, xq[t * ab:(t + 1) * ab].copy(), N, K)
            assert T.norm_err(c[t], y + bias) <= 2e-6
        if N <= 512:
            ch = P.gemm_nt("q6_k", xq, W, bias, M, N, K)      # host-pointer entry point, same kernel
            assert np.array_equal(ch, c)


def test_gemm_mfma_q6_k_extremes():
    """The scaled weight sc * (q - 32) spans [-4064, 4096]; the corners of that
    range and the extreme activations stay exact through the two int8 planes."""
    M, N, K = 64, 64, 512
    W, _, xq = make_case("q6_k", N, K, "rand", 977, tokens=M)
    for ql, qh, sc in ((0x00, 0x00, -128), (0xFF, 0xFF, 127), (0x00, 0x00, 127), (0xFF, 0xFF, -128)):
        Wb = W.copy().reshape(-1, 210)
        Wb[:, 0:128] = ql
        Wb[:, 128:192] = qh
        Wb[:, 192:208] = np.uint8(sc & 0xFF)
        Wb = Wb.reshape(-1)
        for pattern in ("alt", "max", "min"):
            xb = xq.copy().reshape(-1, 292)
            q = {"alt": np.where(np.arange(256) % 2 == 0, -128, 127), "max": np.full(256, 127),
                 "min": np.full(256, -128)}[pattern].astype(np.int8)
            xb[:, 4:260] = q.view(np.uint8)
            xb[:, 260:292] = q.astype(np.int16).reshape(16, 16).sum(axis=1).astype(np.int16).view(np.uint8)
            xb = xb.reshape(-1)
            say("gemm mfma q6_k extremes", ql, sc, pattern)
            ref = T.oracle_gemm_nt("q6_k", xb, Wb, None, M, N, K)
            c = P.dev_gemm_nt("q6_k", P.to_device(xb), P.to_device(Wb), None, M, N, K).cpu().numpy()
            assert T.norm_err(c, ref) <= TOL, (ql, sc, pattern)


def test_gemm_mfma_q6_k_down_projection_shape():
    """M=512, N=4096, K=11008: the oracle on a sample of weight rows for every
    token, and whole rows of C against the GEMV kernel for a few tokens."""
    M, N, K = 512, 4096, 11008
    W = T.synth_weights("q6_k", N, K, seed=6160)
    xf = T.normal(M * K, 0.0, 1.0, seed=6161)
    say("gemm mfma q6_k down projection shape")
    xq_d = P.dev_quantize(P.to_device(xf), "q8_k", rows=M)
    xq = xq_d.cpu().numpy()
    Wd = P.to_device(W)
    c = P.dev_gemm_nt("q6_k", xq_d, Wd, None, M, N, K).cpu().numpy()
    rb = T.row_bytes("q6_k", K)
    rows = np.array([0, 1, 31, 32, 127, 128, 2047, 2048, 4094, 4095])
    Wsub = np.ascontiguousarray(W.reshape(N, rb)[rows]).reshape(-1)
    ref = T.oracle_gemm_nt("q6_k", xq, Wsub, None, M, len(rows), K)
    assert T.norm_err(c[:, rows], ref) <= TOL
    ab = T.row_bytes("q8_k", K)
    for t in (0, 63, 64, 300, 511):
        y = P.dev_gemm_nt("q6_k", P.to_device(xq[t * ab:(t + 1) * ab].copy()), Wd, None, 1, N, K).cpu().numpy().reshape(-1)
        assert T.norm_err(c[t], y) <= 2e-6, t


# ---- fused prefill MLP ------------------------------------------------------------------------

def _q8k_fields(b):
    b = b.reshape(-1, 292)
    return b[:, :4].copy().view(np.float32).reshape(-1), b[:, 4:260].view(np.int8).astype(np.int32), \
        b[:, 260:].copy().view(np.int16).astype(np.int32)


def test_swiglu_q8_k_vs_oracle():
    """SiLU(gate)*up quantized to Q8_K.  The device rounds exp once from double,
    the host's expf is almost always correctly rounded too: block scales agree to
    one unit in the last place, quants differ by at most one in a vanishing
    fraction, and the stored bsums are the sums of the stored quants."""
    rows, k, ld = 37, 1024, 2 * 1024 + 64
    g = T.normal(rows * ld, 0.0, 3.0, seed=4401)
    u = T.normal(rows * ld, 0.0, 1.0, seed=4402)
    g.reshape(rows, ld)[3, 256:512] = 0.0                   # SiLU(0) = 0: a zero block
    g.reshape(rows, ld)[5, :k] *= 30.0                      # saturated SiLU on both sides
    want = np.zeros(rows * (k // 256) * 292, np.uint8)
    T.oracle().orc_swiglu_q8_k(T.ptr(g), T.ptr(u), T.ptr(want), rows, k, ld)
    say("ckq_swiglu_q8_k_dev rows", rows, "k", k, "ld", ld)
    got = P.dev_swiglu_q8_k(P.to_device(g), P.to_device(u), rows, k, ld).cpu().numpy()
    dg, qg, bg = _q8k_fields(got)
    dw, qw, bw = _q8k_fields(want)
    assert np.all(np.abs(dg - dw) <= 1.2e-7 * np.abs(dw))
    assert np.abs(qg - qw).max() <= 1 and np.count_nonzero(qg != qw) <= qg.size // 5000
    assert np.array_equal(bg, qg.reshape(-1, 16, 16).sum(axis=2))
    assert not got.reshape(-1, 292)[3 * (k // 256) + 1].any()


@pytest.mark.parametrize("fmt", ["q4_k", "q6_k"])
def test_fused_mlp_golden_case(fmt):
    """The reference's own output for 70 tokens (host pointers, then device pointers)."""
    G = T.golden()
    SEQ, ED, AED, ID, AID = (int(v) for v in G["mlp_shape"])
    x, w1, b1, b2, w2 = G["mlp_x"], G["mlp_w1"], G["mlp_b1"], G["mlp_b2"], G["mlp_w2_" + fmt]
    want = G["mlp_out_%s_avx2" % fmt].reshape(SEQ, AED)
    say("fused_mlp_swiglu_prefill_w1w2_quant golden", fmt)
    got = P.fused_mlp_swiglu_prefill_w1w2_quant(x, w1, b1, "q8_0", w2, b2, fmt, SEQ, ED, AED, ID, AID)
    assert T.norm_err(got, want) <= TOL
    import torch
    out_d = torch.zeros(SEQ * AED, dtype=torch.float32, device="cuda")
    scr = torch.zeros(16, dtype=torch.uint8, device="cuda")
    d = [P.to_device(a) for a in (x, w1, b1, w2, b2)]          # kept alive across the call
    ckq.lib().fused_mlp_swiglu_prefill_w1w2_quant(
        P._dp(d[0]), P._dp(d[1]), P._dp(d[2]), P.CK_DT["q8_0"], P._dp(d[3]), P._dp(d[4]), P.CK_DT[fmt], P._dp(out_d),
        SEQ, ED, AED, ID, AID, P._dp(scr))
    assert np.array_equal(out_d.cpu().numpy().reshape(SEQ, AED), got)


def test_results_in_device_memory_are_there_when_a_call_returns():
    """The synchronous symbols on device pointers: the result is read at once on another stream, which nothing orders behind the library's, and by a
    copy to the host; short calls and one that takes longer than the library looks for its completion word."""
    import torch
    L = ckq.lib()
    other = torch.cuda.Stream()
    for seq, E, I in [(9, 256, 512), (200, 896, 1024), (4096, 2048, 8192)]:
        x = P.to_device(T.normal(seq * E, 0.0, 1.0, seed=E))
        W1, W2 = P.to_device(T.synth_weights("q8_0", 2 * I, E, seed=85)), P.to_device(T.synth_weights("q4_k", E, I, seed=86))
        scr, want = torch.zeros(16, dtype=torch.uint8, device="cuda"), None
        say("results in device memory", seq, E, I)
        for _ in range(6):
            y = torch.full((seq, E), 7.0, device="cuda")
            torch.cuda.synchronize()
            L.fused_mlp_swiglu_prefill_w1w2_quant(P._dp(x), P._dp(W1), None, P.CK_DT["q8_0"], P._dp(W2), None, P.CK_DT["q4_k"], P._dp(y), seq, E, E, I, I, P._dp(scr))
            with torch.cuda.stream(other):
                seen = y.clone()
            other.synchronize()
            if want is None:
                want = y.cpu()
                assert bool(torch.isfinite(want).all()) and not bool((want == 7.0).any())
            assert torch.equal(seen.cpu(), want) and torch.equal(y.cpu(), want), (seq, E, I)


def test_results_of_every_call_are_there_where_the_caller_reads_them():
    """The five kinds of synchronous call with a result of their own, in ordinary device memory (read at once on another stream, and by a copy) and in
    managed memory (read at once by the CPU): the same bytes as through host memory."""
    import torch
    with open("/proc/self/maps") as f:
        hip = ctypes.CDLL(next(l.split()[-1] for l in f if "libamdhip64" in l))
    L, other = ckq.lib(), torch.cuda.Stream()
    M, K, D, seq, E, I = 96, 1024, 4096, 40, 256, 512
    h = {"W": T.random_blocks("q4_k", M * K // 256, 31), "x": T.oracle_quantize(T.normal(K, 0.0, 1.0, 32), "q8_k"), "f": T.normal(4 * D, 0.0, 1.0, 33),
         "g": T.normal(D, 1.0, 0.1, 34), "xm": T.normal(seq * E, 0.0, 1.0, 35), "W1": T.synth_weights("q8_0", 2 * I, E, seed=36), "W2": T.synth_weights("q4_k", E, I, seed=37),
         "s": np.zeros(16, np.uint8)}
    calls = [("matmul", 4 * M, lambda p, y: L.gemv_q4_k_q8_k(y, p("W"), p("x"), M, K)),
             ("quantize", 4 * D // 256 * 292, lambda p, y: L.quantize_batch_q8_k(p("f"), y, 4, D)),
             ("dequantize", 4 * M * K, lambda p, y: L.dequant_q4_k_row(p("W"), y, M * K)),
             ("rmsnorm", 4 * D // 256 * 292, lambda p, y: L.rmsnorm_q8_k_fused(p("f"), p("g"), y, 4, D, D, 1e-5)),
             ("fused mlp", 4 * seq * E, lambda p, y: L.fused_mlp_swiglu_prefill_w1w2_quant(p("xm"), p("W1"), None, P.CK_DT["q8_0"], p("W2"), None, P.CK_DT["q4_k"], y,
                                                                                           seq, E, E, I, I, p("s")))]
    d = {k: P.to_device(v) for k, v in h.items()}
    managed = ctypes.c_void_p()
    assert hip.hipMallocManaged(ctypes.byref(managed), ctypes.c_size_t(4 * M * K), 1) == 0
    try:
        for name, n, call in calls:
            say("results where the caller reads them", name)
            want = np.zeros(n, np.uint8)
            call(lambda k: T.ptr(h[k]), T.ptr(want))
            for _ in range(4):
                y = torch.full((n,), 0x55, dtype=torch.uint8, device="cuda")
                torch.cuda.synchronize()
                call(lambda k: P._dp(d[k]), P._dp(y))
                with torch.cuda.stream(other):
                    seen = y.clone()
                other.synchronize()
                assert np.array_equal(seen.cpu().numpy(), want) and np.array_equal(y.cpu().numpy(), want), name
                ctypes.memset(managed, 0x55, n)
                call(lambda k: P._dp(d[k]), managed)
                assert ctypes.string_at(managed, n) == want.tobytes(), name
    finally:
        torch.cuda.synchronize()
        assert hip.hipFree(managed) == 0


@pytest.mark.parametrize("fmt,seq,E,I,bias", [("q4_k", 130, 896, 4864, True), ("q6_k", 33, 256, 1024, False),
                                              ("q4_k", 1, 64, 256, True), ("q6_k", 512, 128, 512, True)])
def test_fused_mlp_vs_oracle(fmt, seq, E, I, bias):
    """Stage by stage, each stage of the oracle fed with the device's previous
    stage: between the two GEMMs sits a quantizer, and a last-place difference
    in a gate value (the GEMMs sum in different orders) can move one quant by a
    whole step, which no fp32 tolerance on the end result accounts for.  The
    fused call must equal the chain of its stages bit for bit, and stay within
    a few quantization flips of the all-CPU result end to end."""
    import torch
    x = T.normal(seq * E, 0.0, 1.0, seed=4500 + seq)
    w1 = T.synth_weights("q8_0", 2 * I, E, seed=4501 + seq, std=0.25)
    w2 = T.synth_weights(fmt, E, I, seed=4502 + seq)
    b1 = T.normal(2 * I, 0.0, 0.3, seed=4503) if bias else None
    b2 = T.normal(E, 0.0, 0.3, seed=4504) if bias else None
    say("fused mlp", fmt, "seq", seq, "E", E, "I", I, "bias", bias)
    got = P.fused_mlp_swiglu_prefill_w1w2_quant(x, w1, b1, "q8_0", w2, b2, fmt, seq, E, E, I, I)
    # stage 1: Q8_0 of x, bit-exact
    xq_d = P.dev_quantize(P.to_device(x), "q8_0", rows=seq)
    xq = xq_d.cpu().numpy()
    assert np.array_equal(xq, T.oracle_quantize(x, "q8_0", rows=seq))
    # stage 2: gate and up in one GEMM over the stacked rows
    w1_d, b1_d = P.to_device(w1), (P.to_device(b1) if bias else None)
    gu_d = P.dev_gemm_nt("q8_0", xq_d, w1_d, b1_d, seq, 2 * I, E)
    gu = gu_d.cpu().numpy().reshape(seq, 2 * I)
    assert T.norm_err(gu, T.oracle_gemm_nt("q8_0", xq, w1, b1, seq, 2 * I, E)) <= TOL
    # stage 3: SiLU(gate)*up -> Q8_K, oracle applied to the device's gate and up
    h_d = P.dev_swiglu_q8_k(gu_d, gu_d.view(-1)[I:], seq, I, 2 * I)
    h = h_d.cpu().numpy()
    want_h = np.zeros_like(h)
    guc = np.ascontiguousarray(gu).reshape(-1)
    T.oracle().orc_swiglu_q8_k(T.ptr(guc), T.ptr(guc[I:]), T.ptr(want_h), seq, I, 2 * I)
    dg, qg, _ = _q8k_fields(h)
    dw, qw, _ = _q8k_fields(want_h)
    assert np.all(np.abs(dg - dw) <= 1.2e-7 * np.abs(dw))
    assert np.abs(qg - qw).max() <= 1 and np.count_nonzero(qg != qw) <= max(2, qg.size // 5000)
    # stage 4: the down GEMM on the device's Q8_K
    w2_d, b2_d = P.to_device(w2), (P.to_device(b2) if bias else None)
    out_d = P.dev_gemm_nt(fmt, h_d, w2_d, b2_d, seq, E, I)
    out = out_d.cpu().numpy().reshape(seq, E)
    assert T.norm_err(out, T.oracle_gemm_nt(fmt, h, w2, b2, seq, E, I)) <= TOL
    # the fused entry point is exactly that chain
    assert np.array_equal(got, out)
    # end to end against the all-CPU chain: fp32 tolerance plus a few quantization flips
    want = T.oracle_fused_mlp(x, w1, b1, w2, b2, fmt, seq, E, E, I, I)
    assert T.norm_err(got, want) <= 5e-3
    assert np.mean(np.abs(got - want) <= TOL * np.abs(want).max()) >= 0.98


def test_fused_mlp_argument_errors_leave_output_untouched():
    G = T.golden()
    SEQ, ED, AED, ID, AID = (int(v) for v in G["mlp_shape"])
    x, w1, w2 = G["mlp_x"], G["mlp_w1"], G["mlp_w2_q4_k"]
    mk = lambda: np.full(SEQ * AED, 7.0, np.float32)
    say("fused mlp argument errors")
    for kw in (dict(w1_fmt="q4_k"), dict(w2_fmt="q8_0")):
        out = mk()
        P.fused_mlp_swiglu_prefill_w1w2_quant(x, w1, None, kw.get("w1_fmt", "q8_0"), w2, None, kw.get("w2_fmt", "q4_k"),
                                              SEQ, ED, AED, ID, AID, output=out)
        assert np.all(out == 7.0), kw
    for dims in ((0, ED, AED, ID, AID), (SEQ, ED, AED + 8, ID, AID), (SEQ, ED, AED, ID, AID + 32),
                 (SEQ, AED + 1, AED, ID, AID), (SEQ, ED, AED, AID + 1, AID)):
        out = mk()
        P.fused_mlp_swiglu_prefill_w1w2_quant(x, w1, None, "q8_0", w2, None, "q4_k", *dims, output=out)
        assert np.all(out == 7.0), dims
    out = mk()
    P.fused_mlp_swiglu_prefill_w1w2_quant(x, w1, None, "q8_0", w2, None, "q4_k", SEQ, ED, AED, ID, AID, output=out,
                                          scratch=False)
    assert np.all(out == 7.0)
    assert int(ckq.lib().fused_mlp_swiglu_prefill_w1w2_quant_scratch_size(AED, AID)) == int(G["mlp_scratch_size"][0])


# ---- prefill GEMM on the matrix cores, Q8_0 (token counts above 16) --------------------------

@pytest.mark.parametrize("M,N,K", [(17, 128, 128), (33, 200, 96), (64, 96, 160), (100, 333, 896), (128, 1, 32),
                                   (65, 129, 4096), (130, 1030, 64), (512, 512, 416)])
def test_gemm_mfma_q8_0_vs_oracle(M, N, K):
    bias = T.normal(N, 0.0, 0.5, seed=N)
    for kind in ("rand", "enc"):
        W, _, xq = make_case("q8_0", N, K, kind, 1100 + M + N, tokens=M)
        say("gemm mfma q8_0", kind, "M", M, "N", N, "K", K)
        ref = T.oracle_gemm_nt("q8_0", xq, W, bias, M, N, K)
        c = P.dev_gemm_nt("q8_0", P.to_device(xq), P.to_device(W), P.to_device(bias), M, N, K).cpu().numpy()
        assert T.norm_err(c, ref) <= TOL, (M, N, K, kind)
        # the matrix-core path and the dot4 path agree token by token
        ab = T.row_bytes("q8_0", K)
        for t in (0, M - 1):
            y = P.gemv("q8_0", W, xq[t * ab:(t + 1) * ab].copy(), N, K)
            assert T.norm_err(c[t], y + bias) <= 2e-6
        if N <= 512:
            ch = P.gemm_nt("q8_0", xq, W, None, M, N, K)      # host-pointer entry point, same kernel, no bias
            assert T.norm_err(ch, ref - bias) <= TOL
            ldc = N + 3                                        # unaligned row pitch: scalar stores
            cd = P.to_device(np.full(M * ldc, 5.0, np.float32))
            xq_d, W_d = P.to_device(xq), P.to_device(W)        # kept alive across the call
            P.check(ckq.lib().ckq_gemm_nt_dev(P.FMT["q8_0"], P._dp(xq_d), P._dp(W_d), None, P._dp(cd),
                                              M, N, K, ldc, P._stream()), "ckq_gemm_nt_dev")
            cdn = cd.cpu().numpy().reshape(M, ldc)
            assert np.array_equal(cdn[:, :N], ch) and np.all(cdn[:, N:] == 5.0)


def test_gemm_mfma_q8_0_extremes():
    """All quants at -128 / 127 on both sides and the largest finite fp16 scales
    that keep the result finite: the int32 block sums are exact."""
    M, N, K = 64, 64, 256
    W, _, xq = make_case("q8_0", N, K, "rand", 1177, tokens=M)
    for wq, xqv in ((127, 127), (-128, -128), (-128, 127)):
        Wb = W.copy().reshape(-1, 34)
        Wb[:, 2:] = np.uint8(wq & 0xFF)
        Wb[:, 0:2] = np.array([1.5], np.float16).view(np.uint8)
        xb = xq.copy().reshape(-1, 34)
        xb[:, 2:] = np.uint8(xqv & 0xFF)
        xb[:, 0:2] = np.array([0.75], np.float16).view(np.uint8)
        say("gemm mfma q8_0 extremes", wq, xqv)
        ref = T.oracle_gemm_nt("q8_0", xb.reshape(-1), Wb.reshape(-1), None, M, N, K)
        c = P.dev_gemm_nt("q8_0", P.to_device(xb.reshape(-1)), P.to_device(Wb.reshape(-1)), None, M, N, K).cpu().numpy()
        assert np.array_equal(c, ref)        # every term is exact in fp32 here
        assert c[0, 0] == np.float32(1.5 * 0.75 * wq * xqv * 32 * (K // 32))


# ---- prefill GEMM on the matrix cores, Q5_K (token counts above 16) --------------------------

@pytest.mark.parametrize("M,N,K", [(65, 128, 256), (70, 200, 1024), (66, 96, 512), (100, 333, 2048),
                                   (128, 1, 256), (97, 129, 4864), (512, 896, 1024)])
def test_gemm_mfma_q5_k_vs_oracle(M, N, K):
    bias = T.normal(N, 0.0, 0.5, seed=N)
    for kind in ("rand", "enc"):
        W, _, xq = make_case("q5_k", N, K, kind, 1300 + M + N, tokens=M)
        say("gemm mfma q5_k", kind, "M", M, "N", N, "K", K)
        ref = T.oracle_gemm_nt("q5_k", xq, W, bias, M, N, K)
        c = P.dev_gemm_nt("q5_k", P.to_device(xq), P.to_device(W), P.to_device(bias), M, N, K).cpu().numpy()
        assert T.norm_err(c, ref) <= TOL, (M, N, K, kind)
        # the matrix-core path and the dot4 path agree token by token
        ab = T.row_bytes("q8_k", K)
        for t in (0, M - 1):
            y = P.gemv("q5_k", W, xq[t * ab:(t + 1) * ab].copy(), N, K)
            assert T.norm_err(c[t], y + bias) <= 2e-6
        if N <= 512:
            ch = P.gemm_nt("q5_k", xq, W, bias, M, N, K)      # host-pointer entry point, same kernel
            assert np.array_equal(ch, c)


def test_gemm_mfma_q5_k_stored_bsums_and_extremes():
    """Stored bsums are consumed (zeroed bsums drop the min term), and the
    extreme values (5-bit value 31, scale and min 63, q8 = -128 / 127, bsums at
    both ends of their range) stay exact through the split operands."""
    M, N, K = 96, 64, 512
    W, _, xq = make_case("q5_k", N, K, "rand", 1311, tokens=M)
    xz = xq.copy().reshape(-1, 292)
    xz[:, 260:292] = 0
    xz = xz.reshape(-1)
    say("gemm mfma q5_k zeroed bsums")
    ref = T.oracle_gemm_nt("q5_k", xz, W, None, M, N, K)
    c = P.dev_gemm_nt("q5_k", P.to_device(xz), P.to_device(W), None, M, N, K).cpu().numpy()
    assert T.norm_err(c, ref) <= TOL
    Wb = W.copy().reshape(-1, 176)
    Wb[:, 4:16] = 0xFF          # all scales and mins 63
    Wb[:, 16:] = 0xFF           # all fifth bits and nibbles set: every value 31
    Wb = Wb.reshape(-1)
    for pattern in ("alt", "max", "min"):
        xb = xq.copy().reshape(-1, 292)
        q = {"alt": np.where(np.arange(256) % 2 == 0, -128, 127), "max": np.full(256, 127),
             "min": np.full(256, -128)}[pattern].astype(np.int8)
        xb[:, 4:260] = q.view(np.uint8)
        xb[:, 260:292] = q.astype(np.int16).reshape(16, 16).sum(axis=1).astype(np.int16).view(np.uint8)
        xb = xb.reshape(-1)
        say("gemm mfma q5_k extremes", pattern)
        ref = T.oracle_gemm_nt("q5_k", xb, Wb, None, M, N, K)
        c = P.dev_gemm_nt("q5_k", P.to_device(xb), P.to_device(Wb), None, M, N, K).cpu().numpy()
        assert T.norm_err(c, ref) <= TOL, pattern


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k"])
@pytest.mark.parametrize("M,N,K", [(1, 70, 1280), (5, 300, 512), (13, 96, 2816), (16, 4100, 1024), (24, 200, 512), (30, 2100, 2560), (70, 200, 2304), (100, 130, 512)])
def test_stored_bsums_of_any_sixteen_bits(fmt, M, N, K):
    """Stored bsums that no int8 quants sum to, pairs of them up to +-2^15: eight times a pair of the quantizer's.  Every kernel that serves the size against the oracle, whose
    min term is an integer.  The bar: the rounding of up to eleven fp32 terms and their sums, 16 x 2^-24 of the terms' absolute sum, which is at most some five
    times the largest result here; a part of a pair cut to bf16 that does not fit it errs by 1e-4 and more."""
    W, _, xq = make_case(fmt, N, K, "rand", 1400 + M, tokens=M)
    rng = np.random.default_rng(M + K)
    xb = xq.copy().reshape(-1, 292)
    stored = rng.integers(-16384, 16384, size=(xb.shape[0], 16)).astype(np.int16)
    stored[0], stored[-1] = 16383, -16384
    xb[:, 260:292] = stored.view(np.uint8)
    xb = xb.reshape(-1)
    say("stored bsums of any value", fmt, M, N, K)
    ref = T.oracle_gemm_nt(fmt, xb, W, None, M, N, K)
    L, tag = ckq.lib(), P.FMT[fmt]
    Xd, Wd = P.to_device(xb), P.to_device(W)
    forms = [(0, 0), (2, 0), (2, 16)] + ([(1, v) for v in (0, 16) + ((64, 96) if fmt == "q4_k" else (1, 2))] if M > 8 else [])
    try:
        for policy, variant in forms:
            L.ckq_set_prefill_variant(tag, variant)
            L.ckq_set_gemm_policy(policy)
            c = P.dev_gemm_nt(fmt, Xd, Wd, None, M, N, K).cpu().numpy().reshape(M, N)
            assert T.norm_err(c, ref) <= 5e-6, (policy, variant)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


# ---- loader hook: registered weight regions ---------------------------------------------------

def test_weights_register_manifest_and_ranges(tmp_path):
    """A weight arena laid out by a manifest (as the reference's loader fills it):
    the hook uploads the quantized tensors once; calls with host pointers into
    the arena - whole tensors, row ranges of them, the gate or up half of a
    stacked matrix - are served from those regions without new uploads."""
    L = ckq.lib()
    L.ckq_weights_clear()
    N, K = 48, 512
    wa = T.synth_weights("q4_k", N, K, seed=9101)
    wb = T.synth_weights("q6_k", N, K, seed=9102)
    arena = np.zeros(4096 + len(wa) + 64 + len(wb) + 512, np.uint8)
    oa, ob = 4096, 4096 + len(wa) + 64
    arena[oa:oa + len(wa)] = wa
    arena[ob:ob + len(wb)] = wb
    arena[:4096].view(np.float32)[:] = 1.0                       # an fp32 tensor the hook must skip
    m = tmp_path / "weights_manifest.map"
    m.write_text("# name|dtype|file_offset|size|runtime_offset\n"
                 "model.norm.weight|fp32|8|4096|0\n"
                 "model.layers.0.wq|Q4_K|4104|%d|%d\n"
                 "model.layers.0.wdown|q6k|0x%x|%d|%d\n" % (len(wa), oa, 4104 + len(wa), len(wb), ob))
    say("ckq_weights_register_manifest")
    assert L.ckq_weights_register_manifest(T.ptr(arena), str(m).encode()) == 2
    nbytes = ctypes.c_size_t(0)
    assert L.ckq_weights_resident(ctypes.byref(nbytes)) == 2 and nbytes.value == len(wa) + len(wb)
    xq = T.oracle_quantize(T.normal(K, seed=9103), "q8_k")
    ya = P.gemv("q4_k", arena[oa:oa + len(wa)], xq, N, K)          # views: host pointers into the arena
    yb = P.gemv("q6_k", arena[ob:ob + len(wb)], xq, N, K)
    assert T.norm_err(ya, T.oracle_gemv("q4_k", wa, xq, N, K)) <= TOL
    assert T.norm_err(yb, T.oracle_gemv("q6_k", wb, xq, N, K)) <= TOL
    rb = T.row_bytes("q4_k", K)
    ysub = P.gemv("q4_k", arena[oa + 8 * rb:oa + 40 * rb], xq, 32, K)   # rows 8..39 of the first tensor
    assert np.array_equal(ysub, ya[8:40])
    assert L.ckq_weights_resident(None) == 2                       # nothing new was uploaded
    # a registered region is not re-checked: new content needs invalidate
    arena[oa:oa + len(wa)] = T.synth_weights("q4_k", N, K, seed=9104)
    assert np.array_equal(P.gemv("q4_k", arena[oa:oa + len(wa)], xq, N, K), ya)
    L.ckq_weights_invalidate(T.ptr(arena[oa:]))
    assert L.ckq_weights_resident(None) == 1
    y2 = P.gemv("q4_k", arena[oa:oa + len(wa)], xq, N, K)
    assert T.norm_err(y2, T.oracle_gemv("q4_k", arena[oa:oa + len(wa)].copy(), xq, N, K)) <= TOL
    L.ckq_weights_clear()
    assert L.ckq_weights_resident(None) == 0


# ---- K-split prefill GEMMs ----------------------------------------------------------------------

@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k", "q8_0"])
def test_gemm_split_k_is_deterministic_and_matches_oracle(fmt):
    """Few tiles and a long K: the launch splits K over several blocks per tile
    and sums the partial tiles in a fixed order.  Same bits on every run, the
    oracle's values within the fp32 tolerance, bias added once."""
    M, N, K = 96, 200, 19 * 256          # 4 tiles, 19 (or 38) K-steps: a ragged last split
    bias = T.normal(N, 0.0, 0.5, seed=77)
    W, _, xq = make_case(fmt, N, K, "enc", 1500 + T.FMT[fmt], tokens=M)
    say("split-K gemm", fmt)
    xq_d, W_d, b_d = P.to_device(xq), P.to_device(W), P.to_device(bias)
    c0 = P.dev_gemm_nt(fmt, xq_d, W_d, b_d, M, N, K).cpu().numpy()
    ref = T.oracle_gemm_nt(fmt, xq, W, bias, M, N, K)
    assert T.norm_err(c0, ref) <= TOL
    for _ in range(3):
        assert np.array_equal(P.dev_gemm_nt(fmt, xq_d, W_d, b_d, M, N, K).cpu().numpy(), c0)
    # a second stream gets its own scratch
    import torch
    st = torch.cuda.Stream()
    with torch.cuda.stream(st):
        c1 = P.dev_gemm_nt(fmt, xq_d, W_d, b_d, M, N, K)
    st.synchronize()
    assert np.array_equal(c1.cpu().numpy(), c0)


def test_gemm_mfma_q4_k_two_wave_groups_per_tile():
    """160 tiles and nine K-blocks: one tile per CU, so the launch gives every
    tile two groups of waves that take alternate K-blocks (five and four) and
    add their partial tiles in a fixed order.  The oracle on a sample of weight
    rows for every token, whole rows against the GEMV kernel for a few tokens,
    and the same bits on a second run."""
    M, N, K = 512, 2560, 2304
    W = T.synth_weights("q4_k", N, K, seed=5250)
    xf = T.normal(M * K, 0.0, 1.0, seed=5251)
    bias = T.normal(N, 0.0, 0.5, seed=5252)
    say("gemm mfma q4_k two wave groups")
    xq_d = P.dev_quantize(P.to_device(xf), "q8_k", rows=M)
    xq = xq_d.cpu().numpy()
    Wd, bd = P.to_device(W), P.to_device(bias)
    c = P.dev_gemm_nt("q4_k", xq_d, Wd, bd, M, N, K).cpu().numpy()
    rb = T.row_bytes("q4_k", K)
    rows = np.array([0, 1, 31, 32, 127, 128, 1279, 1280, 2558, 2559])
    Wsub = np.ascontiguousarray(W.reshape(N, rb)[rows]).reshape(-1)
    ref = T.oracle_gemm_nt("q4_k", xq, Wsub, np.ascontiguousarray(bias[rows]), M, len(rows), K)
    assert T.norm_err(c[:, rows], ref) <= TOL
    ab = T.row_bytes("q8_k", K)
    for t in (0, 63, 64, 300, 511):
        y = P.dev_gemm_nt("q4_k", P.to_device(xq[t * ab:(t + 1) * ab].copy()), Wd, bd, 1, N, K).cpu().numpy().reshape(-1)
        assert T.norm_err(c[t], y) <= 2e-6, t
    assert np.array_equal(P.dev_gemm_nt("q4_k", xq_d, Wd, bd, M, N, K).cpu().numpy(), c)


# ---- matrix-core GEMMs on seeded random shapes ---------------------------------------------------

@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k", "q8_0"])
def test_gemm_mfma_random_shapes(fmt):
    """Ragged token counts, row counts that are no multiple of the 32-row wave
    slice or the 128-row tile, K from one block up, with and without bias and
    with a row pitch wider than N: every combination a tile edge can meet."""
    import torch
    rng = np.random.default_rng(20240 + T.FMT[fmt])
    lo = 65 if fmt == "q5_k" else 17
    for case in range(10):
        M = int(rng.integers(lo, 210))
        N = int(rng.integers(1, 300))
        K = int(rng.integers(1, 21)) * 32 if fmt == "q8_0" else int(rng.integers(1, 7)) * 256
        use_bias = bool(case & 1)
        ldc = N + int(rng.integers(0, 9)) if case % 3 == 0 else N
        W, _, xq = make_case(fmt, N, K, "enc" if case & 2 else "rand", 7000 + 31 * case + T.FMT[fmt], tokens=M)
        bias = T.normal(N, 0.0, 0.5, seed=case) if use_bias else None
        say("gemm mfma random", fmt, "M", M, "N", N, "K", K, "ldc", ldc, "bias", use_bias)
        ref = T.oracle_gemm_nt(fmt, xq, W, bias, M, N, K)
        xq_d, W_d = P.to_device(xq), P.to_device(W)
        b_d = P.to_device(bias) if use_bias else None
        c_d = torch.full((M * ldc,), 3.0, dtype=torch.float32, device="cuda")
        P.check(ckq.lib().ckq_gemm_nt_dev(P.FMT[fmt], P._dp(xq_d), P._dp(W_d), P._dp(b_d), P._dp(c_d), M, N, K, ldc,
                                          P._stream()), "ckq_gemm_nt_dev")
        c = c_d.cpu().numpy().reshape(M, ldc)
        assert T.norm_err(c[:, :N], ref) <= TOL, (fmt, M, N, K, ldc)
        assert np.all(c[:, N:] == 3.0), (fmt, M, N, K, ldc)         # nothing written beyond a row's N outputs


# ---- Q5_0 weights x Q8_0 activations ------------------------------------------------------------

def test_q5_0_subblock_dots_and_gemv_k_sweep():
    rows = 41
    for K in (32, 128, 512, 896, 1024, 2048, 4096, 8192, 10240):
        for kind in ("rand", "enc"):
            W, _, xq = make_case("q5_0", rows, K, kind, 60 + K)
            say("q5_0", kind, "rows", rows, "K", K)
            W_d, xq_d = P.to_device(W), P.to_device(xq)
            got = P.dev_subblock_dots("q5_0", W_d, xq_d, rows, K).cpu().numpy()
            assert np.array_equal(got, T.oracle_subdots("q5_0", W, xq, rows, K)), K
            y = P.dev_gemm_nt("q5_0", xq_d, W_d, None, 1, rows, K).cpu().numpy().reshape(-1)
            assert T.norm_err(y, T.oracle_gemv("q5_0", W, xq, rows, K)) <= TOL, (K, kind)


@pytest.mark.parametrize("kind", ["rand", "enc"])
def test_q5_0_golden_fixture(kind):
    G = T.golden()
    M, K, TOK = (int(v) for v in G["shape"])
    W, xq = G["w_q5_0_" + kind], G["act_q80"]
    say("q5_0 golden", kind)
    y = P.gemv("q5_0", W, xq, M, K)
    c = P.gemm_nt("q5_0", xq, W, G["bias"], TOK, M, K)
    for build in ("avx2", "avx512"):
        assert T.norm_err(y, G["y_q5_0_%s_%s" % (kind, build)]) <= TOL
        assert T.norm_err(c, G["c_q5_0_%s_%s" % (kind, build)].reshape(TOK, M)) <= TOL
    s = np.zeros(1, np.float32)
    ckq.lib().vec_dot_q5_0_q8_0(K, T.ptr(s), T.ptr(W), T.ptr(xq))
    assert abs(float(s[0]) - float(G["s_q5_0_%s_vecdot" % kind][0])) <= TOL * np.abs(y).max()
    yp = np.zeros(M, np.float32)
    for ith in range(5):
        ckq.lib().gemv_q5_0_q8_0_parallel_simd(T.ptr(yp), T.ptr(W), T.ptr(xq), M, K, ith, 5)
    assert np.array_equal(yp, y)


def test_q5_0_row_and_token_counts():
    """Token tiles up to eight tokens; above that (forced here, this matrix is
    small) the blocks are rewritten as Q8_0 blocks and the Q8_0 matrix-core GEMM
    runs: the same bits as that GEMM on weights converted by the oracle."""
    K = 896
    for rows in (1, 3, 17, 64, 65, 257):
        W, _, xq = make_case("q5_0", rows, K, "rand", 11 * rows)
        say("q5_0 rows", rows)
        assert T.norm_err(P.gemv("q5_0", W, xq, rows, K), T.oracle_gemv("q5_0", W, xq, rows, K)) <= TOL, rows
    N = 77
    bias = T.normal(N, 0.0, 0.5, seed=8)
    for M in (1, 2, 5, 8, 9, 16, 17, 33, 130, 512):
        W, _, xq = make_case("q5_0", N, K, "enc", 310 + M, tokens=M)
        say("q5_0 gemm_nt tokens", M)
        ref = T.oracle_gemm_nt("q5_0", xq, W, bias, M, N, K)
        c = P.gemm_nt("q5_0", xq, W, bias, M, N, K)
        assert T.norm_err(c, ref) <= TOL, M
        if M > 8:
            w8 = np.zeros(len(W) // 22 * 34, np.uint8)
            T.oracle().orc_q5_0_to_q8_0(T.ptr(W), T.ptr(w8), ctypes.c_size_t(len(W) // 22))
            assert np.array_equal(P.gemm_nt("q8_0", xq, w8, bias, M, N, K), c), M


def test_fused_mlp_q5_0_gate_up_golden_case():
    G = T.golden()
    SEQ, ED, AED, ID, AID = (int(v) for v in G["mlp_shape"])
    say("fused mlp q5_0 gate/up golden")
    got = P.fused_mlp_swiglu_prefill_w1w2_quant(G["mlp_x"], G["mlp_w1_q5_0"], G["mlp_b1"], "q5_0", G["mlp_w2_q4_k"],
                                                G["mlp_b2"], "q4_k", SEQ, ED, AED, ID, AID)
    assert T.norm_err(got, G["mlp_out_q5_0w1_q4_k_avx2"].reshape(SEQ, AED)) <= TOL


@pytest.mark.parametrize("seq,E,I", [(70, 64, 4864), (200, 896, 1024), (129, 928, 1280), (512, 896, 4864), (9, 256, 512)])
def test_fused_mlp_q5_0_equals_its_steps(seq, E, I):
    """Activations quantized and weights rewritten by one launch (gate and up on the matrix cores; even and odd numbers of blocks a row, last
    blocks of either part partly filled; the last size streams): the output is that of the steps called one by one, to the bit."""
    import torch
    L = ckq.lib()
    x = P.to_device(T.normal(seq * E, 0.0, 1.0, seed=E))
    W1, W2 = P.to_device(T.random_blocks("q5_0", 2 * I * E // 32, 81)), P.to_device(T.synth_weights("q4_k", E, I, seed=82))
    b1, b2 = P.to_device(T.normal(2 * I, 0.0, 0.1, seed=83)), P.to_device(T.normal(E, 0.0, 0.1, seed=84))
    y, scr = torch.zeros(seq, E, device="cuda"), torch.zeros(16, dtype=torch.uint8, device="cuda")
    say("fused mlp q5_0, one launch for both operands", seq, E, I)
    L.fused_mlp_swiglu_prefill_w1w2_quant(P._dp(x), P._dp(W1), P._dp(b1), P.CK_DT["q5_0"], P._dp(W2), P._dp(b2), P.CK_DT["q4_k"], P._dp(y),
                                          seq, E, E, I, I, P._dp(scr))
    gu = P.dev_gemm_nt("q5_0", P.dev_quantize(x, "q8_0", rows=seq), W1, b1, seq, 2 * I, E).view(seq, 2 * I)
    h = P.dev_swiglu_q8_k(gu.view(-1), gu.view(-1)[I:], seq, I, 2 * I)
    want = P.dev_gemm_nt("q4_k", h, W2, b2, seq, E, I).view(seq, E)
    assert bool(torch.isfinite(want).all()) and torch.equal(y, want)


# ---- automatic choice between the streaming kernel and the matrix cores --------------------------

@pytest.mark.parametrize("fmt,N,K,expect", [
    ("q4_k", 4096, 4096, {8: "stream", 9: "stream", 16: "stream", 17: "matrix"}),      # 9.4 MB: two passes stream
    ("q4_k", 11008, 4096, {8: "stream", 9: "matrix"}),                                  # 25 MB
    ("q6_k", 1024, 4096, {16: "stream", 40: "stream", 49: "matrix"}),                   # 3.4 MB
    ("q8_0", 4864, 896, {64: "stream", 72: "stream", 73: "matrix"}),                    # 4.6 MB, aligned-load streaming
    ("q8_0", 32000, 4096, {16: "stream", 17: "matrix"}),                                # 139 MB: two passes still stream
    ("q5_k", 4864, 1024, {64: "stream", 96: "stream", 100: "matrix"}),                  # 3.3 MB, 40 MB budget
    ("q5_0", 896, 896, {48: "stream", 57: "matrix"}),                                   # below the 3 MB floor
])
def test_gemm_automatic_kernel_choice(fmt, N, K, expect):
    """With the default policy the library picks the kernel by token count and
    weight size.  Each result matches the oracle on a sample of rows, and equals
    bit for bit what the kernel it should have picked gives when forced."""
    L = ckq.lib()
    W = T.random_blocks(fmt, N * (K // T.ELEMS[fmt]), 4242)
    Wd = P.to_device(W)
    rb = T.row_bytes(fmt, K)
    rows = np.array([0, 1, N // 2, N - 1])
    Wsub = np.ascontiguousarray(W.reshape(N, rb)[rows]).reshape(-1)
    for M, which in expect.items():
        say("automatic kernel choice", fmt, N, K, M, which)
        xq = T.oracle_quantize(T.normal(M * K, 0.0, 1.0, 500 + M), T.act_fmt(fmt), rows=M)
        xd = P.to_device(xq)
        L.ckq_set_gemm_policy(0)
        auto = P.dev_gemm_nt(fmt, xd, Wd, None, M, N, K).cpu().numpy()
        assert T.norm_err(auto[:, rows], T.oracle_gemm_nt(fmt, xq, Wsub, None, M, len(rows), K)) <= TOL, M
        L.ckq_set_gemm_policy(1 if which == "matrix" else 2)
        forced = P.dev_gemm_nt(fmt, xd, Wd, None, M, N, K).cpu().numpy()
        L.ckq_set_gemm_policy(0)
        assert np.array_equal(auto, forced), (M, which)


# ---- sequences: independent entries of one shape share a launch ----------------------------------

@pytest.mark.parametrize("fmt,N,K", [("q4_k", 384, 1024), ("q6_k", 200, 512), ("q8_0", 130, 896), ("q5_k", 96, 768)])
def test_matmul_sequence_groups_independent_entries(fmt, N, K):
    """Q/K/V-like entries (one input, separate weights and outputs, K and V
    narrower than Q) and a pair with separate inputs go out as grouped launches
    at one token; every output has the bits of the same matmul launched alone,
    with and without biases, for one and several tokens, and the oracle's
    values."""
    import torch
    Ns = [N, N // 4 + 1, N // 4 + 1, N, N + 5, 2 * N]
    for M in (1, 3, 8):
        Ws = [T.random_blocks(fmt, Ns[i] * (K // T.ELEMS[fmt]), 700 + i) for i in range(6)]
        xs = [T.oracle_quantize(T.normal(M * K, 0.0, 1.0, 800 + i), T.act_fmt(fmt), rows=M) for i in range(2)]
        bias = [T.normal(Ns[i], 0.0, 0.5, seed=900 + i) if i % 2 else None for i in range(6)]
        Wd = [P.to_device(w) for w in Ws]
        xd = [P.to_device(x) for x in xs]
        bd = [None if b is None else P.to_device(b) for b in bias]
        inp = [0, 0, 0, 1, 0, 1]                       # entries 0-2 share an input; 3-5 alternate
        outs = [torch.full((M * Ns[i],), 7.0, dtype=torch.float32, device="cuda") for i in range(6)]
        say("sequence grouping", fmt, M)
        P.dev_matmul_sequence([(fmt, xd[inp[i]], Wd[i], bd[i], outs[i], M, Ns[i], K) for i in range(6)])
        for i in range(6):
            alone = P.dev_gemm_nt(fmt, xd[inp[i]], Wd[i], bd[i], M, Ns[i], K).cpu().numpy()
            got = outs[i].cpu().numpy().reshape(M, Ns[i])
            assert np.array_equal(got, alone), (M, i)
            assert T.norm_err(got, T.oracle_gemm_nt(fmt, xs[inp[i]], Ws[i], bias[i], M, Ns[i], K)) <= TOL, (M, i)


def test_matmul_sequence_keeps_order_where_entries_depend():
    """Entries that write what a later entry reads, or write the same output,
    stay separate launches in list order: the bytes equal those of the same
    entries issued one call at a time."""
    import torch
    fmt, N, K, M = "q4_k", 1168, 1024, 1
    W1 = P.to_device(T.random_blocks(fmt, N * (K // 256), 31))
    W2 = P.to_device(T.random_blocks(fmt, N * (K // 256), 32))
    x = P.to_device(T.oracle_quantize(T.normal(K, 0.0, 1.0, 33), "q8_k"))
    say("sequence with dependent entries")

    def run(seq_call):
        a = torch.zeros(N, dtype=torch.float32, device="cuda")
        b = torch.zeros(N, dtype=torch.float32, device="cuda")
        ops = [(fmt, x, W1, None, a, M, N, K),
               (fmt, a, W2, None, b, M, N, K),      # reads the first 1168 bytes of `a` as a Q8_K row
               (fmt, x, W2, None, b, M, N, K),      # same output as the entry before: the last one wins
               (fmt, x, W1, None, a, M, N, K)]      # and `a` again
        if seq_call:
            P.dev_matmul_sequence(ops)
        else:
            for o in ops:
                P.dev_matmul_sequence([o])
        torch.cuda.synchronize()
        return a.cpu().numpy().view(np.uint32), b.cpu().numpy().view(np.uint32)

    a1, b1 = run(True)
    a2, b2 = run(False)
    assert np.array_equal(a1, a2) and np.array_equal(b1, b2)
    ref = P.dev_gemm_nt(fmt, x, W2, None, M, N, K).cpu().numpy().reshape(-1).view(np.uint32)
    assert np.array_equal(b1, ref)


def test_host_inputs_stored_straight_into_device_memory_are_never_stale():
    """Host-pointer calls copy small inputs with CPU stores into a device buffer the
    next kernel reads (no upload launch).  3000 calls in a row, each with a
    different activation vector of a different length and, every other call, a
    bias: every result has the bits the device-pointer path gives for the same
    inputs, so no call has read an earlier call's bytes."""
    import torch
    rng = np.random.default_rng(4711)
    N = 384
    Ks = [256, 512, 1024, 2048]
    Wh = {K: T.synth_weights("q4_k", N, K, seed=900 + K) for K in Ks}
    Wd = {K: P.to_device(Wh[K]) for K in Ks}
    pool = {K: [T.oracle_quantize(T.normal(K, 0.0, 1.0 + 0.1 * i, seed=1000 * K + i), "q8_k") for i in range(24)] for K in Ks}
    biases = [T.normal(N, 0.0, 1.0, seed=77 + i) for i in range(4)]
    want = {}
    for K in Ks:
        for i, xq in enumerate(pool[K]):
            for bi in (-1, 0, 1, 2, 3):
                b = None if bi < 0 else P.to_device(biases[bi])
                want[(K, i, bi)] = P.dev_gemm_nt("q4_k", P.to_device(xq), Wd[K], b, 1, N, K).cpu().numpy().reshape(-1)
    torch.cuda.synchronize()
    say("3000 host-pointer calls with changing inputs")
    bad = 0
    for it in range(3000):
        K = Ks[int(rng.integers(len(Ks)))]
        i = int(rng.integers(24))
        bi = int(rng.integers(4)) if it & 1 else -1
        xq = pool[K][i].copy()                      # a fresh host address most of the time
        got = P.gemm_nt("q4_k", xq, Wh[K], None if bi < 0 else biases[bi], 1, N, K).reshape(-1)
        bad += int(not np.array_equal(got, want[(K, i, bi)]))
    assert bad == 0, "%d of 3000 calls read stale inputs" % bad


# ---- fp32 activations on the matrix cores -------------------------------------------------------

@pytest.mark.parametrize("fmt", F32_FMTS)
def test_f32act_matrix_cores_vs_fp64(fmt):
    """The matrix-core kernel (forced; up to 32 tokens per tile) at the edges of its tiles: one token and
    one more than a tile, row counts around 32 and 64, fewer steps of K than the eight waves of a block and
    one more, an odd number of 32-blocks (Q8_0); against dequantize-then-matmul in fp64, with a bias and a
    padded C, and with infinite activations where the exact result is infinite."""
    import torch
    L = ckq.lib()
    blk = 32 if fmt == "q8_0" else 256
    shapes = [(2, 1, blk), (31, 33, 2 * blk), (32, 64, 512), (33, 65, 2304), (70, 31, 17 * blk), (97, 200, 1024), (200, 2085, 768)]
    L.ckq_set_gemm_policy(1)
    try:
        for M, N, K in shapes:
            W, xf, _ = make_case(fmt, N, K, "enc", 9000 + M + K, tokens=M)
            bias = T.normal(N, 0.0, 0.5, seed=N)
            say("f32act matrix cores", fmt, M, N, K)
            ldc = N + 3
            c = torch.full((M, ldc), 7.0, dtype=torch.float32, device="cuda")
            x_d, W_d, b_d = P.to_device(xf), P.to_device(W), P.to_device(bias)
            P.check(L.ckq_gemm_nt_f32act_dev(P.FMT[fmt], P._dp(x_d), P._dp(W_d), P._dp(b_d), P._dp(c), M, N, K, ldc, P._stream()), "f32act")
            got = c.cpu().numpy()
            want = xf.reshape(M, K).astype(np.float64) @ T.np_dequant(fmt, W).reshape(N, K).T + bias
            assert T.norm_err(got[:, :N], want) <= 2e-6, (M, N, K)
            assert np.all(got[:, N:] == 7.0), (M, N, K)
        M, N, K = 40, 64, 512
        W = np.tile(T.synth_weights(fmt, 1, K, seed=5), N)
        w0 = T.np_dequant(fmt, W[:T.row_bytes(fmt, K)])
        x = T.normal(M * K, 0.0, 1.0, seed=6).reshape(M, K)
        k = int(np.argmax(np.abs(w0)))
        x[3, k] = np.inf
        got = P.dev_gemm_nt_f32act(fmt, P.to_device(x.reshape(-1)), P.to_device(W), None, M, N, K).cpu().numpy().reshape(M, N)
        assert np.all(np.isfinite(np.delete(got, 3, axis=0)))
        assert np.all(got[3] == np.copysign(np.inf, w0[k]))
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt", F32_FMTS)
@pytest.mark.parametrize("mean", [0.0, 1.0, 4.0])
def test_f32act_matrix_cores_are_as_exact_as_one_token_at_a_time(fmt, mean):
    """Error of both kernels for fp32 activations against 64 bits, for activations of mean 0, 1 and 4 (the min term of Q4_K is
    then a large part of what the scales sum to): encoded weights, random blocks, and Q4_K blocks whose min is many times the
    scale or has the other sign.  An error is the rms over 512 rows of a row's relative one, of 32 tokens, and within 1 % or so
    of its expectation; the matrix cores' is not the larger one."""
    import torch
    L = ckq.lib()
    M, N = 32, 512
    for kind, K in (("enc", 1024), ("enc", 4096), ("enc", 11008), ("rand", 2048), ("odd", 2048)):
        W = T.synth_weights(fmt, N, K, seed=40 + K) if kind == "enc" else T.random_blocks(fmt, N * K // T.ELEMS[fmt], 43)
        if kind == "odd" and fmt == "q4_k":
            blocks = W.reshape(-1, 144)
            blocks[0::3, 0:2] = (0x01, 0x00)         # d = 2^-24
            blocks[1::3, 3] ^= 0x80                  # dmin negated
        x = T.normal(M * K, mean, 1.0, seed=41 + K)
        want = x.reshape(M, K).astype(np.float64) @ T.np_dequant(fmt, W).reshape(N, K).T
        err = []
        for policy in (2, 1):
            say("fp32 activations, error", fmt, mean, kind, K, policy)
            L.ckq_set_gemm_policy(policy)
            try:
                got = P.dev_gemm_nt_f32act(fmt, P.to_device(x), P.to_device(W), None, M, N, K).cpu().numpy().reshape(M, N)
            finally:
                L.ckq_set_gemm_policy(0)
            err.append(float(np.sqrt(np.mean(np.sum((got - want) ** 2, axis=0) / np.sum(want ** 2, axis=0)))))
        say("   one token at a time %.3e  matrix cores %.3e" % tuple(err))
        assert err[1] <= 1.03 * err[0], (kind, K, err)


@pytest.mark.parametrize("fmt", F32_FMTS)
def test_f32act_matrix_cores_infinite_huge_and_tiny_activations(fmt):
    """Infinities, NaNs (with a payload in the low 16 bits alone), finite activations whose products with the integers pass the
    fp32 range where those with the weights do not, denormal activations, blocks whose scale is zero: what the oracle gives,
    token by token."""
    import torch
    L = ckq.lib()
    M, N, K = 37, 70, 1024
    W = T.synth_weights(fmt, N, K, seed=15)
    rows = W.reshape(N, -1)
    if fmt == "q4_k":
        rows[5, 4:16] &= 0x30                       # some sub-block scales and mins become zero
        rows[6, 0:2] = 0                            # d = 0: every weight of the block is -dmin mn
    x = T.normal(M * K, 0.0, 1.0, seed=16).reshape(M, K)
    x[2, 100] = np.inf
    x[3, 700] = -np.inf
    x[4, 3], x[4, 900] = np.inf, -np.inf
    x[5, 17:18].view(np.uint32)[:] = 0x7F800001
    x[6] *= np.float32(2.0 ** 122)
    x[7, 40] = 3.0e38
    x[8] *= np.float32(2.0 ** 105)
    x[9] *= np.float32(2.0 ** -120)
    x[10] *= np.float32(2.0 ** -130)
    x[11] = 0.0
    x[35, 1023] = np.inf
    with np.errstate(all="ignore"):
        want = T.oracle_gemm_nt_f32act(fmt, x.reshape(-1), W, None, M, N, K)
    L.ckq_set_gemm_policy(1)
    try:
        say("fp32 activations at the ends of the range", fmt)
        got = P.dev_gemm_nt_f32act(fmt, P.to_device(x.reshape(-1)), P.to_device(W), None, M, N, K).cpu().numpy().reshape(M, N)
    finally:
        L.ckq_set_gemm_policy(0)
    for t in range(M):
        fin = np.isfinite(want[t])
        assert np.array_equal(np.isnan(got[t]), np.isnan(want[t])), t
        assert np.array_equal(got[t][np.isinf(want[t])], want[t][np.isinf(want[t])]), t
        if fin.any():
            scale = float(np.abs(want[t][fin]).max())
            # a sum of 1024 fp32 products; denormal terms are rounded to multiples of 2^-149 each
            assert float(np.abs(got[t][fin].astype(np.float64) - want[t][fin]).max()) <= 1e-5 * scale + 1024 * 2.0 ** -149, t


@pytest.mark.parametrize("fmt,blocks", [("q6_k", (1, 2, 7, 8, 9, 17)), ("q8_0", (1, 2, 3, 5, 15, 33, 34, 67))])
@pytest.mark.parametrize("ofs", [0, 2])
def test_f32act_weights_by_runs(fmt, blocks, ofs):
    """Weights that come in runs of one Q6_K or four Q8_0 blocks, from matrices on a dword and two bytes off: block counts that end
    within a run, within a wave's share, or leave waves without one; one and two row tiles per wave, the last row of the matrix
    in each place.  The buffer ends with the matrix.  Against float64; the result of fp32 sums of up to 2176 products has an
    rms error below 2e-7 of the result's, its largest below 2e-6."""
    import torch
    L = ckq.lib()
    B = T.ELEMS[fmt]
    L.ckq_set_gemm_policy(1)
    try:
        for nb in blocks:
            for M, N in ((33, 1), (2, 33), (200, 1793)):
                K = nb * B
                W = T.random_blocks(fmt, N * nb, 50 + nb)
                buf = torch.zeros(W.size + ofs, dtype=torch.uint8, device="cuda")
                buf[ofs:] = P.to_device(W)
                x = T.normal(M * K, 0.5, 1.0, seed=nb)
                x_d = P.to_device(x)
                c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
                say("f32act runs", fmt, nb, M, N, ofs)
                P.check(L.ckq_gemm_nt_f32act_dev(P.FMT[fmt], P._dp(x_d), ctypes.c_void_p(buf.data_ptr() + ofs), None, P._dp(c), M, N, K, N, P._stream()), "f32act")
                want = x_d.view(M, K).double() @ torch.from_numpy(T.np_dequant(fmt, W).reshape(N, K)).cuda().double().T
                rms = float(want.pow(2).mean().sqrt())
                assert float((c - want).pow(2).mean().sqrt()) <= 2e-7 * rms, (nb, M, N)
                assert float((c - want).abs().max()) <= 2e-6 * float(want.abs().max()), (nb, M, N)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt,M,N,K", [("q4_k", 5, 8250, 1280), ("q4_k", 97, 2090, 512), ("q4_k", 70, 5500, 768), ("q6_k", 5, 8250, 2304), ("q6_k", 97, 2090, 1792), ("q6_k", 40, 4128, 256),
                                       ("q6_k", 70, 5500, 2048), ("q8_0", 5, 8250, 1408), ("q8_0", 40, 4128, 1024), ("q8_0", 97, 2090, 5120), ("q8_0", 33, 4128, 4672), ("q8_0", 70, 5500, 2080)])
def test_f32act_row_tiles_by_rounds_of_blocks(fmt, M, N, K):
    """Sizes on both sides of the choice between one and two row tiles a wave: the rows in one call have the bits of two calls of a part each,
    which fill the chip less and choose otherwise."""
    import torch
    L = ckq.lib()
    say("f32act row tiles", fmt, M, N, K)
    x_d = P.to_device(T.normal(M * K, 0.5, 1.0, seed=K))
    W = P.to_device(T.random_blocks(fmt, N * K // T.ELEMS[fmt], 70)).view(N, -1)

    def run(w):
        c = torch.full((M, w.shape[0]), 7.0, dtype=torch.float32, device="cuda")
        P.check(L.ckq_gemm_nt_f32act_dev(P.FMT[fmt], P._dp(x_d), P._dp(w), None, P._dp(c), M, w.shape[0], K, w.shape[0], P._stream()), "f32act")
        return c
    try:
        L.ckq_set_gemm_policy(1)
        assert torch.equal(run(W), torch.cat([run(W[:1056].contiguous()), run(W[1056:].contiguous())], 1))
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt,nb", [("q6_k", 1), ("q6_k", 9), ("q8_0", 5), ("q8_0", 67)])
@pytest.mark.parametrize("ofs", [0, 2])
def test_f32act_bytes_beside_the_weights(fmt, nb, ofs):
    """A matrix of an odd number of blocks, on a dword or two bytes off, between bytes of zeros and between bytes of ones: one set of bits."""
    import torch
    L = ckq.lib()
    L.ckq_set_gemm_policy(1)
    try:
        for M, N in ((33, 1), (200, 1793)):
            K = nb * T.ELEMS[fmt]
            W = T.random_blocks(fmt, N * nb, 60 + nb)
            x_d = P.to_device(T.normal(M * K, 0.5, 1.0, seed=nb))
            got = []
            for fill in (0, 255):
                buf = torch.full((W.size + ofs + 6,), fill, dtype=torch.uint8, device="cuda")
                buf[ofs:ofs + W.size] = P.to_device(W)
                c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
                say("f32act neighbours", fmt, nb, M, N, ofs, fill)
                P.check(L.ckq_gemm_nt_f32act_dev(P.FMT[fmt], P._dp(x_d), ctypes.c_void_p(buf.data_ptr() + ofs), None, P._dp(c), M, N, K, N, P._stream()), "f32act")
                got.append(c)
            assert torch.equal(*got)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt,widths", [("q6_k", (256, 512, 768, 1536, 1792, 2304)),
                                        ("q8_0", (32, 416, 512, 544, 1024, 1280, 1312, 1536, 1568, 2080, 2592))])
def test_f32act_short_rows(fmt, widths):
    """Rows that a block loads once for all its waves, and both sides of the choices around them: widths that end with and within a
    run, waves with none, one and several steps; grids of a block, of a block per CU and of more, at one and two row tiles.  Against
    float64; an output is a sum of at most 41 fp32 additions over 8 waves, each rounded by 2^-24 of a partial sum, which random signs
    keep far below S, the sum of the magnitudes: 3e-7 S is five such roundings of S itself."""
    import torch
    L = ckq.lib()
    B = T.ELEMS[fmt]
    L.ckq_set_gemm_policy(1)
    try:
        for K in widths:
            for M, N in ((1, 1), (3, 35), (64, 4096), (33, 4129), (96, 4097)):
                W = T.random_blocks(fmt, N * K // B, 60 + K // B)
                x = T.normal(M * K, 0.5, 1.0, seed=K)
                W_d, x_d = P.to_device(W), P.to_device(x)
                c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
                say("f32act short", fmt, K, M, N)
                P.check(L.ckq_gemm_nt_f32act_dev(P.FMT[fmt], P._dp(x_d), P._dp(W_d), None, P._dp(c), M, N, K, N, P._stream()), "f32act")
                X, V = x_d.view(M, K).double(), torch.from_numpy(T.np_dequant(fmt, W).reshape(N, K)).cuda().double()
                assert bool(((c - X @ V.T).abs() <= 3e-7 * (X.abs() @ V.abs().T)).all()), (K, M, N)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("K,N,few,more", [(4672, 70, 27, 28), (4672, 5120, 27, 28), (4672, 5121, 27, 28), (4704, 70, 27, 28), (4672, 70, 29, 33),
                                          (4672, 4097, 64, 96), (4608, 4097, 64, 96), (5120, 70, 27, 28)])
def test_f32act_q8_0_token_tiles_partly_filled(K, N, few, more):
    """Both sides of the choice between a row per lane and weights in memory order by tokens, blocks and width: the tokens that both calls
    have keep their bits, and all are right against float64 (a sum of at most 28 additions, as in the test above)."""
    import torch
    L = ckq.lib()
    W = T.random_blocks("q8_0", N * K // 32, 70 + N)
    x = T.normal(more * K, 0.5, 1.0, seed=K)
    W_d, x_d = P.to_device(W), P.to_device(x)
    L.ckq_set_gemm_policy(1)
    try:
        got = []
        for M in (few, more):
            c = torch.full((M, N), 7.0, dtype=torch.float32, device="cuda")
            say("f32act q8_0 partly filled", K, M, N)
            P.check(L.ckq_gemm_nt_f32act_dev(P.FMT["q8_0"], P._dp(x_d), P._dp(W_d), None, P._dp(c), M, N, K, N, P._stream()), "f32act")
            got.append(c)
    finally:
        L.ckq_set_gemm_policy(0)
    assert torch.equal(got[0].view(torch.int32), got[1][:few].view(torch.int32))
    X, V = x_d.view(more, K).double(), torch.from_numpy(T.np_dequant("q8_0", W).reshape(N, K)).cuda().double()
    assert bool(((got[1] - X @ V.T).abs() <= 3e-7 * (X.abs() @ V.abs().T)).all())


# ---- 16-row tiles: a few to a few dozen tokens of the K-quants -------------------------------------

@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_vs_oracle_and_the_kernels_they_stand_in_for(fmt):
    """The kernel forced at the edges of its tiles - two tokens, eight and sixteen and one more, row counts
    around 16, one K-block, more K-blocks than waves, the longest row it takes - against the oracle, with a
    bias and a padded C.  It has the bits of the kernel that would otherwise run: of the streaming kernel at
    these sizes, of the tile kernels, K split and wave groups included, at those of the matrix cores; three
    matrices of one input share a launch."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, K in [(2, 1, 256), (8, 15, 512), (9, 16, 1024), (16, 17, 2304), (17, 33, 43 * 256), (13, 70, 64 * 256), (40, 100, 5 * 256)]:
            W, _, xq = make_case(fmt, N, K, "rand" if N % 2 else "enc", 9100 + M + N, tokens=M)
            bias = T.normal(N, 0.0, 0.5, seed=N)
            say("16-row tiles", fmt, M, N, K)
            L.ckq_set_prefill_variant(tag, 16)
            c = torch.full((M, N + 3), 7.0, dtype=torch.float32, device="cuda")
            x_d, W_d, b_d = P.to_device(xq), P.to_device(W), P.to_device(bias)
            P.check(L.ckq_gemm_nt_dev(tag, P._dp(x_d), P._dp(W_d), P._dp(b_d), P._dp(c), M, N, K, N + 3, P._stream()), "ckq_gemm_nt_dev")
            got = c.cpu().numpy()
            assert T.norm_err(got[:, :N], T.oracle_gemm_nt(fmt, xq, W, bias, M, N, K)) <= TOL, (M, N, K)
            assert np.all(got[:, N:] == 7.0), (M, N, K)
            rb = x_d.numel() // M
            for m in {0, M // 2, M - 1}:
                one = P.dev_gemm_nt(fmt, x_d[m * rb:(m + 1) * rb].clone(), W_d, b_d, 1, N, K)
                assert torch.equal(c[m, :N], one.view(N)), (M, N, K, m)
        for M, N, K in [(9, 11008, 2048), (17, 4096, 4096), (33, 4096, 11008), (12, 32000, 512), (100, 4864, 4096)]:
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
            W = P.to_device(T.random_blocks(fmt, N * K // 256, 9200 + M))
            say("16-row tiles against the tile kernels", fmt, M, N, K)
            L.ckq_set_prefill_variant(tag, 16)
            L.ckq_set_gemm_policy(0)
            a = P.dev_gemm_nt(fmt, xq, W, None, M, N, K).clone()
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(1)
            b = P.dev_gemm_nt(fmt, xq, W, None, M, N, K).clone()
            L.ckq_set_gemm_policy(0)
            budget = (40 if fmt == "q5_k" else 20) << 20
            if (M + 7) // 8 * max(N * T.row_bytes(fmt, K), 3 << 20) > budget:      # the streaming kernel's part ends here
                assert torch.equal(a, b), (M, N, K)
            else:
                assert torch.allclose(a, b, rtol=0, atol=2e-6 * float(b.abs().max())), (M, N, K)
        M, K, Ns = 12, 1024, [640, 33, 16]
        L.ckq_set_prefill_variant(tag, 16)
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=3)), "q8_k", rows=M)
        Ws = [P.to_device(T.synth_weights(fmt, n, K, seed=9300 + i)) for i, n in enumerate(Ns)]
        ys = [torch.zeros(M * n, dtype=torch.float32, device="cuda") for n in Ns]
        for m in (M, 5):
            say("16-row tiles, grouped", fmt, m)
            P.dev_matmul_sequence([(fmt, xq, W, None, y, m, n, K) for W, y, n in zip(Ws, ys, Ns)])
            for W, y, n in zip(Ws, ys, Ns):
                assert torch.equal(y[:m * n].view(m, n), P.dev_gemm_nt(fmt, xq, W, None, m, n, K).view(m, n)), (m, n)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k", "q8_0", "q5_0"])
@pytest.mark.parametrize("N,K", [(7, 256), (250, 1024), (16383, 512), (16385, 512), (1023, 4864), (1025, 4864), (2047, 4096), (2049, 4096), (300, 11008)])
def test_streamed_tokens_have_the_bits_of_single_ones(fmt, N, K):
    """Token tiles of the streaming kernel on both sides of the row counts that take one or two rows per slot and smaller token
    tiles: every token's outputs are those of a call with that token alone - of the K-quants bit for bit, of Q8_0 and Q5_0, whose
    scaling the compiler may contract into a multiply-add or not per instantiation, but for one rounding a block."""
    import torch
    L = ckq.lib()
    W, bias = P.to_device(T.random_blocks(fmt, N * K // ckq.api.BLOCK_ELEMS[fmt], 9700 + N % 97)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
    try:
        L.ckq_set_gemm_policy(2)
        for M in (2, 3, 4, 5, 8):
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), P.act_format(fmt), rows=M)
            rb = xq.numel() // M
            say("streamed tokens", fmt, M, N, K)
            y = P.dev_gemm_nt(fmt, xq, W, bias, M, N, K).view(M, N)
            for m in range(M):
                one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K).view(N)
                same = torch.equal(y[m], one) if fmt[-1] == "k" else torch.allclose(y[m], one, rtol=0, atol=2e-6 * float(one.abs().max()))
                assert same, (M, m)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt,K", [("q8_0", 7232), ("q8_0", 7264), ("q8_0", 7296), ("q8_0", 14528), ("q8_0", 14592), ("q5_0", 7264), ("q5_0", 7296), ("q5_0", 14592), ("q5_0", 30720),
                                   ("q4_k", 7168), ("q4_k", 7424), ("q5_k", 7424), ("q6_k", 14336), ("q6_k", 14592), ("q5_k", 30720)])
def test_streamed_token_tiles_at_the_limit_of_lds(fmt, K):
    """Rows of which eight, four or two tokens just fit the staged tile or just do not, with and without two rows per slot: every token's outputs
    are those of a call with that token alone, in the sense of the test above."""
    import torch
    L = ckq.lib()
    try:
        L.ckq_set_gemm_policy(2)
        for N, M in ((70, 13), (2100, 5)):
            say("streamed tiles at the limit", fmt, M, N, K)
            W = P.to_device(T.random_blocks(fmt, N * K // ckq.api.BLOCK_ELEMS[fmt], 9730 + N % 97))
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), P.act_format(fmt), rows=M).view(M, -1)
            y = P.dev_gemm_nt(fmt, xq.view(-1), W, None, M, N, K).view(M, N)
            for m in range(M):
                one = P.dev_gemm_nt(fmt, xq[m].clone(), W, None, 1, N, K).view(N)
                same = torch.equal(y[m], one) if fmt[-1] == "k" else torch.allclose(y[m], one, rtol=0, atol=2e-6 * float(one.abs().max()))
                assert same, (M, m)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("M,N,K", [(9, 500, 7296), (16, 4100, 7296), (11, 1500, 9728), (13, 300, 11008), (40, 200, 8192)])
def test_q8_0_long_rows_of_several_tokens_stream(M, N, K):
    """The automatic choice for long Q8_0 rows has the streaming kernel's bits, from the entry point that allocates nothing too, and an error
    against 64 bits no larger than that of one token at a time (rms; a tenth for the spread over some thousand outputs)."""
    import torch
    L = ckq.lib()
    say("q8_0 long rows", M, N, K)
    xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_0", rows=M)
    W = P.to_device(T.random_blocks("q8_0", N * K // 32, 9720))
    auto = P.dev_gemm_nt("q8_0", xq, W, None, M, N, K).view(M, N).clone()
    bare = torch.full((M, N), 7.0, device="cuda")
    P.check(L.ckq_gemm_nt_noalloc_dev(P.FMT["q8_0"], P._dp(xq), P._dp(W), None, P._dp(bare), M, N, K, N, P._stream()), "ckq_gemm_nt_noalloc_dev")
    try:
        L.ckq_set_gemm_policy(2)
        streamed = P.dev_gemm_nt("q8_0", xq, W, None, M, N, K).view(M, N)
    finally:
        L.ckq_set_gemm_policy(0)
    assert torch.equal(auto, streamed) and torch.equal(auto, bare)

    def values(blocks, rows):
        b = blocks.cpu().view(rows, K // 32, 34)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        return (b[:, :, 2:].contiguous().view(torch.int8).double() * d).view(rows, K)
    exact = values(xq, M) @ values(W, N).T
    one = torch.stack([P.dev_gemm_nt("q8_0", xq.view(M, -1)[m].clone(), W, None, 1, N, K).view(N) for m in range(M)])

    def rms(y):
        return float((y.double().cpu() - exact).square().mean().sqrt())
    assert rms(auto) <= 1.1 * rms(one)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_of_short_rows_and_several_token_groups(fmt):
    """The kernel that keeps the planes of its weights across token groups: one to eight K-blocks (waves), two groups and many,
    groups dealt evenly to a row tile's blocks and not, the last rows and tokens of the matrix.  In the order of the streaming
    kernel (policy 2) and of the tile kernels (1), bit for bit; and several matrices in one launch."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, K in [(93, 9729, 1024), (70, 12001, 256), (17, 33, 2048), (33, 16, 1792), (21, 20011, 768), (500, 100, 1280)]:
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
            W, bias = P.to_device(T.random_blocks(fmt, N * K // 256, 9400 + M)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
            say("16-row tiles, several token groups", fmt, M, N, K)
            L.ckq_set_prefill_variant(tag, 16)
            L.ckq_set_gemm_policy(2)
            tree = P.dev_gemm_nt(fmt, xq, W, bias, M, N, K).clone().view(M, N)
            L.ckq_set_gemm_policy(1)
            chain = P.dev_gemm_nt(fmt, xq, W, bias, M, N, K).clone()
            L.ckq_set_prefill_variant(tag, 0)
            assert torch.equal(chain, P.dev_gemm_nt(fmt, xq, W, bias, M, N, K)), (M, N, K)
            L.ckq_set_gemm_policy(0)
            rb = xq.numel() // M
            for m in range(0, M, max(1, M // 12)):
                one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K)
                assert torch.equal(tree[m], one.view(N)), (M, N, K, m)
        M, K, Ns = 77, 1024, [9000, 33, 4861, 250]
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=4)), "q8_k", rows=M)
        Ws = [P.to_device(T.random_blocks(fmt, n * K // 256, 9500 + i)) for i, n in enumerate(Ns)]
        for policy in (1, 0):
            L.ckq_set_prefill_variant(tag, 16)
            L.ckq_set_gemm_policy(policy)
            ys = [torch.zeros(M, n, dtype=torch.float32, device="cuda") for n in Ns]
            say("16-row tiles, several token groups, grouped", fmt, policy)
            P.dev_matmul_sequence([(fmt, xq, W, None, y, M, n, K) for W, y, n in zip(Ws, ys, Ns)])
            for W, y, n in zip(Ws, ys, Ns):
                assert torch.allclose(y, P.dev_gemm_nt(fmt, xq, W, None, M, n, K).view(M, n), rtol=0, atol=2e-6 * float(y.abs().max())), (policy, n)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_of_several_token_groups_copied_to_lds(fmt):
    """Where the kernel that keeps its planes copies a group while the one before is at work: three groups and more for one block, one
    to eight waves (sums by part of the waves, by all, by two fours in turn), a last group of one token, and an output pitch past what its
    stores reach, which another kernel serves.  In both orders bit for bit, with a bias and a padded C."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, K, ldy in [(161, 2033, 256, 2040), (49, 5000, 512, 5000), (113, 900, 768, 901), (97, 3001, 1024, 3001), (65, 2100, 1536, 2111), (81, 1300, 2048, 1300),
                             (18, 40, 1024, 1 << 25)]:
            if fmt == "q4_k" and K > 1024:
                continue
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
            W, bias = P.to_device(T.random_blocks(fmt, N * K // 256, 9450 + M)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
            say("16-row tiles, groups copied to LDS", fmt, M, N, K, ldy)

            def call(policy, forced):
                L.ckq_set_prefill_variant(tag, 16 if forced else 0)
                L.ckq_set_gemm_policy(policy)
                c = torch.full(((M - 1) * ldy + N,), 7.0, device="cuda")
                P.check(L.ckq_gemm_nt_dev(tag, P._dp(xq), P._dp(W), P._dp(bias), P._dp(c), M, N, K, ldy, P._stream()), "ckq_gemm_nt_dev")
                return c.as_strided((M, N), (ldy, 1)), c
            (tree, all_), (chain, _), (tiles, _) = call(2, True), call(1, True), call(1, False)
            assert torch.equal(chain, tiles), (M, N, K)
            if ldy > N:
                assert bool((all_[N:ldy] == 7.0).all()), (M, N, K)
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(0)
            rb = xq.numel() // M
            for m in {0, 15, 16, M // 2, M - 1}:
                one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K)
                assert torch.equal(tree[m], one.view(N)), (M, N, K, m)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_k_split_whose_pieces_meet_in_lds(fmt):
    """Two, three and four pieces of K, of two blocks and more, the last one shorter; one token and one row more than a tile, a single row; as many
    blocks as the CUs have places for.  Bit for bit the chains of the tile kernels as the 16-row tiles run them, within the tolerance the oracle's result, nothing outside the
    matrix; and the entry point that allocates nothing refuses what it refused when the partial tiles lay in memory, and takes what the
    16-row tiles took although others go to the K split now."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, nb in [(9, 1, 8), (64, 128, 8), (65, 33, 9), (130, 1000, 11), (512, 2048, 8), (200, 257, 12), (449, 1025, 13), (33, 4096, 15), (512, 896, 19), (70, 130, 16), (500, 900, 28),
                         (509, 1024, 17), (1000, 100, 21)]:
            K = nb * 256
            xh = T.normal(M * K, 0.0, 1.0, seed=M)
            xq, Wh = P.dev_quantize(P.to_device(xh), "q8_k", rows=M), T.synth_weights(fmt, N, K, seed=9700 + nb)
            W, bias = P.to_device(Wh), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
            say("K split, pieces meet in LDS", fmt, M, N, K)

            def call(forced, b=bias):
                L.ckq_set_prefill_variant(tag, 16 if forced else 0)
                L.ckq_set_gemm_policy(1)
                c = torch.full((M + 1, N + 3), 7.0, device="cuda")
                P.check(L.ckq_gemm_nt_dev(tag, P._dp(xq), P._dp(W), None if b is None else P._dp(b), P._dp(c), M, N, K, N + 3, P._stream()), "ckq_gemm_nt_dev")
                assert bool((c[:, N:] == 7.0).all()) and bool((c[M] == 7.0).all()), (M, N, K)
                return c[:M, :N]
            assert torch.equal(call(False), call(True)), (M, N, K)
            assert torch.equal(call(False, None), call(True, None)), (M, N, K)
            if M * N * K < 1 << 28:
                want = T.oracle_gemm_nt(fmt, xq.cpu().numpy(), Wh, bias.cpu().numpy(), M, N, K)
                assert T.norm_err(call(False).cpu().numpy(), want) <= TOL
        for M, N, nb, refused in [(512, 896, 19, True), (65, 33, 9, False), {"q4_k": (172, 3385, 10, False), "q5_k": (182, 3139, 10, False), "q6_k": (191, 3084, 10, False)}[fmt]]:
            K = nb * 256
            xq, W = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=3)), "q8_k", rows=M), P.to_device(T.random_blocks(fmt, N * nb, 9750))
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(0)
            c = torch.full((M, N), 7.0, device="cuda")
            rc = L.ckq_gemm_nt_noalloc_dev(tag, P._dp(xq), P._dp(W), None, P._dp(c), M, N, K, N, P._stream())
            assert (rc != 0) == refused and bool((c == 7.0).all()) == refused, (rc, M, N)
            if not refused:
                assert torch.equal(c, P.dev_gemm_nt(fmt, xq, W, None, M, N, K).view(M, N))
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_with_planes_kept_for_one_group(fmt):
    """Few row tiles and many groups: the kernel that keeps its planes in blocks of one group each, and of two, the last of one; one block a row to
    eight.  In both orders bit for bit."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, K in [(113, 40, 256), (194, 993, 256), (50, 300, 768), (33, 17, 1024), (82, 4630, 512), (250, 90, 2048), (219, 2069, 1280), (256, 16, 1792)]:
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
            W, bias = P.to_device(T.random_blocks(fmt, N * K // 256, 9560 + M)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
            say("16-row tiles, planes kept for one group", fmt, M, N, K)

            def call(policy, forced):
                L.ckq_set_prefill_variant(tag, 16 if forced else 0)
                L.ckq_set_gemm_policy(policy)
                return P.dev_gemm_nt(fmt, xq, W, bias, M, N, K).view(M, N).clone()
            tree, chain, tiles = call(2, True), call(1, True), call(1, False)
            assert torch.equal(chain, tiles), (M, N, K)
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(0)
            rb = xq.numel() // M
            for m in {0, 15, 16, M // 2, M - 1}:
                one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K)
                assert torch.equal(tree[m], one.view(N)), (M, N, K, m)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_alone_on_their_cu(fmt):
    """Row tiles that have a CU each, one token group and rows too few for groups in pairs: blocks of eight waves, of twelve and (rows longer than
    the LDS has room for) in between; fewer 256-blocks than waves in the last turn, one, and none.  In the tile kernels' order bit for bit what
    they give, in the streaming kernel's what one token at a time gives."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, K in [(13, 1500, 12 * 256), (16, 1040, 13 * 256), (9, 4096, 16 * 256), (40, 1033, 17 * 256), (13, 2048, 24 * 256), (8, 1100, 25 * 256), (15, 1056, 32 * 256),
                        (13, 1056, 33 * 256), (12, 1200, 43 * 256), (11, 1200, 64 * 256)]:
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
            W, bias = P.to_device(T.random_blocks(fmt, N * K // 256, 9520 + M)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
            say("16-row tiles, alone on their CU", fmt, M, N, K)

            def call(policy, forced):
                L.ckq_set_prefill_variant(tag, 16 if forced else 0)
                L.ckq_set_gemm_policy(policy)
                c = torch.full((M, N + 3), 7.0, device="cuda")
                P.check(L.ckq_gemm_nt_dev(tag, P._dp(xq), P._dp(W), P._dp(bias), P._dp(c), M, N, K, N + 3, P._stream()), "ckq_gemm_nt_dev")
                assert bool((c[:, N:] == 7.0).all()), (M, N, K)
                return c[:, :N]
            tree = call(2, True)
            if M > 8:
                chain, tiles = call(1, True), call(1, False)
                assert torch.equal(chain, tiles), (M, N, K)
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(0)
            rb = xq.numel() // M
            for m in {0, M // 2, M - 1}:
                one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K)
                assert torch.equal(tree[m], one.view(N)), (M, N, K, m)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_matrices_of_three_to_eight_tokens_share_one_choice_of_kernel(fmt):
    """Groups that go to the 16-row tiles and ones that stream, with rows that some or none of the matrices alone would take there, rows too long for a grouped
    streaming launch and the longest, ragged and tiny matrices: bit for bit what the streaming kernel gives each matrix alone."""
    import torch
    L = ckq.lib()
    try:
        for M, K, Ns in [(8, 4352, (4352, 1088, 1088)), (5, 2560, (2560, 640, 640)), (6, 3072, (3072, 1536, 1536)), (7, 512, (512, 128, 128)), (8, 768, (1000, 17, 1)), (5, 2048, (5632, 5632)),
                         (8, 256, (70, 4000)), (6, 7424, (1500, 1, 300)), (7, 11008, (96, 33)), (5, 16384, (700, 500)), (5, 16640, (64, 32)), (8, 1280, (1280, 320, 320)), (4, 2560, (2560, 640, 640)),
                         (4, 4608, (4608, 1152, 1152)), (3, 8192, (2100, 40)), (3, 14592, (300, 17)), (2, 4608, (4608, 600))]:
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M + K)), "q8_k", rows=M)
            Ws = [P.to_device(T.random_blocks(fmt, n * K // 256, 9700 + i)) for i, n in enumerate(Ns)]
            bs = [P.to_device(T.normal(n, 0.0, 0.5, seed=n)) for n in Ns]
            say("groups of three to eight tokens", fmt, M, K, Ns)
            ys = [torch.full((M, n + 3), 7.0, device="cuda") for n in Ns]
            P.dev_matmul_sequence([(fmt, xq, W, b, y, M, n, K, n + 3) for W, b, y, n in zip(Ws, bs, ys, Ns)])
            L.ckq_set_gemm_policy(2)
            for W, b, y, n in zip(Ws, bs, ys, Ns):
                assert torch.equal(y[:, :n], P.dev_gemm_nt(fmt, xq, W, b, M, n, K).view(M, n)) and bool((y[:, n:] == 7.0).all()), (M, K, n)
            L.ckq_set_gemm_policy(0)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt", ["q5_k", "q6_k"])
def test_groups_of_too_few_tiles_for_a_shared_launch_keep_their_matrices_bits(fmt):
    """Q, K and V of 17 to 313 tokens whose tiles together would leave most of the chip idle, on either side of the line between one launch of 16-row tiles and
    the tile kernels one by one: the bits that each matrix has alone."""
    import torch
    for M, K, Ns in [(105, 2304, (2304, 2304, 2304)), (81, 4352, (4352, 1088, 1088)), (38, 3072, (3072, 3072, 3072)), (17, 5120, (4100, 2561)), (313, 2560, (2560, 320, 320)), (34, 8704, (8704, 1088, 1088))]:
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M + K)), "q8_k", rows=M)
        Ws = [P.to_device(T.random_blocks(fmt, n * K // 256, 9800 + i)) for i, n in enumerate(Ns)]
        bs = [P.to_device(T.normal(n, 0.0, 0.5, seed=n)) for n in Ns]
        say("groups of few tiles", fmt, M, K, Ns)
        ys = [torch.full((M, n + 3), 7.0, device="cuda") for n in Ns]
        P.dev_matmul_sequence([(fmt, xq, W, b, y, M, n, K, n + 3) for W, b, y, n in zip(Ws, bs, ys, Ns)])
        for W, b, y, n in zip(Ws, bs, ys, Ns):
            one = P.dev_gemm_nt(fmt, xq, W, b, M, n, K).view(M, n)
            assert bool((y[:, n:] == 7.0).all())
            if (M + 7) // 8 * max(n * T.row_bytes(fmt, K), 3 << 20) > (40 if fmt == "q5_k" else 20) << 20:
                assert torch.equal(y[:, :n], one), (M, K, n)
            else:                                         # alone it streams, with another order of its sums
                assert torch.allclose(y[:, :n], one, rtol=0, atol=2e-6 * float(one.abs().max())), (M, K, n)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_of_token_groups_in_pairs(fmt):
    """Longer rows, two token groups a block: an even and an odd number of groups, a last group of one token, ragged rows, fewer blocks of the row than
    waves and more, row tiles that just have a CU each as pairs and ones that do not; in the tile kernels' order bit for bit what they
    give, in the streaming kernel's what one token at a time gives, with no, some and all but a few positions that hold two blocks of the row."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]
    try:
        for M, N, K in [(32, 4096, 9 * 256), (33, 3003, 11 * 256), (64, 2039, 16 * 256), (93, 1024, 19 * 256), (17, 4095, 20 * 256), (50, 1500, 24 * 256), (32, 2100, 43 * 256),
                        (70, 9000, 10 * 256), (40, 6001, 16 * 256), (64, 5000, 19 * 256), (129, 700, 9 * 256)]:
            xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
            W, bias = P.to_device(T.random_blocks(fmt, N * K // 256, 9480 + M)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
            say("16-row tiles, token groups in pairs", fmt, M, N, K)

            def call(policy, forced):
                L.ckq_set_prefill_variant(tag, 16 if forced else 0)
                L.ckq_set_gemm_policy(policy)
                c = torch.full((M, N + 3), 7.0, device="cuda")
                P.check(L.ckq_gemm_nt_dev(tag, P._dp(xq), P._dp(W), P._dp(bias), P._dp(c), M, N, K, N + 3, P._stream()), "ckq_gemm_nt_dev")
                assert bool((c[:, N:] == 7.0).all()), (M, N, K)
                return c[:, :N]
            tree, chain, tiles = call(2, True), call(1, True), call(1, False)
            assert torch.equal(chain, tiles), (M, N, K)
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(0)
            rb = xq.numel() // M
            for m in {0, 15, 16, M // 2, M - 1}:
                one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K)
                assert torch.equal(tree[m], one.view(N)), (M, N, K, m)
        M, K, Ns = 40, 4096, [3000, 700, 333]
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=6)), "q8_k", rows=M)
        Ws = [P.to_device(T.random_blocks(fmt, n * K // 256, 9490 + i)) for i, n in enumerate(Ns)]
        for policy in (2, 1, 0):
            L.ckq_set_prefill_variant(tag, 16)
            L.ckq_set_gemm_policy(policy)
            ys = [torch.zeros(M, n, dtype=torch.float32, device="cuda") for n in Ns]
            say("16-row tiles, token groups in pairs, grouped", fmt, policy)
            P.dev_matmul_sequence([(fmt, xq, W, None, y, M, n, K) for W, y, n in zip(Ws, ys, Ns)])
            for W, y, n in zip(Ws, ys, Ns):
                assert torch.allclose(y, P.dev_gemm_nt(fmt, xq, W, None, M, n, K).view(M, n), rtol=0, atol=2e-6 * float(y.abs().max())), (policy, n)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
def test_16_row_tiles_with_held_activations(fmt):
    """The kernel that goes through several row tiles with its activations in registers: one wave a block and sixteen, blocks of one
    tile, of some more than others and of several rounds of the tiles whose terms fit the LDS, last tiles that start early (row counts
    past a multiple of 16), a bias and a padded C, one token short of the group and all sixteen.  In the order of the tile
    kernels (policy 1) bit for bit what they give, in that of the streaming kernel (2) what one token at a time gives; and several matrices in one launch."""
    import torch
    L = ckq.lib()
    tag = P.FMT[fmt]

    def forced(policy, call):
        L.ckq_set_prefill_variant(tag, 16)
        L.ckq_set_gemm_policy(policy)
        try:
            return call()
        finally:
            L.ckq_set_prefill_variant(tag, 0)
            L.ckq_set_gemm_policy(0)
    for M, N, K in [(3, 16, 1024), (16, 4111, 1024), (15, 17, 768), (9, 140001, 256), (16, 33000, 512), (13, 130017, 768), (16, 40007, 1024), (12, 12303, 2048),
                    (16, 16401, 3072), (11, 9001, 3584), (16, 7003, 4096), (8, 21001, 4096)]:
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=M)), "q8_k", rows=M)
        W, bias = P.to_device(T.random_blocks(fmt, N * K // 256, 9600 + M)), P.to_device(T.normal(N, 0.0, 0.5, seed=N))
        say("16-row tiles, held activations", fmt, M, N, K)
        c = torch.full((M, N + 5), 7.0, dtype=torch.float32, device="cuda")
        forced(2, lambda: P.check(L.ckq_gemm_nt_dev(tag, P._dp(xq), P._dp(W), P._dp(bias), P._dp(c), M, N, K, N + 5, P._stream()), "ckq_gemm_nt_dev"))
        assert bool((c[:, N:] == 7.0).all()), (M, N, K)
        rb = xq.numel() // M
        for m in range(0, M, 3):
            one = P.dev_gemm_nt(fmt, xq[m * rb:(m + 1) * rb].clone(), W, bias, 1, N, K)
            assert torch.equal(c[m, :N], one.view(N)), (M, N, K, m)
        if M > 8:
            chain = forced(1, lambda: P.dev_gemm_nt(fmt, xq, W, bias, M, N, K).clone())
            L.ckq_set_gemm_policy(1)
            try:
                tiles = P.dev_gemm_nt(fmt, xq, W, bias, M, N, K)
            finally:
                L.ckq_set_gemm_policy(0)
            assert torch.equal(chain, tiles), (M, N, K)
    for M, K, Ns in ((13, 1024, [9000, 33, 4861, 250]), (16, 4096, [5000, 3003])):
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, seed=5)), "q8_k", rows=M)
        Ws = [P.to_device(T.random_blocks(fmt, n * K // 256, 9650 + i)) for i, n in enumerate(Ns)]
        for policy in (2, 1, 0):
            ys = [torch.zeros(M, n, dtype=torch.float32, device="cuda") for n in Ns]
            say("16-row tiles, held activations, grouped", fmt, M, policy)
            forced(policy, lambda: P.dev_matmul_sequence([(fmt, xq, W, None, y, M, n, K) for W, y, n in zip(Ws, ys, Ns)]))
            for W, y, n in zip(Ws, ys, Ns):
                assert torch.allclose(y, P.dev_gemm_nt(fmt, xq, W, None, M, n, K).view(M, n), rtol=0, atol=2e-6 * float(y.abs().max())), (policy, n)


@pytest.mark.parametrize("blocks", [1, 2, 3, 4, 5, 6, 7, 8, 13, 37, 64])
def test_gemm_mfma_q8_0_row_alignment_and_k_remainders(blocks):
    """Rows of odd and even numbers of 32-blocks (odd ones start on dwords every other row), K ending after one, two, three
    and four blocks of the last step, operands that start two bytes past a dword, an infinite weight scale."""
    import torch
    L = ckq.lib()
    K = 32 * blocks
    try:
        L.ckq_set_gemm_policy(1)
        for M, N, wo, xo in [(9, 5, 0, 0), (64, 128, 2, 0), (70, 200, 0, 2), (65, 131, 2, 2)]:
            W, _, xq = make_case("q8_0", N, K, "rand", 9400 + M + blocks, tokens=M)
            if M == 70:
                W = W.copy()
                W.reshape(N, -1)[3, :2] = (0x00, 0x7C)
            bias = T.normal(N, 0.0, 0.5, seed=N)
            say("q8_0 alignment", M, N, K, wo, xo)
            ref = T.oracle_gemm_nt("q8_0", xq, W, bias, M, N, K)
            wd = torch.zeros(len(W) + 4, dtype=torch.uint8, device="cuda")
            xd = torch.zeros(len(xq) + 4, dtype=torch.uint8, device="cuda")
            wd[wo:wo + len(W)] = P.to_device(W)
            xd[xo:xo + len(xq)] = P.to_device(xq)
            c = torch.full((M, N + 1), 7.0, dtype=torch.float32, device="cuda")
            b = P.to_device(bias)
            P.check(L.ckq_gemm_nt_dev(P.FMT["q8_0"], xd.data_ptr() + xo, wd.data_ptr() + wo, P._dp(b), P._dp(c), M, N, K,
                                      N + 1, P._stream()), "ckq_gemm_nt_dev")
            got = c.cpu().numpy()
            assert np.all(got[:, N] == 7.0)
            ok = np.isfinite(ref)
            assert np.array_equal(np.isnan(got[:, :N]), np.isnan(ref)) and np.array_equal(got[:, :N][~ok & ~np.isnan(ref)], ref[~ok & ~np.isnan(ref)])
            assert T.norm_err(np.where(ok, got[:, :N], 0.0), np.where(ok, ref, 0.0)) <= TOL, (M, N, K)
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("rows", [1, 3, 15, 16, 17, 33, 16384, 16385])
def test_host_results_as_they_arrive(rows):
    """Host-pointer GEMVs whose results the CPU waits for word by word (up to 64 KiB): sizes around its sixteen words at a time and
    its limit, several calls through one twin, inputs of their own each; the bits are the device entry point's."""
    K = 256
    say("arrive", rows)
    W, _, _ = make_case("q4_k", rows, K, "rand", 9500 + rows)
    for seed in range(3):
        xq = P.quantize(T.normal(K, 0.0, 1.0, 9600 + seed))
        assert np.array_equal(xq, T.oracle_quantize(T.normal(K, 0.0, 1.0, 9600 + seed), "q8_k"))
        y = P.gemv("q4_k", W, xq, rows, K)
        ref = P.dev_gemm_nt("q4_k", P.to_device(xq), P.to_device(W), None, 1, rows, K).cpu().numpy().reshape(-1)
        assert np.array_equal(y, ref)


def test_host_result_equal_to_the_mark():
    """Quants that spell the word the CPU takes for "not there yet": the call ends all the same, with the right bytes."""
    x = T.normal(5 * 256, 0.0, 1.0, 9700)
    for b in (0, 2, 4):
        x[256 * b:256 * (b + 1)] = 0.0
        x[256 * b] = -127.0                                     # iscale = 1
        x[256 * b + 60:256 * b + 64] = (-63, -45, -91, 127)     # c1 d3 a5 7f
    for _ in range(2):
        got = P.quantize(x)
        assert np.array_equal(got, T.oracle_quantize(x, "q8_k"))
        assert (got.view(np.uint32) == 0x7FA5D3C1).sum() == 3


@pytest.mark.parametrize("M,N,K", [(9, 131, 64), (33, 300, 192), (63, 1030, 2112), (129, 2050, 576), (192, 21001, 640), (350, 24484, 256), (385, 24499, 320),
                                   (128, 8000, 1984), (16, 21000, 2112), (130, 8001, 1984), (65, 12000, 2240)])
def test_gemm_mfma_q8_0_tiles_and_teams(M, N, K):
    """Tiles of 32, 64 and 96 tokens, one and two teams, K ending inside a step and with one step more for the first team, against
    fp64.  An output is nb terms, each rounded twice and added once: (nb + 4) 2^-24 of the sum of the terms' magnitudes."""
    import torch
    x, w = T.random_blocks("q8_0", M * (K // 32), 9800 + M), T.random_blocks("q8_0", N * (K // 32), 9801 + N)

    def real(b, rows):
        b = P.to_device(b).view(rows, K // 32, 34)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        return (d * b[:, :, 2:].contiguous().view(torch.int8).double()).reshape(rows, K)
    say("q8_0 tiles", M, N, K)
    bias = P.to_device(T.normal(N, 0.0, 0.5, seed=N))
    y = P.dev_gemm_nt("q8_0", P.to_device(x), P.to_device(w), bias, M, N, K).view(M, N).double() - bias.double()
    A, B = real(x, M), real(w, N)
    bound = (A.abs() @ B.abs().T) * (K // 32 + 4) * 2.0 ** -24 + bias.abs().double() * 2.0 ** -23
    assert bool((torch.isfinite(bound)).all())
    assert float(((y - A @ B.T).abs() / bound).max()) <= 1.0


@pytest.mark.parametrize("M,N,K", [(9, 131, 32), (10, 1, 224), (33, 300, 96), (63, 1030, 2080), (129, 2050, 608), (192, 21001, 672), (350, 24484, 288), (385, 24499, 352),
                                   (128, 8000, 1952), (130, 8001, 2016), (65, 12000, 2208), (70, 129, 9248)])
def test_gemm_mfma_q8_0_rows_of_an_odd_number_of_blocks(M, N, K):
    """Rows that start on dwords and two bytes behind them in turn, one block or three after the last whole step, in every form of the kernel and split
    along K: against fp64 at the bound of the test above.  A scale that is infinite makes the outputs of its row what the oracle has."""
    import torch
    x, w = T.random_blocks("q8_0", M * (K // 32), 9850 + M), T.random_blocks("q8_0", N * (K // 32), 9851 + N)

    def real(b, rows):
        b = P.to_device(b).view(rows, K // 32, 34)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        return (d * b[:, :, 2:].contiguous().view(torch.int8).double()).reshape(rows, K)
    say("q8_0, an odd number of blocks", M, N, K)
    bias = P.to_device(T.normal(N, 0.0, 0.5, seed=N))
    L = ckq.lib()
    try:
        L.ckq_set_gemm_policy(1)
        y = P.dev_gemm_nt("q8_0", P.to_device(x), P.to_device(w), bias, M, N, K).view(M, N).double() - bias.double()
        A, B = real(x, M), real(w, N)
        bound = (A.abs() @ B.abs().T) * (K // 32 + 4) * 2.0 ** -24 + bias.abs().double() * 2.0 ** -23
        assert bool((torch.isfinite(bound)).all())
        assert float(((y - A @ B.T).abs() / bound).max()) <= 1.0
        if M * N * K < 1 << 21:
            rows = w.reshape(N, -1)
            rows[N // 2, 34 * (K // 64):34 * (K // 64) + 2] = (0, 0x7C)
            got = P.dev_gemm_nt("q8_0", P.to_device(x), P.to_device(w), None, M, N, K).cpu().numpy().reshape(M, N)
            with np.errstate(all="ignore"):
                want = T.oracle_gemm_nt("q8_0", x, w, None, M, N, K)
            assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want)) and not np.isfinite(want[:, N // 2]).any()
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("K", [160, 192, 224, 256, 1056, 1088, 1120])
@pytest.mark.parametrize("M,Ns", [(257, (4100, 1, 129)), (70, (9100, 1027, 130)), (333, (3000, 777))])
def test_grouped_q8_0_rows_of_every_number_of_blocks(M, Ns, K):
    """One launch for several matrices whose rows end one, two, three or no blocks after the last whole step, one of a single row and odd ones among them (160 tiles and more: never split along K):
    against fp64 at the bound of the tests of single matrices, and nothing beside C's columns."""
    import torch
    assert sum(-(-n // 128) for n in Ns) * -(-M // 64) >= 160
    x = T.random_blocks("q8_0", M * (K // 32), 9870 + M)
    ws = [T.random_blocks("q8_0", n * (K // 32), 9871 + n) for n in Ns]

    def real(b, rows):
        b = P.to_device(b).view(rows, K // 32, 34)
        d = b[:, :, :2].contiguous().view(torch.float16).double()
        return (d * b[:, :, 2:].contiguous().view(torch.int8).double()).reshape(rows, K)
    say("q8_0 groups, blocks of a row", M, Ns, K)
    xd, Ws = P.to_device(x), [P.to_device(w) for w in ws]
    bs = [P.to_device(T.normal(n, 0.0, 0.5, seed=n)) for n in Ns]
    ys = [torch.full((M, n + 3), 7.0, device="cuda") for n in Ns]
    L = ckq.lib()
    try:
        L.ckq_set_gemm_policy(1)
        P.dev_matmul_sequence([("q8_0", xd, W, b, y, M, n, K, n + 3) for W, b, y, n in zip(Ws, bs, ys, Ns)])
    finally:
        L.ckq_set_gemm_policy(0)
    A = real(x, M)
    for w, b, y, n in zip(ws, bs, ys, Ns):
        B = real(w, n)
        bound = (A.abs() @ B.abs().T) * (K // 32 + 4) * 2.0 ** -24 + b.abs().double() * 2.0 ** -23
        assert bool(torch.isfinite(bound).all()) and bool((y[:, n:] == 7.0).all())
        assert float(((y[:, :n].double() - b.double() - A @ B.T).abs() / bound).max()) <= 1.0, n


@pytest.mark.parametrize("fmt,M,D,N", [("q4_k", 1, 768, (768, 64, 64)), ("q5_k", 1, 1024, (1024, 128, 128)), ("q6_k", 1, 2048, (2048, 17)), ("q5_k", 2, 1280, (200, 130, 7, 64)),
                                       ("q4_k", 3, 1024, (1000, 128, 1)), ("q5_k", 4, 1024, (1024, 128, 128)), ("q6_k", 4, 1792, (31,)), ("q4_k", 5, 1024, (130, 130)),
                                       ("q5_k", 8, 768, (65, 3)), ("q4_k", 1, 512, (512,)), ("q6_k", 4, 256, (300, 9)), ("q4_k", 1, 2304, (300,)), ("q5_k", 1, 1024, (40000,))])
@pytest.mark.parametrize("step", ["rms", "quantize"])
def test_sequence_producer_joined_with_its_matmuls(fmt, M, D, N, step):
    """A producer step and the matmuls behind it, narrow ones among them, on both sides of the sizes that share a launch: every buffer has the bits
    of the steps one by one.  Rows of zeros, a row stride, bias, and results that overlap the input (never one launch)."""
    import torch
    L = ckq.lib()
    ld = D + 8 if step == "rms" else D
    tag = P.STEP["rmsnorm_q8_k" if step == "rms" else "quantize_q8_k"]
    x = T.normal(M * ld, 0.0, 1.0, 9900 + D).reshape(M, ld)
    if M > 1:
        x[1, :] = 0.0
    x[0, 256:512] = 0.0
    gamma = P.to_device(T.normal(D, 1.0, 0.2, 9901))
    Ws = [P.to_device(T.random_blocks(fmt, n * (D // 256), 9902 + n)) for n in N]
    bias = P.to_device(T.normal(N[0], 0.0, 0.5, 9903))

    def run(one_by_one, overlap):
        xd = P.to_device(x.reshape(-1))
        xq = torch.full((M * (D // 256) * 292,), 77, dtype=torch.uint8, device="cuda")
        ys = [torch.full((M, n + 3), 7.0, device="cuda") for n in N]
        ops = [P.MatmulOp(tag, M, 0, D, ld, xd.data_ptr(), gamma.data_ptr() if step == "rms" else None, None, xq.data_ptr(), 1e-5)]
        for i, n in enumerate(N):
            y = xd if overlap and i == 0 else ys[i]
            ops.append(P.MatmulOp(P.FMT[fmt], M, n, D, n + 3, xq.data_ptr(), Ws[i].data_ptr(), bias.data_ptr() if i == 0 else None, y.data_ptr(), 0.0))
        for part in ([[o] for o in ops] if one_by_one else [ops]):
            arr = (P.MatmulOp * len(part))(*part)
            P.check(L.ckq_matmul_sequence_dev(ctypes.cast(arr, ctypes.c_void_p), len(part), 1, P._stream()), "sequence")
        return [xd, xq] + ys
    say("joined", fmt, M, D, N, step)
    for overlap in (False, True):
        if overlap and (N[0] + 3) * M > M * ld:
            continue
        for a, b in zip(run(False, overlap), run(True, overlap)):
            assert torch.equal(a, b)


@pytest.mark.parametrize("fmt,M,D,N", [("q4_k", 2, 1024, (8192, 64, 64)), ("q5_k", 4, 1024, (8000, 40, 40)), ("q6_k", 3, 768, (7990, 33, 5)), ("q4_k", 2, 512, (11000, 70, 9)),
                                       ("q5_k", 3, 512, (11000, 70, 9)), ("q6_k", 2, 1280, (2800, 33, 16)), ("q5_k", 2, 2048, (3000, 500, 64)), ("q4_k", 2, 1024, (16384,)),
                                       ("q4_k", 5, 256, (13113,))])
def test_producer_joined_with_two_rows_a_slot(fmt, M, D, N):
    """Wide matrices, narrow ones beside them, that take one launch with their producer at two rows a slot: it is taken, and every buffer has the
    bits of the steps one by one."""
    import torch
    L = ckq.lib()
    n, nb = len(N), D // 256
    say("joined, two rows", fmt, M, D, N)
    x = P.to_device(T.normal(M * D, 0.0, 1.0, 9910 + D))
    gamma = P.to_device(T.normal(D, 1.0, 0.2, 9911))
    Ws = [P.to_device(T.random_blocks(fmt, r * nb, 9912 + r)) for r in N]
    bias = P.to_device(T.normal(N[0], 0.0, 0.5, 9913))

    def buffers():
        return [torch.full((M * nb * 292,), 77, dtype=torch.uint8, device="cuda")] + [torch.full((M, r), 7.0, device="cuda") for r in N]
    one, two = buffers(), buffers()
    P.check(L.ckq_rmsnorm_q8_k_fused_dev(P._dp(x), P._dp(gamma), P._dp(one[0]), M, D, D, 1e-5, P._stream()), "rmsnorm")
    for i, r in enumerate(N):
        P.check(L.ckq_gemm_nt_dev(P.FMT[fmt], P._dp(one[0]), P._dp(Ws[i]), P._dp(bias) if i == 0 else None, P._dp(one[1 + i]), M, r, D, r, P._stream()), "gemm")
    ptrs = ctypes.c_void_p * n
    rc = L.ckq_launch_gemv_pro(P.FMT[fmt], n, ptrs(*[y.data_ptr() for y in two[1:]]), ptrs(*[W.data_ptr() for W in Ws]), ptrs(bias.data_ptr(), *[None] * (n - 1)),
                               (ctypes.c_int * n)(*N), (ctypes.c_long * n)(*N), D, M, P._dp(x), P._dp(gamma), ctypes.c_float(1e-5), ctypes.c_long(D), P._dp(two[0]), P._stream())
    assert rc == 0
    for a, b in zip(one, two):
        assert torch.equal(a, b)


@pytest.mark.parametrize("M,Ns,K", [(97, (22016,), 1024), (160, (16777,), 1024), (192, (11008,), 768), (512, (5120,), 1536), (481, (6100,), 1024), (300, (6701,), 2816),
                                    (90, (26000,), 1024), (225, (9728, 9728), 1536), (288, (4096, 1024, 1024, 3000), 1280), (512, (6400,), 512)])
def test_gemm_q4_k_token_tile_choice(M, Ns, K):
    """Sizes on both sides of the choice between 64- and 96-token tiles (blocks of an XCD on its CUs), single matrices and groups: the bits of
    64-token tiles."""
    import torch
    L = ckq.lib()
    say("q4_k tile choice", M, Ns, K)
    xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, 9950)), "q8_k", M)
    Ws = [P.to_device(T.random_blocks("q4_k", n * (K // 256), 9951 + n)) for n in Ns]
    got = {}
    try:
        L.ckq_set_gemm_policy(1)
        for tile in (0, 64, 96):
            L.ckq_set_prefill_variant(P.FMT["q4_k"], tile)
            ys = [torch.full((M, n), 7.0, device="cuda") for n in Ns]
            P.dev_matmul_sequence([("q4_k", xq, W, None, y, M, n, K) for W, y, n in zip(Ws, ys, Ns)])
            got[tile] = ys
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(P.FMT["q4_k"], 0)
    for tile in (0, 96):
        for a, b in zip(got[tile], got[64]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("fmt", FMTS)
@pytest.mark.parametrize("M", [9, 65, 129, 200, 673])
def test_gemm_mfma_tiles_over_the_xcds(fmt, M):
    """Every tile is computed once whatever the numbers of tiles: 1 to 17 tiles of weight rows, 1 to 11 of tokens, split along K and not, one
    matrix and a group.  Against the streaming kernel, whose terms and order differ: the bar of the other parity tests."""
    import torch
    L = ckq.lib()
    for K in (256, 2304):
        xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, 9960)), T.act_fmt(fmt), M)
        Ns = (1, 129, 700, 900, 1100, 2049, 2100)
        Ws = [P.to_device(T.random_blocks(fmt, n * (K // T.ELEMS[fmt]), 9961 + n)) for n in Ns]
        say("tiles over the XCDs", fmt, M, K)

        def run(policy, group):
            L.ckq_set_gemm_policy(policy)
            ys = [torch.full((M, n), 7.0, device="cuda") for n in Ns]
            ops = [(fmt, xq, W, None, y, M, n, K) for W, y, n in zip(Ws, ys, Ns)]
            for part in ([ops[:4], ops[4:]] if group else [[o] for o in ops]):
                P.dev_matmul_sequence(part)
            return ys
        try:
            want, one, grp = run(2, False), run(1, False), run(1, True)
        finally:
            L.ckq_set_gemm_policy(0)
        for w, a, b in zip(want, one, grp):
            bar = TOL * float(w.abs().max())
            assert float((a - w).abs().max()) <= bar and float((b - w).abs().max()) <= bar


PIECES_OF_K = [(65, 1100, 7936), (40, 300, 5376), (65, 650, 11008), (129, 1200, 1664), (129, 1200, 5376), (129, 1200, 6656), (129, 1500, 7168), (65, 129, 16384), (200, 2700, 2304), (385, 1700, 3328)]


def _pieces_of_k(tiles, steps):
    """(pieces, steps of each but the last) of a launch of `tiles` tiles that is split along K."""
    s = max(1, min(256 // tiles, steps // 4, 16)) if tiles < 160 and steps >= 8 else 1
    per = -(-steps // s)
    return -(-steps // per), per


def test_sizes_of_the_pieces_of_k_are_uneven():
    """Of the first five sizes below the 64-token tiles of the K-quants, and of the first three and the fourth the 32-, 64- and 96-token tiles of Q8_0: more than four pieces (fewer may be waves of
    one block instead), a shorter last one, and a number of pieces of all tiles that eight does not divide."""
    for M, N, K in PIECES_OF_K[:3] + PIECES_OF_K[4:6]:
        tiles = -(-M // 64) * -(-N // 128)
        pieces, per = _pieces_of_k(tiles, K // 256)
        assert pieces > 4 and tiles * pieces % 8 and K // 256 % per, (M, N, K)
    for M, N, K in PIECES_OF_K[:4]:
        for tokens in (32, 64, 96):
            tiles = -(-M // tokens) * -(-N // 128)
            pieces, per = _pieces_of_k(tiles, -(-K // 128))
            assert pieces > 1 and tiles * pieces % 8 and -(-K // 128) % per, (M, N, K, tokens)


@pytest.mark.parametrize("fmt,M,N,K", [(fmt, *size) for fmt in FMTS for size in PIECES_OF_K if size[2] % T.ELEMS[fmt] == 0])
def test_gemm_pieces_of_k_dealt_with_their_tiles(fmt, M, N, K):
    """Every piece of K of every tile is computed once, where eight XCDs divide neither the number of pieces nor that of the tiles and the last piece is shorter (the test above); where they do
    (36 tiles in seven equal pieces, of Q8_0 in more; 4 in sixteen); and where the K-quants' pieces are waves of one block instead (two of 5 and of 7 blocks, the last two sizes).
    Against the streaming kernel, whose terms and order differ: the bar of the other parity tests."""
    import torch
    L = ckq.lib()
    say("pieces of K over the XCDs", fmt, M, N, K)
    xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, 9963)), T.act_fmt(fmt), M)
    W = P.to_device(T.random_blocks(fmt, N * (K // T.ELEMS[fmt]), 9964))
    try:
        L.ckq_set_gemm_policy(2)
        want = P.dev_gemm_nt(fmt, xq, W, None, M, N, K).clone()
        L.ckq_set_gemm_policy(1)
        got = P.dev_gemm_nt(fmt, xq, W, None, M, N, K)
    finally:
        L.ckq_set_gemm_policy(0)
    assert float((got - want).abs().max()) <= TOL * float(want.abs().max())


@pytest.mark.parametrize("fmt,variants", [("q5_k", (2, 1)), ("q4_k", (64, 96))])
@pytest.mark.parametrize("M,Ns,K", [(405, (11008, 11008), 768), (65, (17000,), 512), (88, (9000, 7700), 256), (282, (7041,), 1024), (257, (6657, 300), 512)])
def test_gemm_ragged_token_tiles_dealt_last(fmt, variants, M, Ns, K):
    """Launches whose ragged token tiles come last, one matrix and two, with a bias and a padded C: the bits of the other tile kernel of the
    format, which deals its tiles otherwise, and nothing beside C's columns."""
    import torch
    L = ckq.lib()
    say("ragged tiles last", fmt, M, Ns, K)
    xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, 9990)), "q8_k", M)
    Ws = [P.to_device(T.random_blocks(fmt, n * (K // 256), 9991 + n)) for n in Ns]
    bs = [P.to_device(T.normal(n, 0.0, 0.5, 9992 + n)) for n in Ns]
    got = []
    try:
        L.ckq_set_gemm_policy(1)
        for v in variants:
            L.ckq_set_prefill_variant(P.FMT[fmt], v)
            ys = [torch.full((M, n + 3), 7.0, device="cuda") for n in Ns]
            P.dev_matmul_sequence([(fmt, xq, W, b, y, M, n, K, n + 3) for W, b, y, n in zip(Ws, bs, ys, Ns)])
            got.append(ys)
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(P.FMT[fmt], 0)
    for a, b, n in zip(got[0], got[1], Ns):
        assert torch.equal(a, b) and bool((a[:, n:] == 7.0).all())


@pytest.mark.parametrize("M,Ns,K", [(64, (20000,), 512), (40, (16700,), 1024), (160, (10000,), 768), (190, (4096, 2048, 3000), 512), (345, (10391,), 512), (266, (9000, 9000), 768),
                                    (247, (10593,), 2304), (129, (16300,), 256), (600, (3000,), 1280)])
def test_gemm_q6_k_kernel_choice(M, Ns, K):
    """Sizes on the sides of the choice between 64-token, 128-token and paired tiles, single matrices and groups, not split along K: one set of
    bits, that of the paired kernel."""
    import torch
    L = ckq.lib()
    say("q6_k kernel choice", M, Ns, K)
    xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, 9970)), "q8_k", M)
    Ws = [P.to_device(T.random_blocks("q6_k", n * (K // 256), 9971 + n)) for n in Ns]
    got = {}
    try:
        L.ckq_set_gemm_policy(1)
        for variant in (0, 1, 2):
            L.ckq_set_prefill_variant(P.FMT["q6_k"], variant)
            ys = [torch.full((M, n), 7.0, device="cuda") for n in Ns]
            P.dev_matmul_sequence([("q6_k", xq, W, None, y, M, n, K) for W, y, n in zip(Ws, ys, Ns)])
            got[variant] = ys
    finally:
        L.ckq_set_gemm_policy(0)
        L.ckq_set_prefill_variant(P.FMT["q6_k"], 0)
    for variant in (0, 1):
        for a, b in zip(got[variant], got[2]):
            assert torch.equal(a, b)


@pytest.mark.parametrize("N,K", [(128, 2048), (128, 3072), (300, 5120), (64, 7168), (132, 8192), (260, 16384), (200, 9216)])
def test_gemm_split_k_partials_added(N, K):
    """K splits of two to sixteen, added four outputs a thread where rows of C start on 16 bytes and one elsewhere, with a bias that is and is not
    so aligned and without: one set of bits, the same as on a second call."""
    import torch
    L = ckq.lib()
    M = 70
    xq = P.dev_quantize(P.to_device(T.normal(M * K, 0.0, 1.0, 9980)), "q8_k", M)
    W = P.to_device(T.random_blocks("q4_k", N * (K // 256), 9981))
    b = P.to_device(T.normal(N + 1, 0.0, 0.5, 9982))
    say("split partials", N, K)

    def run(ldc, bias):
        c = torch.full((M, ldc), 7.0, device="cuda")
        P.check(L.ckq_gemm_nt_dev(P.FMT["q4_k"], P._dp(xq), P._dp(W), bias, P._dp(c), M, N, K, ldc, P._stream()), "ckq_gemm_nt_dev")
        assert bool((c[:, N:] == 7.0).all())
        return c[:, :N].clone()
    try:
        L.ckq_set_gemm_policy(1)
        plain = run(N, None)
        assert torch.equal(plain, run(N + 1, None)) and torch.equal(plain, run(N, None))
        for ofs in (0, 1):
            p = ctypes.c_void_p(b.data_ptr() + 4 * ofs)
            want = plain + b[ofs:ofs + N]
            assert torch.equal(run(N, p), want) and torch.equal(run(N + 3, p), want)
    finally:
        L.ckq_set_gemm_policy(0)
