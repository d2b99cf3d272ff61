"""CPU checks of the C-ABI library: it loads, exports every declared symbol,
and the host logic that needs no device (argument screening) behaves like the
reference.  No kernel is launched here."""
import ctypes
import importlib
import os
import subprocess

import numpy as np
import pytest

ckq = importlib.import_module("c-kernel-engine_amd")


@pytest.fixture(scope="module")
def L():
    if not os.path.exists(ckq.lib_path()):
        ckq.build()
    return ckq.lib()


def test_every_declared_symbol_is_exported(L):
    names = ckq.declared_symbols()
    assert len(names) >= 60
    missing = [n for n in names if not hasattr(L, n)]
    assert not missing, missing
    # and the binding table covers the header
    from importlib import import_module
    api = import_module("c-kernel-engine_amd.api")
    assert sorted(api._SIGS) == names


def test_reference_symbol_names_present(L):
    # the symbols a generated libmodel.so resolves for this path
    # (reference include/ckernel_engine.h:192-363)
    for n in ["quantize_row_q8_k", "quantize_batch_q8_k", "quantize_row_q8_0", "gemv_q4_k_q8_k",
              "gemv_q4_k_q8_k_parallel_simd", "gemm_nt_q4_k_q8_k", "gemv_q5_k", "gemm_nt_q5_k",
              "gemv_q6_k_q8_k", "gemv_q6_k_q8_k_parallel_simd", "gemm_nt_q6_k_q8_k", "gemv_q8_0_q8_0",
              "gemv_q8_0", "gemm_nt_q8_0_q8_0", "vec_dot_q6_k_q8_k", "vec_dot_q8_0_q8_0"]:
        assert hasattr(L, n)
    # the parity scripts' wrappers (reference include/ck_parity_api.h:42-56, 193-201)
    for n in ["ck_test_dequant_q4_k", "ck_test_dequant_q6_k", "ck_test_quantize_q8_k", "ck_test_gemv_q4_k",
              "ck_test_gemv_q6_k", "ck_test_gemm_q4_k", "ck_test_gemm_q6_k", "ck_test_gemm_q8_0"]:
        assert hasattr(L, n)


def test_block_size_getters(L):
    assert L.ck_get_block_q4_k_size() == 144
    assert L.ck_get_block_q6_k_size() == 210
    assert L.ck_get_block_q8_k_size() == 292
    assert L.ck_get_qk_k() == 256


def test_bad_arguments_return_without_touching_output(L):
    """NULL pointer or non-positive dimension: silent return
    (reference gemm_kernels_q4k_q8k.c:188-190, :221-223, :307-312)."""
    y = np.full(8, 7.0, np.float32)
    w = np.zeros(8 * 144, np.uint8)
    x = np.zeros(292, np.uint8)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    L.gemv_q4_k_q8_k(p(y), None, p(x), 8, 256)
    L.gemv_q4_k_q8_k(p(y), p(w), None, 8, 256)
    L.gemv_q4_k_q8_k(p(y), p(w), p(x), 0, 256)
    L.gemv_q4_k_q8_k(p(y), p(w), p(x), 8, -256)
    L.gemv_q4_k_q8_k_parallel(p(y), p(w), p(x), 8, 256, 3, 3)   # ith >= nth
    L.gemv_q4_k_q8_k_parallel(p(y), p(w), p(x), 8, 256, -1, 3)
    L.gemv_q4_k_q8_k_parallel_simd(p(y), p(w), p(x), 8, 256, 0, 0)
    L.gemv_q6_k_q8_k_parallel(p(y), p(w), p(x), 8, 256, 5, 2)
    L.gemv_q8_0_q8_0_parallel_simd(p(y), p(w), p(x), 8, 256, 2, 2)
    L.gemm_nt_q4_k_q8_k(None, p(w), None, p(y), 1, 8, 256)
    L.gemm_nt_q6_k_q8_k(p(x), p(w), None, p(y), 1, 0, 256)
    L.gemv_q5_k_q8_k(p(y), p(w), p(x), 8, 200)                   # K % 256 != 0 (gemm_kernels_q5_k.c:313-315)
    L.vec_dot_q6_k_q8_k(0, p(y), p(w), p(x))
    L.quantize_row_q8_k(None, p(x), 256)
    L.quantize_row_q8_k(p(y), p(x), 0)
    assert np.all(y == 7.0)
    assert L.ckq_last_error() == 0


def test_dev_entry_points_reject_bad_shapes(L):
    # status codes come back before anything touches a device
    one = ctypes.c_void_p(16)
    assert L.ckq_gemv_q4_k_q8_k_dev(one, one, one, 4, 100, None) == -2
    assert L.ckq_gemv_q4_k_q8_k_dev(None, one, one, 4, 256, None) == -1
    assert L.ckq_gemm_nt_dev(9, one, one, None, one, 1, 4, 256, 4, None) == -3
    assert L.ckq_quantize_q8_k_dev(one, one, 1, 100, None) == -2
    assert L.ckq_quantize_q8_0_dev(one, one, 0, 32, None) == -1
    assert b"multiple" in L.ckq_error_string(-2)


def test_manifest_hook_parses_without_touching_a_device(L, tmp_path):
    """The loader hook reads the reference's manifest format; tensors of other
    dtypes are skipped, so a manifest without quantized weights needs no device;
    unreadable files and malformed lines are reported as argument errors."""
    base = np.zeros(64, np.uint8)
    p = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    m = tmp_path / "weights_manifest.map"
    m.write_text("# name|dtype|file_offset|size|runtime_offset\n\n"
                 "model.norm.weight|fp32|8|3584|0\n"
                 "model.rope.cache|f16|0x1000|128|4096\n")
    assert L.ckq_weights_register_manifest(p(base), str(m).encode()) == 0
    assert L.ckq_weights_register_manifest(p(base), str(tmp_path / "missing.map").encode()) == -1
    assert L.ckq_weights_register_manifest(None, str(m).encode()) == -1
    bad = tmp_path / "bad.map"
    bad.write_text("model.norm.weight|fp32|8|3584\n")
    assert L.ckq_weights_register_manifest(p(base), str(bad).encode()) == -1
    assert L.ckq_last_error() == 0
    nbytes = ctypes.c_size_t(7)
    assert L.ckq_weights_resident(ctypes.byref(nbytes)) == 0 and nbytes.value == 0


def test_header_compiles_next_to_the_reference_headers(tmp_path):
    """One translation unit with the reference's own headers and this library's:
    every shared prototype must be declaration-compatible (the fused MLP takes
    the reference's CKDataType, include/ckernel_engine.h:666-680)."""
    ref_inc = "/root/reference/include"
    if not os.path.exists(os.path.join(ref_inc, "ckernel_engine.h")):
        pytest.skip("reference checkout not present")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    src = tmp_path / "tu.c"
    src.write_text('#include "ckernel_engine.h"\n#include "ckernel_quant.h"\n#include "ck_parity_api.h"\n'
                   '#include "ckernel_quant_hip.h"\n'
                   'void (*p)(const float *, const void *, const float *, CKDataType, const void *, const float *,\n'
                   '          CKDataType, float *, int, int, int, int, int, void *) = fused_mlp_swiglu_prefill_w1w2_quant;\n'
                   'int main(void) { return 0; }\n')
    r = subprocess.run(["gcc", "-std=gnu11", "-Wall", "-Werror", "-I" + ref_inc, "-I" + os.path.join(root, "include"),
                        "-c", str(src), "-o", str(tmp_path / "tu.o")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    # and on its own, as C and as C++
    alone = tmp_path / "alone.c"
    alone.write_text('#include "ckernel_quant_hip.h"\nint main(void) { return (int)sizeof(ckq_ck_dtype) - 4; }\n')
    for cc, std in (("gcc", "-std=gnu11"), ("g++", "-std=c++17")):
        r = subprocess.run([cc, std, "-Wall", "-Werror", "-x", "c" if cc == "gcc" else "c++",
                            "-I" + os.path.join(root, "include"), "-c", str(alone), "-o", str(tmp_path / "a.o")],
                           capture_output=True, text=True)
        assert r.returncode == 0, r.stderr


def test_grid_chunk_index_arithmetic(L):
    """Launches whose token tiles exceed gridDim.y's 65 535 are issued in chunks;
    the chunks must tile [0, total) exactly, in order, without overlap."""
    L.ckq_grid_chunk.restype = None
    L.ckq_grid_chunk.argtypes = [ctypes.c_long] * 3 + [ctypes.POINTER(ctypes.c_long)] * 2
    for total, per in ((1, 65535), (65535, 65535), (65536, 65535), (70000, 65535), (131072, 65535),
                       (8 * 65535 + 3, 8 * 65535), (200000, 2 * 65535)):
        covered, c = 0, 0
        while c * per < total:
            first, count = ctypes.c_long(), ctypes.c_long()
            L.ckq_grid_chunk(total, per, c, ctypes.byref(first), ctypes.byref(count))
            assert first.value == covered and 0 < count.value <= per
            covered += count.value
            c += 1
        assert covered == total and c == -(-total // per)


STREAM, TILES, ROWS16_STREAM, ROWS16_TILES = range(4)
ROUTE_SHAPES = [(n, k) for n in (1, 128, 1000, 4096, 16383, 32000) for k in (256, 512, 1024, 4096, 11008, 16640)]
ROUTE_TOKENS = (1, 2, 3, 4, 5, 8, 9, 16, 33, 93, 512)


def route(L, fmt, n, k, tokens, f32=False, aligned=1):
    tag = {"q4_k": 17, "q6_k": 18, "q8_0": 16}[fmt] if f32 else ckq.parity.FMT[fmt]
    return L.ckq_launch_route(tag, n, k, tokens, aligned)


def test_forced_policies_keep_their_kernels(L):
    """STREAM streams at every token count, MATRIX takes the tile kernels above eight tokens (fp32 activations: from two on), over
    all formats and sizes; the automatic choice uses the 16-row tiles somewhere at either side of eight tokens."""
    fmts = [(f, False) for f in ("q4_k", "q5_k", "q6_k", "q8_0", "q5_0")] + [(f, True) for f in ("q4_k", "q6_k", "q8_0")]
    try:
        seen = set()
        for fmt, f32 in fmts:
            for n, k in ROUTE_SHAPES:
                for t in ROUTE_TOKENS:
                    L.ckq_set_gemm_policy(0)
                    seen.add((route(L, fmt, n, k, t, f32), t > 8))
                    L.ckq_set_gemm_policy(2)
                    assert route(L, fmt, n, k, t, f32) == STREAM, (fmt, f32, n, k, t)
                    L.ckq_set_gemm_policy(1)
                    if t > (1 if f32 else 8):
                        assert route(L, fmt, n, k, t, f32) == TILES, (fmt, f32, n, k, t)
        assert {(ROWS16_STREAM, False), (ROWS16_STREAM, True), (ROWS16_TILES, True)} <= seen
    finally:
        L.ckq_set_gemm_policy(0)


@pytest.mark.parametrize("fmt,variants", [("q4_k", (64, 96)), ("q5_k", (1, 2)), ("q6_k", (1, 2))])
def test_forced_variants_keep_their_kernels(L, fmt, variants):
    """A tile kernel that was asked for serves every size that the automatic policy takes off the streaming kernel; variant 16
    sends everything from two tokens on (K up to 16384) to the 16-row tiles, in the order of the kernel they stand in for."""
    tag = ckq.parity.FMT[fmt]
    try:
        for n, k in ROUTE_SHAPES:
            for t in ROUTE_TOKENS:
                L.ckq_set_prefill_variant(tag, 0)
                auto = route(L, fmt, n, k, t)
                for v in variants:
                    L.ckq_set_prefill_variant(tag, v)
                    assert route(L, fmt, n, k, t) == (TILES if auto in (TILES, ROWS16_TILES) else auto), (v, n, k, t)
                L.ckq_set_prefill_variant(tag, 16)
                if t >= 2 and k <= 16384:
                    assert route(L, fmt, n, k, t) == (ROWS16_TILES if auto in (TILES, ROWS16_TILES) else ROWS16_STREAM), (n, k, t)
                else:
                    assert route(L, fmt, n, k, t) == auto
    finally:
        L.ckq_set_prefill_variant(tag, 0)


@pytest.mark.parametrize("fmt,n,k,tokens,want", [
    ("q5_k", 290, 1792, 25, STREAM), ("q6_k", 435, 1536, 13, STREAM), ("q4_k", 1024, 1024, 16, STREAM),
    ("q5_k", 4096, 8192, 4, STREAM), ("q4_k", 4096, 11008, 4, STREAM), ("q6_k", 4096, 8192, 4, STREAM),
    ("q6_k", 4096, 11008, 4, ROWS16_STREAM), ("q5_k", 5000, 1024, 24, ROWS16_STREAM), ("q4_k", 5345, 1280, 26, ROWS16_STREAM),
    ("q6_k", 4096, 4096, 13, ROWS16_TILES), ("q5_k", 4864, 1024, 93, ROWS16_STREAM), ("q4_k", 11008, 4096, 512, TILES),
    ("q6_k", 3759, 6912, 111, TILES), ("q6_k", 7371, 6912, 29, TILES), ("q6_k", 292, 6400, 1138, TILES), ("q6_k", 7534, 2560, 10, ROWS16_TILES),
    ("q4_k", 27284, 256, 120, TILES), ("q4_k", 10244, 768, 110, TILES), ("q4_k", 17582, 256, 176, TILES), ("q5_k", 26823, 256, 117, TILES), ("q5_k", 3199, 1792, 185, ROWS16_TILES),
    ("q4_k", 6552, 1024, 64, ROWS16_TILES), ("q5_k", 5029, 1792, 104, ROWS16_TILES), ("q6_k", 28565, 1024, 62, TILES), ("q6_k", 5000, 2048, 64, ROWS16_TILES),
    ("q5_k", 1141, 256, 64, ROWS16_STREAM), ("q5_k", 948, 256, 80, ROWS16_STREAM), ("q5_k", 3258, 256, 24, ROWS16_STREAM), ("q6_k", 368, 2048, 47, ROWS16_STREAM),
    ("q6_k", 454, 1792, 34, ROWS16_STREAM), ("q6_k", 1458, 512, 44, ROWS16_STREAM), ("q4_k", 1284, 512, 36, ROWS16_STREAM), ("q4_k", 438, 1024, 36, STREAM), ("q5_k", 177, 1024, 20, STREAM)])
def test_16_row_tiles_where_they_are_the_faster_ones(L, fmt, n, k, tokens, want):
    """Shapes at which the kernels were timed against each other; the faster one is taken."""
    assert route(L, fmt, n, k, tokens) == want


@pytest.mark.parametrize("fmt,n,k,tokens,want", [
    ("q4_k", 2304, 2304, 8, ROWS16_STREAM), ("q4_k", 1792, 4608, 7, ROWS16_STREAM), ("q4_k", 1024, 3072, 8, STREAM), ("q5_k", 3328, 3328, 8, ROWS16_STREAM), ("q5_k", 1280, 5632, 8, ROWS16_STREAM),
    ("q5_k", 1024, 2560, 6, STREAM), ("q6_k", 3584, 10752, 5, ROWS16_STREAM), ("q6_k", 1024, 3328, 5, STREAM), ("q6_k", 1792, 1792, 8, STREAM),
    ("q5_k", 3328, 13568, 3, ROWS16_STREAM), ("q6_k", 4352, 4352, 4, ROWS16_STREAM), ("q6_k", 2560, 2560, 4, STREAM), ("q4_k", 3840, 3840, 4, STREAM), ("q6_k", 14336, 14336, 2, STREAM)])
def test_16_row_tiles_at_two_to_eight_tokens(L, fmt, n, k, tokens, want):
    """Single matrices on either side of the line, where both kernels were timed."""
    assert route(L, fmt, n, k, tokens) == want


@pytest.mark.parametrize("n,k,tokens,want", [(11493, 11008, 4, ROWS16_STREAM), (15968, 10496, 3, ROWS16_STREAM), (17034, 6912, 4, ROWS16_STREAM), (16040, 14080, 4, ROWS16_STREAM),
                                             (567, 9984, 3, STREAM), (8520, 4096, 3, STREAM), (576, 14592, 4, STREAM)])
def test_q6_k_long_rows_at_three_and_four_tokens(L, n, k, tokens, want):
    """Rows of two to four passes of the streaming kernel, weights of some megabytes: both kernels were timed (as one matrix or as several of as many rows), the faster one by a seventh and more is taken."""
    assert route(L, "q6_k", n, k, tokens) == want


@pytest.mark.parametrize("n,k,tokens,want", [(8695, 1024, 8, ROWS16_STREAM), (7479, 1024, 8, ROWS16_STREAM), (7256, 1024, 5, ROWS16_STREAM), (7434, 1024, 8, ROWS16_STREAM), (15500, 512, 6, ROWS16_STREAM),
                                             (9500, 768, 7, ROWS16_STREAM), (3500, 1024, 8, STREAM), (7500, 512, 8, STREAM), (3500, 768, 6, STREAM)])
def test_q4_k_short_rows_at_five_to_eight_tokens(L, n, k, tokens, want):
    """Rows of two to four blocks on either side of the line, where both kernels were timed."""
    assert route(L, "q4_k", n, k, tokens) == want


APART = -7


def group_route(L, fmt, tokens, k, ns):
    return L.ckq_launch_group_route(ckq.parity.FMT[fmt], len(ns), (ctypes.c_int * len(ns))(*ns), k, tokens)


@pytest.mark.parametrize("fmt", ["q4_k", "q5_k", "q6_k"])
@pytest.mark.parametrize("tokens,k,ns,want", [
    (8, 4352, (4352, 1088, 1088), ROWS16_STREAM), (5, 2560, (2560, 640, 640), ROWS16_STREAM), (6, 3072, (3072, 1536, 1536), ROWS16_STREAM), (5, 2048, (5632, 5632), ROWS16_STREAM),
    (8, 1280, (1280, 320, 320), ROWS16_STREAM), (6, 7424, (1500, 1, 300), ROWS16_STREAM), (5, 16384, (700, 500), ROWS16_STREAM), (4, 4608, (4608, 1152, 1152), ROWS16_STREAM),
    (7, 512, (512, 128, 128), STREAM), (8, 768, (1000, 17, 1), STREAM), (8, 256, (70, 4000), STREAM), (7, 11008, (96, 33), STREAM), (5, 16640, (64, 32), STREAM),
    (4, 2560, (2560, 640, 640), STREAM), (3, 8192, (2100, 40), STREAM), (3, 14592, (300, 17), STREAM), (2, 4608, (4608, 600), STREAM)])
def test_groups_of_few_tokens_have_one_kernel(L, fmt, tokens, k, ns, want):
    """The sizes whose bits are compared on the GPU (test_matrices_of_three_to_eight_tokens_share_one_choice_of_kernel) lie on both sides of the line."""
    assert group_route(L, fmt, tokens, k, ns) == want


@pytest.mark.parametrize("fmt,tokens,k,ns,want", [
    # three and four tokens, long rows
    ("q6_k", 4, 11008, (3831, 3831, 3831), ROWS16_STREAM), ("q6_k", 3, 10496, (7984, 7984), ROWS16_STREAM), ("q6_k", 4, 6912, (8517, 4258, 4258), ROWS16_STREAM),
    # too few tiles for a shared launch: one launch of 16-row tiles, or one by one
    ("q5_k", 105, 2304, (2304, 2304, 2304), ROWS16_TILES), ("q6_k", 105, 2304, (2304, 2304, 2304), ROWS16_TILES), ("q5_k", 98, 3072, (3072, 1536, 1536), ROWS16_TILES),
    ("q6_k", 64, 5120, (5120, 1280, 1280), ROWS16_TILES), ("q5_k", 313, 2560, (2560, 320, 320), ROWS16_TILES), ("q6_k", 17, 5120, (4100, 2561), ROWS16_TILES),
    ("q5_k", 34, 8704, (8704, 1088, 1088), APART), ("q6_k", 34, 8704, (8704, 1088, 1088), APART), ("q5_k", 81, 4352, (4352, 1088, 1088), APART), ("q5_k", 17, 5120, (4100, 2561), APART),
    # Q4_K against one launch of unsplit tiles, and against single launches
    ("q4_k", 65, 1536, (6912, 6912), TILES), ("q4_k", 133, 1280, (3840, 3840), TILES), ("q4_k", 32, 3840, (11008, 11008), TILES), ("q4_k", 257, 768, (3584, 3584), TILES),
    ("q4_k", 32, 1280, (10240, 10240), ROWS16_TILES), ("q4_k", 98, 2816, (2816, 1408, 1408), ROWS16_TILES)])
def test_groups_go_where_they_were_timed_to_be_faster(L, fmt, tokens, k, ns, want):
    assert group_route(L, fmt, tokens, k, ns) == want


def test_group_route_refuses_what_is_no_group(L):
    assert group_route(L, "q4_k", 8, 4096, (4096,)) == -1 and group_route(L, "q8_0", 8, 4096, (4096, 4096)) == -1
    assert group_route(L, "q4_k", 8, 4000, (64, 64)) == -1 and group_route(L, "q4_k", 0, 4096, (64, 64)) == -1


@pytest.mark.parametrize("M,Ns,last", [(405, (11008, 11008), True), (276, (7680, 7680), True), (139, (5888, 5888), True), (282, (7041,), True), (65, (17000,), True),
                                       (88, (9000, 7700), True), (341, (6912, 6912), False), (384, (11008, 11008), False), (227, (8960, 8960), False),
                                       (405, (4096, 1024, 1024), False), (9, (34000,), False), (400, (28672,), False)])
def test_ragged_token_tiles_dealt_last(L, M, Ns, last):
    """Sizes at which the order of a launch's tiles was timed.  Dealt last, the ragged tiles have the highest block ids, every tile
    has one block, and an XCD (block id modulo 8) has at most two more of a matrix than another."""
    N, out = (ctypes.c_int * len(Ns))(*Ns), [ctypes.c_int() for _ in range(3)]

    def tile(i):
        grid = L.ckq_launch_ragged_last(M, len(Ns), N, i, *map(ctypes.byref, out))
        return grid, tuple(o.value for o in out)
    grid = tile(0)[0]
    assert bool(grid) == last
    if last:
        dealt = [(i, t) for i, t in ((i, tile(i)[1]) for i in range(grid)) if t[0] >= 0]
        whole, tiles = M // 64, [-(-n // 128) for n in Ns]
        assert sorted(t for _, t in dealt) == [(p, r, c) for p, n in enumerate(tiles) for r in range(n) for c in range(whole + 1)]
        order = [c == whole for _, (_, _, c) in dealt]
        assert order == sorted(order)
        per_xcd = [sum(i % 8 == x for i, _ in dealt) for x in range(8)]
        assert max(per_xcd) - min(per_xcd) <= 2 * len(Ns)


@pytest.mark.parametrize("n,k,tokens,want", [(11000, 1280, 65, TILES), (20480, 1280, 32, ROWS16_TILES), (20480, 1280, 48, TILES), (13824, 1536, 65, TILES), (7680, 1280, 133, TILES),
                                             (22016, 2816, 24, TILES), (32000, 2048, 40, TILES), (25000, 1536, 20, TILES), (28000, 768, 100, TILES), (8192, 4096, 16, ROWS16_TILES)])
def test_q4_k_unsplit_tiles_or_16_row_tiles(L, n, k, tokens, want):
    """160 tiles of 64 tokens and more: sizes at which both kernels were timed, the faster one (within 4 %) is taken; one token group keeps its own rule."""
    assert route(L, "q4_k", n, k, tokens) == want


def test_q8_0_order_of_sums_does_not_hang_on_the_width(L):
    """Long rows on dwords stream where shorter rows of as many bytes do, up to 16 tokens always: the tile kernel's chains of additions are longer, and
    it may need scratch for a split along K.  Host arithmetic of the same line."""
    for k in (3648, 7232, 7296, 8192, 9728, 11008, 16384):
        for n in (200, 600, 1200, 4096, 16532):
            mb = n * (k // 32) * 34e-6
            for t in (9, 11, 16, 17, 24, 40, 64):
                tiles = 4.8 + -(-t // 8) * mb / 5.0 > max(14.0, 9.0 + mb / 2.5)
                assert route(L, "q8_0", n, k, t) == (TILES if tiles else STREAM), (n, k, t)
                assert t > 16 or not tiles


@pytest.mark.parametrize("M,N,K,form", [(326, 17318, 2816, 2), (252, 8318, 1280, 2), (162, 10958, 2816, 2), (600, 31833, 1536, 2), (266, 35817, 768, 2), (512, 11008, 4096, 2),
                                        (247, 10593, 3584, 1), (241, 13644, 5632, 1), (105, 28675, 4864, 1), (48, 32000, 4096, 0), (160, 10000, 4096, 0), (93, 4096, 4096, 0)])
def test_q6_k_kernel_is_the_fastest_one(L, M, N, K, form):
    """Sizes at which the three kernels were timed against each other; the fastest one is taken."""
    assert L.ckq_launch_q6k_form(M, N, K) == form


@pytest.mark.parametrize("fmt,n_row,rows,elems,width", [
    ("q4_k", 256, 512, 4, 64), ("q4_k", 512, 2048, 4, 128), ("q4_k", 4096, 384, 4, 256), ("q4_k", 5120, 384, 4, 256), ("q4_k", 1024, 6000, 4, 256), ("q4_k", 8192, 2048, 16, 256),
    ("q4_k", 6144, 1024, 16, 192), ("q4_k", 4096, 1500, 16, 256), ("q6_k", 256, 40000, 4, 64), ("q6_k", 1024, 2048, 4, 256), ("q6_k", 512, 10000, 4, 128), ("q6_k", 5120, 1024, 16, 192),
    ("q6_k", 4096, 700, 16, 256), ("q6_k", 4096, 512, 4, 256), ("q8_0", 896, 20000, 4, 256), ("q8_0", 32, 1, 4, 64)])
def test_dequantizer_form_is_the_faster_one(L, fmt, n_row, rows, elems, width):
    """Sizes at which four and sixteen elements a thread were timed against each other; blocks no larger than their share of the row needs."""
    w = ctypes.c_int()
    assert (L.ckq_launch_dequant_form(ckq.parity.FMT[fmt], n_row, rows, ctypes.byref(w)), w.value) == (elems, width)


def test_workspace_slot_bookkeeping(L):
    """Slot choice of the per-(device, stream, kind) scratch table of the K-split
    GEMMs: a known key finds its slot, a new key takes the first free slot, and
    with every slot taken the least recently used one is handed out for
    recycling - more distinct streams than slots must not fail."""
    n = 8
    U64 = ctypes.c_uint64 * n
    L.ckq_workspace_pick.restype = ctypes.c_int
    L.ckq_workspace_pick.argtypes = [U64, U64, ctypes.c_int, ctypes.c_uint64]
    keys, use = U64(), U64()
    clock = 0
    where = {}
    for k in range(1, 3 * n + 1):                    # 24 distinct "streams" through 8 slots
        key = (1 << 63) | (0x7f0000001000 + 64 * k)
        i = L.ckq_workspace_pick(keys, use, n, key)
        assert 0 <= i < n
        if k <= n:
            assert keys[i] == 0 and i == k - 1       # first free slot, in order
        else:
            assert use[i] == min(use)                # least recently used
            where = {kk: ii for kk, ii in where.items() if ii != i}
        keys[i] = key
        clock += 1
        use[i] = clock
        where[key] = i
        # a key that is present is found again, whatever its age
        for kk, ii in where.items():
            assert L.ckq_workspace_pick(keys, use, n, kk) == ii
    # touching an old entry protects it from being the next victim
    oldest = min(range(n), key=lambda j: use[j])
    clock += 1
    use[oldest] = clock
    assert L.ckq_workspace_pick(keys, use, n, (1 << 63) | 0x1234) != oldest


def test_no_device_fails_loudly():
    """Without a GPU a compute call must not succeed silently: the library
    reports the HIP error and aborts the process."""
    import torch
    if torch.cuda.is_available():
        pytest.skip("a GPU is present")
    code = (
        "import importlib, numpy as np, ctypes\n"
        "ckq = importlib.import_module('c-kernel-engine_amd')\n"
        "x = np.ones(256, np.float32); y = np.zeros(292, np.uint8)\n"
        "ckq.lib().quantize_row_q8_k(x.ctypes.data_as(ctypes.c_void_p), y.ctypes.data_as(ctypes.c_void_p), 256)\n"
        "print('survived')\n"
    )
    r = subprocess.run(["python", "-c", code], capture_output=True, text=True,
                       cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
    assert r.returncode != 0
    assert "survived" not in r.stdout
    assert "no CPU fallback" in r.stderr


def test_dpp_hazard_checker(tmp_path):
    """csrc/check_dpp.py, the build's check of the GEMMs' hand-written DPP
    instructions: a VALU write of the broadcast register one instruction before
    is a hazard, the same write behind an s_nop 1 or by an LDS read is not, and
    a VALU write of EXEC needs five wait states."""
    import importlib.util
    path = os.path.join(os.path.dirname(ckq.lib_path()), "check_dpp.py")
    spec = importlib.util.spec_from_file_location("check_dpp", path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    dpp = "\tv_fmac_f32_dpp v10, v5, v7 row_newbcast:3 row_mask:0xf bank_mask:0xf\n"
    cases = {
        "valu_adjacent": ("\tv_cvt_f32_f16_e32 v5, v9\n" + dpp, 1),
        "valu_two_back": ("\tv_cvt_f32_f16_e32 v5, v9\n\tv_mov_b32_e32 v1, v2\n" + dpp, 1),
        "valu_three_back": ("\tv_cvt_f32_f16_e32 v5, v9\n\tv_mov_b32_e32 v1, v2\n\tv_mov_b32_e32 v3, v2\n" + dpp, 0),
        "valu_then_nop": ("\tv_cvt_f32_f16_e32 v5, v9\n\ts_nop 1\n" + dpp, 0),
        "lds_read": ("\tds_read_b32 v5, v9\n\ts_waitcnt lgkmcnt(0)\n" + dpp, 0),
        "wide_write": ("\tv_pk_mul_lo_u16 v[4:5], v1, v2\n" + dpp, 1),
        "other_register": ("\tv_mov_b32_e32 v6, v9\n" + dpp, 0),
        "valu_exec": ("\tv_cmpx_lt_i32_e32 v1, v2\n\tv_mov_b32_e32 v1, v2\n\tv_mov_b32_e32 v3, v2\n" + dpp, 1),
        "salu_exec": ("\ts_or_b64 exec, exec, s[6:7]\n" + dpp, 0),
    }
    for name, (text, want) in cases.items():
        f = tmp_path / (name + ".s")
        f.write_text(text)
        count, bad = mod.check(str(f))
        assert count == 1 and bad == want, (name, count, bad)
