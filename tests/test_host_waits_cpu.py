"""How the synchronous symbols wait for a result in the caller's own memory, with a HIP runtime that does nothing (hip_stub.c) under the
real host layer: no GPU, no kernel."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "c-kernel-engine_amd", "csrc")
ROCM = os.environ.get("ROCM", "/opt/rocm")
DEVICE, MANAGED = 2, 3                          # hipMemoryTypeDevice, hipMemoryTypeManaged
THIS_GPU, ANOTHER_GPU = 1, 0                    # the stub's current device is 1


@pytest.fixture(scope="module")
def L(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("host") / "libhost_stub.so")
    subprocess.run(["gcc", "-O1", "-fPIC", "-shared", "-std=gnu11", "-w", "-D__HIP_PLATFORM_AMD__", "-I" + os.path.join(ROCM, "include"),
                    "-I" + os.path.join(HERE, "..", "include"), "-I" + CSRC, "-Wl,-Bsymbolic", "-o", so, os.path.join(CSRC, "ckq_host.c"),
                    os.path.join(CSRC, "ckq_pure.c"), os.path.join(HERE, "hip_stub.c"), "-lpthread"], check=True)
    lib = ctypes.CDLL(so)
    lib.stub_memory.argtypes = [ctypes.c_void_p, ctypes.c_size_t, ctypes.c_int, ctypes.c_int, ctypes.c_uint]
    return lib


def calls(L, P):
    """The five kinds of call with a result of their own: name, and a function of the result's address; inputs are all at `a`."""
    i, f = ctypes.c_int, ctypes.c_float
    v = ctypes.c_void_p
    return [
        ("matmul", lambda a, y: L.gemv_q4_k_q8_k(v(y), v(a), v(a), i(4), i(256))),
        ("quantize", lambda a, y: L.quantize_row_q8_k(v(a), v(y), i(512))),
        ("dequantize", lambda a, y: L.dequant_q4_k_row(v(a), v(y), ctypes.c_size_t(512))),
        ("rmsnorm", lambda a, y: L.rmsnorm_q8_k_fused(v(a), v(a), v(y), i(2), i(256), i(256), f(1e-5))),
        ("fused mlp", lambda a, y: L.fused_mlp_swiglu_prefill_w1w2_quant(v(a), v(a), None, i(P.CK_DT["q8_0"]), v(a), None, i(P.CK_DT["q4_k"]), v(y), i(2), i(64), i(64),
                                                                         i(256), i(256), v(a))),
    ]


@pytest.mark.parametrize("what,kind,device,flags,word", [
    ("device memory", DEVICE, THIS_GPU, 0, True), ("managed", MANAGED, THIS_GPU, 0, False), ("fine-grained", DEVICE, THIS_GPU, 1, False),
    ("uncached", DEVICE, THIS_GPU, 3, False), ("another GPU's", DEVICE, ANOTHER_GPU, 0, False)])
def test_only_this_gpus_ordinary_memory_is_left_without_the_synchronisation_call(L, what, kind, device, flags, word):
    """A result that the CPU may read where it lies, or that lies behind another GPU, is returned after the stream synchronisation, which promises that they
    see it; ordinary memory of the library's own GPU after the completion word."""
    import importlib
    P = importlib.import_module("c-kernel-engine_amd").parity
    a, y = np.zeros(1 << 16, np.uint8), np.zeros(1 << 16, np.uint8)
    for name, call in calls(L, P):
        L.stub_reset()
        L.stub_memory(a.ctypes.data, a.nbytes, DEVICE, THIS_GPU, 0)
        L.stub_memory(y.ctypes.data, y.nbytes, kind, device, flags)
        call(a.ctypes.data, y.ctypes.data)
        words, syncs = (ctypes.c_int.in_dll(L, n).value for n in ("stub_words", "stub_syncs"))
        assert (words > 0, syncs > 0) == (word, not word), (name, what, words, syncs)
