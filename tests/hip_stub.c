/* A HIP runtime and kernel launches that do nothing, for tests of the host layer (csrc/ckq_host.c) without a GPU: the test says what
 * kind of memory an address is, and reads back how a call waited. */
#include <stdint.h>
#include <stdlib.h>
#include <string.h>

#include <hip/hip_runtime_api.h>

static struct { const uint8_t *p; size_t bytes; int type, device; unsigned flags; } g_mem[16];
static int g_mems;
int stub_words, stub_syncs;             /* completion words written, stream synchronisations */

void stub_memory(const void *p, size_t bytes, int type, int device, unsigned flags)
{
    g_mem[g_mems].p = p;
    g_mem[g_mems].bytes = bytes;
    g_mem[g_mems].type = type;
    g_mem[g_mems].device = device;
    g_mem[g_mems++].flags = flags;
}
void stub_reset(void) { g_mems = stub_words = stub_syncs = 0; }

hipError_t hipPointerGetAttributes(hipPointerAttribute_t *at, const void *p)
{
    memset(at, 0, sizeof *at);
    for (int i = 0; i < g_mems; ++i)
        if ((uintptr_t)p - (uintptr_t)g_mem[i].p < g_mem[i].bytes) {
            at->type = (enum hipMemoryType)g_mem[i].type;
            at->device = g_mem[i].device;
            at->isManaged = at->type == hipMemoryTypeManaged;
            at->allocationFlags = g_mem[i].flags;
            return hipSuccess;
        }
    return hipErrorInvalidValue;
}
hipError_t hipStreamWriteValue32(hipStream_t s, void *p, uint32_t v, unsigned flags)
{
    (void)s; (void)flags;
    ++stub_words;
    *(volatile uint32_t *)p = v;
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { (void)s; ++stub_syncs; return hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { *n = 2; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = 1; return hipSuccess; }
hipError_t hipGetDeviceProperties(hipDeviceProp_t *p, int d)
{
    (void)d;
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned flags) { (void)flags; *s = (hipStream_t)(uintptr_t)8; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t n) { *p = malloc(n); return hipSuccess; }
hipError_t hipExtMallocWithFlags(void **p, size_t n, unsigned flags) { (void)p; (void)n; (void)flags; return hipErrorOutOfMemory; }
hipError_t hipHostMalloc(void **p, size_t n, unsigned flags) { (void)flags; *p = calloc(1, n); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned flags) { (void)flags; *d = h; return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
const char *hipGetErrorString(hipError_t e) { (void)e; return "stub"; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t st) { (void)d; (void)s; (void)n; (void)k; (void)st; return hipSuccess; }
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k, hipStream_t st)
{
    (void)d; (void)dp; (void)s; (void)sp; (void)w; (void)h; (void)k; (void)st;
    return hipSuccess;
}

#define LAUNCH(name) int name() { return 0; }
LAUNCH(ckq_launch_copy) LAUNCH(ckq_launch_dequant_rows) LAUNCH(ckq_launch_gemm_block_sums) LAUNCH(ckq_launch_gemm_group) LAUNCH(ckq_launch_gemv)
LAUNCH(ckq_launch_gemv_group) LAUNCH(ckq_launch_gemv_noalloc) LAUNCH(ckq_launch_gemv_pro) LAUNCH(ckq_launch_noalloc_setup) LAUNCH(ckq_launch_quantize_gemv_q8_0)
LAUNCH(ckq_launch_quantize_q8_0) LAUNCH(ckq_launch_quantize_q8_k) LAUNCH(ckq_launch_read) LAUNCH(ckq_launch_read_tuned) LAUNCH(ckq_launch_release_stream)
LAUNCH(ckq_launch_rmsnorm_q8_k_fused) LAUNCH(ckq_launch_set_gemm_policy) LAUNCH(ckq_launch_set_q4k_tile) LAUNCH(ckq_launch_set_q5k_variant)
LAUNCH(ckq_launch_set_q6k_variant) LAUNCH(ckq_launch_set_rows16) LAUNCH(ckq_launch_swiglu_q8_k)
