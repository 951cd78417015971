// The library's host code over a stand-in for the HIP runtime: device memory is
// host memory, kernels do nothing, and every allocation is counted.  The checks
// at the end look at decisions that the C interface does not show.  Built for
// the host only and loaded by tests/test_host_logic.py, on machines without a
// GPU.
#include "../../w2dynamics_amd/csrc/ctqmc_engine.hip"

#include <cstdlib>

namespace {

long long g_allocs = 0;        // allocations of device memory so far
size_t g_live = 0;             // bytes of device memory held
size_t g_limit = (size_t)1 << 40;
char g_symbol[1 << 16];        // what symbols name

struct Block {
    size_t n;
    char pad[256 - sizeof(size_t)];
};

}  // namespace

extern "C" {

char __hip_fatbin[16];
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *)
{
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}

hipError_t hipMalloc(void **p, size_t n)
{
    if (n > g_limit - g_live) return hipErrorOutOfMemory;
    Block *b = static_cast<Block *>(std::calloc(1, sizeof(Block) + n));
    if (!b) return hipErrorOutOfMemory;
    b->n = n;
    ++g_allocs;
    g_live += n;
    *p = b + 1;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!p) return hipSuccess;
    Block *b = static_cast<Block *>(p) - 1;
    g_live -= b->n;
    std::free(b);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p) { return std::free(p), hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *p, unsigned) { return *d = p, hipSuccess; }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { return std::memmove(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) { return hipMemcpy(d, s, n, k); }
hipError_t hipMemcpy2D(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind)
{
    for (size_t i = 0; i < h; ++i)
        std::memmove(static_cast<char *>(d) + i * dp, static_cast<const char *>(s) + i * sp, w);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t dp, const void *s, size_t sp, size_t w, size_t h, hipMemcpyKind k, hipStream_t)
{
    return hipMemcpy2D(d, dp, s, sp, w, h, k);
}
hipError_t hipMemset(void *p, int v, size_t n) { return std::memset(p, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t) { return hipMemset(p, v, n); }
hipError_t hipMemset2DAsync(void *p, size_t pitch, int v, size_t w, size_t h, hipStream_t)
{
    for (size_t i = 0; i < h; ++i) std::memset(static_cast<char *>(p) + i * pitch, v, w);
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetSymbolAddress(void **p, const void *) { return *p = g_symbol, hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
// one compute unit of an MI355X
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t a, int)
{
    *v = a == hipDeviceAttributeMultiprocessorCount ? 1 : 160 * 1024;
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s) { return *s = nullptr, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return *g = nullptr, hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    return *e = nullptr, hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return *e = nullptr, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) { return *ms = 1.0f, hipSuccess; }

// --- what the tests look at ---------------------------------------------------
// device memory: allocations so far, bytes held
void host_memory(long long *allocs, long long *live) { *allocs = g_allocs, *live = (long long)g_live; }
// no further device memory
void host_memory_full(int on) { g_limit = on ? g_live : (size_t)1 << 40; }

// operators of the LDS lists, whether they are cut short, LDS bytes of a
// workgroup (dynamic, and with the kernels' own variables), the limit
void host_layout(const w2d_ctqmc *h, long long *v)
{
    v[0] = h->L.lcap_lds, v[1] = h->L.lcap_short, v[2] = h->L.lds_bytes;
    v[3] = h->L.lds_bytes + (long long)sizeof(w2d::WalkEnv), v[4] = h->lds_max, v[5] = h->L.cap, v[6] = h->full_lists;
}

// chain c stops for room with k pairs in every flavour
void host_halt(w2d_ctqmc *h, int c, int k)
{
    w2d::ChainHdr *x = reinterpret_cast<w2d::ChainHdr *>(h->chains + h->L.hdrs) + c;
    x->halt = w2d::HALT_CAP;
    x->nop = 2 * 2 * h->model.nbands * k;
    for (int f = 0; f < 2 * h->model.nbands; ++f) x->kf[f] = k;
}
int host_resume(w2d_ctqmc *h, int *again)
{
    std::vector<w2d::ChainHdr> hd;
    int st = read_headers(h, hd);
    if (st) return st;
    long long from;
    bool a;
    st = resume_halted(h, hd, from, a);
    *again = a;
    return st;
}
// why chain c stopped, its error
void host_chain(const w2d_ctqmc *h, int c, int *halt, int *err)
{
    const w2d::ChainHdr *x = reinterpret_cast<const w2d::ChainHdr *>(h->chains + h->L.hdrs) + c;
    *halt = x->halt, *err = x->err;
}

}  // extern "C"
