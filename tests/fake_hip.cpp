// A HIP runtime without a device, for tests of the library's host side: what it
// allocates, which kernels it launches with which grids and events, and what it
// does when an allocation is refused.  Loaded with global symbols before libjev,
// whose HIP calls then land here: device memory is host memory under a limit that
// the test sets, copies are memcpy, kernels are written down and do not run.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

namespace {
std::map<const void *, std::string> g_kernels;
std::map<void *, size_t> g_blocks;
size_t g_live = 0, g_limit = ~(size_t)0;
int g_refused = 0;
std::string g_log;
hipError_t g_last = hipSuccess;
struct Call {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
} g_call;
long g_handles = 0;
template <typename T> hipError_t handle(T *out)
{
    *out = (T)(intptr_t)(++g_handles * 16);
    return hipSuccess;
}
// name|x|y|z|start event|stop event
hipError_t launch(const void *f, dim3 grid, hipEvent_t e0, hipEvent_t e1)
{
    const dim3 g = grid;
    g_log += g_kernels[f] + "|" + std::to_string(g.x) + "|" + std::to_string(g.y) + "|" + std::to_string(g.z) + "|" +
             std::to_string((intptr_t)e0) + "|" + std::to_string((intptr_t)e1) + "\n";
    return hipSuccess;
}
char g_symbol[64 << 20];
} // namespace

extern "C" {
// for the test
void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_live(void) { return g_live; }
int fake_refused(void) { return g_refused; }
const char *fake_log(void) { return g_log.c_str(); }
void fake_clear(void)
{
    g_log.clear();
    g_refused = 0;
}

void **__hipRegisterFatBinary(const void *)
{
    static void *module;
    return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *)
{
    g_kernels[host] = name;
}
void __hipRegisterVar(void **, void *, char *, const char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s)
{
    g_call = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *lds, hipStream_t *s)
{
    *grid = g_call.grid;
    *block = g_call.block;
    *lds = g_call.lds;
    *s = g_call.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t) { return launch(f, grid, nullptr, nullptr); }
hipError_t hipExtLaunchKernel(const void *f, dim3 grid, dim3, void **, size_t, hipStream_t, hipEvent_t e0, hipEvent_t e1, int)
{
    return launch(f, grid, e0, e1);
}

hipError_t hipMalloc(void **p, size_t n)
{
    *p = nullptr;
    if (n > g_limit || g_live > g_limit - n || !(*p = std::malloc(n))) {
        g_refused++;
        return g_last = hipErrorOutOfMemory;
    }
    g_blocks[*p] = n;
    g_live += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    auto it = g_blocks.find(p);
    if (it == g_blocks.end()) return p ? g_last = hipErrorInvalidValue : hipSuccess;
    g_live -= it->second;
    g_blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return (*p = std::calloc(1, n)) ? hipSuccess : hipErrorOutOfMemory; }
hipError_t hipHostFree(void *p)
{
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    *p = g_symbol;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *, size_t, const void *, size_t, size_t, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t n, hipStream_t)
{
    std::memset(p, v, n);
    return hipSuccess;
}

hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipGetLastError(void)
{
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipStreamCreate(hipStream_t *s) { return handle(s); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { return handle(g); }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { return handle(e); }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.f;
    return hipSuccess;
}
}
