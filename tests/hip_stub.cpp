// A HIP runtime for tests of the library's host code on machines without a GPU: memory is the
// host's, kernels do nothing, and every call is recorded with its stream.  Loaded ahead of
// libcrt.so it takes the place of the symbols that the library imports from the HIP runtime.
#include <hip/hip_runtime_api.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {

std::mutex               mu;
std::string              phase = "-", text;
std::map<void *, size_t> live;
size_t                   live_bytes = 0;
long                     calls = 0, fail_at = -1, handles = 0;
hipError_t               last = hipSuccess;
uintptr_t                next_handle = 0x1000;

// Records a call; the one that stub_fail chose fails.
hipError_t call(const char *name, const void *stream = nullptr, bool can_fail = true)
{
    std::lock_guard<std::mutex> g(mu);
    char line[160];
    std::snprintf(line, sizeof line, "%s %s %p\n", phase.c_str(), name, stream);
    text += line;
    if (can_fail && calls++ == fail_at) return last = hipErrorUnknown;
    return hipSuccess;
}

hipError_t take(void **p, size_t n)
{
    std::lock_guard<std::mutex> g(mu);
    *p = std::calloc(1, n ? n : 1);
    live[*p] = n;
    live_bytes += n;
    return hipSuccess;
}

hipError_t give(void *p)
{
    std::lock_guard<std::mutex> g(mu);
    auto it = live.find(p);
    if (it == live.end()) return hipErrorInvalidValue;
    live_bytes -= it->second;
    live.erase(it);
    std::free(p);
    return hipSuccess;
}

template <class T>
hipError_t handle(T *h)
{
    std::lock_guard<std::mutex> g(mu);
    *h = reinterpret_cast<T>(next_handle += 16);
    ++handles;
    return hipSuccess;
}

hipError_t drop()
{
    std::lock_guard<std::mutex> g(mu);
    --handles;
    return hipSuccess;
}

}  // namespace

extern "C" {

void        stub_phase(const char *name) { phase = name; }
const char *stub_log() { return text.c_str(); }
void        stub_clear() { text.clear(); }
// the k-th call from now on that can fail does (-1: none)
void        stub_fail(long k)
{
    if (k >= 0) calls = 0;
    fail_at = k;
    last    = hipSuccess;
}
int         stub_reached(long k) { return calls > k; }   // whether the call chosen last was made
size_t      stub_live() { return live_bytes; }
long        stub_handles() { return handles; }   // streams, events and graphs

#define TRY(...)                                            \
    do {                                                    \
        const hipError_t e_ = call(__func__, ##__VA_ARGS__); \
        if (e_ != hipSuccess) return e_;                    \
    } while (0)

hipError_t hipMalloc(void **p, size_t n)
{
    TRY();
    return take(p, n);
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    TRY();
    return take(p, n);
}
hipError_t hipFree(void *p)
{
    (void)call(__func__, nullptr, false);
    return p ? give(p) : hipSuccess;
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    TRY();
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st)
{
    TRY(st);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t st)
{
    TRY(st);
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemsetD32Async(hipDeviceptr_t d, int v, size_t n, hipStream_t st)
{
    TRY(st);
    for (size_t i = 0; i < n; ++i) static_cast<int *>(d)[i] = v;
    return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    TRY();
    return handle(s);
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    (void)call(__func__, s, false);
    return drop();
}
hipError_t hipStreamSynchronize(hipStream_t s) { return call(__func__, s); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t, unsigned) { return call(__func__, s); }
hipError_t hipStreamBeginCapture(hipStream_t s, hipStreamCaptureMode) { return call(__func__, s); }
hipError_t hipStreamEndCapture(hipStream_t s, hipGraph_t *g)
{
    TRY(s);
    return handle(g);
}
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    TRY();
    return handle(e);
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t s) { return call(__func__, s); }
hipError_t hipGraphDestroy(hipGraph_t) { return drop(); }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return drop(); }
hipError_t hipEventCreate(hipEvent_t *e)
{
    TRY();
    return handle(e);
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    TRY();
    return handle(e);
}
hipError_t hipEventDestroy(hipEvent_t) { return drop(); }
hipError_t hipEventRecord(hipEvent_t, hipStream_t s) { return call(__func__, s); }
hipError_t hipEventSynchronize(hipEvent_t) { return call(__func__); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    std::memset(p, 0, sizeof *p);
    std::strcpy(p->name, "stub");
    std::strcpy(p->gcnArchName, "gfx950");
    p->multiProcessorCount = 256;
    return hipSuccess;
}
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return call(__func__); }
hipError_t hipGetSymbolAddress(void **p, const void *)
{
    static void *block = std::calloc(1, 64);   // no kernel runs: never read
    *p = block;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t  hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t s) { return call(__func__, s); }

static thread_local struct { dim3 g, b; size_t n; hipStream_t s; } config;
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s)
{
    config = {g, b, n, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s)
{
    *g = config.g;
    *b = config.b;
    *n = config.n;
    *s = config.s;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *)
{
    static void *h = nullptr;
    return &h;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
