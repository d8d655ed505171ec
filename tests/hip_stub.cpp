// The HIP runtime calls libch4g.so makes, on host memory and without running
// any kernel: for tests of the library's host side (what it allocates, launches
// and gives back, and what it does when an allocation fails) where there is no
// GPU.  Loaded with global visibility before the library, so that its symbols
// are found first.  Copies copy, kernels are counted by name.
#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>

namespace {

std::map<const void *, std::string> kernel_names;
std::map<std::string, long> launched;
std::map<void *, size_t> device;  // live allocations
std::set<void *> streams, events;
long mallocs = 0, fail_from = -1, fail_to = -1, streams_made = 0, captures = 0;
size_t fail_bytes = 0, live_bytes = 0, peak_bytes = 0;
hipError_t last = hipSuccess;

struct Config {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
thread_local Config pushed;

hipError_t ret(hipError_t e)
{
    if (e != hipSuccess) last = e;
    return e;
}

}  // namespace

extern "C" {

// ---- what the tests ask
long stub_launches(const char *part)
{
    long n = 0;
    for (auto &k : launched)
        if (k.first.find(part) != std::string::npos) n += k.second;
    return n;
}
size_t stub_live_bytes() { return live_bytes; }
size_t stub_peak_bytes() { return peak_bytes; }  // since stub_reset
long stub_streams_made() { return streams_made; }
long stub_captures() { return captures; }
// device allocations fail: those of at least `bytes`, from the `first` such
// one counted from now, `count` of them (0: none)
void stub_fail(size_t bytes, long first, long count)
{
    mallocs = 0;
    fail_bytes = bytes;
    fail_from = first;
    fail_to = first + count;
}
void stub_reset()
{
    launched.clear();
    streams_made = captures = 0;
    peak_bytes = live_bytes;
}

// ---- the runtime
void **__hipRegisterFatBinary(const void *) { return (void **)malloc(8); }
void __hipUnregisterFatBinary(void **m) { free(m); }
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *,
                           int *)
{
    kernel_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t t)
{
    pushed = {g, b, s, t};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *t)
{
    *g = pushed.grid;
    *b = pushed.block;
    *s = pushed.shared;
    *t = pushed.stream;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t s)
{
    if (!kernel_names.count(f)) return ret(hipErrorInvalidDeviceFunction);
    if (!g.x || !g.y || !g.z || !b.x || b.x * b.y * b.z > 1024) return ret(hipErrorInvalidConfiguration);
    if (s && !streams.count(s)) return ret(hipErrorInvalidHandle);
    launched[kernel_names[f]]++;
    return hipSuccess;
}

hipError_t hipMalloc(void **p, size_t n)
{
    if (n >= fail_bytes) {
        const long k = mallocs++;
        if (k >= fail_from && k < fail_to) return ret(hipErrorOutOfMemory);
    }
    *p = calloc(1, n ? n : 1);
    if (!*p) return ret(hipErrorOutOfMemory);
    device[*p] = n;
    live_bytes += n;
    if (live_bytes > peak_bytes) peak_bytes = live_bytes;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    auto d = device.find(p);
    if (d == device.end()) return ret(hipErrorInvalidValue);
    live_bytes -= d->second;
    device.erase(d);
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    *p = calloc(1, n);
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t *f, size_t *t)
{
    *f = *t = (size_t)1 << 34;
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t)
{
    memset(d, v, n);
    return hipSuccess;
}

hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned)
{
    *s = (hipStream_t)malloc(8);
    streams.insert(*s);
    streams_made++;
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s)
{
    if (!streams.erase(s)) return ret(hipErrorInvalidHandle);
    free(s);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return s && !streams.count(s) ? ret(hipErrorInvalidHandle) : hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = (hipEvent_t)malloc(8);
    events.insert(*e);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e)
{
    if (!events.erase(e)) return ret(hipErrorInvalidHandle);
    free(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    return !events.count(e) || (s && !streams.count(s)) ? ret(hipErrorInvalidHandle) : hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) { return events.count(e) ? hipSuccess : ret(hipErrorInvalidHandle); }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t)
{
    *ms = 0.f;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned)
{
    return !events.count(e) || !streams.count(s) ? ret(hipErrorInvalidHandle) : hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode)
{
    captures++;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g)
{
    *g = (hipGraph_t)malloc(8);
    return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g)
{
    free(g);
    return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t)
{
    *x = (hipGraphExec_t)malloc(8);
    return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t x)
{
    free(x);
    return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }

hipError_t hipGetDeviceCount(int *n)
{
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d)
{
    *d = 0;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
int hipGetStreamDeviceId(hipStream_t) { return 0; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int)
{
    *v = 64;
    return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int)
{
    memset(p, 0, sizeof *p);
    strcpy(p->gcnArchName, "gfx950");
    p->warpSize = 64;
    p->multiProcessorCount = 256;
    p->maxThreadsPerBlock = 1024;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *s)
{
    *p = (void *)s;
    return hipSuccess;
}
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError()
{
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}

}  // extern "C"
