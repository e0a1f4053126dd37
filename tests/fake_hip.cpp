// A HIP runtime without a GPU, for tests of the library's host code: loaded before
// libcpwgpu.so with global symbols, it takes the place of the functions that the library
// calls.  Device memory is host memory, copies are made at once, kernels are not run
// but cost time on a clock that the events read (fake_cost).  Streams and events belong
// to the device that was current when they were made; an event that is recorded on a
// stream of another device is an error, as in the real runtime.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

namespace {
struct Stream { int dev; };
struct Event { int dev; double us; };
struct Cost { std::string part; double first, later; long after; };
struct Config { dim3 g, b; size_t s; hipStream_t q; };
std::recursive_mutex mu;
int ndev = 1;
thread_local int cur = 0;
thread_local std::vector<Config> configs;
double clock_us = 0.0;
long since_sync = 0, fail_host_malloc = 0, live = 0;
std::map<const void *, std::string> names;
std::map<const void *, size_t> vars;
std::map<const void *, void *> var_mem;
std::vector<Cost> costs;
std::string text;
Stream null_stream{0};
Stream *stream(hipStream_t s) { return s ? reinterpret_cast<Stream *>(s) : &null_stream; }
void log(const char *what) { text += what; text += '\n'; }
void synced(const char *what) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    since_sync = 0;
    log(what);
}
hipError_t launch(const void *f) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    since_sync++;
    const auto it = names.find(f);
    const std::string n = it == names.end() ? "?" : it->second;
    double us = 1.0;
    for (const Cost &c : costs)
        if (n.find(c.part) != std::string::npos) us = since_sync > c.after ? c.later : c.first;
    clock_us += us;
    log(("launch " + n).c_str());
    return hipSuccess;
}
}  // namespace

extern "C" {
// ---- the tests' side ---------------------------------------------------------
void fake_devices(int n) { ndev = n; }
void fake_fail_host_malloc(long n) { fail_host_malloc = n; }  // the next n allocations
// kernels whose name holds part: first us, and later us once `after` launches went out since the last wait
void fake_cost(const char *part, double first, double later, long after) { costs.push_back({part, first, later, after}); }
void fake_clear() { std::lock_guard<std::recursive_mutex> lk(mu); text.clear(); }
const char *fake_log() { return text.c_str(); }
long fake_live() { return live; }  // allocations, device and pinned, not given back

// ---- the runtime ---------------------------------------------------------------
hipError_t hipGetDeviceCount(int *n) { *n = ndev; return hipSuccess; }
hipError_t hipGetDevice(int *d) { *d = cur; return hipSuccess; }
hipError_t hipSetDevice(int d) { if (d < 0 || d >= ndev) return hipErrorInvalidDevice; cur = d; return hipSuccess; }
hipError_t hipDeviceSynchronize() { synced("device sync"); return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "fake error"; }
hipError_t hipMalloc(void **p, size_t n) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    *p = calloc(1, n ? n : 1);
    live += *p != nullptr;
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipFree(void *p) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    live -= p != nullptr;
    free(p);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (fail_host_malloc > 0) { fail_host_malloc--; return hipErrorOutOfMemory; }
    *p = malloc(n);
    live++;
    return hipSuccess;
}
hipError_t hipHostFree(void *p) { return hipFree(p); }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = reinterpret_cast<hipStream_t>(new Stream{cur}); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { synced("stream sync"); return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = reinterpret_cast<hipEvent_t>(new Event{cur, 0.0}); return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
hipError_t hipEventDestroy(hipEvent_t e) { delete reinterpret_cast<Event *>(e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    Event *v = reinterpret_cast<Event *>(e);
    if (s && stream(s)->dev != v->dev) return hipErrorInvalidHandle;
    v->us = clock_us;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { synced("event sync"); return hipSuccess; }
hipError_t hipEventElapsedTime(float *ms, hipEvent_t a, hipEvent_t b) {
    *ms = (float)((reinterpret_cast<Event *>(b)->us - reinterpret_cast<Event *>(a)->us) * 1e-3);
    return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind k, hipStream_t) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    log(k == hipMemcpyHostToDevice ? "copy in" : k == hipMemcpyDeviceToHost ? "copy out" : "copy");
    memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpy2DAsync(void *d, size_t ld, const void *s, size_t ls, size_t w, size_t h, hipMemcpyKind k, hipStream_t) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    log(k == hipMemcpyHostToDevice ? "copy in" : k == hipMemcpyDeviceToHost ? "copy out" : "copy");
    for (size_t i = 0; i < h; i++) memcpy((char *)d + i * ld, (const char *)s + i * ls, w);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) { return launch(f); }
hipError_t hipExtLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t, hipEvent_t, hipEvent_t, int) { return launch(f); }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t s, hipStream_t q) { configs.push_back({g, b, s, q}); return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *s, hipStream_t *q) {
    const Config c = configs.back();
    configs.pop_back();
    *g = c.g; *b = c.b; *s = c.s; *q = c.q;
    return hipSuccess;
}
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *f, char *, const char *name, unsigned, void *, void *, dim3 *, dim3 *, int *) {
    names[f] = name;
}
void __hipRegisterVar(void **, void *v, char *, char *, int, size_t n, int, int) { vars[v] = n; }
hipError_t hipGetSymbolAddress(void **p, const void *v) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    if (!var_mem.count(v)) var_mem[v] = calloc(1, vars[v]);
    *p = var_mem[v];
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { log("capture"); return hipSuccess; }
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { log("capture end"); *g = reinterpret_cast<hipGraph_t>(&null_stream); return hipSuccess; }
hipError_t hipGraphInstantiate(hipGraphExec_t *e, hipGraph_t, hipGraphNode_t *, char *, size_t) { *e = reinterpret_cast<hipGraphExec_t>(&null_stream); return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { log("graph launch"); return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
}
