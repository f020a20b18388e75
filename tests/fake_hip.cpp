// The HIP runtime functions that the engine library calls, without a GPU: memory is host memory with a
// capacity, copies are memcpy, kernels do nothing. Every call is written to a log, and a test sets what
// a GPU would decide: which streams are under capture, which events are done, how much memory there is.
// Loaded with RTLD_GLOBAL before the engine, so that the engine's references resolve to it.
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>

namespace {
std::recursive_mutex mu;
std::map<void *, size_t> live;
std::map<const void *, std::string> kernels;
std::map<const void *, size_t> vars;
std::set<void *> captured;   // streams under capture
std::set<void *> exclusive;  // ... of which these forbid hipMalloc and hipFree meanwhile (the global mode)
uint64_t capacity = 288ull << 30, used = 0;
bool events_done = true;
uintptr_t next_handle = 0x1000;
hipError_t last = hipSuccess;
std::string text, out;
thread_local hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;

void log(const char *fmt, ...) {
    char b[1024];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(b, sizeof b, fmt, ap);
    va_end(ap);
    text += b;
    text += '\n';
}
hipError_t ret(hipError_t e) {
    if (e != hipSuccess) last = e;
    return e;
}
hipError_t alloc(void **p, size_t n) {
    if (used + n > capacity) return hipErrorOutOfMemory;
    *p = aligned_alloc(4096, (n + 4095) / 4096 * 4096);
    if (!*p) return hipErrorOutOfMemory;
    live[*p] = n;
    used += n;
    return hipSuccess;
}
void dealloc(void *p) {
    auto it = live.find(p);
    if (it == live.end()) {
        fprintf(stderr, "fake_hip: free of unknown address %p\n", p);
        abort();
    }
    used -= it->second;
    live.erase(it);
    free(p);
}
}  // namespace

#define F extern "C" __attribute__((visibility("default")))
#define LOCK std::lock_guard<std::recursive_mutex> lk(mu)

// ---- the test's side
F void fake_capacity(uint64_t n) { capacity = n; }
F uint64_t fake_used() { return used; }
// on: 0 ends the capture, 1 begins one in the relaxed mode, 2 in the global mode
F void fake_capture(void *s, int on) {
    LOCK;
    captured.erase(s);
    exclusive.erase(s);
    if (on) captured.insert(s);
    if (on == 2) exclusive.insert(s);
}
F void fake_events_done(int on) { events_done = on; }
F const char *fake_log() {  // and clears it
    LOCK;
    out.swap(text);
    text.clear();
    return out.c_str();
}

F const char *fake_kernels() {  // the names of the kernels in the library
    LOCK;
    static std::string names;
    names.clear();
    for (auto &k : kernels) names += k.second + '\n';
    return names.c_str();
}

// ---- the runtime
F hipError_t hipMalloc(void **p, size_t n) {
    LOCK;
    const hipError_t e = !exclusive.empty() && mode != hipStreamCaptureModeRelaxed ? hipErrorStreamCaptureUnsupported : alloc(p, n);
    log("malloc %zu %s", n, e == hipSuccess ? "ok" : "failed");
    return ret(e);
}
F hipError_t hipFree(void *p) {
    LOCK;
    if (!p) return hipSuccess;
    if (!exclusive.empty() && mode != hipStreamCaptureModeRelaxed) return ret(hipErrorStreamCaptureUnsupported);
    log("free %zu", live.count(p) ? live[p] : 0);
    dealloc(p);
    return hipSuccess;
}
F hipError_t hipMallocAsync(void **p, size_t n, hipStream_t s) {
    LOCK;
    const hipError_t e = alloc(p, n);
    log("malloc_async %zu %s%s", n, e == hipSuccess ? "ok" : "failed", captured.count(s) ? " captured" : "");
    return ret(e);
}
F hipError_t hipFreeAsync(void *p, hipStream_t s) {
    LOCK;
    log("free_async%s", captured.count(s) ? " captured" : "");
    dealloc(p);
    return hipSuccess;
}
F hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    LOCK;
    memcpy(d, s, n);
    return hipSuccess;
}
F hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
F hipError_t hipSetDevice(int) { return hipSuccess; }
F hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
    memset(p, 0, sizeof *p);
    strcpy(p->name, "no GPU");
    strcpy(p->gcnArchName, "gfx950:sramecc+:xnack-");
    p->multiProcessorCount = 256;
    p->totalGlobalMem = capacity;
    return hipSuccess;
}
F hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
F hipError_t hipDeviceSynchronize() { LOCK; log("device_synchronize"); return hipSuccess; }
F hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
F const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : e == hipErrorInvalidValue ? "invalid argument" : "error"; }
F hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
F hipError_t hipGetSymbolAddress(void **p, const void *sym) {
    LOCK;
    static void *mem = aligned_alloc(4096, vars[sym]);
    *p = mem;
    return hipSuccess;
}
F hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { LOCK; *s = (hipStream_t)(next_handle += 16); return hipSuccess; }
F hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
F hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus *st) {
    LOCK;
    *st = captured.count(s) ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
F hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode *m) { std::swap(*m, mode); return hipSuccess; }
F hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
F hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t *g) { LOCK; *g = (hipGraph_t)(next_handle += 16); return hipSuccess; }
F hipError_t hipGraphInstantiate(hipGraphExec_t *x, hipGraph_t, hipGraphNode_t *, char *, size_t) { LOCK; *x = (hipGraphExec_t)(next_handle += 16); return hipSuccess; }
F hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
F hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
F hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
F hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { LOCK; *e = (hipEvent_t)(next_handle += 16); return hipSuccess; }
F hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
F hipError_t hipEventQuery(hipEvent_t) { return events_done ? hipSuccess : hipErrorNotReady; }
F hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { LOCK; log("record %p on %p", (void *)e, (void *)s); return hipSuccess; }
F hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { LOCK; log("wait %p on %p", (void *)e, (void *)s); return hipSuccess; }
F hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *f, int, size_t) {
    LOCK;
    log("occupancy %s", kernels[f].c_str());
    *n = 2;
    return hipSuccess;
}
F hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t s) {
    LOCK;
    log("launch %s grid %u %u block %u on %p", kernels[f].c_str(), g.x, g.y, b.x, (void *)s);
    return hipSuccess;
}
F hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **, size_t, hipStream_t s, hipEvent_t, hipEvent_t stop, int) {
    LOCK;
    log("launch %s grid %u %u block %u on %p done %p", kernels[f].c_str(), g.x, g.y, b.x, (void *)s, (void *)stop);
    return hipSuccess;
}

namespace {
struct Config { dim3 g, b; size_t n; hipStream_t s; };
thread_local Config pushed;
}
F hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t n, hipStream_t s) { pushed = {g, b, n, s}; return hipSuccess; }
F hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *n, hipStream_t *s) {
    *g = pushed.g;
    *b = pushed.b;
    *n = pushed.n;
    *s = pushed.s;
    return hipSuccess;
}
F void **__hipRegisterFatBinary(const void *) { static void *p; return &p; }
F void __hipUnregisterFatBinary(void **) {}
F void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *, void *, int *) {
    LOCK;
    kernels[host] = name;
}
F void __hipRegisterVar(void **, void *host, char *, const char *, int, size_t n, int, int) { LOCK; vars[host] = n; }
