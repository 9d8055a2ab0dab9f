// A HIP runtime of host memory for tests of what the library asks of the runtime: allocations, launches,
// events and streams are logged in order, kernels do not run.  Loaded with RTLD_GLOBAL before the library,
// whose HIP calls it then answers.
#ifndef __HIP_PLATFORM_AMD__
#define __HIP_PLATFORM_AMD__
#endif
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::vector<std::string> g_log;
std::map<void const*, std::string> g_names;
std::map<void*, size_t> g_live;
size_t g_total = 0, g_limit = size_t(1) << 40;
hipStream_t g_capturing = nullptr;
hipError_t g_last = hipSuccess;
double g_clock = 1e6, g_step = 1.0;
struct Call {
    dim3 grid, block;
    size_t shared;
    hipStream_t stream;
};
std::vector<Call> g_calls;

template <class... A> void log(char const* f, A... a) {
    char b[512];
    std::snprintf(b, sizeof(b), f, a...);
    g_log.push_back(b);
}
hipError_t fail(hipError_t e) { return g_last = e; }
} // namespace

extern "C" {
// controls
void fake_clear() { g_log.clear(); }
void fake_room(size_t bytes) { g_limit = g_total + bytes; } // device memory left
void fake_capture(void* s) { g_capturing = hipStream_t(s); } // the stream under capture
void fake_step(double ms) { g_step = ms; } // every timed interval is this much longer than the one before
size_t fake_log(char* out, size_t n) {
    std::string s;
    for (auto const& l : g_log) s += l + "\n";
    if (s.size() < n) std::memcpy(out, s.c_str(), s.size() + 1);
    return s.size() + 1;
}

hipError_t hipMalloc(void** p, size_t n) {
    if (g_capturing) return fail(hipErrorStreamCaptureUnsupported);
    if (g_total + n > g_limit) {
        log("nomem %zu", n);
        return fail(hipErrorOutOfMemory);
    }
    *p = std::calloc(n, 1);
    g_total += g_live[*p] = n;
    log("malloc %p %zu", *p, n);
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    log("free %p", p);
    g_total -= g_live[p];
    g_live.erase(p);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void* d, void const* s, size_t n, hipMemcpyKind) {
    if (g_capturing) return fail(hipErrorStreamCaptureUnsupported);
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, void const* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return s == g_capturing && s ? fail(hipErrorStreamCaptureUnsupported) : hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t s, hipStreamCaptureStatus* st) {
    *st = s && s == g_capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    log("wait %p %p", (void*)s, (void*)e);
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t* e) {
    *e = hipEvent_t(std::malloc(1));
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t e) {
    std::free((void*)e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    log("record %p %p", (void*)s, (void*)e);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = float(g_clock += g_step);
    log("elapsed %.0f", g_clock);
    return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
    *d = 0;
    return hipSuccess;
}
hipError_t hipGetLastError() {
    const hipError_t e = g_last;
    g_last = hipSuccess;
    return e;
}
char const* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, void const*, int, size_t) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, void const* s) {
    *p = const_cast<void*>(s);
    return hipSuccess;
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t s) {
    g_calls.push_back({g, b, sh, s});
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* sh, hipStream_t* s) {
    const Call c = g_calls.back();
    g_calls.pop_back();
    *g = c.grid;
    *b = c.block;
    *sh = c.shared;
    *s = c.stream;
    return hipSuccess;
}
void __hipRegisterFunction(void**, void const* host, char*, char const* name, unsigned, void*, void*, void*, void*, int*) {
    g_names[host] = name;
}
void** __hipRegisterFatBinary(void const*) {
    static void* handle;
    return &handle;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t hipLaunchKernel(void const* f, dim3 g, dim3 b, void** args, size_t, hipStream_t s) {
    std::string const& n = g_names[f];
    // the buffer between the two kernels (facet slots, traces) is the third argument of all four
    const bool two = n.find("poisson_trace") != n.npos || n.find("poisson_element") != n.npos ||
                     n.find("elasticity_facet_kernel") != n.npos || n.find("elasticity_element_kernel") != n.npos;
    log("launch %s grid %ux%u block %u stream %p between %p", n.c_str(), g.x, g.y, b.x, (void*)s,
        two ? *static_cast<void**>(args[2]) : nullptr);
    return hipSuccess;
}
}
