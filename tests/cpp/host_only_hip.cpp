// A HIP runtime without a GPU, for tests of what the host side asks of the device: device memory is host memory, kernels
// are not run, and every launch and allocation is written down. Preloaded before libfastlanes_amd.so (tests/host_hip.py).
// Streams are numbers: stream 0x100 * k + n belongs to device k; the null stream (0), hipStreamLegacy (1) and
// hipStreamPerThread (2) to the current device.
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>
#include <utility>

namespace {
struct Config {
    dim3        g, b;
    size_t      lds;
    hipStream_t s;
};
struct Var {
    std::string name;
    size_t      size;
};
std::map<const void*, std::string>                    kernels;
std::map<const void*, Var>                            vars;
std::map<std::pair<const void*, int>, void*>          symbols;  // a variable's copy on a device
std::string                                           log_;
thread_local Config                                   cfg;
thread_local int                                      current = 0;
void                                                  say(const char* what, unsigned long long a) {
    char t[64];
    std::snprintf(t, sizeof t, "%s %llu\n", what, a);
    log_ += t;
}
int device_of(hipStream_t s) { return (uintptr_t)s > 2 ? (int)((uintptr_t)s >> 8) : current; }
}  // namespace

extern "C" {
const char* host_hip_log() { return log_.c_str(); }
void        host_hip_clear() { log_.clear(); }

void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    kernels[f] = name;
}
void __hipRegisterVar(void**, void* var, char*, char* name, int, size_t size, int, int) { vars[var] = {name, size}; }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t s) { return cfg = {g, b, lds, s}, hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* s) {
    return *g = cfg.g, *b = cfg.b, *lds = cfg.lds, *s = cfg.s, hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t lds, hipStream_t s) {
    char t[96];
    std::snprintf(t, sizeof t, " %u %u %zu %d\n", g.x, b.x, lds, device_of(s));
    log_ += "launch " + kernels[f] + t;
    return hipSuccess;
}

hipError_t hipGetLastError() { return hipSuccess; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipGetDevice(int* d) { return *d = current, hipSuccess; }
hipError_t hipSetDevice(int d) { return current = d, hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t s, hipDevice_t* d) {
    if (s == hipStreamLegacy) std::abort();  // the real one takes the handle for a pointer
    return *d = device_of(s), hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
    std::memset(p, 0, sizeof *p);
    p->multiProcessorCount = 256, p->sharedMemPerBlock = 160 << 10, p->maxThreadsPerMultiProcessor = 2048;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) { return say("malloc", n), *p = std::calloc(n + 1, 1), hipSuccess; }
hipError_t hipMallocAsync(void** p, size_t n, hipStream_t s) {
    return say("malloc_async_on", device_of(s)), *p = std::calloc(n + 1, 1), hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return say("host_malloc", n), *p = std::calloc(n + 1, 1), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipFreeAsync(void* p, hipStream_t) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) { return std::memcpy(d, s, n), hipSuccess; }
hipError_t hipMemset(void* d, int v, size_t n) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { return std::memset(d, v, n), hipSuccess; }
hipError_t hipGetSymbolAddress(void** p, const void* var) {
    say("symbol_on", current);
    void*& at = symbols[{var, current}];
    if (!at) at = std::calloc(vars[var].size + 1, 1);
    return *p = at, hipSuccess;
}
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return *s = (hipStream_t)1, hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = (hipEvent_t)1, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int* n, const void*, int, size_t) { return *n = 8, hipSuccess; }
}
