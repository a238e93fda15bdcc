// A HIP runtime that runs nothing, preloaded in front of the real one: device memory is host memory, copies copy, launches are written down (thread, kernel, grid). What the library's host code
// asks for, and in what order, can then be checked without a device.
#include <hip/hip_runtime.h>
#include <cxxabi.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <unistd.h>
#include <map>
#include <mutex>
#include <string>
#include <vector>

struct Launch { int thread; const void * kernel; dim3 grid, block; };
static std::mutex mu;
static std::vector<Launch> seen;
static std::map<const void *, std::string> & names() { static std::map<const void *, std::string> m; return m; }
static std::map<void *, size_t> & blocks() { static std::map<void *, size_t> m; return m; }
static size_t refuse = 0, held = 0;
static useconds_t pause_us = 0;
static hipError_t last = hipSuccess;
static thread_local int me = 0;
static thread_local struct { dim3 grid, block; size_t lds; hipStream_t st; } cfg;

static hipError_t take(void ** p, size_t n, bool device) {
    std::lock_guard<std::mutex> lk(mu);
    *p = nullptr;
    if (device && n == refuse) return last = hipErrorOutOfMemory;
    if (posix_memalign(p, 4096, n ? n : 1)) return last = hipErrorOutOfMemory;
    memset(*p, 0, n);
    if (device) { blocks()[*p] = n; held += n; }
    return hipSuccess;
}

#pragma GCC visibility push(default)
extern "C" {
// ---- what the tests ask
void shim_thread(int id) { me = id; }
void shim_pause(int us) { pause_us = (useconds_t) us; }
void shim_refuse(size_t bytes) { refuse = bytes; }                  // device allocations of exactly this size fail
size_t shim_held() { return held; }
int shim_last() { return (int) last; }
void shim_forget() { std::lock_guard<std::mutex> lk(mu); seen.clear(); }
long shim_launches() { std::lock_guard<std::mutex> lk(mu); return (long) seen.size(); }
// launch i: thread, grid (x, y, z), the kernel's name with its template arguments
void shim_launch(long i, int * out4, char * name, long n) {
    std::lock_guard<std::mutex> lk(mu);
    const Launch & l = seen[(size_t) i];
    out4[0] = l.thread; out4[1] = (int) l.grid.x; out4[2] = (int) l.grid.y; out4[3] = (int) l.grid.z;
    const auto at = names().find(l.kernel);
    int rc = 0;
    char * d = at == names().end() ? nullptr : abi::__cxa_demangle(at->second.c_str(), nullptr, nullptr, &rc);
    snprintf(name, (size_t) n, "%s", d ? d : at == names().end() ? "?" : at->second.c_str());
    free(d);
}

// ---- registration and launches
void ** __hipRegisterFatBinary(const void *) { static void * h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void * host, char *, const char * device, unsigned, void *, void *, void *, void *, int *) { names()[host] = device; }
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t st) { cfg = {grid, block, lds, st}; return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 * grid, dim3 * block, size_t * lds, hipStream_t * st) { *grid = cfg.grid; *block = cfg.block; *lds = cfg.lds; *st = cfg.st; return hipSuccess; }
hipError_t hipLaunchKernel(const void * f, dim3 grid, dim3 block, void **, size_t, hipStream_t) {
    { std::lock_guard<std::mutex> lk(mu); seen.push_back({me, f, grid, block}); }
    if (pause_us) usleep(pause_us);                                 // (another thread's turn)
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }

// ---- memory
hipError_t hipMalloc(void ** p, size_t n) { return take(p, n, true); }
hipError_t hipHostMalloc(void ** p, size_t n, unsigned) { return take(p, n, false); }
hipError_t hipHostFree(void * p) { free(p); return hipSuccess; }
hipError_t hipFree(void * p) {
    std::lock_guard<std::mutex> lk(mu);
    const auto at = blocks().find(p);
    if (at != blocks().end()) { held -= at->second; blocks().erase(at); }
    free(p);
    return hipSuccess;
}
hipError_t hipMemGetInfo(size_t * f, size_t * t) { *f = *t = (size_t) 64 << 30; return hipSuccess; }
hipError_t hipMemcpy(void * d, const void * s, size_t n, hipMemcpyKind) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemcpyAsync(void * d, const void * s, size_t n, hipMemcpyKind, hipStream_t) { memcpy(d, s, n); return hipSuccess; }
hipError_t hipMemset(void * d, int v, size_t n) { memset(d, v, n); return hipSuccess; }
hipError_t hipMemsetAsync(void * d, int v, size_t n, hipStream_t) { memset(d, v, n); return hipSuccess; }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t * a, const void *) { memset(a, 0, sizeof(*a)); return hipSuccess; }

// ---- device, streams, events
hipError_t hipGetDevice(int * d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDeviceCount(int * n) { *n = 1; return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 * p, int) { memset(p, 0, sizeof(*p)); p->multiProcessorCount = 256; return hipSuccess; }
const char * hipGetErrorString(hipError_t) { return "shim"; }
hipError_t hipGetLastError() { const hipError_t e = last; last = hipSuccess; return e; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t * s, unsigned) { *s = (hipStream_t) malloc(8); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free((void *) s); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamWaitEvent(hipStream_t, hipEvent_t, unsigned) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t * e, unsigned) { *e = (hipEvent_t) malloc(8); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free((void *) e); return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
}
