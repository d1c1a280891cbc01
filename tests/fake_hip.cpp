// A stand-in for the HIP runtime, for tests of the host code of librender_hip on the CPU.
//
// It carries out no kernel: "device" memory is ordinary memory, copies and fills take place at once, and
// every call is written down, one line each, in the order it was made.  A chosen call can be made to fail.
// Loaded with its symbols global before librender_hip.so, whose HIP calls then end here.
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>

namespace {

std::recursive_mutex lock;
std::string lines;
std::map<const void*, std::string> kernels;             // host stub -> mangled name
std::map<uintptr_t, std::pair<size_t, int>> blocks;     // address -> bytes, type of memory
std::string fail_what;                                  // calls whose line contains this ...
int fail_nth = 0;                                       // ... the n-th of them fails (1: the next)
hipError_t last = hipSuccess;
uintptr_t next_handle = 0x1000;
bool capturing = false;

// Writes the call down; what it returns.
hipError_t call(const char* fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    std::vsnprintf(buf, sizeof(buf), fmt, ap);
    va_end(ap);
    std::lock_guard<std::recursive_mutex> lk(lock);
    const bool fails = fail_nth > 0 && std::strstr(buf, fail_what.c_str()) && --fail_nth == 0;
    lines += buf;
    lines += fails ? " FAILED\n" : "\n";
    if (fails) last = hipErrorLaunchFailure;
    return fails ? hipErrorLaunchFailure : hipSuccess;
}

hipError_t get(void** p, size_t n, int type) {
    std::lock_guard<std::recursive_mutex> lk(lock);
    *p = std::aligned_alloc(4096, (n + 4095) & ~(size_t)4095);
    if (!*p) return hipErrorOutOfMemory;
    if (n < ((size_t)64 << 20)) std::memset(*p, 0, n);
    blocks[(uintptr_t)*p] = {n ? n : 1, type};
    return hipSuccess;
}

hipError_t give_back(void* p) {
    std::lock_guard<std::recursive_mutex> lk(lock);
    blocks.erase((uintptr_t)p);
    std::free(p);
    return hipSuccess;
}

template <typename T>
hipError_t handle(T* h) {
    std::lock_guard<std::recursive_mutex> lk(lock);
    *h = reinterpret_cast<T>(next_handle += 16);
    return hipSuccess;
}

struct {
    dim3 grid, block;
    size_t lds;
    hipStream_t s;
} config;

}  // namespace

extern "C" {

// ---- for the test -------------------------------------------------------------------------
const char* fake_lines() { return lines.c_str(); }
void fake_clear() { lines.clear(); }
void fake_fail(const char* what, int nth) {
    fail_what = what;
    fail_nth = nth;
}

// ---- registration and launches ------------------------------------------------------------
void** __hipRegisterFatBinary(const void*) {
    static void* module;
    return &module;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* host, char*, const char* name, unsigned, void*, void*, dim3*, dim3*, int*) {
    kernels[host] = name;
}
void __hipRegisterVar(void**, void*, char*, char*, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t lds, hipStream_t s) {
    config = {grid, block, lds, s};
    return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* grid, dim3* block, size_t* lds, hipStream_t* s) {
    *grid = config.grid;
    *block = config.block;
    *lds = config.lds;
    *s = config.s;
    return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3 b, void**, size_t, hipStream_t s) {
    return call("%s %s grid %u block %u stream %p", capturing ? "capture" : "launch", kernels[f].c_str(), g.x * g.y * g.z,
                b.x * b.y * b.z, (void*)s);
}

// ---- memory -------------------------------------------------------------------------------
hipError_t hipMalloc(void** p, size_t n) {
    const hipError_t e = call("malloc %zu", n);
    return e != hipSuccess ? e : get(p, n, hipMemoryTypeDevice);
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    const hipError_t e = call("hostmalloc %zu", n);
    return e != hipSuccess ? e : get(p, n, hipMemoryTypeHost);
}
hipError_t hipFree(void* p) {
    call("free %p", p);
    return give_back(p);
}
hipError_t hipHostFree(void* p) {
    call("hostfree %p", p);
    return give_back(p);
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind k, hipStream_t st) {
    const hipError_t e = call("copy %s %p from %p bytes %zu stream %p", k == hipMemcpyHostToDevice ? "in" : "out", d, s, n, (void*)st);
    if (e == hipSuccess) std::memcpy(d, s, n);
    return e;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
    std::memset(d, v, n);
    return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::recursive_mutex> lk(lock);
    std::memset(a, 0, sizeof(*a));
    a->type = hipMemoryTypeUnregistered;
    auto it = blocks.upper_bound((uintptr_t)p);
    if (it != blocks.begin() && (--it)->first + it->second.first > (uintptr_t)p) a->type = (hipMemoryType)it->second.second;
    return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void*) {
    static void* mem = nullptr;
    if (!mem) get(&mem, (size_t)128 << 20, hipMemoryTypeDevice);
    *p = mem;
    return hipSuccess;
}

// ---- streams, events, graphs --------------------------------------------------------------
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return handle(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t s) { return call("sync stream %p", (void*)s); }
hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) { return call("wait event %p stream %p", (void*)e, (void*)s); }
hipError_t hipEventCreate(hipEvent_t* e) { return handle(e); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return handle(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return call("record event %p stream %p", (void*)e, (void*)s); }
hipError_t hipEventSynchronize(hipEvent_t e) { return call("sync event %p", (void*)e); }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
    *ms = 1.0f;
    return hipSuccess;
}
hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
    capturing = true;
    return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
    capturing = false;
    return handle(g);
}
hipError_t hipGraphInstantiate(hipGraphExec_t* x, hipGraph_t, hipGraphNode_t*, char*, size_t) { return handle(x); }
hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
hipError_t hipGraphLaunch(hipGraphExec_t x, hipStream_t s) { return call("graph %p stream %p", (void*)x, (void*)s); }

// ---- device -------------------------------------------------------------------------------
hipError_t hipGetDeviceCount(int* n) {
    *n = 1;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
    *v = 256;
    return hipSuccess;
}
hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    std::memset(p, 0, sizeof(*p));
    p->multiProcessorCount = 256;
    return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int v) { return call("attribute %s %d", kernels[f].c_str(), v); }
hipError_t hipGetLastError(void) {
    const hipError_t e = last;
    last = hipSuccess;
    return e;
}
const char* hipGetErrorString(hipError_t) { return "a failure asked for by the test"; }

}  // extern "C"
