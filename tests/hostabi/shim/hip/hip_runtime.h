// Host stand-in for the HIP runtime, for the CPU build of the renderer's host
// code (pt_renderer.cpp): "device" memory is host memory with a limit, a high
// water mark and a switch that refuses pinned memory; streams and events are
// names, everything queued on them runs at once.
#pragma once
#include "../../../hostpath/shim/hip/hip_runtime.h"

#include <cstdlib>
#include <mutex>

struct uchar4 { unsigned char x, y, z, w; };
enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2, hipErrorNotReady = 600 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipStreamNonBlocking = 1, hipHostMallocDefault = 0 };
enum hipStreamCaptureMode { hipStreamCaptureModeThreadLocal };
typedef struct ihipEvent_t* hipEvent_t;
typedef struct ihipGraph_t* hipGraph_t;
typedef struct ihipGraphExec_t* hipGraphExec_t;
struct hipDeviceProp_t { int multiProcessorCount; size_t sharedMemPerBlock, totalGlobalMem; };

namespace fake {
constexpr size_t MARK = 0x9e3779b97f4a7c15;
struct State {
    std::mutex m;
    size_t used = 0, peak = 0, limit = SIZE_MAX, pinned = 0;
    bool refuse_pinned = false;
    int streams = 0;
};
inline State& state() {
    static State s;
    return s;
}
}  // namespace fake

inline const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int) {
    *p = hipDeviceProp_t{256, 65536, size_t{288} << 30};
    return hipSuccess;
}
// A header of one cache line before each allocation: its size and a mark.
inline hipError_t hipMalloc(void** p, size_t n) {
    fake::State& s = fake::state();
    std::lock_guard<std::mutex> g(s.m);
    *p = nullptr;
    if (n > s.limit || s.used > s.limit - n) return hipErrorOutOfMemory;
    size_t* at = static_cast<size_t*>(std::malloc(n + 64));  // untouched pages cost nothing
    if (!at) return hipErrorOutOfMemory;
    at[0] = n;
    at[1] = fake::MARK;
    *p = reinterpret_cast<char*>(at) + 64;
    s.used += n;
    if (s.used > s.peak) s.peak = s.used;
    return hipSuccess;
}
inline hipError_t hipFree(void* p) {
    fake::State& s = fake::state();
    std::lock_guard<std::mutex> g(s.m);
    size_t* at = reinterpret_cast<size_t*>(static_cast<char*>(p) - 64);
    if (at[1] != fake::MARK) std::abort();  // not ours, or freed twice
    at[1] = 0;
    s.used -= at[0];
    std::free(at);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    fake::State& s = fake::state();
    std::lock_guard<std::mutex> g(s.m);
    size_t* at = s.refuse_pinned ? nullptr : static_cast<size_t*>(std::malloc(n + 64));
    *p = at ? reinterpret_cast<char*>(at) + 64 : nullptr;
    if (!at) return hipErrorOutOfMemory;
    at[0] = n;
    s.pinned += n;
    return hipSuccess;
}
inline hipError_t hipHostFree(void* p) {
    fake::State& s = fake::state();
    std::lock_guard<std::mutex> g(s.m);
    size_t* at = reinterpret_cast<size_t*>(static_cast<char*>(p) - 64);
    s.pinned -= at[0];
    std::free(at);
    return hipSuccess;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind) { std::memcpy(d, s, n); return hipSuccess; }
inline hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
    std::memcpy(d, s, n);
    return hipSuccess;
}
inline hipError_t hipMemcpy2DAsync(void* d, size_t dp, const void* s, size_t sp, size_t w, size_t h, hipMemcpyKind,
                                   hipStream_t) {
    for (size_t i = 0; i < h; ++i) std::memcpy(static_cast<char*>(d) + i * dp, static_cast<const char*>(s) + i * sp, w);
    return hipSuccess;
}
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) {
    std::lock_guard<std::mutex> g(fake::state().m);
    *s = reinterpret_cast<hipStream_t>(static_cast<intptr_t>(++fake::state().streams));
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 0.f; return hipSuccess; }
inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { return hipSuccess; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = nullptr; return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, void*, char*, size_t) { *e = nullptr; return hipSuccess; }
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
