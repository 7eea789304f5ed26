// A stand-in for the HIP runtime, for host code only: device memory is host
// memory, streams run every operation at once, and a test can make allocations
// fail and look at the copies that were asked for.
#pragma once

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#define __host__
#define __device__
#define __forceinline__ inline
#define __align__(n) __attribute__((aligned(n)))

struct float4 { float x, y, z, w; };
struct uint2 { uint32_t x, y; };
struct uint4 { uint32_t x, y, z, w; };

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2, hipErrorInvalidDevice = 101,
                  hipErrorInvalidSymbol = 13 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipDeviceAttribute_t { hipDeviceAttributeWallClockRate };
enum hipStreamCaptureMode { hipStreamCaptureModeThreadLocal };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
constexpr unsigned hipStreamNonBlocking = 1, hipHostMallocDefault = 0, hipEventDisableTiming = 2;
using hipStream_t = struct FakeStream*;
using hipEvent_t = struct FakeEvent*;
using hipGraph_t = struct FakeGraph*;
using hipGraphExec_t = struct FakeGraphExec*;
struct hipDeviceProp_t { int multiProcessorCount; char name[256], gcnArchName[256]; };
struct hipPointerAttribute_t { hipMemoryType type; };

namespace fake {
struct Copy { const void* dst; const void* src; size_t bytes; };
struct State {
    std::mutex mu;
    std::map<const char*, size_t> device, pinned;   // live allocations
    size_t device_bytes = 0, device_limit = ~size_t(0), device_peak = 0;
    int pinned_fail_from = 1 << 30, pinned_calls = 0;  // the pinned allocation from which on all fail
    int copy_fail_at = 1 << 30, copy_calls = 0;        // the copy that fails
    std::vector<Copy> copies;
    int num_cus = 256;
    int captures = 0, replays = 0, threads = 0;
};
inline State& state() { static State s; return s; }
inline thread_local hipError_t last_error = hipSuccess;
inline hipError_t note(hipError_t e) { if (e != hipSuccess) last_error = e; return e; }
inline hipError_t take(std::map<const char*, size_t>& where, void** p, size_t bytes)
{
    char* m = static_cast<char*>(std::calloc(std::max<size_t>(bytes, 1), 1));
    if (!m) return hipErrorOutOfMemory;
    where[m] = bytes;
    *p = m;
    return hipSuccess;
}
}  // namespace fake

template <class T> hipError_t hipMalloc(T** p, size_t bytes)
{
    auto& s = fake::state();
    std::lock_guard<std::mutex> lock(s.mu);
    if (bytes > s.device_limit || s.device_bytes > s.device_limit - bytes) return fake::note(hipErrorOutOfMemory);
    void* m = nullptr;
    const hipError_t e = fake::take(s.device, &m, bytes);
    if (e != hipSuccess) return fake::note(e);
    s.device_bytes += bytes;
    s.device_peak = std::max(s.device_peak, s.device_bytes);
    *p = static_cast<T*>(m);
    return hipSuccess;
}
inline hipError_t hipFree(void* p)
{
    auto& s = fake::state();
    std::lock_guard<std::mutex> lock(s.mu);
    auto it = s.device.find(static_cast<char*>(p));
    if (it == s.device.end()) std::abort();          // freed twice, or never allocated
    s.device_bytes -= it->second;
    s.device.erase(it);
    std::free(p);
    return hipSuccess;
}
template <class T> hipError_t hipHostMalloc(T** p, size_t bytes, unsigned)
{
    auto& s = fake::state();
    std::lock_guard<std::mutex> lock(s.mu);
    if (++s.pinned_calls >= s.pinned_fail_from) return fake::note(hipErrorOutOfMemory);
    void* m = nullptr;
    const hipError_t e = fake::take(s.pinned, &m, bytes);
    *p = static_cast<T*>(m);
    return fake::note(e);
}
inline hipError_t hipHostFree(void* p)
{
    auto& s = fake::state();
    std::lock_guard<std::mutex> lock(s.mu);
    if (!s.pinned.erase(static_cast<char*>(p))) std::abort();
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p)
{
    auto& s = fake::state();
    std::lock_guard<std::mutex> lock(s.mu);
    auto in = [&](const std::map<const char*, size_t>& m) {
        auto it = m.upper_bound(static_cast<const char*>(p));
        return it != m.begin() && static_cast<const char*>(p) < (--it)->first + it->second;
    };
    a->type = in(s.pinned) ? hipMemoryTypeHost : (in(s.device) ? hipMemoryTypeDevice : hipMemoryTypeUnregistered);
    return a->type == hipMemoryTypeUnregistered ? fake::note(hipErrorInvalidValue) : hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t)
{
    auto& s = fake::state();
    {
        std::lock_guard<std::mutex> lock(s.mu);
        if (++s.copy_calls == s.copy_fail_at) return fake::note(hipErrorInvalidValue);
        if (!dst || !src || bytes > (size_t(1) << 40)) return fake::note(hipErrorInvalidValue);
        s.copies.push_back({dst, src, bytes});
    }
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
inline hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
inline hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) { std::memset(d, v, n); return hipSuccess; }
inline hipError_t hipGetLastError() { const hipError_t e = fake::last_error; fake::last_error = hipSuccess; return e; }
inline const char* hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "invalid argument"; }
inline hipError_t hipGetDeviceCount(int* n) { *n = 1; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetDeviceProperties(hipDeviceProp_t* p, int)
{
    *p = hipDeviceProp_t{fake::state().num_cus, "fake", "fake"};
    return hipSuccess;
}
inline hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) { *v = 100000; return hipSuccess; }
inline hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { *s = nullptr; return hipSuccess; }
inline hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
inline hipError_t hipEventCreate(hipEvent_t* e) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return hipEventCreate(e); }
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
inline hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) { *ms = 1.0f; return hipSuccess; }
inline hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) { ++fake::state().captures; return hipSuccess; }
inline hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) { *g = reinterpret_cast<hipGraph_t>(1); return hipSuccess; }
inline hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t, void*, void*, size_t)
{
    *e = reinterpret_cast<hipGraphExec_t>(1);
    return hipSuccess;
}
inline hipError_t hipGraphLaunch(hipGraphExec_t, hipStream_t) { ++fake::state().replays; return hipSuccess; }
inline hipError_t hipGraphDestroy(hipGraph_t) { return hipSuccess; }
inline hipError_t hipGraphExecDestroy(hipGraphExec_t) { return hipSuccess; }
#define HIP_SYMBOL(x) static_cast<const void*>(x)
inline hipError_t hipGetSymbolAddress(void** p, const void* symbol) { *p = const_cast<void*>(symbol); return hipSuccess; }
