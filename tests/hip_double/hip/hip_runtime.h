// Test double of the HIP calls that csrc/host_copy.hip makes, for a host compiler.  "Device"
// memory is host memory, and a stream runs nothing by itself: its work is queued and runs
// when something waits for the stream or for an event on it, so whatever a caller does not
// wait for is still pending.  One call of a kind can be made to fail (hip_double::fail).
#pragma once
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>

enum hipError_t { hipSuccess = 0, hipErrorInvalidDevice = 101, hipErrorUnknown = 999 };
enum hipMemcpyKind { hipMemcpyHostToDevice, hipMemcpyDeviceToHost };
enum { hipHostMallocDefault = 0, hipEventDisableTiming = 2 };

namespace hip_double {
enum Call { NONE, EVENT_RECORD, STREAM_SYNC, EVENT_SYNC };
inline Call fail = NONE;  // the next call of this kind fails
inline std::mutex mu;
inline bool failing(Call c) {
    if (fail != c) return false;
    fail = NONE;
    return true;
}
struct Stream {
    std::deque<std::function<void()>> work;
    long done = 0, queued = 0;
    void run(long upto) {
        for (; done < upto; ++done) {
            work.front()();
            work.pop_front();
        }
    }
    void add(std::function<void()> f) {
        work.push_back(std::move(f));
        ++queued;
    }
};
struct Event { Stream* stream = nullptr; long at = 0; };
struct Index { unsigned x; };
}  // namespace hip_double
typedef hip_double::Stream* hipStream_t;
typedef hip_double::Event* hipEvent_t;
inline thread_local hip_double::Index blockIdx, threadIdx;
struct dim3 { unsigned x; dim3(unsigned n) : x(n) {} };
#define __global__
#define __launch_bounds__(n)

inline const char* hipGetErrorString(hipError_t) { return "error of the test double"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipMalloc(void** p, size_t n) { *p = std::calloc(1, n); return hipSuccess; }
inline hipError_t hipFree(void* p) { std::free(p); return hipSuccess; }
inline hipError_t hipHostMalloc(void** p, size_t n, unsigned) { return hipMalloc(p, n); }
inline hipError_t hipHostFree(void* p) { return hipFree(p); }
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { *e = new hip_double::Event; return hipSuccess; }
inline hipError_t hipEventDestroy(hipEvent_t e) { delete e; return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    std::lock_guard<std::mutex> lk(hip_double::mu);
    if (hip_double::failing(hip_double::EVENT_RECORD)) return hipErrorUnknown;
    e->stream = s;
    e->at = s->queued;
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
    std::lock_guard<std::mutex> lk(hip_double::mu);
    if (hip_double::failing(hip_double::EVENT_SYNC)) return hipErrorUnknown;
    if (e->stream) e->stream->run(e->at);
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    std::lock_guard<std::mutex> lk(hip_double::mu);
    if (hip_double::failing(hip_double::STREAM_SYNC)) return hipErrorUnknown;
    s->run(s->queued);
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t s) {
    std::lock_guard<std::mutex> lk(hip_double::mu);
    s->add([=] { std::memcpy(dst, src, n); });
    return hipSuccess;
}
inline hipError_t hipMemsetAsync(void* dst, int v, size_t n, hipStream_t s) {
    std::lock_guard<std::mutex> lk(hip_double::mu);
    s->add([=] { std::memset(dst, v, n); });
    return hipSuccess;
}
template <class F, class A, class B>
inline void hipLaunchKernelGGL(F kernel, dim3 grid, dim3 threads, size_t, hipStream_t s, A a, B b) {
    std::lock_guard<std::mutex> lk(hip_double::mu);
    s->add([=] {
        for (blockIdx.x = 0; blockIdx.x < grid.x; ++blockIdx.x)
            for (threadIdx.x = 0; threadIdx.x < threads.x; ++threadIdx.x) kernel(a, b);
    });
}
