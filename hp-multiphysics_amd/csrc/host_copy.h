// Copies between a caller's (pageable) host arrays and device arrays.
//
// A pageable hipMemcpy costs about 20 us however small it is, and a large one into pages
// that were never touched (a fresh numpy array) runs at the speed of one thread's page
// faults: at 512 x 512, p = 4, reading the state back (101 MB) took 10.4 ms, 3.9 ms now.
// Both go through pinned staging slots here instead:
//   small (a residual call of a small mesh): one kernel moves every segment between the
//     slot and the device arrays, so three arrays cost one launch and no copy engine;
//   large, to the host: up to 8 threads each walk their own chunks, two staging halves per
//     thread, so page faults and host copies run in parallel with the transfers;
//   the rest (middle sizes, large ones to the device) copies directly.
// Slots belong to a pool shared by the contexts of a process: at most POOL_SLOTS (of
// SLOT_BYTES) exist at once, a call that finds none free copies directly, and the pool is
// freed when the last object that uses it is destroyed.  Thread safe; a slot that a copy
// to the device may still read is waited for (its event) before it is used again.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstring>
#include <stdexcept>
#include <string>
#include <vector>

namespace hpg {

struct HostSeg {
    void* host;
    void* dev;
    size_t bytes;  // a multiple of 4
};

// every segment host -> device (returns when the host arrays may be reused; the device
// side is ordered on the stream) or device -> host (returns when the data has arrived);
// throws std::runtime_error on a HIP error
void copy_to_device(hipStream_t stream, const HostSeg* seg, int n);
void copy_to_host(hipStream_t stream, const HostSeg* seg, int n);

// counts the objects that use the pool (contexts, networks)
struct HostCopyUser {
    HostCopyUser();
    ~HostCopyUser();
    HostCopyUser(const HostCopyUser&) = delete;
    HostCopyUser& operator=(const HostCopyUser&) = delete;
};

// Device arrays of a context, zeroed at allocation.  While a context is being built, small
// arrays share 1 MiB chunks with a host mirror that takes their initial contents, and
// flush() sends each chunk's used part once: a context of a small mesh is a few allocations
// and copies instead of about 120 allocations, 120 clears and 60 pageable copies.  Large
// arrays, and everything after flush(), are allocated and copied on their own.
class DeviceArrays {
    static constexpr size_t CHUNK = size_t(1) << 20, ALIGN = 256;
    std::vector<void*> allocs;
    std::vector<char> mirror;
    char* chunk = nullptr;
    bool building = true;

    static void ok(hipError_t e, const char* what) {
        if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
    }
    void send(hipStream_t st) {
        if (!chunk) return;
        ok(hipMemcpyAsync(chunk, mirror.data(), mirror.size(), hipMemcpyHostToDevice, st), "H2D");
        ok(hipStreamSynchronize(st), "sync");
        chunk = nullptr;
    }
    void* get(hipStream_t st, size_t bytes, const void* init) {
        if (building && bytes <= CHUNK / 8) {
            bytes = (bytes + ALIGN - 1) / ALIGN * ALIGN;
            if (chunk && mirror.size() + bytes > CHUNK) send(st);
            if (!chunk) {
                void* p = nullptr;
                ok(hipMalloc(&p, CHUNK), "hipMalloc");
                allocs.push_back(p);
                chunk = static_cast<char*>(p);
                mirror.clear();
                mirror.reserve(CHUNK);
            }
            const size_t o = mirror.size();
            mirror.resize(o + bytes, 0);
            return chunk + o;
        }
        void* p = nullptr;
        ok(hipMalloc(&p, bytes), "hipMalloc");
        allocs.push_back(p);
        if (!init) ok(hipMemsetAsync(p, 0, bytes, st), "memset");
        return p;
    }

public:
    template <class T>
    T* alloc(hipStream_t st, size_t n) {
        return static_cast<T*>(get(st, (n ? n : 1) * sizeof(T), nullptr));
    }
    template <class T>
    T* upload(hipStream_t st, const T* h, size_t n) {
        if (n == 0) return alloc<T>(st, 0);
        char* p = static_cast<char*>(get(st, n * sizeof(T), h));
        if (chunk && p >= chunk && p < chunk + CHUNK) std::memcpy(mirror.data() + (p - chunk), h, n * sizeof(T));
        else ok(hipMemcpyAsync(p, h, n * sizeof(T), hipMemcpyHostToDevice, st), "H2D");
        return reinterpret_cast<T*>(p);
    }
    // the end of construction: every array holds its initial contents
    void flush(hipStream_t st) {
        send(st);
        building = false;
        std::vector<char>().swap(mirror);
        ok(hipStreamSynchronize(st), "sync");
    }
    void release() {
        for (void* p : allocs) (void)hipFree(p);
        allocs.clear();
    }
};

}  // namespace hpg
