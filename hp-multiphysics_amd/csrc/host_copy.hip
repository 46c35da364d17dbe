// See host_copy.h.
#include "host_copy.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

namespace hpg {
namespace {

constexpr int THREADS = 8, HALVES = 2, POOL_SLOTS = 4, MAX_SEG = 4;
constexpr size_t CHUNK = size_t(1) << 20;                  // staging unit of a large copy
constexpr size_t SLOT_BYTES = CHUNK * THREADS * HALVES;    // 16 MiB
// Measured, staged / direct, us.  To the device (a host array new to the runtime takes what a
// repeated one does, within 6 us up to 1 MB and 4 % above): 64 KB 14 / 34, 128 KB 16 / 60,
// 256 KB 20 / 16, 512 KB 28 / 27, 2 MB 96 / 79, 16 MB 571 / 460: direct from 256 KB up.  To
// the host, into pages touched before: 64 KB 14 / 36, 256 KB 22 / 19, 1 MB 61 / 64, with the
// threads 2 MB 126 / 127, 4 MB 224 / 251, 64 MB 2 256 / 3 910; into pages never touched (the
// page faults cost more than the copy): 64 KB 23 / 45, 256 KB 54 / 52, 1 MB 242 / 236, with
// the threads 2 MB 349 / 471, 4 MB 445 / 967, 64 MB 3 681 / 15 161.
constexpr size_t SMALL = size_t(1) << 18;
constexpr size_t LARGE = size_t(2) << 20;

void hip(hipError_t e, const char* what) {
    if (e != hipSuccess) throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}

struct Slot {
    int dev = 0;
    char* p = nullptr;
    hipEvent_t ev[THREADS * HALVES] = {};
    bool pending = false;  // a copy to the device on `stream` may still read the slot (ev[0])
    hipStream_t stream = nullptr;
    void wait() {
        if (!pending) return;
        hip(hipEventSynchronize(ev[0]), "staging wait");
        pending = false;
    }
    ~Slot() {
        if (pending) (void)hipEventSynchronize(ev[0]);
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
        if (p) (void)hipHostFree(p);
    }
};

struct Pool {
    std::mutex mu;
    std::vector<std::unique_ptr<Slot>> free;
    int made = 0, users = 0;
};
Pool& pool() {
    static Pool* p = new Pool;  // never destroyed: objects may outlive static destruction
    return *p;
}

std::unique_ptr<Slot> take() {
    int dev = 0;
    hip(hipGetDevice(&dev), "hipGetDevice");
    Pool& q = pool();
    {
        std::lock_guard<std::mutex> lk(q.mu);
        for (size_t k = 0; k < q.free.size(); ++k)
            if (q.free[k]->dev == dev) {
                std::unique_ptr<Slot> s = std::move(q.free[k]);
                q.free.erase(q.free.begin() + k);
                return s;
            }
        if (q.made >= POOL_SLOTS) return nullptr;
        ++q.made;
    }
    std::unique_ptr<Slot> s(new Slot);
    s->dev = dev;
    bool ok = hipHostMalloc((void**)&s->p, SLOT_BYTES, hipHostMallocDefault) == hipSuccess;
    for (hipEvent_t& e : s->ev) ok = ok && hipEventCreateWithFlags(&e, hipEventDisableTiming) == hipSuccess;
    if (ok) return s;
    (void)hipGetLastError();  // no pinned memory: the caller copies directly
    s.reset();
    std::lock_guard<std::mutex> lk(q.mu);
    --q.made;
    return nullptr;
}

// returns the slot to the pool on every path
struct Held {
    std::unique_ptr<Slot> s;
    Held() : s(take()) {}
    // a copy failed with work of this slot perhaps still queued on the stream: wait for it,
    // or, where that fails too, keep the slot out of the pool (it stays counted there, so
    // no more than POOL_SLOTS are ever lost)
    void settle(hipStream_t st) {
        if (hipStreamSynchronize(st) != hipSuccess) (void)s.release();
    }
    ~Held() {
        if (!s) return;
        Pool& q = pool();
        std::lock_guard<std::mutex> lk(q.mu);
        q.free.push_back(std::move(s));
    }
};

struct Segs {
    unsigned* dev[MAX_SEG];
    unsigned end[MAX_SEG];  // running word counts
    int n;
};

template <bool TO_DEV>
__global__ __launch_bounds__(256) void k_stage(Segs g, unsigned* __restrict__ slot) {
    const unsigned k = blockIdx.x * 256 + threadIdx.x;
    unsigned b = 0;
    for (int i = 0; i < g.n; ++i) {
        if (k >= b && k < g.end[i]) {
            if (TO_DEV) g.dev[i][k - b] = slot[k];
            else slot[k] = g.dev[i][k - b];
        }
        b = g.end[i];
    }
}

void direct(hipStream_t st, const HostSeg* seg, int n, bool to_dev) {
    for (int i = 0; i < n; ++i) {
        if (!seg[i].bytes) continue;
        if (to_dev) hip(hipMemcpyAsync(seg[i].dev, seg[i].host, seg[i].bytes, hipMemcpyHostToDevice, st), "H2D");
        else hip(hipMemcpyAsync(seg[i].host, seg[i].dev, seg[i].bytes, hipMemcpyDeviceToHost, st), "D2H");
    }
    hip(hipStreamSynchronize(st), "sync");
}

void small(hipStream_t st, const HostSeg* seg, int n, bool to_dev, Slot& s) {
    // the same stream's earlier copy out of the slot runs before this call's kernel; the
    // host's own writes have to wait for it
    if (to_dev || s.stream != st) s.wait();
    Segs g{};
    g.n = n;
    unsigned end = 0;
    for (int i = 0; i < n; ++i) {
        if (to_dev && seg[i].bytes) std::memcpy(s.p + 4 * (size_t)end, seg[i].host, seg[i].bytes);
        end += (unsigned)(seg[i].bytes / 4);
        g.dev[i] = static_cast<unsigned*>(seg[i].dev);
        g.end[i] = end;
    }
    const dim3 grid((end + 255) / 256), th(256);
    if (to_dev) {
        hipLaunchKernelGGL(k_stage<true>, grid, th, 0, st, g, reinterpret_cast<unsigned*>(s.p));
        hip(hipGetLastError(), "staging launch");
        hip(hipEventRecord(s.ev[0], st), "hipEventRecord");
        s.pending = true;
        s.stream = st;
        return;
    }
    hipLaunchKernelGGL(k_stage<false>, grid, th, 0, st, g, reinterpret_cast<unsigned*>(s.p));
    hip(hipGetLastError(), "staging launch");
    hip(hipStreamSynchronize(st), "sync");
    s.pending = false;
    size_t o = 0;
    for (int i = 0; i < n; ++i) {
        if (seg[i].bytes) std::memcpy(seg[i].host, s.p + o, seg[i].bytes);
        o += seg[i].bytes;
    }
}

void large(hipStream_t st, const HostSeg* seg, int n, Slot& s, size_t total) {
    struct Piece { char* host; char* dev; size_t bytes; };
    s.wait();
    std::vector<Piece> pieces;
    for (int i = 0; i < n; ++i)
        for (size_t o = 0; o < seg[i].bytes; o += CHUNK)
            pieces.push_back({static_cast<char*>(seg[i].host) + o, static_cast<char*>(seg[i].dev) + o,
                              std::min(CHUNK, seg[i].bytes - o)});
    const int nt = (int)std::max<size_t>(1, std::min<size_t>(THREADS, total / CHUNK));
    std::atomic<int> failed{0};
    auto work = [&](int j) {
        if (hipSetDevice(s.dev) != hipSuccess) { failed = (int)hipErrorInvalidDevice; return; }
        auto ok = [&](hipError_t e) { if (e != hipSuccess) failed = (int)e; return e == hipSuccess; };
        Piece wait[HALVES] = {};  // pieces in flight per half
        bool used[HALVES] = {};
        int h = 0;
        auto finish = [&](int b) {
            if (!used[b]) return true;
            used[b] = false;
            if (!ok(hipEventSynchronize(s.ev[j * HALVES + b]))) return false;
            std::memcpy(wait[b].host, s.p + (size_t)(j * HALVES + b) * CHUNK, wait[b].bytes);
            return true;
        };
        for (size_t k = j; k < pieces.size() && !failed; k += nt, h ^= 1) {
            const Piece& c = pieces[k];
            if (!finish(h)) break;
            if (!ok(hipMemcpyAsync(s.p + (size_t)(j * HALVES + h) * CHUNK, c.dev, c.bytes, hipMemcpyDeviceToHost, st)))
                break;
            wait[h] = c;
            used[h] = true;
            if (!ok(hipEventRecord(s.ev[j * HALVES + h], st))) {
                used[h] = false;
                break;
            }
        }
        finish(h);
        finish(h ^ 1);
    };
    std::vector<std::thread> th;
    int started = 1;
    try {
        for (; started < nt; ++started) th.emplace_back(work, started);
    } catch (...) {  // no more threads: this one does the rest of the shares
    }
    work(0);
    for (int j = started; j < nt; ++j) work(j);
    for (std::thread& t : th) t.join();
    hip((hipError_t)failed.load(), "D2H");
}

void exchange(hipStream_t st, const HostSeg* seg, int n, bool to_dev) {
    size_t total = 0;
    for (int i = 0; i < n; ++i) {
        if (seg[i].bytes && (!seg[i].host || !seg[i].dev)) throw std::runtime_error("copy: null array");
        total += seg[i].bytes;
    }
    if (total == 0) {
        if (!to_dev) hip(hipStreamSynchronize(st), "sync");
        return;
    }
    if (n > MAX_SEG || (total > SMALL && (to_dev || total < LARGE))) {
        direct(st, seg, n, to_dev);
        return;
    }
    Held h;
    if (!h.s) {
        direct(st, seg, n, to_dev);
        return;
    }
    try {
        if (total <= SMALL) small(st, seg, n, to_dev, *h.s);
        else large(st, seg, n, *h.s, total);
    } catch (...) {
        h.settle(st);
        throw;
    }
}

}  // namespace

void copy_to_device(hipStream_t stream, const HostSeg* seg, int n) { exchange(stream, seg, n, true); }
void copy_to_host(hipStream_t stream, const HostSeg* seg, int n) { exchange(stream, seg, n, false); }

HostCopyUser::HostCopyUser() {
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    ++q.users;
}
HostCopyUser::~HostCopyUser() {
    std::vector<std::unique_ptr<Slot>> drop;
    Pool& q = pool();
    std::lock_guard<std::mutex> lk(q.mu);
    if (--q.users == 0) {
        q.made -= (int)q.free.size();
        drop.swap(q.free);
    }
}

}  // namespace hpg
