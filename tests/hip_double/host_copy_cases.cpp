// Cases of csrc/host_copy.hip on the test double: prints the failing expectation, or "ok".
#include "host_copy.h"

#include <cstdio>

using namespace hpg;

namespace {
constexpr size_t N = 1024, BIG = (size_t(3) << 20) / 4;  // words: a staged upload, a threaded download
hip_double::Stream& stream() { return *new hip_double::Stream; }  // outlives the slots that were used on it
std::vector<unsigned> fill(size_t n, unsigned x) { return std::vector<unsigned>(n, x); }
template <class T>
HostSeg seg(std::vector<T>& h, std::vector<T>& d) { return {h.data(), d.data(), h.size() * sizeof(T)}; }
bool all(const std::vector<unsigned>& v, unsigned x) {
    for (unsigned k : v)
        if (k != x) return false;
    return true;
}
template <class F>
bool throws(F f) {
    try { f(); } catch (const std::exception&) { return true; }
    return false;
}
int bad = 0;
void expect(bool ok, const char* what) {
    if (ok) return;
    std::printf("FAILED: %s\n", what);
    ++bad;
}
}  // namespace

int main() {
    HostCopyUser user;
    // a call that fails after its kernel was queued leaves no slot behind that the kernel
    // still uses: another call on another stream keeps its own data, and so does the first
    for (hip_double::Call what : {hip_double::EVENT_RECORD, hip_double::STREAM_SYNC, hip_double::EVENT_SYNC}) {
        hip_double::Stream &a = stream(), &b = stream();
        auto h1 = fill(N, 1), d1 = fill(N, 0), h2 = fill(N, 2), d2 = fill(N, 0), h3 = fill(N, 0), d3 = fill(N, 3);
        const HostSeg up1 = seg(h1, d1), up2 = seg(h2, d2), down3 = seg(h3, d3);
        if (what == hip_double::EVENT_RECORD) {
            hip_double::fail = what;
            expect(throws([&] { copy_to_device(&a, &up1, 1); }), "a failing event record is reported");
            copy_to_device(&b, &up2, 1);
            hipStreamSynchronize(&b);
            hipStreamSynchronize(&a);
            expect(all(d1, 1), "the upload whose event record failed keeps its own data");
            expect(all(d2, 2), "the next upload keeps its own data");
        } else if (what == hip_double::STREAM_SYNC) {
            hip_double::fail = what;
            expect(throws([&] { copy_to_host(&a, &down3, 1); }), "a failing wait is reported");
            copy_to_device(&b, &up2, 1);
            hipStreamSynchronize(&a);  // the download's kernel, if it is still queued
            hipStreamSynchronize(&b);
            expect(all(d2, 2), "an upload after the failed download keeps its own data");
        } else {
            // the wait for an earlier upload fails: the slot is still in use, whoever takes it
            copy_to_device(&a, &up1, 1);
            hip_double::fail = what;
            expect(throws([&] { copy_to_device(&b, &up2, 1); }), "a failing wait for a slot is reported");
            copy_to_device(&b, &up2, 1);
            hipStreamSynchronize(&b);
            hipStreamSynchronize(&a);
            expect(all(d1, 1), "the earlier upload keeps its own data");
            expect(all(d2, 2), "the upload tried again keeps its own data");
        }
    }
    // a wait that fails in a threaded download
    {
        hip_double::Stream &a = stream(), &b = stream();
        auto h = fill(BIG, 0), d = fill(BIG, 5), h2 = fill(N, 2), d2 = fill(N, 0);
        const HostSeg down = seg(h, d), up2 = seg(h2, d2);
        hip_double::fail = hip_double::EVENT_SYNC;
        expect(throws([&] { copy_to_host(&a, &down, 1); }), "a failing wait of a large download is reported");
        copy_to_device(&b, &up2, 1);
        hipStreamSynchronize(&a);
        hipStreamSynchronize(&b);
        expect(all(d2, 2), "an upload after the failed large download keeps its own data");
        copy_to_host(&a, &down, 1);
        expect(all(h, 5), "the large download tried again");
    }
    if (!bad) std::printf("ok\n");
    return bad ? 1 : 0;
}
