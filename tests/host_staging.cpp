// Test program of staging.h on a stand-in HIP runtime: device memory is host memory, and the work of the one stream
// is queued and runs only where the caller waits for it, so a slot that is filled again or read too early shows.
// test_host_staging.py builds it and runs one case per call; exit status 0: as it should be.
#include "staging.h"

#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <string>
#include <vector>

namespace {
std::vector<std::function<void()>> g_queue;       // the stream's work in order
size_t g_done = 0;                                 // entries already run
std::vector<size_t> g_events;                      // queue position each event stands for
bool g_refuse_pinned = false, g_refuse_launch = false;
hipError_t g_last = hipSuccess;
int g_kernels = 0, g_memcpys = 0;
std::vector<std::pair<const unsigned char *, size_t>> g_known;   // memory the runtime knows

void run_to(size_t n) {
    for (; g_done < n; g_done++) g_queue[g_done]();
}
hipError_t fail(hipError_t e) { return g_last = e; }
}  // namespace

extern "C" {
hipError_t hipHostMalloc(void ** p, size_t n, unsigned) {
    if (g_refuse_pinned) return fail(hipErrorOutOfMemory);
    *p = malloc(n);
    return hipSuccess;
}
hipError_t hipHostFree(void * p) { run_to(g_queue.size()); free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t * e, unsigned) {
    g_events.push_back(0);
    *e = (hipEvent_t) (uintptr_t) g_events.size();
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { g_events[(uintptr_t) e - 1] = g_queue.size(); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e) { run_to(g_events[(uintptr_t) e - 1]); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { run_to(g_queue.size()); return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMemcpyAsync(void * d, const void * s, size_t n, hipMemcpyKind, hipStream_t) {
    g_memcpys++;
    g_queue.push_back([=] { memcpy(d, s, n); });
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t * a, const void * p) {
    *a = {};
    a->type = hipMemoryTypeUnregistered;
    for (const auto & k : g_known)
        if (p >= k.first && p < k.first + k.second) a->type = hipMemoryTypeHost;
    return hipSuccess;
}
}

void jepa_log(const char * fmt, ...) {
    va_list a;
    va_start(a, fmt);
    vfprintf(stderr, fmt, a);
    va_end(a);
}
std::recursive_mutex & jepa_hip_mutex() {
    static std::recursive_mutex m;
    return m;
}
bool launch_copy_bytes(const void * s, void * d, size_t n, hipStream_t) {
    if (g_refuse_launch) return false;
    g_kernels++;
    g_queue.push_back([=] { memcpy(d, s, n); });
    return true;
}

namespace {
#define CHECK(x) do { if (!(x)) { fprintf(stderr, "line %d: %s\n", __LINE__, #x); return 1; } } while (0)

std::vector<unsigned char> bytes_of(size_t n, unsigned seed) {
    std::vector<unsigned char> v(n);
    for (size_t i = 0; i < n; i++) v[i] = (unsigned char) ((i * 2654435761u + seed * 40503u) >> 11);
    return v;
}

// several transfers each way through one object, with pieces before and past the eight slots; the source of a
// gathering upload, and of one that takes the slots, is overwritten as soon as the call returns
int round_trips(bool plain) {
    host_staging st;
    const size_t slot = host_staging::SLOT;
    unsigned seed = 1;
    for (size_t n : {(size_t) 4, slot - 4, slot, slot + 4, 3 * slot, 8 * slot + 1024, 21 * slot + 12}) {
        const std::vector<unsigned char> a = bytes_of(n, seed++);
        std::vector<unsigned char> src = a, dev(n, 0), back(n, 0);
        if (plain) CHECK(st.upload(dev.data(), src.data(), n, nullptr));
        else CHECK(st.upload(dev.data(), n, nullptr, [&](void * p, size_t at, size_t k) { memcpy(p, src.data() + at, k); }));
        if (plain) run_to(g_queue.size());
        std::fill(src.begin(), src.end(), 0xee);
        CHECK(st.download(back.data(), dev.data(), n, nullptr));
        CHECK(back == a);
    }
    return 0;
}
}  // namespace

int main(int argc, char ** argv) {
    const std::string c = argc > 1 ? argv[1] : "";
    if (c == "slots") return round_trips(true) + round_trips(false);
    if (c == "refused") {
        g_refuse_pinned = true;
        if (round_trips(false) || round_trips(true)) return 1;
        CHECK(g_kernels == 0 && g_memcpys > 0);
        CHECK(g_last == hipSuccess);      // nothing left behind for the forward's own check
        g_refuse_pinned = false;          // granted later: the slots are used
        g_kernels = 0;
        CHECK(round_trips(true) == 0 && g_kernels > 0);
        return 0;
    }
    if (c == "direct") {
        // one copy from where the source is: more than a slot, or memory the runtime knows, of any size
        host_staging st;
        const size_t slot = host_staging::SLOT;
        std::vector<unsigned char> src = bytes_of(2 * slot, 5), dev(2 * slot, 0);
        auto takes = [&](const unsigned char * p, size_t n, int kernels, int memcpys) {
            g_kernels = g_memcpys = 0;
            std::fill(dev.begin(), dev.end(), 0);
            if (!st.upload(dev.data(), p, n, nullptr)) return false;
            run_to(g_queue.size());
            return g_kernels == kernels && g_memcpys == memcpys && memcmp(dev.data(), p, n) == 0;
        };
        CHECK(takes(src.data(), 4, 1, 0) && takes(src.data(), slot, 1, 0));
        CHECK(takes(src.data(), slot + 4, 0, 1) && takes(src.data(), 2 * slot, 0, 1));
        g_known.push_back({src.data() + slot, slot});
        CHECK(takes(src.data() + slot, 4, 0, 1) && takes(src.data() + slot + 400, slot - 400, 0, 1));
        CHECK(takes(src.data(), slot, 1, 0));
        return 0;
    }
    if (c == "stale") {
        CHECK(round_trips(true) == 0);
        g_last = hipErrorInvalidDevice;   // left by some earlier call of the program
        CHECK(round_trips(true) == 0);
        g_last = hipErrorInvalidDevice;
        CHECK(round_trips(false) == 0);
        g_last = hipSuccess;              // a launch that fails is still reported
        g_refuse_launch = true;
        host_staging st;
        unsigned char a[8] = {}, b[8];
        CHECK(!st.upload(b, a, 8, nullptr) && !st.download(a, b, 8, nullptr));
        return 0;
    }
    fprintf(stderr, "no case %s\n", c.c_str());
    return 2;
}
