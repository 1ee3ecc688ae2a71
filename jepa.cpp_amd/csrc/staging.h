// staging.h - host <-> device transfers of a context's host-buffer calls through its own pinned memory.
//
// A copy to pageable memory goes through the runtime's staging buffer, one piece after the other, and the call
// waits for it. Here the CPU copy of one piece runs while the one before is on its way: eight slots of 512 KB,
// made on first use and freed with the context; each slot has an event that says when its last copy is done. The
// device side of a copy is a kernel that reads or writes the pinned memory: hipMemcpyAsync costs more per piece.
// Where the system grants no pinned memory the copies go through the runtime.
//
// us of one transfer, hipMemcpyAsync / slots, waited for (hot: the same host buffer each time; cold: more buffers
// than the CPU's cache holds):
//   down, cold     64 KB 36 / 14, 512 KB 31 / 34, 2 MB 122 / 117, 4 MB 243 / 222, 16 MB 979 / 867; hot 4 MB 237 / 134
//   up, hot        16 KB 18 / 13, 64 KB 33 / 14, 256 KB 15 / 20 (one box 109 / 20), 600 KB 27 / 37, 2 MB 80 / 89,
//                  4 MB 133 / 157, 16 MB 460 / 570
//   up, cold       600 KB 32 / 42, 2 MB 102 / 93, 4 MB 179 / 164, 16 MB 608 / 576
//   up, registered 600 KB 20 / 36, 4 MB 83 / 157, 16 MB 301 / 564
// So every download takes the slots, and so do uploads of at most one slot and uploads that gather their source.
// Above one slot the runtime pins the source's pages and copies from there: no CPU copy, which is what bounds the
// slots (~30 GB/s). Memory that the runtime already knows (pinned, registered, managed, device) is copied from
// where it is at any size.
#pragma once
#include "common.h"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstddef>
#include <cstdlib>
#include <cstring>

// n bytes (a multiple of 4, both ends 4-byte aligned) between memory the device can address (misc.hip); false: not
// launched
bool launch_copy_bytes(const void * src, void * dst, size_t n, hipStream_t s);

struct host_staging {
    static constexpr size_t SLOT = 512 * 1024;
    static constexpr int N = 8;

    ~host_staging() {
        for (hipEvent_t & e : done)
            if (e) hipEventDestroy(e);
        if (mem) hipHostFree(mem);
    }

    // dst[0, bytes) on the device, enqueued on s; fill(p, at, n) writes bytes [at, at + n) of the source
    // to p, before the call returns
    template <class F>
    bool upload(void * dst, size_t bytes, hipStream_t s, F && fill) {
        if (!ready()) return upload_pageable(dst, bytes, s, fill);
        for (size_t at = 0; at < bytes; at += SLOT) {
            const size_t n = std::min(SLOT, bytes - at);
            const int k = next++ % N;
            if (!settle(k)) return false;
            unsigned char * p = mem + (size_t) k * SLOT;
            fill(p, at, n);
            if (!launch_copy_bytes(p, (char *) dst + at, n, s) || !mark(k, s)) return false;
        }
        return true;
    }
    // the source may be read until the work enqueued on s is done
    bool upload(void * dst, const void * src, size_t bytes, hipStream_t s) {
        if (bytes > SLOT || known(src)) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s) == hipSuccess;
        return upload(dst, bytes, s, [&](void * p, size_t at, size_t n) { memcpy(p, (const char *) src + at, n); });
    }

    // src[0, bytes) on the device to host memory, after the work enqueued on s; returns when dst is whole
    bool download(void * dst, const void * src, size_t bytes, hipStream_t s) {
        if (!ready())
            return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s) == hipSuccess && hipStreamSynchronize(s) == hipSuccess;
        const size_t pieces = (bytes + SLOT - 1) / SLOT;
        const unsigned first = next;
        auto ask = [&](size_t i) {
            const int k = (int) ((first + i) % N);
            if (!settle(k)) return false;
            return launch_copy_bytes((const char *) src + i * SLOT, mem + (size_t) k * SLOT, std::min(SLOT, bytes - i * SLOT), s) && mark(k, s);
        };
        for (size_t i = 0; i < std::min<size_t>(N, pieces); i++)
            if (!ask(i)) return false;
        for (size_t i = 0; i < pieces; i++) {
            const int k = (int) ((first + i) % N);
            if (!settle(k)) return false;
            memcpy((char *) dst + i * SLOT, mem + (size_t) k * SLOT, std::min(SLOT, bytes - i * SLOT));
            if (i + N < pieces && !ask(i + N)) return false;
        }
        next = first + (unsigned) pieces;
        return true;
    }

private:
    unsigned char * mem = nullptr;
    hipEvent_t done[N] = {};
    bool busy[N] = {};
    unsigned next = 0;

    // the slots are there (made on first use); if not, the next call asks again
    bool ready() {
        if (mem) return true;
        std::lock_guard<std::recursive_mutex> lk(jepa_hip_mutex());
        bool ok = true;
        for (hipEvent_t & e : done)
            if (ok && !e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) { e = nullptr; ok = false; }
        void * p = nullptr;
        ok = ok && hipHostMalloc(&p, SLOT * N, hipHostMallocDefault) == hipSuccess;
        if (ok) mem = (unsigned char *) p;
        else (void) hipGetLastError();   // (the forward takes an error left on the thread for one of its launches)
        return ok;
    }
    // memory of the HIP runtime's own: pinned or registered host memory, managed or device memory
    static bool known(const void * p) {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type != hipMemoryTypeUnregistered;
        (void) hipGetLastError();
        return false;
    }
    template <class F>
    static bool upload_pageable(void * dst, size_t bytes, hipStream_t s, F && fill) {
        unsigned char * p = (unsigned char *) malloc(std::min(SLOT, bytes));
        bool ok = p != nullptr;
        for (size_t at = 0; ok && at < bytes; at += SLOT) {
            const size_t n = std::min(SLOT, bytes - at);
            fill(p, at, n);
            ok = hipMemcpyAsync((char *) dst + at, p, n, hipMemcpyHostToDevice, s) == hipSuccess && hipStreamSynchronize(s) == hipSuccess;
        }
        free(p);
        return ok;
    }
    bool settle(int k) {   // slot k is free again
        if (busy[k] && hipEventSynchronize(done[k]) != hipSuccess) return false;
        busy[k] = false;
        return true;
    }
    bool mark(int k, hipStream_t s) {   // slot k is in use until the work enqueued on s so far is done
        busy[k] = hipEventRecord(done[k], s) == hipSuccess;
        if (!busy[k]) (void) hipStreamSynchronize(s);
        return busy[k];
    }
};
