// staging.h - host <-> device transfers of a context's host-buffer calls through its own pinned memory.
//
// A copy from or to pageable memory goes through the runtime's staging buffer, one piece after the
// other, and the call waits for it: 4 MB took 137 us up and 255 us down where the same bytes take 86 us
// between pinned memory and the device (measured, one MI355X box). Here the CPU copy of one piece
// runs while the one before is on its way. Eight slots of 512 KB, made on first use and freed with
// the context; each slot has an event that says when its last copy is done. The device side of a copy is
// a kernel that reads or writes the pinned memory: at this size hipMemcpyAsync costs more per piece
// (1.77 MB up / down, CPU copies included: 64 / 64 us against 72 / 89; 4 MB 126 / 129 against 153 / 192;
// pieces of 256 KB and 1 MB are slower for the kernel). Where the system grants no pinned memory the copies go
// through the runtime's staging buffer.
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
    // to p. The source is read before the call returns.
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
    bool upload(void * dst, const void * src, size_t bytes, hipStream_t s) {
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
