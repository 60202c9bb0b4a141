// cmf_xfer.hpp -- host <-> device transfers in chunks through pinned slots.
//
// A pageable copy runs at 17.6 GB/s to the host and 35.6 GB/s from it here, in one
// thread, and costs about 25 us however small; PCIe carries 54 GB/s. So kernels
// write what the host asked for straight into pinned slots, many arrays per launch,
// and several threads copy between the slots and the caller's memory (which also
// spreads the page faults of fresh arrays over them).
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <system_error>
#include <thread>
#include <vector>

namespace cmf {

constexpr int XFER_THREADS = 4;                     // 8 copy no faster (144 MB to the host: 3.5 ms both)
constexpr int XFER_SLOTS = 2 * XFER_THREADS;        // two per thread: one on the GPU, one copied by the host

// pinned memory of a handle, grown to what a call needs; GPU stores to it are seen by
// the host once the kernel has ended
struct Pinned {
    char* p = nullptr;
    size_t cap = 0;
    hipError_t grow(size_t bytes) {
        if (bytes <= cap) return hipSuccess;
        void* q = nullptr;
        const hipError_t e = hipHostMalloc(&q, bytes, hipHostMallocCoherent);
        if (e != hipSuccess) return e;
        release();
        p = static_cast<char*>(q);
        cap = bytes;
        return hipSuccess;
    }
    void release() {
        if (p) (void)hipHostFree(p);
        p = nullptr;
        cap = 0;
    }
};

// The first touch of a page of pinned memory by the host costs 1.5 us, 0.4 ms per MB:
// done by other threads while this one has something else to do, until it leaves the
// scope.
struct Prefault {
    std::vector<std::thread> th;
    Prefault(char* p, size_t bytes) {
        const size_t part = (bytes / XFER_THREADS + 4095) & ~(size_t)4095;
        if (bytes < (size_t)1 << 20) return;        // dearer to start the threads
        try {
            for (size_t at = 0; at < bytes; at += part)
                th.emplace_back([p, at, end = at + part < bytes ? at + part : bytes] {
                    for (size_t q = at; q < end; q += 4096) *(volatile char*)(p + q) = 0;
                });
        } catch (const std::exception&) {
            // no more threads: the transfers touch the rest
        }
    }
    ~Prefault() {
        for (std::thread& t : th) t.join();
    }
};

// f(worker) on up to nw threads, this one among them; the first error
template <class F>
hipError_t run_workers(int nw, int device, F f) {
    hipError_t rc[XFER_THREADS] = {};
    std::vector<std::thread> th;
    try {
        for (int w = 1; w < nw; ++w)
            th.emplace_back([&rc, &f, device, w] {
                rc[w] = hipSetDevice(device);
                if (rc[w] == hipSuccess) rc[w] = f(w);
            });
    } catch (const std::exception&) {
        // no more threads: those there are take the chunks
    }
    rc[0] = f(0);
    for (std::thread& t : th) t.join();
    for (hipError_t e : rc)
        if (e != hipSuccess) return e;
    return hipSuccess;
}

// Chunks 0 .. nc-1, each started on the GPU from a slot (start) and finished by the
// host once its event has passed (finish); every worker keeps two in flight.
template <class S, class F>
hipError_t run_chunks(int nc, int device, S start, F finish) {
    std::atomic<int> next{0};
    const int nw = nc / 2 < XFER_THREADS ? (nc / 2 > 0 ? nc / 2 : 1) : XFER_THREADS;
    return run_workers(nw, device, [&](int w) -> hipError_t {
        hipEvent_t ev[2] = {nullptr, nullptr};
        int at[2] = {-1, -1};
        hipError_t e = hipSuccess;
        for (int k = 0; k < 2 && e == hipSuccess; ++k) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
        for (int k = 0; e == hipSuccess; k ^= 1) {
            if (at[k] >= 0) {
                e = hipEventSynchronize(ev[k]);
                if (e == hipSuccess) finish(at[k], 2 * w + k);
                at[k] = -1;
                if (e != hipSuccess) break;
            }
            const int c = next.fetch_add(1);
            if (c < nc) {
                e = start(c, 2 * w + k, ev[k]);
                if (e == hipSuccess) at[k] = c;
            } else if (at[k ^ 1] < 0) {
                break;
            }
        }
        for (hipEvent_t x : ev)
            if (x) (void)hipEventDestroy(x);
        return e;
    });
}

}  // namespace cmf
