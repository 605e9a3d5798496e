// lh_hostcopy.h -- large device-to-host copies into pageable memory.
//
// A plain hipMemcpy into the pageable array of a caller stages through one
// thread and faults every page on the way: 92 MB of saves (11 states of 2049 × 256
// bins) took 9.2 ms, three times the propagation they came from.
// Here the pages are made present while the GPU works (HostPages), and two
// threads then empty a ring of four 4 MiB page-locked slots: 2.1 ms, near the
// link's rate (3.8 ms where the pages are not present; slots of 1 MiB 3.0 ms,
// of 256 KiB 6.8 ms; four threads 2.1 ms).
#pragma once
#include <hip/hip_runtime.h>
#include <sys/mman.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <thread>
#include <utility>
#include <vector>

// Copies below this go to hipMemcpy: 8 MiB takes 0.54 ms there, and the ring's
// allocation and threads cost up to that.
static constexpr size_t LH_COPY_LARGE = (size_t)16 << 20;
static constexpr size_t LH_COPY_SLOT = (size_t)4 << 20;
static constexpr int LH_COPY_THREADS = 2;

// Makes the pages of large output arrays present, from four threads of its own,
// between start() and wait(); contents stay as they are (MADV_POPULATE_WRITE; a
// kernel or a mapping without it leaves the faults to the copy).
class HostPages {
    std::vector<std::pair<char*, size_t>> pieces;
    std::atomic<size_t> next{0};
    std::vector<std::thread> th;

  public:
    void add(void* p, size_t bytes) {
        if (!p || bytes < LH_COPY_LARGE) return;
        const uintptr_t huge = (uintptr_t)2 << 20, page = 4096;
        uintptr_t a = ((uintptr_t)p + page - 1) & ~(page - 1);
        const uintptr_t e = ((uintptr_t)p + bytes) & ~(page - 1);
        while (a < e) {
            const uintptr_t b = std::min(e, (a + huge) & ~(huge - 1));
            try {
                pieces.push_back({(char*)a, b - a});
            } catch (...) {  // the rest is left to the copy
                return;
            }
            a = b;
        }
    }
    void start() {
        if (pieces.empty()) return;
        try {
            for (int i = 0; i < 4; i++)
                th.emplace_back([this] {
                    for (;;) {
                        const size_t k = next.fetch_add(1);
                        constexpr int populate_write = 23;  // MADV_POPULATE_WRITE
                        if (k >= pieces.size() || madvise(pieces[k].first, pieces[k].second, populate_write)) return;
                    }
                });
        } catch (...) {  // no more threads or memory: what was started does it
        }
    }
    void wait() {
        for (auto& t : th) t.join();
        th.clear();
    }
    ~HostPages() { wait(); }
};

// dst ← src (device memory whose writers are done or ordered before s).
static hipError_t copy_to_host(void* dst, const void* src, size_t bytes, int device, hipStream_t s) {
    if (bytes < LH_COPY_LARGE) return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
    hipPointerAttribute_t at;
    if (hipPointerGetAttributes(&at, dst) != hipSuccess)
        (void)hipGetLastError();  // pageable memory
    else if (at.type != hipMemoryTypeUnregistered)
        return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);  // page-locked already
    constexpr int NS = 2 * LH_COPY_THREADS;
    char* ring = nullptr;
    hipEvent_t ev[NS] = {};
    bool ready = hipHostMalloc((void**)&ring, NS * LH_COPY_SLOT, hipHostMallocDefault) == hipSuccess;
    for (int i = 0; i < NS && ready; i++) ready = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming) == hipSuccess;
    const size_t nch = (bytes + LH_COPY_SLOT - 1) / LH_COPY_SLOT;
    std::atomic<int> err{(int)hipSuccess};
    // thread i: slots 2i and 2i+1 in turn, chunks i, i + LH_COPY_THREADS, ...
    auto work = [&](int i) {
        const auto size = [&](size_t c) { return std::min(LH_COPY_SLOT, bytes - c * LH_COPY_SLOT); };
        const auto issue = [&](size_t c, int q) {
            if (c >= nch) return hipSuccess;
            hipError_t e = hipMemcpyAsync(ring + q * LH_COPY_SLOT, (const char*)src + c * LH_COPY_SLOT, size(c),
                                          hipMemcpyDeviceToHost, s);
            return e == hipSuccess ? hipEventRecord(ev[q], s) : e;
        };
        hipError_t e = hipSetDevice(device);
        int q = 2 * i;
        if (e == hipSuccess) e = issue(i, q);
        if (e == hipSuccess) e = issue(i + LH_COPY_THREADS, q + 1);
        for (size_t c = i; c < nch && e == hipSuccess; c += LH_COPY_THREADS, q ^= 1) {
            e = hipEventSynchronize(ev[q]);
            if (e != hipSuccess) break;
            memcpy((char*)dst + c * LH_COPY_SLOT, ring + q * LH_COPY_SLOT, size(c));
            e = issue(c + 2 * LH_COPY_THREADS, q);
        }
        if (e != hipSuccess) err = (int)e;
    };
    if (ready) {
        std::vector<std::thread> th;
        int begun = 0;
        try {
            for (int i = 1; i < LH_COPY_THREADS; i++, begun++) th.emplace_back(work, i);
        } catch (...) {  // this thread does the rest
        }
        work(0);
        for (auto& t : th) t.join();
        for (int i = begun + 1; i < LH_COPY_THREADS; i++) work(i);
        const hipError_t e = hipStreamSynchronize(s);  // nothing in flight into the ring
        if (e != hipSuccess && err == (int)hipSuccess) err = (int)e;
    } else {
        (void)hipGetLastError();
        err = (int)hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
    }
    for (int i = 0; i < NS; i++)
        if (ev[i]) (void)hipEventDestroy(ev[i]);
    if (ring) (void)hipHostFree(ring);
    return (hipError_t)(int)err;
}
