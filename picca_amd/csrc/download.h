// Results from the device to the caller's arrays through a ring of pinned buffers.
//
// A copy into the caller's pageable pages runs at 18 GB/s, one thread filling fresh memory for
// it at 4 to 5 GB/s; a copy into pinned memory runs at 57 GB/s, and the host threads move (or
// add) a chunk on while the next is copied.  A 5000 x 5000 matrix (forest x quasar distortion,
// 3000 forests) takes the call from 64 ms to 21 ms, a 2500 x 2500 one (covariance of 1196
// samples, whose inputs are now scanned by all threads) from 8.3 ms to 4.3 ms, the six results
// of 20 000 continuum fits in one copy from 0.76 ms to 0.71 ms.  Chunks of 4 MB: 4.8 ms for the
// covariance.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <cstring>
#include <system_error>
#include <thread>
#include <vector>

namespace picca_host {

// The ring of one context: allocated with the first download, 16 MB, freed with the context.
struct DownloadRing {
    static constexpr int SLOTS = 2;
    static constexpr int64_t BYTES = (int64_t)8 << 20;
    char *slot[SLOTS] = {nullptr, nullptr};
    hipEvent_t copied[SLOTS] = {nullptr, nullptr};
    bool pinned = false;
    ~DownloadRing() { release(); }
    void release() {
        for (int k = 0; k < SLOTS; ++k) {
            if (copied[k]) (void)hipEventDestroy(copied[k]);
            copied[k] = nullptr;
        }
        if (pinned)
            (void)hipHostFree(slot[0]);
        else
            std::free(slot[0]);
        slot[0] = nullptr;
    }
    hipError_t ensure() {
        if (slot[0]) return hipSuccess;
        for (int k = 0; k < SLOTS; ++k)
            if (!copied[k]) {
                const hipError_t err = hipEventCreateWithFlags(&copied[k], hipEventDisableTiming);
                if (err != hipSuccess) return err;
            }
        pinned = hipHostMalloc((void **)&slot[0], SLOTS * BYTES) == hipSuccess;
        if (!pinned) {   // no pinned memory left: pageable memory does as well, slower
            (void)hipGetLastError();
            slot[0] = (char *)std::malloc(SLOTS * BYTES);
            if (!slot[0]) return hipErrorOutOfMemory;
        }
        for (int k = 1; k < SLOTS; ++k) slot[k] = slot[0] + k * BYTES;
        return hipSuccess;
    }
};

// Calls take(src, lo, hi) for pieces [lo, hi) that cover the first `bytes` bytes at the device
// pointer `from`, src the host copy of byte lo; on several threads when there is more than a
// chunk.  The copies follow the stream's work; every piece is taken when it returns.
template <class Take>
hipError_t download(DownloadRing &ring, const void *from, int64_t bytes, hipStream_t stream,
                    const Take &take) {
    if (bytes <= 0) return hipSuccess;
    hipError_t err = ring.ensure();
    if (err != hipSuccess) return err;
    constexpr int SLOTS = DownloadRing::SLOTS;
    constexpr int64_t CHUNK = DownloadRing::BYTES;
    const int64_t chunks = (bytes + CHUNK - 1) / CHUNK;
    auto issue = [&](int64_t c) {
        const int64_t lo = c * CHUNK, n = std::min(CHUNK, bytes - lo);
        hipError_t e = hipMemcpyAsync(ring.slot[c % SLOTS], (const char *)from + lo, (size_t)n,
                                      hipMemcpyDeviceToHost, stream);
        return e == hipSuccess ? hipEventRecord(ring.copied[c % SLOTS], stream) : e;
    };
    std::atomic<int64_t> ready{0};    // chunks copied
    std::atomic<bool> failed{false};
    std::vector<std::atomic<int>> taken((size_t)chunks);   // threads done with a chunk
    for (auto &t : taken) t.store(0, std::memory_order_relaxed);
    int workers = 1;
    if (chunks > 1) {
        const unsigned hw = std::thread::hardware_concurrency();
        workers = (int)std::max<unsigned>(1, std::min<unsigned>(hw, 16));
    }
    // slice w of chunk c, in whole 4 KiB pages
    auto work = [&](int64_t c, int w) {
        const int64_t lo = c * CHUNK, n = std::min(CHUNK, bytes - lo);
        const int64_t step = ((n + workers - 1) / workers + 4095) & ~(int64_t)4095;
        const int64_t a = std::min(n, w * step), b = std::min(n, a + step);
        if (a < b) take((const char *)ring.slot[c % SLOTS] + a, lo + a, lo + b);
        taken[(size_t)c].fetch_add(1, std::memory_order_release);
    };
    std::vector<std::thread> pool;
    std::atomic<int> started{0};   // 0: the number of workers is not settled
    try {
        for (int w = 1; w < workers; ++w)
            pool.emplace_back([&, w] {
                while (started.load(std::memory_order_acquire) == 0) std::this_thread::yield();
                for (int64_t c = 0; c < chunks; ++c) {
                    while (ready.load(std::memory_order_acquire) <= c) {
                        if (failed.load(std::memory_order_acquire)) return;
                        std::this_thread::yield();
                    }
                    work(c, w);
                }
            });
    } catch (const std::system_error &) {   // fewer threads
    }
    workers = (int)pool.size() + 1;
    started.store(1, std::memory_order_release);
    for (int64_t c = 0; c < std::min<int64_t>(SLOTS, chunks) && err == hipSuccess; ++c)
        err = issue(c);
    for (int64_t c = 0; c < chunks && err == hipSuccess; ++c) {
        err = hipEventSynchronize(ring.copied[c % SLOTS]);
        if (err != hipSuccess) break;
        ready.store(c + 1, std::memory_order_release);
        work(c, 0);
        while (taken[(size_t)c].load(std::memory_order_acquire) < workers)
            std::this_thread::yield();
        if (c + SLOTS < chunks) err = issue(c + SLOTS);
    }
    if (err != hipSuccess) failed.store(true, std::memory_order_release);
    for (auto &t : pool) t.join();
    if (err != hipSuccess) (void)hipStreamSynchronize(stream);   // no copy into the ring is left
    return err;
}

// out[k] = (ADD: out[k] +) from[k]
template <bool ADD>
hipError_t download_values(DownloadRing &ring, const double *from, int64_t n, hipStream_t stream,
                           double *out) {
    return download(ring, from, n * 8, stream, [out](const char *src, int64_t lo, int64_t hi) {
        const double *s = (const double *)src;
        double *o = out + lo / 8;
        const int64_t m = (hi - lo) / 8;
        if (ADD)
            for (int64_t k = 0; k < m; ++k) o[k] += s[k];
        else
            std::memcpy(o, s, (size_t)(hi - lo));
    });
}

}  // namespace picca_host
