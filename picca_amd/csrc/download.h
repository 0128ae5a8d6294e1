// Results from the device to the caller's arrays through a ring of pinned buffers.
//
// A copy into the caller's pageable pages runs at 18 GB/s, one thread filling fresh memory for
// it at 4 to 5 GB/s; a copy into pinned memory runs at 57 GB/s, and the host threads move (or
// add) a chunk on while the next is copied.  A 5000 x 5000 matrix (forest x quasar distortion,
// 3000 forests) takes the call from 64 ms to 19 ms, a 2500 x 2500 one (covariance of 1196
// samples, whose inputs are now scanned by all threads) from 8.2 ms to 4.4 ms, the six results
// of 20 000 continuum fits in one copy from 0.76 ms to 0.69 ms.  Chunks of 4 MB instead of 8: 4.8 ms
// against 4.3 ms for the covariance.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace picca_host {

// The pinned memory of one context, freed with it: one block of the largest result so far (a power
// of two from 64 KB) up to 1 MB, two chunks of 1 MB for results up to 16 MB, which the calling
// thread moves on, two of 8 MB beyond, on several threads (12.5 MB: 0.73 ms, with threads 0.83 to
// 1.24 ms; 18 MB: 1.1 ms with threads, 1.38 ms as one pageable copy).  The first reading of fresh
// pinned pages takes the host 0.4 ms a MB, as much as a small result's whole call.
struct DownloadRing {
    static constexpr int SLOTS = 2;
    static constexpr int64_t SMALL = (int64_t)1 << 20, LARGE = (int64_t)8 << 20;   // a chunk
    static constexpr int64_t ONE_THREAD = 2 * LARGE;   // results that take no other threads
    char *memory = nullptr;
    hipEvent_t copied[SLOTS] = {nullptr, nullptr};
    int64_t room = 0;   // bytes of memory
    bool pinned = false;
    ~DownloadRing() { release(); }
    // bytes of one chunk of a result that takes several
    static int64_t chunk(int64_t bytes) { return bytes <= ONE_THREAD ? SMALL : LARGE; }
    void release() {
        for (int k = 0; k < SLOTS; ++k) {
            if (copied[k]) (void)hipEventDestroy(copied[k]);
            copied[k] = nullptr;
        }
        release_memory();
    }
    void release_memory() {
        if (memory && pinned)
            (void)hipHostFree(memory);
        else
            std::free(memory);
        memory = nullptr;
        room = 0;
    }
    // Room for a result of `bytes` bytes; no copy into the memory is under way.
    hipError_t ensure(int64_t bytes) {
        int64_t want = (int64_t)64 << 10;
        while (want < bytes && want < SMALL) want <<= 1;
        if (bytes > SMALL) {
            want = SLOTS * chunk(bytes);
            for (int k = 0; k < SLOTS; ++k)
                if (!copied[k]) {
                    const hipError_t err =
                        hipEventCreateWithFlags(&copied[k], hipEventDisableTiming);
                    if (err != hipSuccess) return err;
                }
        }
        if (room >= want) return hipSuccess;
        release_memory();
        pinned = hipHostMalloc((void **)&memory, (size_t)want) == hipSuccess;
        if (!pinned) {   // no pinned memory left: pageable memory does as well, slower
            (void)hipGetLastError();
            memory = (char *)std::malloc((size_t)want);
            if (!memory) return hipErrorOutOfMemory;
        }
        room = want;
        return hipSuccess;
    }
    // The first n <= SMALL bytes at `from`, in memory when it returns.
    hipError_t fetch(const void *from, int64_t n, hipStream_t stream) {
        hipError_t err = ensure(n);
        if (err == hipSuccess)
            err = hipMemcpyAsync(memory, from, (size_t)n, hipMemcpyDeviceToHost, stream);
        const hipError_t done = hipStreamSynchronize(stream);
        return err == hipSuccess ? done : err;
    }
};

// Calls take(src, lo, hi) for pieces [lo, hi) that cover the first `bytes` bytes at the device
// pointer `from`, src the host copy of byte lo; on several threads beyond ONE_THREAD bytes.  The copies
// follow the stream's work; every piece is taken when it returns.
template <class Take>
hipError_t download(DownloadRing &ring, const void *from, int64_t bytes, hipStream_t stream,
                    const Take &take) {
    if (bytes <= 0) return hipSuccess;
    constexpr int SLOTS = DownloadRing::SLOTS;
    if (bytes <= DownloadRing::SMALL) {
        const hipError_t one = ring.fetch(from, bytes, stream);
        if (one == hipSuccess) take((const char *)ring.memory, (int64_t)0, bytes);
        return one;
    }
    const int64_t CHUNK = DownloadRing::chunk(bytes);
    auto slot = [&](int64_t c) { return ring.memory + (c % SLOTS) * CHUNK; };
    hipError_t err = ring.ensure(bytes);
    if (err != hipSuccess) return err;
    const int64_t chunks = (bytes + CHUNK - 1) / CHUNK;
    auto issue = [&](int64_t c) {
        const int64_t lo = c * CHUNK, n = std::min(CHUNK, bytes - lo);
        hipError_t e = hipMemcpyAsync(slot(c), (const char *)from + lo, (size_t)n,
                                      hipMemcpyDeviceToHost, stream);
        return e == hipSuccess ? hipEventRecord(ring.copied[c % SLOTS], stream) : e;
    };
    // chunks copied, pieces taken over all chunks; a thread takes its slice of a chunk once, and
    // the next chunk is not ready before every slice of this one is taken
    std::mutex lock;
    std::condition_variable copied, took;
    int64_t ready = 0, taken = 0;
    bool settled = false, failed = false;   // settled: the number of workers is known
    const unsigned hw = std::thread::hardware_concurrency();
    int workers = bytes <= DownloadRing::ONE_THREAD
                      ? 1 : (int)std::max<unsigned>(1, std::min<unsigned>(hw, 16));
    // slice w of chunk c, in whole 4 KiB pages
    auto work = [&](int64_t c, int w) {
        const int64_t lo = c * CHUNK, n = std::min(CHUNK, bytes - lo);
        const int64_t step = ((n + workers - 1) / workers + 4095) & ~(int64_t)4095;
        const int64_t a = std::min(n, w * step), b = std::min(n, a + step);
        if (a < b) take((const char *)slot(c) + a, lo + a, lo + b);
    };
    std::vector<std::thread> pool;
    try {
        pool.reserve((size_t)workers);
        for (int w = 1; w < workers; ++w)
            pool.emplace_back([&, w] {
                for (int64_t c = 0; c < chunks; ++c) {
                    {
                        std::unique_lock<std::mutex> hold(lock);
                        copied.wait(hold, [&] { return settled && (failed || ready > c); });
                        if (failed) return;
                    }
                    work(c, w);
                    std::lock_guard<std::mutex> hold(lock);
                    if (++taken == (c + 1) * (workers - 1)) took.notify_one();
                }
            });
    } catch (const std::exception &) {   // fewer threads
    }
    {
        std::lock_guard<std::mutex> hold(lock);
        workers = (int)pool.size() + 1;
        settled = true;
    }
    for (int64_t c = 0; c < std::min<int64_t>(SLOTS, chunks) && err == hipSuccess; ++c)
        err = issue(c);
    for (int64_t c = 0; c < chunks && err == hipSuccess; ++c) {
        err = hipEventSynchronize(ring.copied[c % SLOTS]);
        if (err != hipSuccess) break;
        {
            std::lock_guard<std::mutex> hold(lock);
            ready = c + 1;
        }
        copied.notify_all();
        work(c, 0);
        {
            std::unique_lock<std::mutex> hold(lock);
            took.wait(hold, [&] { return taken == (c + 1) * (workers - 1); });
        }
        if (c + SLOTS < chunks) err = issue(c + SLOTS);
    }
    if (err != hipSuccess) {
        {
            std::lock_guard<std::mutex> hold(lock);
            failed = true;
        }
        copied.notify_all();
    }
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
