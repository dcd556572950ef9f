// copyout.hpp -- large results into the caller's pageable memory.
//
// A device-to-host copy into memory that the caller has just allocated is
// bound by one host thread that faults the pages in and copies: 10 GB/s for
// 85 MB (64 potentials of a 24^3 cell, 8.3 ms beside 0.2 ms of kernels),
// against 57 GB/s into pinned memory.  Here the chunks land in a pinned ring
// and a few threads move them on, so the faults run in parallel: 8.4 -> 5.9
// ms (chunks of 1 MB 7.8, of 512 KB 10: the threads wake each other too often).
#pragma once

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <exception>
#include <thread>
#include <vector>

// below this a single copy is as fast (starting the threads costs 0.1 ms)
#define COPY_OUT_MIN ((size_t)16 << 20)
#define COPY_OUT_CHUNK ((size_t)2 << 20)
#define COPY_OUT_SLOTS 16
#define COPY_OUT_THREADS 8

// whether the host cannot read or write at p, which the copy engine can
static bool device_only(const void* p)
{
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) == hipSuccess) return a.type == hipMemoryTypeDevice;
    (void)hipGetLastError(); // memory that HIP does not know: the host's
    return false;
}

struct CopyOut
{
    char* ring = nullptr; // COPY_OUT_SLOTS pinned chunks
    hipEvent_t ev[COPY_OUT_SLOTS] = {};
    int ensure()
    {
        for (auto& e : ev)
            if (!e) HIP_TRY(hipEventCreateWithFlags(&e, hipEventDisableTiming));
        if (!ring && hipHostMalloc(reinterpret_cast<void**>(&ring),
                                   COPY_OUT_CHUNK * COPY_OUT_SLOTS) != hipSuccess)
        {
            (void)hipGetLastError(); // plain copies then; no launch shall report it
            ring = nullptr;
            return LELPH_ERR_ALLOC;
        }
        return LELPH_OK;
    }
    void release()
    {
        if (ring) (void)hipHostFree(ring);
        ring = nullptr;
        for (auto& e : ev)
        {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
    }

    // bytes of src (device) to dst (host) after the work on st; both are done
    // on return.  The threads live in this call and touch the ring and dst
    // only; every HIP call stays on the calling thread.
    int run(void* dst, const void* src, size_t bytes, hipStream_t st)
    {
        const size_t n = (bytes + COPY_OUT_CHUNK - 1) / COPY_OUT_CHUNK;
        const unsigned cpus = std::thread::hardware_concurrency();
        if (bytes < COPY_OUT_MIN || cpus < 4 || device_only(dst) || ensure() != LELPH_OK)
        {
            HIP_TRY(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st));
            HIP_TRY(hipStreamSynchronize(st));
            return LELPH_OK;
        }
        struct Shared
        {
            std::mutex mu;
            std::condition_variable cv;
            size_t landed = 0; // chunks in the ring
            std::vector<char> moved;
            size_t next = 0;
            bool stop = false;
        } sh;
        sh.moved.assign(n, 0);
        auto size_of = [&](size_t i) {
            return std::min(COPY_OUT_CHUNK, bytes - i * COPY_OUT_CHUNK);
        };
        // takes chunk after chunk; false once there is none left
        auto step = [&]() -> bool {
            size_t i;
            {
                std::unique_lock<std::mutex> lk(sh.mu);
                if (sh.next >= n) return false;
                i = sh.next++;
                sh.cv.wait(lk, [&] { return sh.stop || sh.landed > i; });
                if (sh.landed <= i) return false;
            }
            std::memcpy(static_cast<char*>(dst) + i * COPY_OUT_CHUNK,
                        ring + (i % COPY_OUT_SLOTS) * COPY_OUT_CHUNK, size_of(i));
            {
                std::lock_guard<std::mutex> lk(sh.mu);
                sh.moved[i] = 1;
            }
            sh.cv.notify_all();
            return true;
        };
        std::vector<std::thread> pool;
        const unsigned want = std::min<unsigned>(COPY_OUT_THREADS, cpus / 2);
        try
        {
            pool.reserve(want);
            for (unsigned t = 0; t < want; ++t)
                pool.emplace_back([&] {
                    while (step())
                        ;
                });
        }
        catch (const std::exception&)
        {
            // fewer threads, or none: then this thread moves the chunks
        }
        auto issue = [&](size_t i) -> bool {
            const size_t slot = i % COPY_OUT_SLOTS;
            return hipMemcpyAsync(ring + slot * COPY_OUT_CHUNK,
                                  static_cast<const char*>(src) + i * COPY_OUT_CHUNK, size_of(i),
                                  hipMemcpyDeviceToHost, st) == hipSuccess &&
                   hipEventRecord(ev[slot], st) == hipSuccess;
        };
        bool ok = true;
        size_t issued = 0;
        for (; ok && issued < std::min<size_t>(n, COPY_OUT_SLOTS); ++issued) ok = issue(issued);
        for (size_t i = 0; ok && i < n; ++i)
        {
            ok = hipEventSynchronize(ev[i % COPY_OUT_SLOTS]) == hipSuccess;
            if (!ok) break;
            {
                std::lock_guard<std::mutex> lk(sh.mu);
                sh.landed = i + 1;
            }
            sh.cv.notify_all();
            if (pool.empty()) step();
            // the chunk whose slot the next copy takes
            if (issued < n && issued == i + COPY_OUT_SLOTS)
            {
                std::unique_lock<std::mutex> lk(sh.mu);
                sh.cv.wait(lk, [&] { return sh.moved[i] != 0; });
                lk.unlock();
                ok = issue(issued++);
            }
        }
        {
            std::lock_guard<std::mutex> lk(sh.mu);
            sh.stop = true;
        }
        sh.cv.notify_all();
        for (auto& t : pool) t.join();
        if (!ok) (void)hipStreamSynchronize(st);
        return ok ? LELPH_OK : LELPH_ERR_HIP;
    }
};
