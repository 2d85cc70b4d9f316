// Copies between device memory and pageable host arrays through a ring of
// pinned slots: the DMA engine works on some slots while host threads empty
// (or fill) the others.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <thread>
#include <vector>

// [p, p + bytes) lies in one pinned (page-locked, hipHostMalloc) host
// allocation: the DMA engine can write it directly.
static inline bool host_pinned(const void *p, size_t bytes)
{
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();   // pageable memory: the query reports invalid value
        return false;
    }
    if (a.type != hipMemoryTypeHost) return false;
    void *start = nullptr;
    size_t size = 0;
    if (hipPointerGetAttribute(&start, HIP_POINTER_ATTRIBUTE_RANGE_START_ADDR, (hipDeviceptr_t)p) != hipSuccess ||
        hipPointerGetAttribute(&size, HIP_POINTER_ATTRIBUTE_RANGE_SIZE, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return (const char *)p >= (const char *)start && (const char *)p + bytes <= (const char *)start + size;
}

// The runtime moves pageable memory with one thread: 30 GB/s to the device,
// 18 GB/s to the host and 10 GB/s into fresh pages, where the link carries 57.
// Here a transfer is cut into slots of at most SLOT bytes, aligned to SLOT in
// the host array so that no two threads fault the same huge page, and THREADS
// host threads copy slots while the next ones are on the link.  52 MB into a
// new array 5.2 -> 1.9 ms, 16 MB 0.94 -> 0.50; 36 MB to the device, 1.2 -> 0.9.
// Slots of 1 MB: 2.0 ms and 1.8 in place of 1.5 for a whole replay of 36 MB,
// of 0.5 MB 2.7 and 2.3; 8 slots and threads 1.7 and 1.6, but each MB of the
// ring adds 0.07 ms to its first use.
// The ring is SLOTS * SLOT bytes, made at the first transfer that needs it and
// freed with its owner; no thread outlives a call.  Small transfers stay with
// the runtime: starting the threads costs 0.1 ms, which an upload makes up for
// only from about 16 MB.
struct HostCopy {
    static constexpr size_t SLOT = size_t(1) << 21;
    static constexpr int SLOTS = 4;
    static constexpr unsigned THREADS = 4;
    static constexpr size_t MIN_TO_HOST = size_t(8) << 20;
    static constexpr size_t MIN_TO_DEVICE = size_t(16) << 20;

    struct Piece {
        char *host;
        char *dev;
        size_t bytes;
    };

    char *ring = nullptr;
    hipEvent_t ev[SLOTS] = {};
    bool busy[SLOTS] = {};    // ev[s] is recorded and the slot's DMA not known to be over

    // Move bytes, host <- dev (to_host) or dev <- host, after the work that is
    // on the stream.  On return the data has arrived (to_host) or a pageable
    // array has been read and later work on the stream sees it.
    hipError_t run(char *host, char *dev, size_t bytes, bool to_host, hipStream_t stream)
    {
        if (bytes < (to_host ? MIN_TO_HOST : MIN_TO_DEVICE) || host_pinned(host, bytes) || !prepare())
            return plain(host, dev, bytes, to_host, stream);
        std::vector<Piece> part;
        for (size_t a = 0; a < bytes;) {
            const size_t edge = SLOT - (size_t)((uintptr_t)(host + a) & (SLOT - 1));
            const size_t b = std::min(bytes, a + edge);
            part.push_back({host + a, dev + a, b - a});
            a = b;
        }
        const int64_t n = (int64_t)part.size();
        // ready: copies below it may be made (to_host: their DMA is over; to the
        // device: their slot is free); copied[i]: made
        std::atomic<int64_t> ready{0}, claim{0};
        std::vector<std::atomic<bool>> copied(n);
        for (auto &x : copied) x.store(false, std::memory_order_relaxed);
        std::atomic<bool> stop{false};
        auto copy = [&](int64_t i) {
            char *const s = ring + (size_t)(i % SLOTS) * SLOT;
            if (to_host) memcpy(part[i].host, s, part[i].bytes);
            else memcpy(s, part[i].host, part[i].bytes);
            copied[i].store(true, std::memory_order_release);
        };
        std::vector<std::thread> th;
        th.reserve(THREADS);
        auto start = [&] {
            const unsigned hw = std::max(1u, std::thread::hardware_concurrency());
            try {
                for (unsigned t = 0; t < std::min(THREADS, hw); ++t)
                    th.emplace_back([&] {
                        for (int64_t i; (i = claim.fetch_add(1)) < n; copy(i))
                            while (ready.load(std::memory_order_acquire) <= i) {
                                if (stop.load(std::memory_order_relaxed)) return;
                                std::this_thread::yield();
                            }
                    });
            } catch (...) {   // as many as the system gives; none: the caller copies
            }
            return !th.empty();
        };
        hipError_t e = settle(0, SLOTS);
        if (e == hipSuccess)
            e = to_host ? drain(part, stream, ready, copied, start, copy) : feed(part, stream, ready, copied, start, copy);
        stop.store(true);
        for (auto &x : th) x.join();
        return e;
    }

    void release()
    {
        if (ring) {
            for (int s = 0; s < SLOTS; ++s) if (busy[s]) (void)hipEventSynchronize(ev[s]);
            (void)hipHostFree(ring);
        }
        for (int s = 0; s < SLOTS; ++s) if (ev[s]) (void)hipEventDestroy(ev[s]);
        *this = HostCopy();
    }

private:
    bool prepare()
    {
        if (ring) return true;
        bool ok = true;
        for (int s = 0; s < SLOTS && ok; ++s)
            if (!ev[s]) ok = hipEventCreateWithFlags(&ev[s], hipEventDisableTiming) == hipSuccess;
        void *p = nullptr;
        if (ok) ok = hipHostMalloc(&p, SLOTS * SLOT, hipHostMallocDefault) == hipSuccess;
        if (!ok) { (void)hipGetLastError(); return false; }
        ring = (char *)p;
        return true;
    }

    static hipError_t plain(char *host, char *dev, size_t bytes, bool to_host, hipStream_t stream)
    {
        if (!to_host) return hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream);
        const hipError_t e = hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream);
        return e == hipSuccess ? hipStreamSynchronize(stream) : e;
    }

    hipError_t settle(int a, int b)
    {
        for (int s = a; s < b; ++s) {
            if (!busy[s]) continue;
            const hipError_t e = hipEventSynchronize(ev[s]);
            if (e != hipSuccess) return e;
            busy[s] = false;
        }
        return hipSuccess;
    }

    template <class Start, class Copy>
    hipError_t drain(const std::vector<Piece> &part, hipStream_t stream, std::atomic<int64_t> &ready,
                     std::vector<std::atomic<bool>> &copied, Start start, Copy copy)
    {
        const int64_t n = (int64_t)part.size();
        int64_t next = 0;
        bool threads = false;
        for (int64_t i = 0; i < n; ++i) {
            while (next < std::min(n, i + SLOTS)) {
                if (next >= SLOTS && !copied[next - SLOTS].load(std::memory_order_acquire)) {
                    if (next > i) break;
                    std::this_thread::yield();
                    continue;
                }
                const int s = (int)(next % SLOTS);
                hipError_t e = hipMemcpyAsync(ring + (size_t)s * SLOT, part[next].dev, part[next].bytes,
                                              hipMemcpyDeviceToHost, stream);
                if (e == hipSuccess) e = hipEventRecord(ev[s], stream);
                if (e != hipSuccess) { (void)hipStreamSynchronize(stream); return e; }
                busy[s] = true;
                ++next;
            }
            if (i == 0) threads = start();   // while the first slots are on the link
            const int s = (int)(i % SLOTS);
            const hipError_t e = settle(s, s + 1);
            if (e != hipSuccess) return e;
            if (threads) ready.store(i + 1, std::memory_order_release);
            else copy(i);
        }
        for (int64_t i = std::max<int64_t>(0, n - SLOTS); i < n; ++i)
            while (!copied[i].load(std::memory_order_acquire)) std::this_thread::yield();
        return hipSuccess;
    }

    template <class Start, class Copy>
    hipError_t feed(const std::vector<Piece> &part, hipStream_t stream, std::atomic<int64_t> &ready,
                    std::vector<std::atomic<bool>> &copied, Start start, Copy copy)
    {
        const int64_t n = (int64_t)part.size();
        const bool threads = start();
        int64_t freed = 0;   // copies whose DMA is over
        ready.store(std::min<int64_t>(n, SLOTS), std::memory_order_release);
        for (int64_t i = 0; i < n; ++i) {
            while (!copied[i].load(std::memory_order_acquire)) {
                if (!threads && i < freed + SLOTS) {
                    copy(i);
                } else if (freed < i) {
                    const int s = (int)(freed % SLOTS);
                    const hipError_t e = freed + SLOTS <= i ? hipEventSynchronize(ev[s]) : hipEventQuery(ev[s]);
                    if (e == hipErrorNotReady) { (void)hipGetLastError(); continue; }
                    if (e != hipSuccess) return e;
                    busy[s] = false;
                    ++freed;
                    ready.store(std::min(n, freed + SLOTS), std::memory_order_release);
                } else {
                    std::this_thread::yield();
                }
            }
            const int s = (int)(i % SLOTS);
            hipError_t e = hipMemcpyAsync(part[i].dev, ring + (size_t)s * SLOT, part[i].bytes, hipMemcpyHostToDevice,
                                          stream);
            if (e == hipSuccess) e = hipEventRecord(ev[s], stream);
            if (e != hipSuccess) { (void)hipStreamSynchronize(stream); return e; }
            busy[s] = true;
        }
        return hipSuccess;
    }
};
