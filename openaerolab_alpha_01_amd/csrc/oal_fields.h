// The density and velocity download's chunks, slots and worker threads (host; no HIP: the device comes as a
// template argument).
//
// The kernel writes chunks of cells into pinned slots over the link, several in flight, while worker threads copy
// finished slots to the caller's arrays: with one thread that copy (and the first touch of the caller's fresh
// pages) is the bound, 10 GB/s, against the link's rate.  Up to 4 MiB are copied by the calling thread alone:
// starting a thread costs about as much as copying half of that.  256^3 (537 MB) 52 -> 12.4 ms, 12 ragged boxes
// (637 MB) 61 -> 14.6 ms; 8^3 blocks 200 x 120 x 104, regrouped by the kernel instead of the host, 33 -> 2.3 ms;
// 48 x 32 x 32 0.13 -> 0.10 ms (no device allocation per call).  Where the host has no memory to pin, the chunks go
// through device memory, one after the other.
#pragma once

#include <sched.h>
#include <stddef.h>
#include <stdint.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace oal {

constexpr uint32_t FIELD_CHUNK = 65536;   // cells: 2 MiB of rho and u
constexpr int FIELD_SLOTS = 12;

struct FieldChunks {
    size_t total, count;
    uint32_t cells;   // of a chunk (the last may be shorter)
    int slots;
    explicit FieldChunks(size_t n) : total(n) {
        cells = (uint32_t)std::min<size_t>(std::max<size_t>((n + 15) / 16, 4096), FIELD_CHUNK);
        count = (n + cells - 1) / cells;
        slots = (int)std::min<size_t>((count + 3) / 4 + 1, FIELD_SLOTS);
    }
    uint32_t size(size_t c) const { return (uint32_t)std::min<size_t>(cells, total - c * cells); }
};

// rho [total], u [3][total], either may be null.  DEV, whose errors are 0 for none:
//   reserve(cells, slots)      slots of 4 `cells` doubles each, or an error: no memory to pin
//   slots(), slot(i)           how many, and where
//   issue(i, c0, n)            writes [4][n] (rho, ux, uy, uz) of the cells [c0, c0 + n) to slot i, asynchronously
//   wait(i)                    until slot i is written
//   direct(c0, n, dst)         the same through device memory: rho to dst[0], ux to dst[1], ..., unless null
//   drain()                    until nothing writes any slot
template <class DEV>
typename DEV::error download_fields(DEV& dev, size_t total, double* rho, double* u) {
    using error = typename DEV::error;
    const FieldChunks fc(total);
    if (dev.reserve(fc.cells, fc.slots) != error(0)) {
        for (size_t c = 0; c < fc.count; ++c) {
            const size_t at = c * fc.cells;
            double* dst[4] = {rho ? rho + at : nullptr, nullptr, nullptr, nullptr};
            if (u)
                for (size_t a = 0; a < 3; ++a) dst[a + 1] = u + a * total + at;
            const error e = dev.direct((uint32_t)at, fc.size(c), dst);
            if (e != error(0)) return e;
        }
        return error(0);
    }
    const size_t slots = dev.slots();
    auto copy_out = [&](size_t c) {
        const size_t n = fc.size(c), at = c * fc.cells;
        const double* s = dev.slot(c % slots);
        if (rho) std::memcpy(rho + at, s, n * 8);
        if (u)
            for (size_t a = 0; a < 3; ++a) std::memcpy(u + a * total + at, s + (a + 1) * n, n * 8);
    };
    // workers: take finished chunks from the queue
    std::mutex mu;
    std::condition_variable work, freed;
    std::vector<size_t> queue;
    size_t taken = 0;                       // chunks taken from the queue
    std::vector<char> busy(slots, 0);       // a slot is in flight or being copied
    bool stop = false;
    std::vector<std::thread> pool;
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    const size_t want = total <= 2 * FIELD_CHUNK ? 0 : std::min<size_t>({total / FIELD_CHUNK, 8, (size_t)std::max(cpus - 1, 0)});
    auto worker = [&] {
        std::unique_lock<std::mutex> lk(mu);
        for (;;) {
            work.wait(lk, [&] { return stop || taken < queue.size(); });
            if (taken >= queue.size()) return;
            const size_t c = queue[taken++];
            lk.unlock();
            copy_out(c);
            lk.lock();
            busy[c % slots] = 0;
            freed.notify_one();
        }
    };
    try {
        queue.reserve(fc.count);
        pool.reserve(want);
        for (size_t i = 0; i < want; ++i) pool.emplace_back(worker);
    } catch (...) {   // fewer threads, or none
    }
    error e = error(0);
    size_t issued = 0, ready = 0;
    while (ready < fc.count && e == error(0)) {
        for (;;) {
            bool open;
            {
                std::unique_lock<std::mutex> lk(mu);
                if (issued == ready && issued < fc.count) freed.wait(lk, [&] { return !busy[issued % slots]; });
                open = issued < fc.count && !busy[issued % slots];
                if (open) busy[issued % slots] = 1;
            }
            if (!open) break;
            e = dev.issue(issued % slots, (uint32_t)(issued * fc.cells), fc.size(issued));
            if (e != error(0)) break;
            ++issued;
        }
        if (e == error(0)) e = dev.wait(ready % slots);
        if (e != error(0)) break;
        if (pool.empty()) {
            copy_out(ready);
            busy[ready % slots] = 0;
        } else {
            std::lock_guard<std::mutex> lk(mu);
            queue.push_back(ready);
            work.notify_one();
        }
        ++ready;
    }
    {
        std::lock_guard<std::mutex> lk(mu);
        stop = true;
    }
    work.notify_all();
    for (std::thread& t : pool) t.join();
    if (e != error(0)) dev.drain();
    return e;
}

}  // namespace oal
