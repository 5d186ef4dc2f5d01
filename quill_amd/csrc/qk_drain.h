// qk_drain.h -- results on their way to the caller's arrays (host side).
//
// A read-back is a list of blocks.  For each, `launch` enqueues a kernel (or
// copy) that writes the block into a pinned slot, and `take` moves the slot
// into the caller's array (widening FP32 to FP64).  Every worker owns two
// slots and has its next block on the stream while it takes the previous
// one, so the link, the conversion and the page faults of a fresh array
// overlap.  A single-threaded conversion from pageable copies took 564 ms
// for the four fields of 512x256x256 cells (3.2 GB in FP64): most of it the
// first touch of the caller's pages, which threads share.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <exception>
#include <thread>
#include <vector>

namespace qk {

// the caller's current device, back in place at the end of the scope
class DeviceScope {
public:
    explicit DeviceScope(int device)
    {
        if (hipGetDevice(&before_) != hipSuccess) before_ = -1;
        if (before_ != device) (void)hipSetDevice(device);
        else before_ = -1;
    }
    ~DeviceScope()
    {
        if (before_ >= 0) (void)hipSetDevice(before_);
    }
    DeviceScope(const DeviceScope &) = delete;
    DeviceScope &operator=(const DeviceScope &) = delete;

private:
    int before_ = -1;
};

class Drain {
public:
    // Bytes per slot and most workers: 8 workers write fresh huge pages at
    // 96 GB/s (16: 104), against 110 GB/s of widened numbers from the link.
    static constexpr size_t kSlot = (size_t)2 << 20;
    static constexpr int kWorkers = 8;
    // Reads below kSmall take slots of kSmallSlot: pinned allocations up to
    // 1 MiB cost 20 us, larger ones 340 us or more, and a short run reads
    // its fields once.
    static constexpr size_t kSmall = (size_t)12 << 20, kSmallSlot = (size_t)256 << 10;

    static size_t slot_bytes(size_t total) { return total < kSmall ? kSmallSlot : kSlot; }

    // launch(block, slot) -> hipError_t; take(block, slot).  `total` is the
    // size of the whole read in the slots' format; `device` is current in the
    // calling thread.  On return the stream has no work left that writes a
    // slot.
    template <class Launch, class Take>
    hipError_t run(int device, hipStream_t st, size_t total, int64_t nblocks, Launch &&launch, Take &&take)
    {
        if (nblocks <= 0) return hipSuccess;
        const size_t slot = slot_bytes(total);
        // a worker for every two blocks, at least 1 MiB each
        int nw = (int)std::min<int64_t>(std::min<int64_t>(kWorkers, (nblocks + 1) / 2), (int64_t)(total >> 20) + 1);
        nw = std::max(1, std::min(nw, (int)std::max(1u, std::thread::hardware_concurrency())));
        if (hipError_t e = reserve(slot * 2 * nw, 2 * nw)) return e;
        std::atomic<int64_t> next{0};
        std::atomic<int> err{hipSuccess};
        auto work = [&](int w) {
            hipError_t e = w > 0 ? hipSetDevice(device) : hipSuccess;   // a new thread starts on device 0
            auto start = [&](int64_t b, int h) {
                if (e == hipSuccess) e = launch(b, pin_ + slot * (2 * w + h));
                if (e == hipSuccess) e = hipEventRecord(ev_[2 * w + h], st);
            };
            int64_t b = next++;
            int h = 0;
            if (b < nblocks) start(b, h);
            while (b < nblocks && e == hipSuccess && err.load() == hipSuccess) {
                const int64_t b2 = next++;
                if (b2 < nblocks) start(b2, h ^ 1);
                if (e == hipSuccess) e = hipEventSynchronize(ev_[2 * w + h]);
                if (e == hipSuccess) take(b, pin_ + slot * (2 * w + h));
                b = b2;
                h ^= 1;
            }
            if (e != hipSuccess) err.store((int)e);
        };
        std::vector<std::thread> helpers;
        try {
            helpers.reserve((size_t)nw);
            for (int w = 1; w < nw; ++w) helpers.emplace_back(work, w);
        } catch (const std::exception &) {
            // fewer workers than asked for: the ones that started and this
            // thread take all blocks
        }
        work(0);
        for (auto &t : helpers) t.join();
        const hipError_t e = hipStreamSynchronize(st);
        return err.load() != hipSuccess ? (hipError_t)err.load() : e;
    }

    hipError_t release()
    {
        hipError_t first = pin_ ? hipHostFree(pin_) : hipSuccess;
        pin_ = nullptr;
        cap_ = 0;
        for (hipEvent_t ev : ev_) {
            const hipError_t e = hipEventDestroy(ev);
            if (first == hipSuccess) first = e;
        }
        ev_.clear();
        return first;
    }

private:
    hipError_t reserve(size_t bytes, int events)
    {
        if (cap_ < bytes) {
            if (pin_) {
                if (hipError_t e = hipHostFree(pin_)) return e;
            }
            pin_ = nullptr;
            cap_ = 0;
            void *p = nullptr;
            if (hipError_t e = hipHostMalloc(&p, bytes)) return e;
            pin_ = (char *)p;
            cap_ = bytes;
        }
        while ((int)ev_.size() < events) {
            hipEvent_t ev;
            if (hipError_t e = hipEventCreateWithFlags(&ev, hipEventDisableTiming)) return e;
            ev_.push_back(ev);
        }
        return hipSuccess;
    }

    char *pin_ = nullptr;   // the workers' slots
    size_t cap_ = 0;
    std::vector<hipEvent_t> ev_;
};

}  // namespace qk
