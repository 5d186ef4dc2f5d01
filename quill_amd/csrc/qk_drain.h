// qk_drain.h -- results on their way to the caller's arrays (host side).
//
// A read-back is a list of blocks.  For each, `launch` enqueues a kernel that
// writes the block into a pinned slot and then the slot's flag, and `take`
// moves the slot into the caller's array (widening FP32 to FP64).  Every
// worker owns two slots and has its next block on the stream while it takes
// the previous one, so the link, the conversion and the page faults of a
// fresh array overlap; the workers are the calling thread and the context's
// helpers.  A single-threaded conversion from pageable copies took 564 ms
// for the four fields of 512x256x256 cells (3.2 GB in FP64), most of it the
// first touch of the caller's pages, which threads share: 46 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <exception>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "qk_kernels.h"

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

// Until a kernel on st has stored `want` to the pinned flag f.  Should the
// stream end without it, the launch failed.
inline hipError_t wait_flag(hipStream_t st, const unsigned *flag, unsigned want)
{
    const std::atomic<unsigned> *f = (const std::atomic<unsigned> *)flag;
    for (unsigned spins = 1; f->load(std::memory_order_acquire) != want; ++spins) {
        if (spins % 65536 == 0) {
            const hipError_t e = hipStreamQuery(st);
            if (e == hipErrorNotReady) {
                (void)hipGetLastError();   // not an error of a later launch
                continue;
            }
            if (e != hipSuccess) return e;
            return f->load(std::memory_order_acquire) == want ? hipSuccess : hipErrorLaunchFailure;
        }
#if defined(__x86_64__)
        __builtin_ia32_pause();
#endif
    }
    return hipSuccess;
}

// Until event e is reached: polled for a while, then waited for.  The stream
// synchronization sleeps after some microseconds and is woken late, which a
// call of a few small steps notices.
inline hipError_t wait_event(hipEvent_t e)
{
    const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(400);
    do {
        const hipError_t r = hipEventQuery(e);
        if (r != hipErrorNotReady) return r;
        (void)hipGetLastError();
    } while (std::chrono::steady_clock::now() < until);
    return hipEventSynchronize(e);
}

class Drain {
public:
    // Bytes per slot and most workers: 8 workers write fresh huge pages at
    // 96 GB/s (16: 104), against 110 GB/s of widened numbers from the link.
    static constexpr size_t kSlot = (size_t)2 << 20;
    static constexpr int kWorkers = 8;
    // A read of less than kShare is taken by the calling thread alone, and no
    // read waits for a helper that has not woken up yet: with the caller's own
    // thread pool still spinning (torch after a parallel region) a new thread
    // got a CPU only after 3 ms, against 0.4 ms for the whole read of
    // 64x32x32 cells.  It has one slot, a small one (pinned allocations up to
    // 1 MiB cost 20 us, larger ones 340 us or more, and a short run reads
    // once), and sleeps in the stream's synchronization instead of polling.
    //
    // The workers' slots, their threads and their page faults in arrays of a
    // few MB cost a context's first shared read 2 ms, with the caller's pool
    // spinning 4 ms.  So a context shares its reads from where it has read
    // kFields bytes, or kRecords for records.  First reads, ms, into fresh
    // pages and into pages that the allocator had kept (spinning in brackets):
    //                   MB   alone       shared                     pageable copies
    //     fields         9   2.4, 1.0    3.2 (3.9), 2.8 (2.3)        2.7,  1.4
    //                   24   4.8, 3.2    3.7 (6.1), 4.1 (5.3)        5.9,  4.4
    //                   30   5.8, 3.9    4.0 (6.2), 4.7 (6.1)        7.4,  7.7
    //     records       12   3.0, 2.0    3.3 (4.3), 3.6 (3.2)        5.5,  2.6
    //                   24   5.7, 5.4    3.9 (6.4), 3.8 (6.7)       10.4,  6.8
    //     node charges  24   2.9, 1.8    3.8 (5.5), 2.4 (3.9)        2.2,  2.1
    //                   44   4.9, 4.6    4.4 (4.1), 1.7 (7.2)        5.2,  5.1
    // and later ones: fields of 24 MB alone 4.7, 3.0, shared 1.5 (3.2), 1.8
    // (3.7), but charges of 24 MB with the pool spinning 2.8, 1.7 and 2.3, 2.8:
    // these, and rows by id, which are numbers too, are shared from kNumbers on.
    static constexpr size_t kShare = (size_t)8 << 20, kAloneSlot = (size_t)960 << 10;
    static constexpr size_t kFields = (size_t)28 << 20, kRecords = (size_t)12 << 20, kNumbers = (size_t)40 << 20;

    // whether to share a read of `total` bytes (in the slots' format)
    bool shares(size_t total, size_t from)
    {
        if (total < kShare) return false;
        read_ += total;
        return read_ > from;
    }

    static size_t slot_bytes(bool shared) { return shared ? kSlot : kAloneSlot; }

    // launch(block, slot, done) -> hipError_t; take(block, slot), a block of at
    // most slot_bytes(shared).  `device` is current in the calling thread.  On
    // return the stream is idle.
    template <class Launch, class Take>
    hipError_t run(int device, hipStream_t st, bool shared, int64_t nblocks, Launch &&launch, Take &&take)
    {
        if (nblocks <= 0) return hipSuccess;
        const size_t slot = slot_bytes(shared);
        if (!shared) {
            if (hipError_t e = reserve(st, slot)) return e;
            void *at = pin_ + kFlagBytes;
            for (int64_t b = 0; b < nblocks; ++b) {
                if (hipError_t e = launch(b, at, ReadDone{arrived_, flag(0), ++seq_[0]})) return e;
                if (hipError_t e = hipStreamSynchronize(st)) return e;
                take(b, at);
            }
            return hipSuccess;
        }
        // a worker for every two blocks
        int nw = (int)std::min<int64_t>(kWorkers, (nblocks + 1) / 2);
        nw = std::max(1, std::min(nw, (int)std::thread::hardware_concurrency()));
        if (hipError_t e = reserve(st, slot * 2 * nw)) return e;
        std::atomic<int64_t> next{0};
        std::atomic<int> err{hipSuccess};
        auto work = [&](int w) {
            hipError_t e = w > 0 ? hipSetDevice(device) : hipSuccess;   // a new thread starts on device 0
            auto at = [&](int h) { return pin_ + kFlagBytes + slot * (2 * w + h); };
            auto start = [&](int64_t b, int h) {
                const int s = 2 * w + h;
                if (e == hipSuccess) e = launch(b, (void *)at(h), ReadDone{arrived_ + s, flag(s), ++seq_[s]});
            };
            int64_t b = next++;
            int h = 0;
            if (b < nblocks) start(b, h);
            while (b < nblocks && e == hipSuccess && err.load() == hipSuccess) {
                const int64_t b2 = next++;
                if (b2 < nblocks) start(b2, h ^ 1);
                if (e == hipSuccess) e = wait(st, 2 * w + h);
                if (e == hipSuccess) take(b, (void *)at(h));
                b = b2;
                h ^= 1;
            }
            if (e != hipSuccess) err.store((int)e);
        };
        open_job(nw, work);
        work(0);
        close_job();
        const hipError_t e = hipStreamSynchronize(st);
        return err.load() != hipSuccess ? (hipError_t)err.load() : e;
    }

    hipError_t release()
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            stop_ = true;
        }
        wake_.notify_all();
        for (auto &t : helpers_) t.join();
        helpers_.clear();
        hipError_t first = pin_ ? hipHostFree(pin_) : hipSuccess;
        if (arrived_) {
            const hipError_t e = hipFree(arrived_);
            if (first == hipSuccess) first = e;
        }
        pin_ = nullptr;
        arrived_ = nullptr;
        cap_ = 0;
        return first;
    }

private:
    // each slot's flag in a cache line of its own, before the slots
    static constexpr size_t kFlagLine = 128, kFlagBytes = kFlagLine * 2 * kWorkers;
    unsigned *flag(int s) const { return (unsigned *)(pin_ + kFlagLine * s); }

    // until slot s holds its block
    hipError_t wait(hipStream_t st, int s) { return wait_flag(st, flag(s), seq_[s]); }

    // helpers sleep between reads and live as long as the context
    void open_job(int nw, std::function<void(int)> work)
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            work_ = std::move(work);
            want_ = nw;
            index_ = 1;   // worker 0 is the calling thread
        }
        try {
            while ((int)helpers_.size() < nw - 1) helpers_.emplace_back([this] { help(); });
        } catch (const std::exception &) {
            // fewer helpers than asked for: those that started and the
            // calling thread take all blocks
        }
        wake_.notify_all();
    }

    void close_job()
    {
        std::unique_lock<std::mutex> lock(mu_);
        want_ = 0;
        idle_.wait(lock, [this] { return busy_ == 0; });
    }

    void help()
    {
        std::unique_lock<std::mutex> lock(mu_);
        for (;;) {
            wake_.wait(lock, [this] { return stop_ || index_ < want_; });
            if (stop_) return;
            const int w = index_++;
            ++busy_;
            lock.unlock();
            work_(w);
            lock.lock();
            if (--busy_ == 0) idle_.notify_one();
        }
    }

    hipError_t reserve(hipStream_t st, size_t slots)
    {
        if (!arrived_) {
            void *p = nullptr;
            if (hipError_t e = hipMalloc(&p, 2 * kWorkers * sizeof(unsigned))) return e;
            arrived_ = (unsigned *)p;
            if (hipError_t e = launch_fill_int(st, (int *)arrived_, 2 * kWorkers, 0)) return e;
        }
        const size_t bytes = kFlagBytes + slots;
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
            for (int s = 0; s < 2 * kWorkers; ++s) {
                seq_[s] = 0;
                *flag(s) = 0;
            }
        }
        return hipSuccess;
    }

    char *pin_ = nullptr;   // flags, then the workers' slots
    size_t cap_ = 0;
    size_t read_ = 0;       // bytes of the reads of kShare or more
    unsigned *arrived_ = nullptr;   // workgroups of each slot's launch that are done
    unsigned seq_[2 * kWorkers] = {};
    std::mutex mu_;
    std::condition_variable wake_, idle_;
    std::vector<std::thread> helpers_;
    std::function<void(int)> work_;
    int want_ = 0, index_ = 0, busy_ = 0;   // workers of the open read, the next one's index, those at work
    bool stop_ = false;
};

}  // namespace qk
