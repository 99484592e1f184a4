// The second thread of long reads (host.cpp): pieces that the GPU leaves in pinned memory, each with a
// flag behind it, on their way to their destination. Nothing of the GPU's runtime in here.
#pragma once
#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

namespace zhip {

inline void pause_cpu() {
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
    __builtin_ia32_pause();
#endif
}

// A read on its way from its staging, which the GPU fills piece by piece, to its destination.
struct Handover {
    uint8_t *dst;
    const uint8_t *src;
    uint64_t size, piece;
    const uint64_t *flags;
    uint64_t ticket;  // (of 64 bits: a process that submits for days would come round to one that a flag still holds)
    uint64_t pieces() const { return (size + piece - 1u) / piece; }
    bool arrived(uint64_t p) const { return __atomic_load_n(flags + p, __ATOMIC_ACQUIRE) == ticket; }
    void copy(uint64_t p) const { memcpy(dst + p * piece, src + p * piece, std::min(piece, size - p * piece)); }
};

// A second thread for long reads: one copies 28 GB/s from pinned memory, the bus brings 54. Pieces
// go to whichever of the two is free, in order, also before they have arrived, so that the two take turns (taken
// only once they had arrived, by either: 8 MB 224 us in half of the processes, 257 in the others). A piece that the
// thread still waits for is the caller's to take back: finish() waits for one copy at most, whatever
// has become of the GPU. The thread sleeps but for the time between start() and finish(), and looks at
// nothing of the context.
class HandoverThread {
  public:
    // (no thread to be had: the caller copies alone)
    void start(const Handover &job) {
        std::lock_guard<std::mutex> hold(lock_);
        job_ = job;
        taken_.store(0, std::memory_order_relaxed);
        open_.store(true, std::memory_order_relaxed);
        if (!thread_.joinable()) {
            try {
                thread_ = std::thread([this] { run(); });
            } catch (const std::system_error &) {
            }
        }
        wake_.notify_one();
    }
    // The caller's next piece: the first that nobody has taken, then the one that the thread has but waits for,
    // then kNone.
    static constexpr uint32_t kNone = ~0u;
    uint32_t take() {
        uint64_t t = taken_.load(std::memory_order_relaxed);
        for (;;) {
            const uint32_t next = (uint32_t)t, held = (uint32_t)(t >> 32);
            const bool fresh = next < job_.pieces();
            if (!fresh && held == 0u) return kNone;
            if (taken_.compare_exchange_weak(t, fresh ? t + 1u : (uint64_t)next, std::memory_order_relaxed)) return fresh ? next : held - 1u;
        }
    }
    // When this returns the thread copies nothing any more, whether or not all pieces were taken.
    void finish() {
        std::unique_lock<std::mutex> hold(lock_);
        open_.store(false, std::memory_order_relaxed);
        idle_.wait(hold, [this] { return !busy_; });
    }
    ~HandoverThread() {
        {
            std::lock_guard<std::mutex> hold(lock_);
            stop_ = true;
        }
        wake_.notify_one();
        if (thread_.joinable()) thread_.join();
    }

  protected:
    void run() {
        std::unique_lock<std::mutex> hold(lock_);
        for (;;) {
            wake_.wait(hold, [this] { return stop_ || open_.load(std::memory_order_relaxed); });
            if (stop_) return;
            const Handover job = job_;
            busy_ = true;
            hold.unlock();
            while (copy_one(job)) {}
            hold.lock();
            busy_ = false;
            open_.store(false, std::memory_order_relaxed);
            idle_.notify_one();
        }
    }
    // Takes a piece, waits for it and copies it, unless the caller took it back; false once nothing is left.
    bool copy_one(const Handover &job) {
        uint64_t t = taken_.load(std::memory_order_relaxed);
        do {
            if ((uint32_t)t >= job.pieces()) return false;
        } while (!taken_.compare_exchange_weak(t, (t + 1u) | (t + 1u) << 32, std::memory_order_relaxed));
        const uint32_t p = (uint32_t)t;
        while (!job.arrived(p)) {
            if (!open_.load(std::memory_order_relaxed)) return false;
            pause_cpu();
        }
        t = taken_.load(std::memory_order_relaxed);
        do {
            if (t >> 32 != p + 1u) return false;  // (taken back: it was the last)
        } while (!taken_.compare_exchange_weak(t, (uint64_t)(uint32_t)t, std::memory_order_relaxed));
        job.copy(p);
        return true;
    }
    std::mutex lock_;
    std::condition_variable wake_, idle_;
    std::thread thread_;
    Handover job_{};
    std::atomic<uint64_t> taken_{0};  // the first piece that nobody has taken; from bit 32 on, one more than the piece that the thread waits for, or 0
    std::atomic<bool> open_{false};
    bool busy_ = false, stop_ = false;
};

}  // namespace zhip
