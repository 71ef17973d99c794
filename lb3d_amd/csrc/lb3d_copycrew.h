// lb3d_copycrew.h -- copies between the caller's memory and transfer buffers by
// several threads (host code only).
#pragma once

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstring>
#include <mutex>
#include <thread>

namespace lb3d {

// Copies between the caller's memory and pinned memory, by the calling thread
// and, for large transfers, a few helpers that live for the transfer: one
// thread writes fresh pages at 15 GB/s, a fourth of what PCIe brings.  A helper
// without work looks for it for SPIN, longer than a piece of 8 MiB takes to be
// converted and to cross PCIe (0.2 ms), so that it is there at once for the
// first piece and between two; then it is parked, and leaves its processor alone while the caller
// waits for the device.
class CopyCrew {
  public:
    explicit CopyCrew(size_t total)
    {
        if (total < (size_t)(16u << 20)) return;
        const unsigned hw = std::thread::hardware_concurrency();
        const int want = hw >= 8 ? MAX_HELPERS : (hw >= 4 ? 1 : 0);
        try {
            for (; n_ < want; n_++) th_[n_] = std::thread([this, i = n_] { work(i); });
        } catch (...) {  // no thread to be had: fewer helpers
        }
    }
    CopyCrew(const CopyCrew &) = delete;
    CopyCrew &operator=(const CopyCrew &) = delete;
    ~CopyCrew()
    {
        {
            std::lock_guard<std::mutex> lock(mu_);
            stop_.store(true, std::memory_order_release);
        }
        wake_.notify_all();
        for (int i = 0; i < n_; i++) th_[i].join();
    }
    void copy(void *d, const void *s, size_t n)
    {
        if (n_ == 0 || n < (size_t)(1u << 20)) {
            std::memcpy(d, s, n);
            return;
        }
        d_ = (char *)d;
        s_ = (const char *)s;
        bytes_ = n;
        done_.store(0, std::memory_order_relaxed);
        parts_ = n_ + 1;
        {
            std::lock_guard<std::mutex> lock(mu_);
            job_.fetch_add(1, std::memory_order_release);
        }
        wake_.notify_all();
        slice(parts_ - 1);
        while (done_.load(std::memory_order_acquire) != n_) std::this_thread::yield();
    }

  private:
    static constexpr int MAX_HELPERS = 3;
    static constexpr std::chrono::microseconds SPIN{500};
    void slice(int i) const
    {
        // whole pages per helper
        const size_t per = ((bytes_ + parts_ - 1) / parts_ + 4095) & ~(size_t)4095;
        const size_t at = per * (size_t)i;
        if (at < bytes_) std::memcpy(d_ + at, s_ + at, bytes_ - at < per ? bytes_ - at : per);
    }
    void work(int i)
    {
        unsigned seen = 0;
        for (;;) {
            const auto until = std::chrono::steady_clock::now() + SPIN;
            while (job_.load(std::memory_order_acquire) == seen && !stop_.load(std::memory_order_acquire) &&
                   std::chrono::steady_clock::now() < until)
                std::this_thread::yield();
            unsigned j = job_.load(std::memory_order_acquire);
            if (j == seen) {
                std::unique_lock<std::mutex> lock(mu_);
                wake_.wait(lock, [&] {
                    return (j = job_.load(std::memory_order_relaxed)) != seen || stop_.load(std::memory_order_relaxed);
                });
                if (j == seen) return;
            }
            seen = j;
            slice(i);
            done_.fetch_add(1, std::memory_order_release);
        }
    }
    std::mutex mu_;
    std::condition_variable wake_;
    std::thread th_[MAX_HELPERS];
    int n_ = 0, parts_ = 1;
    char *d_ = nullptr;
    const char *s_ = nullptr;
    size_t bytes_ = 0;
    std::atomic<unsigned> job_{0};
    std::atomic<int> done_{0};
    std::atomic<bool> stop_{false};
};

}  // namespace lb3d
