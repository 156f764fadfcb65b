// Host threads behind copies to pageable memory (host_copy.hip).
#pragma once

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace ibfs {

// Host threads that copy the parts of one transfer, each thread its slice of
// every part.  They are woken once per transfer.  In a short one they then poll
// for the next part (a wake-up of eight sleeping threads costs about as much as
// copying 8 MB), but for SPIN_US at most, then they sleep; in a long one, and
// between transfers, they sleep at once.  They live as long as the process.
class CopyPool {
 public:
  static constexpr int THREADS = 8;
  static constexpr int SPIN_US = 1000;  // the DMA of a part of 16 MiB takes 300
  struct Part {
    char *dst;
    const char *src;
    size_t bytes;
    std::atomic<int> left{THREADS};
  };

  CopyPool() {
    for (int k = 0; k < THREADS; ++k) th_.emplace_back([this, k] { run(k); });
  }

  // Starts a transfer of n parts; part j is copied once ready(j + 1) was called.
  // spin: the threads poll for a part before they sleep.
  void begin(Part *parts, int n, bool spin) {
    std::lock_guard<std::mutex> lk(mu_);
    parts_ = parts;
    n_ = n;
    spin_ = spin;
    ready_.store(0);
    left_ = THREADS;
    ++gen_;
    go_.notify_all();
  }
  void ready(int n) {
    ready_.store(n);
    // a thread counts itself asleep before it looks at ready_ a last time
    if (asleep_.load() > 0) {
      std::lock_guard<std::mutex> lk(mu_);
      part_.notify_all();
    }
  }
  void wait_part(int j) {
    for (unsigned i = 1; parts_[j].left.load(std::memory_order_acquire) > 0; ++i)
      if ((i & 255) == 0) std::this_thread::yield();
  }
  // Ends the transfer (parts not yet ready are dropped): no thread touches
  // the parts afterwards.
  void end() {
    ready(-1);
    std::unique_lock<std::mutex> lk(mu_);
    done_.wait(lk, [this] { return left_ == 0; });
  }

 private:
  // Waits until part j is ready or the transfer has ended (< 0).
  int wait_ready(int j, bool spin) {
    int r = ready_.load();
    if (spin && r >= 0 && r <= j) {
      const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(SPIN_US);
      for (unsigned i = 1;; ++i) {
        r = ready_.load();
        if (r > j || r < 0) return r;
        if ((i & 255) == 0) {
          if (std::chrono::steady_clock::now() >= until) break;
          std::this_thread::yield();
        }
      }
    }
    if (r > j || r < 0) return r;
    std::unique_lock<std::mutex> lk(mu_);
    asleep_.fetch_add(1);
    part_.wait(lk, [&] { return (r = ready_.load()) > j || r < 0; });
    asleep_.fetch_sub(1);
    return r;
  }

  void run(int k) {
    uint64_t seen = 0;
    for (;;) {
      Part *p;
      int n;
      bool spin;
      {
        std::unique_lock<std::mutex> lk(mu_);
        go_.wait(lk, [&] { return gen_ != seen; });
        seen = gen_;
        p = parts_;
        n = n_;
        spin = spin_;
      }
      for (int j = 0; j < n; ++j) {
        if (wait_ready(j, spin) < 0) break;
        const size_t b = p[j].bytes;
        const size_t lo = b * (size_t)k / THREADS, hi = b * (size_t)(k + 1) / THREADS;
        if (hi > lo) std::memcpy(p[j].dst + lo, p[j].src + lo, hi - lo);
        p[j].left.fetch_sub(1, std::memory_order_release);
      }
      std::lock_guard<std::mutex> lk(mu_);
      if (--left_ == 0) done_.notify_one();
    }
  }

  std::vector<std::thread> th_;
  std::mutex mu_;
  std::condition_variable go_, part_, done_;
  Part *parts_ = nullptr;
  int n_ = 0;
  bool spin_ = false;
  std::atomic<int> ready_{0}, asleep_{0};
  int left_ = 0;
  uint64_t gen_ = 0;
};

}  // namespace ibfs
