// Copies a large result out of two staging buffers with a few threads (host
// only; rtg_runtime.cpp: copy_out).
#pragma once
#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace rtg {

// Copies dst[0, bytes) from chunks that the main thread announces, chunk i
// lying in buffer i % 2; each chunk is split between the main thread and up to
// kHelpers helper threads (fewer where the process has fewer processors).
// While the chunks are still being computed the helpers make dst's pages
// present, which leaves its contents as they are, and then sleep until the
// first chunk; from there on they poll (a chunk takes about 0.1 ms).
class CopyTeam {
 public:
  static constexpr int kHelpers = 3;
  CopyTeam(char* d, size_t n, size_t c, const char* b0, const char* b1)
      : chunk(c),
        dst_(d),
        bytes_(n),
        buf_{b0, b1},
        parts_(1 + std::max(0, std::min(kHelpers, (int)std::thread::hardware_concurrency() - 1))) {
    try {
      threads_.reserve(parts_ - 1);
      for (size_t i = 1; i < parts_; ++i) threads_.emplace_back([this, i] { helper(i); });
    } catch (const std::exception&) {
      // no more threads to be had: the main thread takes their parts
    }
  }
  ~CopyTeam() {
    {
      std::lock_guard<std::mutex> g(mu_);
      stop_.store(true, std::memory_order_release);
    }
    cv_.notify_all();
    for (auto& t : threads_) t.join();
  }
  CopyTeam(const CopyTeam&) = delete;
  CopyTeam& operator=(const CopyTeam&) = delete;

  const size_t chunk;
  size_t count() const { return (bytes_ + chunk - 1) / chunk; }
  size_t size(size_t i) const { return std::min(chunk, bytes_ - i * chunk); }

  // Main thread, before the first chunk: makes its own part's pages present.
  void touch() { touch(0); }
  // Main thread: chunk i has arrived in its buffer; returns once it is in dst.
  void copy(size_t i) {
    if (i == 0) {
      std::lock_guard<std::mutex> g(mu_);
      ready_.store(1, std::memory_order_release);
    } else {
      ready_.store(i + 1, std::memory_order_release);
    }
    if (i == 0) cv_.notify_all();
    part(i, 0);
    for (size_t p = threads_.size() + 1; p < parts_; ++p) part(i, p);
    while (done_.load(std::memory_order_acquire) < (i + 1) * threads_.size()) std::this_thread::yield();
  }

 private:
  static constexpr size_t kPage = 4096;
  char* const dst_;
  const size_t bytes_;
  const char* const buf_[2];
  const size_t parts_;
  std::atomic<size_t> ready_{0}, done_{0};
  std::atomic<bool> stop_{false};
  std::mutex mu_;
  std::condition_variable cv_;
  std::vector<std::thread> threads_;

  // Part p of chunk i: its range of the chunk.
  void range(size_t i, size_t p, size_t* a, size_t* b) const {
    const size_t n = size(i), each = ((n + parts_ - 1) / parts_ + kPage - 1) / kPage * kPage;
    *a = std::min(n, p * each);
    *b = std::min(n, *a + each);
  }
  void part(size_t i, size_t p) {
    size_t a, b;
    range(i, p, &a, &b);
    memcpy(dst_ + i * chunk + a, buf_[i & 1] + a, b - a);
  }
  // A write to every page of part p of all chunks that changes nothing: an
  // atomic or with 0, which the compiler cannot see is 0.
  void touch(size_t p) {
    char zero = 0;
    asm volatile("" : "+r"(zero));
    for (size_t i = 0; i < count(); ++i) {
      size_t a, b;
      range(i, p, &a, &b);
      for (; a < b; a += kPage) __atomic_fetch_or(dst_ + i * chunk + a, zero, __ATOMIC_RELAXED);
    }
  }
  void helper(size_t p) {
    touch(p);
    {
      std::unique_lock<std::mutex> g(mu_);
      cv_.wait(g, [this] { return ready_.load(std::memory_order_relaxed) > 0 || stop_.load(std::memory_order_relaxed); });
    }
    for (size_t i = 0; i < count(); ++i) {
      while (ready_.load(std::memory_order_acquire) <= i) {
        if (stop_.load(std::memory_order_acquire)) return;
        std::this_thread::yield();
      }
      part(i, p);
      done_.fetch_add(1, std::memory_order_acq_rel);
    }
  }
};

}  // namespace rtg
