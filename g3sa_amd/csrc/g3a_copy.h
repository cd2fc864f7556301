// Copies between a caller's pageable memory and page-locked slots by several
// threads, in step with the DMA of the slots.
//
// What bounds a large upload or download is the copy: one thread moves 23 to 28
// GB/s between pageable and page-locked memory, the link 57.  Here the calling
// thread issues and awaits the transfers in order, and a few helpers copy, a
// chunk of 4 MB in eight pieces, so that the first and the last chunk are done
// quickly and a chunk's calls stay few (in chunks of 1 and 2 MB, or with six or
// eight helpers, it was slower).  250,000 reads of 150 bases: upload 1.65 ->
// 1.05 ms, names and qualities 2.17 -> 1.25 ms, 93 MB of records 3.9 -> 2.3 ms.
// The helpers belong to one context, sleep between transfers and are joined
// with it.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace g3a {

class CopyCrew {
 public:
  static constexpr int kSlots = 8, kHelpers = 4;
  static constexpr size_t kPieces = 8;  // a chunk is copied in so many pieces, each by whoever is free
  CopyCrew() = default;
  CopyCrew(const CopyCrew &) = delete;
  CopyCrew &operator=(const CopyCrew &) = delete;
  ~CopyCrew() {
    {
      std::lock_guard<std::mutex> l(m_);
      quit_ = true;
    }
    cv_.notify_all();
    for (auto &t : threads_) t.join();
  }
  // the helpers, started on first use; false when there is none
  bool ready() {
    if (threads_.empty() && !failed_) {
      try {
        for (int i = 0; i < kHelpers; ++i) threads_.emplace_back([this] { help(); });
      } catch (const std::exception &) {  // no thread, or no memory for one
        failed_ = threads_.empty();
      }
    }
    return !threads_.empty();
  }

  // `bytes` from user memory through the slots (slot(i): chunk bytes each):
  // a chunk is copied in, then issue(i, offset, size) starts its transfer and
  // wait(i) awaits it.  Returns the first error of issue or wait.
  template <class Slot, class Issue, class Wait>
  int in(const uint8_t *user, size_t bytes, size_t chunk, Slot slot, Issue issue, Wait wait) {
    Job j;
    auto copy = [&](size_t i, size_t at, size_t m) { std::memcpy(slot(i) + at, user + i * chunk + at, m); };
    start(j, bytes, chunk, copy, kSlots);
    int rc = 0;
    for (size_t i = 0; i < j.n && !rc; ++i) {
      j.await(i);
      rc = issue(i, i * chunk, j.size(i));
      // the slots whose transfers are done by now, half of them behind
      if (!rc && i >= kSlots / 2) {
        rc = wait(i - kSlots / 2);
        j.limit.store(i - kSlots / 2 + 1 + kSlots, std::memory_order_release);
      }
    }
    finish(j);
    return rc;
  }
  // and out: issue(i, ...) fills slot i, wait(i) awaits it, and it is copied out
  template <class Slot, class Issue, class Wait>
  int out(uint8_t *user, size_t bytes, size_t chunk, Slot slot, Issue issue, Wait wait) {
    Job j;
    auto copy = [&](size_t i, size_t at, size_t m) { std::memcpy(user + i * chunk + at, slot(i) + at, m); };
    start(j, bytes, chunk, copy, 0);
    int rc = 0;
    size_t sent = 0;
    for (; sent < j.n && sent < kSlots && !rc; ++sent) rc = issue(sent, sent * chunk, j.size(sent));
    for (size_t i = 0; i < j.n && !rc; ++i) {
      rc = wait(i);
      if (rc) break;
      j.limit.store(i + 1, std::memory_order_release);
      // keep half of the slots in flight: the oldest copied out by now
      if (sent < j.n && i >= kSlots / 2) {
        j.await(sent - kSlots);
        rc = issue(sent, sent * chunk, j.size(sent));
        ++sent;
      }
    }
    if (!rc)
      for (size_t i = j.n > kSlots ? j.n - kSlots : 0; i < j.n; ++i) j.await(i);
    finish(j);
    return rc;
  }

 private:
  struct Job {
    size_t n = 0, bytes = 0, chunk = 0;
    void *ctx = nullptr;
    void (*copy)(void *, size_t, size_t, size_t) = nullptr;
    std::atomic<size_t> next{0}, limit{0};
    std::atomic<size_t> done[kSlots];
    std::atomic<bool> over{false};
    size_t size(size_t i) const { return bytes - i * chunk < chunk ? bytes - i * chunk : chunk; }
    void await(size_t i) const {
      while (done[i % kSlots].load(std::memory_order_acquire) < (i / kSlots + 1) * kPieces) std::this_thread::yield();
    }
    void work() {
      while (!over.load(std::memory_order_acquire)) {
        size_t p = next.load(std::memory_order_relaxed);
        const size_t i = p / kPieces;
        if (i >= n) return;
        if (i >= limit.load(std::memory_order_acquire)) {
          std::this_thread::yield();
          continue;
        }
        if (!next.compare_exchange_weak(p, p + 1)) continue;
        const size_t m = size(i), per = (m + kPieces - 1) / kPieces, at = p % kPieces * per;
        if (at < m) copy(ctx, i, at, m - at < per ? m - at : per);
        done[i % kSlots].fetch_add(1, std::memory_order_release);
      }
    }
  };

  // copy lives on the caller's stack until finish()
  template <class C>
  void start(Job &j, size_t bytes, size_t chunk, C &copy, size_t limit) {
    j.ctx = &copy;
    j.copy = [](void *c, size_t i, size_t at, size_t m) { (*static_cast<C *>(c))(i, at, m); };
    j.n = (bytes + chunk - 1) / chunk;
    j.bytes = bytes;
    j.chunk = chunk;
    for (auto &d : j.done) d.store(0);
    j.limit.store(limit);
    {
      std::lock_guard<std::mutex> l(m_);
      job_ = &j;
      ++turn_;
    }
    cv_.notify_all();
  }
  // no helper is at the job after this
  void finish(Job &j) {
    j.over.store(true, std::memory_order_release);
    std::unique_lock<std::mutex> l(m_);
    job_ = nullptr;
    idle_.wait(l, [this] { return active_ == 0; });
  }
  void help() {
    uint64_t seen = 0;
    std::unique_lock<std::mutex> l(m_);
    for (;;) {
      cv_.wait(l, [&] { return quit_ || (job_ && turn_ != seen); });
      if (quit_) return;
      seen = turn_;
      Job *j = job_;
      ++active_;
      l.unlock();
      j->work();
      l.lock();
      if (--active_ == 0) idle_.notify_all();
    }
  }

  std::vector<std::thread> threads_;
  std::mutex m_;
  std::condition_variable cv_, idle_;
  Job *job_ = nullptr;
  uint64_t turn_ = 0;
  int active_ = 0;
  bool quit_ = false, failed_ = false;
};

}  // namespace g3a
