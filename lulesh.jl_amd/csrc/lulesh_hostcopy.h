// Copies to (and from) the host through pinned staging memory, one per
// context.
//
// A copy straight into pageable memory costs the runtime a pass of its own
// over the destination, page by page and on one thread: a fresh array's pages
// are not there yet, and 7 MB take 1.1 ms where the bus needs 0.15.  Here the
// device copies into pinned chunks and a few threads move them on, each
// meeting its own share of the page faults; a field of less than a chunk
// takes one copy and one wait.  The eleven state fields into fresh arrays, with
// the scalars the caller reads known on the host: s=16 500 -> 165 us, s=30 470
// -> 260, s=63 4.7 -> 2.4 ms, s=96 11.0 -> 4.7, s=192 63.6 -> 21.6.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace lulesh {

class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy &) = delete;
  HostCopy &operator=(const HostCopy &) = delete;
  ~HostCopy() {
    {
      std::lock_guard<std::mutex> l(m_);
      stop_ = true;
    }
    cv_.notify_all();
    for (std::thread &w : workers_) w.join();
    for (hipEvent_t e : ev_)
      if (e) (void)hipEventDestroy(e);
    if (pin_) (void)hipHostFree(pin_);
  }

  // dst[0, bytes) = device src; on return the copy is done and `st` idle.
  hipError_t fetch(hipStream_t st, void *dst, const void *src, size_t bytes) {
    std::lock_guard<std::mutex> l(one_);
    if (bytes > kChunk) return fetch_chunks(st, (char *)dst, (const char *)src, bytes);
    hipError_t e = ready(bytes, 0);
    if (e == hipSuccess && bytes) e = hipMemcpyAsync(pin_, src, bytes, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e == hipSuccess && bytes) memcpy(dst, pin_, bytes);
    return e;
  }

  // device dst = src[0, bytes); on return the copy is done and `st` idle.
  // (Beyond a chunk the runtime's own copy does; below, it takes 60 us where
  // this takes 15.)
  hipError_t send(hipStream_t st, void *dst, const void *src, size_t bytes) {
    std::lock_guard<std::mutex> l(one_);
    const bool staged = bytes <= kChunk;
    hipError_t e = staged ? ready(bytes, 0) : hipSuccess;
    if (e == hipSuccess && staged && bytes) memcpy(pin_, src, bytes);
    if (e == hipSuccess && bytes) e = hipMemcpyAsync(dst, staged ? pin_ : src, bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    return e;
  }

  // f(v, stride, m), in order, for the next m values of every one of
  // `arrays` arrays of n values that follow one another on the device:
  // v + k * stride holds array k's.  Nothing but staging memory is written.
  template <class F>
  hipError_t stream(hipStream_t st, const double *src, int arrays, int64_t n, F f) {
    std::lock_guard<std::mutex> l(one_);
    const int64_t m = (int64_t)(kChunk / sizeof(double)), chunks = (n + m - 1) / m;
    if (arrays * n <= m) {
      hipError_t e = ready((size_t)(arrays * n) * sizeof(double), 0);
      if (e == hipSuccess && n > 0)
        e = hipMemcpyAsync(pin_, src, (size_t)(arrays * n) * sizeof(double), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e == hipSuccess) f((const double *)pin_, n, n);
      return e;
    }
    hipError_t e = ready((size_t)(2 * arrays) * kChunk, 2);
    auto ask = [&](int64_t k) {
      for (int a = 0; a < arrays && e == hipSuccess; ++a)
        e = hipMemcpyAsync(slot((int)(k & 1) * arrays + a), src + a * n + k * m,
                           (size_t)std::min(m, n - k * m) * sizeof(double), hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipEventRecord(ev_[k & 1], st);
    };
    if (e == hipSuccess && chunks > 0) ask(0);
    for (int64_t k = 0; k < chunks && e == hipSuccess; ++k) {
      if (k + 1 < chunks) ask(k + 1);
      if (e == hipSuccess) e = hipEventSynchronize(ev_[k & 1]);
      if (e == hipSuccess) f((const double *)slot((int)(k & 1) * arrays), m, std::min(m, n - k * m));
    }
    const hipError_t e2 = hipStreamSynchronize(st);
    return e != hipSuccess ? e : e2;
  }

 private:
  // A copy command costs the stream about 15 us whatever it moves (57 MB in
  // chunks of 128 KiB 7.3 ms, 256 KiB 4.3, 512 KiB 2.7, 1 MiB 2.05); the
  // threads share a chunk by pieces, so that a few chunks occupy them all (57
  // MB with 4, 6, 16 chunks in flight 2.17, 1.95, 1.92 ms; six are pinned in
  // the time of one download of 7 MB).
  static constexpr size_t kChunk = 1 << 20, kPiece = 1 << 17;
  static constexpr int kSlots = 6, kWorkers = 7, kJobs = kSlots * (int)(kChunk / kPiece);
  struct Job {
    char *dst;
    const char *src;
    size_t bytes;
    int slot;
  };
  std::mutex one_;  // threads that read one context's fields take turns
  char *pin_ = nullptr;
  size_t pinned_ = 0;  // bytes at pin_
  hipEvent_t ev_[kSlots] = {};
  std::atomic<int> busy_[kSlots] = {};  // jobs that still read the slot
  std::mutex m_;
  std::condition_variable cv_;
  Job jobs_[kJobs];  // ring of landed pieces
  int head_ = 0, count_ = 0;
  bool stop_ = false;
  std::vector<std::thread> workers_;

  char *slot(int i) { return pin_ + (size_t)i * kChunk; }

  // at least `bytes` of pinned memory, and `events` events
  hipError_t ready(size_t bytes, int events) {
    hipError_t e = hipSuccess;
    for (int i = 0; i < events && e == hipSuccess; ++i)
      if (!ev_[i]) e = hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming);
    if (e != hipSuccess || bytes <= pinned_) return e;
    size_t want = 1 << 16;  // (a power of two while it is less than a chunk)
    while (want < bytes && want < kChunk) want *= 2;
    want = std::max(want, bytes);
    if (pin_) (void)hipHostFree(pin_);
    pin_ = nullptr;
    pinned_ = 0;
    e = hipHostMalloc((void **)&pin_, want, hipHostMallocDefault);
    if (e != hipSuccess) pin_ = nullptr;
    else pinned_ = want;
    return e;
  }

  bool take(Job &j) {
    if (!count_) return false;
    j = jobs_[head_];
    head_ = (head_ + 1) % kJobs;
    --count_;
    return true;
  }
  void move(const Job &j) {
    memcpy(j.dst, j.src, j.bytes);
    busy_[j.slot].fetch_sub(1, std::memory_order_release);
  }
  bool help() {
    Job j;
    {
      std::lock_guard<std::mutex> l(m_);
      if (!take(j)) return false;
    }
    move(j);
    return true;
  }
  void work() {
    std::unique_lock<std::mutex> l(m_);
    for (;;) {
      Job j;
      if (take(j)) {
        l.unlock();
        move(j);
        l.lock();
      } else if (stop_) {
        return;
      } else {
        cv_.wait(l);
      }
    }
  }

  hipError_t fetch_chunks(hipStream_t st, char *dst, const char *src, size_t bytes) {
    hipError_t e = ready(kSlots * kChunk, kSlots);
    if (e != hipSuccess) return e;
    if (workers_.empty()) {
      const int n = std::min<int>(kWorkers, (int)std::thread::hardware_concurrency() - 1);
      try {
        for (int i = 0; i < n; ++i) workers_.emplace_back([this] { work(); });
      } catch (const std::system_error &) {
        // fewer threads: this one moves what they do not
      }
    }
    const int64_t chunks = (int64_t)((bytes + kChunk - 1) / kChunk);
    auto size = [&](int64_t k) { return std::min(kChunk, bytes - (size_t)k * kChunk); };
    int64_t asked = 0, landed = 0;
    while (landed < chunks && e == hipSuccess) {
      while (asked < chunks && asked - landed < kSlots && e == hipSuccess &&
             !busy_[asked % kSlots].load(std::memory_order_acquire)) {
        const int s = (int)(asked % kSlots);
        e = hipMemcpyAsync(slot(s), src + (size_t)asked * kChunk, size(asked), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(ev_[s], st);
        if (e == hipSuccess) ++asked;
      }
      if (e != hipSuccess) break;
      if (landed < asked) {
        const int s = (int)(landed % kSlots);
        e = hipEventSynchronize(ev_[s]);
        if (e != hipSuccess) break;
        const size_t all = size(landed);
        busy_[s].store((int)((all + kPiece - 1) / kPiece), std::memory_order_relaxed);
        {
          std::lock_guard<std::mutex> l(m_);
          for (size_t o = 0; o < all; o += kPiece, ++count_)
            jobs_[(head_ + count_) % kJobs] =
                Job{dst + (size_t)landed * kChunk + o, slot(s) + o, std::min(kPiece, all - o), s};
        }
        cv_.notify_all();
        ++landed;
      } else if (!help()) {
        std::this_thread::yield();
      }
    }
    // no thread writes dst and no copy is under way once this returns
    while (help()) {
    }
    for (std::atomic<int> &b : busy_)
      while (b.load(std::memory_order_acquire)) std::this_thread::yield();
    const hipError_t e2 = hipStreamSynchronize(st);
    return e != hipSuccess ? e : e2;
  }
};

}  // namespace lulesh
