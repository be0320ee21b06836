// Copies to (and from) the host through pinned staging memory, one per
// context.
//
// A copy straight into pageable memory costs the runtime a pass of its own
// over the destination, page by page and on one thread: a fresh array's pages
// are not there yet, and 7 MB take 1.1 ms where the bus needs 0.15.  Here the
// device copies into pinned chunks and the process's few threads for that
// (lulesh_copypool.h) move them on, each meeting its own share of the page
// faults; a field of less than a chunk takes one copy and one wait.  The eleven state fields into fresh arrays, with
// the scalars the caller reads known on the host: s=16 500 -> 165 us, s=30 470
// -> 260, s=63 4.7 -> 2.4 ms, s=96 11.0 -> 4.7, s=192 63.6 -> 21.6.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <memory>
#include <mutex>
#include <thread>

#include "lulesh_copypool.h"

namespace lulesh {

class HostCopy {
 public:
  HostCopy() = default;
  HostCopy(const HostCopy &) = delete;
  HostCopy &operator=(const HostCopy &) = delete;
  ~HostCopy() {
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
  static constexpr int kSlots = 6;
  static_assert(kSlots * (int)(kChunk / kPiece) <= CopyPool::kPieces, "a queue holds what is in flight");
  std::mutex one_;  // threads that read one context's fields take turns
  char *pin_ = nullptr;
  size_t pinned_ = 0;  // bytes at pin_
  hipEvent_t ev_[kSlots] = {};
  std::atomic<int> busy_[kSlots] = {};  // pieces that still read the slot
  std::shared_ptr<CopyPool> pool_;      // from the first large field on
  CopyPool::Queue queue_;

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

  hipError_t fetch_chunks(hipStream_t st, char *dst, const char *src, size_t bytes) {
    hipError_t e = ready(kSlots * kChunk, kSlots);
    if (e != hipSuccess) return e;
    if (!pool_) pool_ = CopyPool::get();
    pool_->attach(queue_);
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
        pool_->push(queue_, dst + (size_t)landed * kChunk, slot(s), size(landed), kPiece, &busy_[s]);
        ++landed;
      } else if (!pool_->help(queue_)) {
        std::this_thread::yield();
      }
    }
    // no thread writes dst and no copy is under way once this returns
    while (pool_->help(queue_)) {
    }
    for (std::atomic<int> &b : busy_)
      while (b.load(std::memory_order_acquire)) std::this_thread::yield();
    pool_->detach(queue_);
    const hipError_t e2 = hipStreamSynchronize(st);
    return e != hipSuccess ? e : e2;
  }
};

}  // namespace lulesh
