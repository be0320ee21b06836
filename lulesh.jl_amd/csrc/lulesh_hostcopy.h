// Copies to (and from) the host through pinned staging memory, one per
// context.  What a small field takes is allocated with the context, in one
// piece with its scalars: pinned memory that the process has none of left over
// takes up to 350 us, a 2 MiB page of it, and a context of s=20 that was read
// twice paid it twice (its first two fields 327 and 339 us instead of 32 and
// 29).
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
    if (slots_) (void)hipHostFree(slots_);
    if (wide_) (void)hipHostFree(wide_);
  }

  // whether a field of `bytes` takes one copy through the staging memory
  static bool small(size_t bytes) { return bytes <= kChunk; }
  // staging for a context whose largest such field has `bytes`
  static size_t staging(size_t bytes) { return std::max(bytes, kLeast); }
  // pinned memory of that size, which the caller frees after its last call here
  void use(void *pinned, size_t bytes) {
    pin_ = (char *)pinned;
    pinned_ = bytes;
  }

  // dst[0, bytes) = device src; on return the copy is done and `st` idle.
  hipError_t fetch(hipStream_t st, void *dst, const void *src, size_t bytes) {
    std::lock_guard<std::mutex> l(one_);
    if (!small(bytes)) return fetch_chunks(st, (char *)dst, (const char *)src, bytes);
    char *to = nullptr;
    hipError_t e = room(bytes, &to);
    if (e == hipSuccess && bytes) e = hipMemcpyAsync(to, src, bytes, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e == hipSuccess && bytes) memcpy(dst, to, bytes);
    return e;
  }

  // device dst = src[0, bytes); on return the copy is done and `st` idle.
  // (Beyond a chunk the runtime's own copy does; below, it takes 60 us where
  // this takes 15.)
  hipError_t send(hipStream_t st, void *dst, const void *src, size_t bytes) {
    std::lock_guard<std::mutex> l(one_);
    const bool staged = small(bytes);
    char *to = nullptr;
    hipError_t e = staged ? room(bytes, &to) : hipSuccess;
    if (e == hipSuccess && staged && bytes) memcpy(to, src, bytes);
    if (e == hipSuccess && bytes) e = hipMemcpyAsync(dst, staged ? to : src, bytes, hipMemcpyHostToDevice, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    return e;
  }

  // f(v, stride, m), in order, for the next m values of every one of
  // `arrays` arrays (at most three) of n values that follow one another on the
  // device: v + k * stride holds array k's.  Nothing but staging memory is written.
  template <class F>
  hipError_t stream(hipStream_t st, const double *src, int arrays, int64_t n, F f) {
    std::lock_guard<std::mutex> l(one_);
    const int64_t m = (int64_t)(kChunk / sizeof(double)), chunks = (n + m - 1) / m;
    const size_t all = (size_t)(arrays * n) * sizeof(double);
    if (small(all)) {
      char *to = nullptr;
      hipError_t e = room(all, &to);
      if (e == hipSuccess && n > 0) e = hipMemcpyAsync(to, src, all, hipMemcpyDeviceToHost, st);
      if (e == hipSuccess) e = hipStreamSynchronize(st);
      if (e == hipSuccess) f((const double *)to, n, n);
      return e;
    }
    hipError_t e = ready();
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
  static constexpr size_t kChunk = 1 << 20, kPiece = 1 << 17, kLeast = 1 << 16;
  static constexpr int kSlots = 6;
  static_assert(kSlots * (int)(kChunk / kPiece) <= CopyPool::kPieces, "a queue holds what is in flight");
  std::mutex one_;  // threads that read one context's fields take turns
  char *pin_ = nullptr;    // the staging memory of small fields
  size_t pinned_ = 0;
  char *wide_ = nullptr;   // for what that does not hold, while there are no chunks
  size_t wide_bytes_ = 0;
  char *slots_ = nullptr;  // kSlots chunks
  hipEvent_t ev_[kSlots] = {};
  std::atomic<int> busy_[kSlots] = {};  // pieces that still read the slot
  std::shared_ptr<CopyPool> pool_;      // from the first large field on
  CopyPool::Queue queue_;

  char *slot(int i) { return slots_ + (size_t)i * kChunk; }

  // staging memory of at least `bytes`, at most a chunk
  hipError_t room(size_t bytes, char **to) {
    if (bytes > pinned_ && !slots_ && bytes > wide_bytes_) {
      if (wide_) (void)hipHostFree(wide_);
      wide_ = nullptr;
      wide_bytes_ = 0;
      const hipError_t e = hipHostMalloc((void **)&wide_, bytes, hipHostMallocDefault);
      if (e != hipSuccess) {
        wide_ = nullptr;
        return e;
      }
      wide_bytes_ = bytes;
    }
    *to = bytes <= pinned_ ? pin_ : slots_ ? slots_ : wide_;
    return hipSuccess;
  }

  // the chunks and their events
  hipError_t ready() {
    hipError_t e = hipSuccess;
    for (int i = 0; i < kSlots && e == hipSuccess; ++i)
      if (!ev_[i]) e = hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming);
    if (e != hipSuccess || slots_) return e;
    e = hipHostMalloc((void **)&slots_, kSlots * kChunk, hipHostMallocDefault);
    if (e != hipSuccess) slots_ = nullptr;
    return e;
  }

  hipError_t fetch_chunks(hipStream_t st, char *dst, const char *src, size_t bytes) {
    hipError_t e = ready();
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
