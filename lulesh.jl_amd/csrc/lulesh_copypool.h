// Threads that copy pieces of host memory: one set for the whole process,
// shared by the contexts that move large fields to the host.  It is started
// by the first of them and joined when the last is destroyed.  (With a set to
// each context, every one that had read a large field held seven threads of
// its own until it was destroyed.)
#pragma once

#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <memory>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace lulesh {

class CopyPool {
 public:
  static constexpr int kWorkers = 7, kPieces = 48;
  struct Piece {
    char *dst;
    const char *src;
    size_t bytes;
    std::atomic<int> *left;  // counted down when the piece is copied
  };
  // What one copier has for the threads to do; at most kPieces at a time, and
  // its owner pushes and helps from one thread at a time.
  class Queue {
    friend class CopyPool;
    Piece pieces_[kPieces];
    int head_ = 0, count_ = 0;
    Queue *next_ = nullptr;
  };

  // the process's pool (kept by every copier that asked for it)
  static std::shared_ptr<CopyPool> get() {
    static std::mutex m;
    static std::weak_ptr<CopyPool> shared;
    std::lock_guard<std::mutex> l(m);
    std::shared_ptr<CopyPool> p = shared.lock();
    if (!p) {
      p = std::make_shared<CopyPool>();
      p->start();
      shared = p;
    }
    return p;
  }

  CopyPool() = default;
  CopyPool(const CopyPool &) = delete;
  CopyPool &operator=(const CopyPool &) = delete;
  ~CopyPool() {
    {
      std::lock_guard<std::mutex> l(m_);
      stop_ = true;
    }
    cv_.notify_all();
    for (std::thread &w : workers_) w.join();
  }

  void attach(Queue &q) {
    std::lock_guard<std::mutex> l(m_);
    q.next_ = queues_;
    queues_ = &q;
  }
  // (its owner has waited for its pieces)
  void detach(Queue &q) {
    std::lock_guard<std::mutex> l(m_);
    Queue **p = &queues_;
    while (*p != &q) p = &(*p)->next_;
    *p = q.next_;
    q.next_ = nullptr;
  }

  // dst[0, bytes) = src, in pieces of `piece` bytes
  void push(Queue &q, char *dst, const char *src, size_t bytes, size_t piece, std::atomic<int> *left) {
    left->store((int)((bytes + piece - 1) / piece), std::memory_order_relaxed);
    {
      std::lock_guard<std::mutex> l(m_);
      for (size_t o = 0; o < bytes; o += piece, ++q.count_)
        q.pieces_[(q.head_ + q.count_) % kPieces] = Piece{dst + o, src + o, std::min(piece, bytes - o), left};
    }
    cv_.notify_all();
  }

  // one of q's own pieces, by the calling thread; false: none is waiting
  bool help(Queue &q) {
    Piece p;
    {
      std::lock_guard<std::mutex> l(m_);
      if (!take(q, p)) return false;
    }
    copy(p);
    return true;
  }

 private:
  std::mutex m_;
  std::condition_variable cv_;
  Queue *queues_ = nullptr;
  bool stop_ = false;
  std::vector<std::thread> workers_;

  void start() {
    const int n = std::min<int>(kWorkers, (int)std::thread::hardware_concurrency() - 1);
    try {
      for (int i = 0; i < n; ++i) workers_.emplace_back([this] { work(); });
    } catch (const std::system_error &) {
      // fewer threads: the copiers move what they do not
    } catch (const std::bad_alloc &) {
    }
  }

  static bool take(Queue &q, Piece &p) {
    if (!q.count_) return false;
    p = q.pieces_[q.head_];
    q.head_ = (q.head_ + 1) % kPieces;
    --q.count_;
    return true;
  }
  static void copy(const Piece &p) {
    memcpy(p.dst, p.src, p.bytes);
    p.left->fetch_sub(1, std::memory_order_release);
  }
  void work() {
    std::unique_lock<std::mutex> l(m_);
    for (;;) {
      Piece p;
      Queue *q = queues_;
      while (q && !take(*q, p)) q = q->next_;
      if (q) {
        l.unlock();
        copy(p);
        l.lock();
      } else if (stop_) {
        return;
      } else {
        cv_.wait(l);
      }
    }
  }
};

}  // namespace lulesh
