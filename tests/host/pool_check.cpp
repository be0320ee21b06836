// CopyPool (lulesh_copypool.h) under the thread sanitizer: several copiers at
// once, each pushing runs of pieces as field downloads do, a new pool after
// the last owner is gone, and never more threads than one pool's.
#include <dirent.h>

#include <chrono>
#include <cstdio>
#include <vector>

#include "lulesh_copypool.h"

using lulesh::CopyPool;

static int threads() {
  int n = 0;
  DIR *d = opendir("/proc/self/task");
  while (d && readdir(d)) ++n;
  if (d) closedir(d);
  return n - 2;  // . and ..
}
// a joined thread's entry may outlive the join for a moment
static bool threads_fall_to(int n) {
  for (int i = 0; i < 1000 && threads() > n; ++i) std::this_thread::sleep_for(std::chrono::milliseconds(1));
  return threads() <= n;
}

static bool copier(int seed, int rounds) {
  const size_t piece = 100, slot = 8 * piece;
  std::vector<char> src(4 * slot), dst(src.size());
  std::shared_ptr<CopyPool> pool = CopyPool::get();
  CopyPool::Queue q;
  std::atomic<int> left[4] = {};
  for (int r = 0; r < rounds; ++r) {
    for (size_t i = 0; i < src.size(); ++i) src[i] = (char)(seed + r + (int)i * 7);
    std::fill(dst.begin(), dst.end(), 0);
    pool->attach(q);
    for (int s = 0; s < 4; ++s)  // the last one ends inside a piece
      pool->push(q, dst.data() + s * slot, src.data() + s * slot, s == 3 ? slot - 37 : slot, piece, &left[s]);
    while (pool->help(q)) {
    }
    for (auto &l : left)
      while (l.load(std::memory_order_acquire)) std::this_thread::yield();
    pool->detach(q);
    for (size_t i = 0; i < src.size(); ++i)
      if (dst[i] != (i < src.size() - 37 ? src[i] : 0)) return false;
  }
  return true;
}

int main() {
  int bad = 0;
  std::thread([] {}).join();  // the sanitizer starts a thread of its own with the first
  std::this_thread::sleep_for(std::chrono::milliseconds(50));
  const int base = threads();
  for (int life = 0; life < 3; ++life) {
    std::vector<std::shared_ptr<CopyPool>> owners;
    for (int k = 0; k < 5; ++k) owners.push_back(CopyPool::get());
    if (threads() > base + CopyPool::kWorkers) ++bad;
    std::atomic<int> wrong{0};
    std::vector<std::thread> t;
    for (int k = 0; k < 4; ++k)
      t.emplace_back([&, k] {
        if (!copier(k, 50)) ++wrong;
      });
    for (auto &x : t) x.join();
    bad += wrong;
    owners.clear();
    if (!threads_fall_to(base)) ++bad;  // given back
  }
  std::printf("failures %d\n", bad);
  return bad != 0;
}
