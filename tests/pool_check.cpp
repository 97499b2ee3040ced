// Host check of the idle-handle pool (stride_pool.h): one handle serves calls
// that follow one another, a device's handles stay its own, no handle is with
// two takers at once, and no more than the bound stay idle.
//
//   pool_check
//
// Exit status: 0 ok, else the check that failed.
#include <atomic>
#include <thread>
#include <vector>

#include "../meshpress_amd/csrc/stride_pool.h"

using stride::IdlePool;

int main() {
  IdlePool<int, 4> pool;
  std::atomic<int> made{0};
  auto use = [&](int device, auto&& work) {
    int h = 0;
    if (!pool.take(device, h)) h = 100 * device + ++made;
    work(h);
    return pool.put(device, h);
  };
  for (int i = 0; i < 50; ++i)
    if (!use(0, [](int) {})) return 2;
  if (made != 1) return 3;
  bool own = true;
  for (int i = 0; i < 50; ++i) use(i % 3, [&](int h) { own &= h / 100 == i % 3; });
  if (made != 3 || !own) return 4;
  // eight threads: each handle with one taker at a time
  std::vector<std::atomic<int>> busy(16004);   // at most a handle a turn
  std::atomic<bool> shared{false};
  std::vector<std::thread> th;
  for (int t = 0; t < 8; ++t)
    th.emplace_back([&] {
      for (int i = 0; i < 2000; ++i)
        use(0, [&](int h) {
          if (busy[h]++) shared = true;
          --busy[h];
        });
    });
  for (auto& x : th) x.join();
  if (shared) return 5;
  int idle = 0;
  for (int h = 0; pool.take(0, h);) ++idle;
  return idle >= 1 && idle <= 4 ? 0 : 6;
}
