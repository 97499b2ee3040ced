// Host check of the DPR4 writer's threads (write_dup, stride_host.cpp): the
// bytes do not depend on their number, and an allocation that fails, in a
// worker or at any point of the calling thread, reaches the caller as
// std::bad_alloc, after which the writer works as before.
//
//   write_check
//
// Prints how many failing allocations were met.  Exit status: 0 ok, 3 bytes
// differ, 4 a failed allocation was swallowed.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <thread>

static const std::thread::id kMain = std::this_thread::get_id();
static std::atomic<bool> g_fail_workers{false};
static std::atomic<long> g_main_left{-1};   // the calling thread's allocations until one fails; -1: none
static std::atomic<long> g_failed{0};

void* operator new(std::size_t n) {
  const bool here = std::this_thread::get_id() == kMain;
  if (here ? (g_main_left >= 0 && g_main_left-- == 0) : g_fail_workers.load()) {
    ++g_failed;
    throw std::bad_alloc();
  }
  void* p = std::malloc(n ? n : 1);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }

#include "../meshpress_amd/csrc/stride_host.cpp"

using namespace stride;

int main() {
  const int n_m = 300;   // meshlets of one triangle each
  Prep P;
  Residuals R;
  Header H{};
  P.n_t = n_m;
  std::vector<uint8_t> tagk;
  R.off.push_back(0);
  for (int m = 0; m < n_m; ++m) {
    Plan pl;
    pl.l2g = {0, 1, 2};
    pl.tris_local = {0, 1, 2};
    pl.strip_len = {1};
    pl.strip_tris = {0};
    P.plans.push_back(pl);
    P.walks.push_back({{0, 0, 0, 0, 0}, {1, 0, 0, 0, 0}, {2, 0, 0, 0, 0}});
    for (int d = 0; d < 3; ++d) {
      R.anchor.push_back(m + d);
      R.vals.push_back(m % 50 - 25);
      R.vals.push_back(7 * d - m % 11);
    }
    R.n_delta.push_back(2);
    R.n_para.push_back(0);
    R.off.push_back((int64_t)R.vals.size());
    for (int s = 0; s < 6; ++s) {
      tagk.push_back((uint8_t)(1 + (s + m) % 2));
      tagk.push_back((uint8_t)(m % 5));
    }
  }
  for (int d = 0; d < 3; ++d) H.g_bits[d] = 12;
  const std::vector<uint8_t> want = write_dup(P, R, H, tagk.data(), 1);
  for (int nt : {2, 3, 8, 64})
    if (write_dup(P, R, H, tagk.data(), nt) != want) return 3;
  // in the workers
  g_fail_workers = true;
  bool thrown = false;
  try {
    (void)write_dup(P, R, H, tagk.data(), 8);
  } catch (const std::bad_alloc&) {
    thrown = true;
  }
  g_fail_workers = false;
  if (!thrown) return 4;
  // at the calling thread's n-th allocation, until none is left to fail
  for (long n = 0;; ++n) {
    const long before = g_failed;
    std::vector<uint8_t> got;
    thrown = false;
    g_main_left = n;
    try {
      got = write_dup(P, R, H, tagk.data(), 8);
    } catch (const std::bad_alloc&) {
      thrown = true;
    }
    g_main_left = -1;
    const bool met = g_failed != before;
    // a thread that could not be started is no failure: its range runs here
    if (thrown ? !met : got != want) return thrown ? 4 : 3;
    if (!met) break;
  }
  std::printf("%ld\n", g_failed.load());
  return 0;
}
