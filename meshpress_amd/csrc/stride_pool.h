// A bounded list of idle handles per device, shared by every thread of the
// process.  take() hands out one that is idle on the device; put() keeps one
// for the next taker, or returns false when `Keep` are idle there already:
// the caller then destroys it.  A handle is the taker's alone until put().
#pragma once

#include <cstddef>
#include <mutex>
#include <utility>
#include <vector>

namespace stride {

template <class Handle, std::size_t Keep>
class IdlePool {
 public:
  bool take(int device, Handle& h) {
    std::lock_guard<std::mutex> lock(mu_);
    for (auto it = idle_.begin(); it != idle_.end(); ++it)
      if (it->first == device) {
        h = it->second;
        idle_.erase(it);
        return true;
      }
    return false;
  }
  bool put(int device, Handle h) {
    std::lock_guard<std::mutex> lock(mu_);
    std::size_t n = 0;
    for (const auto& x : idle_) n += x.first == device ? 1 : 0;
    if (n >= Keep) return false;
    idle_.emplace_back(device, h);
    return true;
  }

 private:
  std::mutex mu_;
  std::vector<std::pair<int, Handle>> idle_;
};

}  // namespace stride
