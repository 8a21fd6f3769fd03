// once_per_device.hpp -- what has to be done once for a kernel on each device.
// Plain C++: checked on the CPU.
#pragma once

#include <mutex>
#include <set>
#include <utility>

namespace lbm {

class OncePerDevice {
  public:
    // Whether `what` is set up on `device`; f() sets it up (false: it could
    // not be, and is tried again the next time).
    template <class F>
    bool operator()(const void *what, int device, F &&f) {
        const std::lock_guard<std::mutex> lock(mutex_);
        if (done_.count({what, device})) return true;
        if (!f()) return false;
        done_.insert({what, device});
        return true;
    }

  private:
    std::mutex mutex_;
    std::set<std::pair<const void *, int>> done_;
};

}  // namespace lbm
