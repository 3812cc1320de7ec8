// The LDS that a kernel's launches may ask for beyond what every launch has: raised to what the largest of them asked for, on
// each device by itself, and never lowered, whatever threads launch the kernel at the same time.
#pragma once

#include <cstddef>
#include <mutex>

namespace pyre {

class LdsLimit {
 public:
  static constexpr size_t kPlain = 64 * 1024;  // what a launch has without asking

  // Whether launches of `bytes` may go to `device`; set(bytes) asks the device and says whether it agrees.
  template <typename Set>
  bool allow(int device, size_t bytes, Set&& set) {
    if (bytes <= kPlain) return true;
    if (device < 0 || device >= kDevices) return false;
    const std::lock_guard<std::mutex> held(lock_);  // while the device is asked, or a smaller limit could be set behind a larger one
    if (bytes <= most_[device]) return true;
    if (!set(bytes)) return false;
    most_[device] = bytes;
    return true;
  }

 private:
  static constexpr int kDevices = 64;
  std::mutex lock_;
  size_t most_[kDevices] = {};
};

}  // namespace pyre
