// One-time work per device.  A kernel's attributes (its limit of dynamic LDS) belong to the device that is current when
// they are set, and handles may be made on several devices and from several threads: the first caller on a device does
// the work while later ones of that device wait for it, a failure is reported and tried again by the next caller.
#pragma once

#include <mutex>

namespace xabe {

constexpr int kMaxDevices = 64;  // (ordinals past it: the work is done on every call)

class DeviceOnce {
 public:
  // `work` returns 0 when it is done; the return value is the caller's
  template <typename Work>
  int run(int device, Work work) {
    if (device < 0 || device >= kMaxDevices) return work();
    std::lock_guard<std::mutex> lock(mutex_);
    if (done_[device]) return 0;
    const int status = work();
    done_[device] = status == 0;
    return status;
  }

 private:
  std::mutex mutex_;
  bool done_[kMaxDevices] = {};
};

}  // namespace xabe
