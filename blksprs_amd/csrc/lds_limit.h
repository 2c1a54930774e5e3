// The limit of dynamic LDS of a kernel (hipFuncAttributeMaxDynamicSharedMemorySize), raised on demand.  The attribute belongs
// to the code object that a device has loaded, so what was raised is remembered per device, and only once the call that
// raised it has succeeded.  Host code without HIP: the calls are handed in.
#pragma once
#include <atomic>
#include <mutex>

namespace bsa {

// One object per kernel (or per set of kernels raised together), as a function-local static next to the launch.
class LdsLimit {
 public:
  // set(): raises the kernel's limit on the current device, which is `device`, to `bytes`; 0 on success.  Not called
  // where the limit is that high already.  Calls of several threads come one after the other, so a smaller demand never
  // lowers a larger one.
  template <typename Set>
  int raise(int device, int bytes, Set set) {
    if (device < 0 || device >= kDevices) return set();
    if (raised_[device].load(std::memory_order_acquire) >= bytes) return 0;
    const std::lock_guard<std::mutex> lock(mutex_);
    if (raised_[device].load(std::memory_order_relaxed) >= bytes) return 0;
    if (const int rc = set()) return rc;
    raised_[device].store(bytes, std::memory_order_release);
    return 0;
  }

 private:
  static constexpr int kDevices = 64;
  std::atomic<int> raised_[kDevices]{};
  std::mutex mutex_;
};

}  // namespace bsa
