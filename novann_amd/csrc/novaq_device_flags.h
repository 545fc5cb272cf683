// What has been done once on each device: a flag a device, set and read by
// any thread.  Plain C++ (no HIP types) so that a host compiler can build it on
// its own.
#ifndef NOVAQ_DEVICE_FLAGS_H
#define NOVAQ_DEVICE_FLAGS_H

#include <atomic>
#include <cstdint>

namespace novaq {

// (devices past the 64th have no flag: theirs reads unset, so what it guards is
// done again, which is harmless)
class DeviceFlags {
 public:
  bool test(int device) const {
    return device >= 0 && device < 64 &&
           (bits_.load(std::memory_order_acquire) >> device & 1) != 0;
  }
  void set(int device) {
    if (device >= 0 && device < 64)
      bits_.fetch_or(std::uint64_t{1} << device, std::memory_order_release);
  }

 private:
  std::atomic<std::uint64_t> bits_{0};
};

}  // namespace novaq

#endif  // NOVAQ_DEVICE_FLAGS_H
