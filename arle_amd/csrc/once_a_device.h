// What a process does once for each of its GPUs.  Plain C++: nothing here needs a GPU.
#pragma once
#include <atomic>
#include <cstdint>

namespace arle {

class OnceADevice {
 public:
  // Whether it has been done on this device; devices past the 64th are never remembered.
  bool done(int device) const { return device >= 0 && device < 64 && (devices_.load(std::memory_order_acquire) >> device & 1u); }
  void mark(int device) {
    if (device >= 0 && device < 64) devices_.fetch_or(std::uint64_t{1} << device, std::memory_order_release);
  }

 private:
  std::atomic<std::uint64_t> devices_{0};
};

}  // namespace arle
