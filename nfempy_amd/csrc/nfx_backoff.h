// What the outcome of a cooperative launch means, and when a device that refused one is asked again. Host code.
#pragma once

#include <hip/hip_runtime_api.h>

#include <atomic>
#include <cstdint>

namespace nfx {

enum class GridLaunch {
  ran,
  busy,   // another process holds the device's cooperative launches (measured: this code, after 35-46 ms)
  no,     // the device does not have, or cannot give now, what the launch needs
  error,
};

inline GridLaunch grid_outcome(hipError_t e) {
  switch (e) {
    case hipSuccess:
      return GridLaunch::ran;
    case hipErrorIllegalState:
      return GridLaunch::busy;
    case hipErrorCooperativeLaunchTooLarge:
    case hipErrorLaunchOutOfResources:
    case hipErrorOutOfMemory:
    case hipErrorNotSupported:
      return GridLaunch::no;
    default:
      return GridLaunch::error;
  }
}

// Per device of the process: until when it is not asked (a device beyond the table is always asked).
struct GridBackoff {
  static constexpr int kDevices = 64;
  bool waits(int device, int64_t now) const {
    return device >= 0 && device < kDevices && until[device].load(std::memory_order_relaxed) > now;
  }
  void note(int device, int64_t now, int64_t pause) {
    if (device >= 0 && device < kDevices) until[device].store(now + pause, std::memory_order_relaxed);
  }
  std::atomic<int64_t> until[kDevices] = {};
};

}  // namespace nfx
