// What the launch rules ask about the device.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>

// Compute units of the current device (256 on MI355X), asked for once a device: the launch
// rules below were measured there and are stated in compute units, not as numbers of that chip.
static inline int compute_units() {
  constexpr int MAX_DEVICES = 64;
  static std::atomic<int> cached[MAX_DEVICES];        // (launches may come from several threads)
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    (void)hipGetLastError();
    return 256;
  }
  int n = cached[dev].load(std::memory_order_relaxed);
  if (n == 0) {
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      (void)hipGetLastError();
      n = 256;
    }
    cached[dev].store(n, std::memory_order_relaxed);
  }
  return n;
}
