// What the launch rules ask about the device.
#pragma once
#include <hip/hip_runtime.h>

// Compute units of the current device (256 on MI355X), asked for once a device: the launch
// rules below were measured there and are stated in compute units, not as numbers of that chip.
static inline int compute_units() {
  constexpr int MAX_DEVICES = 64;
  static int cached[MAX_DEVICES];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX_DEVICES) {
    (void)hipGetLastError();
    return 256;
  }
  if (cached[dev] == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0) {
      (void)hipGetLastError();
      n = 256;
    }
    cached[dev] = n;
  }
  return cached[dev];
}
