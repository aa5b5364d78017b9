// What the launch rules ask about the device, and what a launch asks of it once.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <mutex>

constexpr int MAX_DEVICES = 64;

// The current device, -1 where there is none to be had or it lies beyond the tables below.
static inline int current_device() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();
    return -1;
  }
  return dev >= 0 && dev < MAX_DEVICES ? dev : -1;
}

// Compute units of the current device (256 on MI355X), asked for once a device: the launch
// rules below were measured there and are stated in compute units, not as numbers of that chip.
static inline int compute_units() {
  static std::atomic<int> cached[MAX_DEVICES];        // (launches may come from several threads)
  const int dev = current_device();
  if (dev < 0) return 256;
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

// More dynamic LDS than a kernel gets unasked (64 KB) has to be asked for, for every device the kernel is
// launched on. One of these a kernel (static, in its launcher) remembers what each device has been asked for.
struct LdsAllowance {
  std::atomic<int> granted[MAX_DEVICES] = {};
  std::mutex asking;                                  // (a smaller size asked for meanwhile must not come last)

  bool ask(const void* kernel, size_t bytes) {
    const int dev = current_device();
    if (dev >= 0 && (int)bytes <= granted[dev].load(std::memory_order_relaxed)) return true;
    std::lock_guard<std::mutex> guard(asking);
    if (dev >= 0 && (int)bytes <= granted[dev].load(std::memory_order_relaxed)) return true;
    if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    if (dev >= 0) granted[dev].store((int)bytes, std::memory_order_relaxed);
    return true;
  }
};
