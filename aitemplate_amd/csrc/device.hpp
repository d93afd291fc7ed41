// Host-side facts about the device that the launchers reckon with.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>

namespace aitamd {

// Compute units of a device, looked up once per device (256 where the device cannot be asked).  The GEMM
// launcher's grid and split-K factor, the instance choice and the choice of an attention form all use this one figure.
inline int device_cus(int dev) {
  constexpr int kSlots = 64;
  static std::atomic<int> cus[kSlots] = {};
  if (dev < 0) dev = 0;
  int v = cus[dev % kSlots].load(std::memory_order_relaxed);
  if (v == 0) {
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cus[dev % kSlots].store(v, std::memory_order_relaxed);
  }
  return v;
}
inline int current_device_cus() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) {
    (void)hipGetLastError();  // no device: the instance choice still answers, priced for a 256-CU part
    return 256;
  }
  return device_cus(dev);
}

}  // namespace aitamd
