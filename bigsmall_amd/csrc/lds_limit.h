// What a launch asks of the current device, once per device and safely from any
// number of host threads: a kernel's dynamic-LDS limit above the 64 KiB default,
// and the number of compute units.
#pragma once

#include "simt.h"
#include <stdint.h>

#include <atomic>

namespace bs_internal {

// Bit d of `done` records that `fn` was configured on device d. The attribute
// call is idempotent, so two threads racing on the first launch both set it;
// the mask only saves the call on later launches. Devices beyond 63 set it on
// every launch. A failure is left to the launch itself, which then reports
// the error through hipGetLastError.
inline void ensure_lds_limit(const void* fn, uint32_t bytes, std::atomic<uint64_t>& done) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) dev = -1;
  const uint64_t bit = (dev >= 0 && dev < 64) ? (1ull << dev) : 0ull;
  if (bit && (done.load(std::memory_order_acquire) & bit)) return;
  if (hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes) == hipSuccess && bit)
    done.fetch_or(bit, std::memory_order_acq_rel);
}

// Compute units of the current device, asked once per device (devices 0..63);
// 2^32-1 when unknown.
inline std::atomic<uint32_t> g_cus[64];
inline uint32_t device_cus() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64) return 0xFFFFFFFFu;
  uint32_t v = g_cus[dev].load(std::memory_order_relaxed);
  if (v == 0) {
    int n = 0;
    if (hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
      return 0xFFFFFFFFu;
    v = (uint32_t)n;
    g_cus[dev].store(v, std::memory_order_relaxed);
  }
  return v;
}

}  // namespace bs_internal
