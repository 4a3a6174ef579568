// Dynamic LDS beyond 64 KB is allowed per kernel and device: asked for at a kernel's first launch on a device, not at each one.
#pragma once
#include <atomic>

#include "common.h"

// `devices`: bit d is set once device d has allowed `bytes` for the kernel (several threads may ask at once; the answer is the same)
inline hipError_t allow_lds(const void* kernel, size_t bytes, std::atomic<uint64_t>& devices) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  const uint64_t bit = dev < 64 ? (uint64_t)1 << dev : 0;
  if (devices.load(std::memory_order_acquire) & bit) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  if (e == hipSuccess) devices.fetch_or(bit, std::memory_order_release);
  return e;
}
