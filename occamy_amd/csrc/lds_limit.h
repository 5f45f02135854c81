// More than 64 KiB of LDS per workgroup has to be asked for, once per kernel and device.
#pragma once
#include <hip/hip_runtime_api.h>
#include <stdint.h>

#include <atomic>

namespace dnnrt {

// The devices that a kernel's limit has been raised on (one per kernel, static): a bit for each of the first 64, any
// further one is asked for at every launch.  Two threads that both find the bit unset both ask, which is harmless.
struct LdsRaised {
  std::atomic<uint64_t> devices{0};
};

inline bool raise_lds(LdsRaised &raised, int device, const void *kernel, int bytes) {
  const uint64_t bit = device >= 0 && device < 64 ? (uint64_t)1 << device : 0;
  if (raised.devices.load(std::memory_order_acquire) & bit) return true;
  if (hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes) != hipSuccess) return false;
  raised.devices.fetch_or(bit, std::memory_order_release);
  return true;
}

}  // namespace dnnrt
