// Shared by the translation units of the library: the per-thread HIP error behind
// marian_hip_last_hip_error(), and what launchers keep per device.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>

#include "../../include/marian_hip_int8.h"

namespace marian_hip {

// Remembers hipError_t `e` for the calling thread and returns MARIAN_HIP_ERR_HIP.
int record_hip_error(int e);

// Launches the abs-max pass over n floats (n % 4 == 0) on `stream`: partials (at least 4 KB of
// workspace) receives *n_partials values whose maximum is max|A|.  Returns a status code.
int launch_absmax_partials(const float* A, unsigned long n, float* partials, int* n_partials, void* stream);

constexpr int kMaxDevices = 64;

// The current device, as an index into the per-device caches below.
inline int current_device(int* dev) {
  const hipError_t e = hipGetDevice(dev);
  if(e != hipSuccess) return record_hip_error((int)e);
  if(*dev < 0 || *dev >= kMaxDevices) return MARIAN_HIP_ERR_RANGE;
  return MARIAN_HIP_OK;
}

// Raises a kernel's dynamic LDS limit, once per kernel and device (`done`: one bit per device).
template <typename KernelT>
int allow_lds(KernelT kernel, int bytes, std::atomic<uint64_t>& done) {
  if(bytes <= 48 * 1024) return MARIAN_HIP_OK;
  int dev = 0;
  int st = current_device(&dev);
  if(st != MARIAN_HIP_OK) return st;
  const uint64_t bit = 1ull << dev;
  if(done.load(std::memory_order_acquire) & bit) return MARIAN_HIP_OK;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if(e != hipSuccess) return record_hip_error((int)e);
  done.fetch_or(bit, std::memory_order_release);
  return MARIAN_HIP_OK;
}

}  // namespace marian_hip
