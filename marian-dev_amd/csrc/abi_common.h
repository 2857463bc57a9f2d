// Shared by the translation units of the library: the per-thread HIP error behind
// marian_hip_last_hip_error(), and what launchers keep per device.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdint>
#include <initializer_list>

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

// What the kernels that normalize their input ask of it: few, short rows, whole vectors, an output that no
// workgroup still reads.  (A: the M x K values the norm starts from.)
inline int norm_input_check(const marian_hip_norm_input* n, const float* A, int64_t M, int64_t K) {
  if(M > MARIAN_HIP_NORM_MAX_ROWS || K > MARIAN_HIP_NORM_MAX_COLS || K % 64 != 0) return MARIAN_HIP_ERR_SHAPE;
  if(!n->add || !n->gamma || !n->beta || !n->out) return MARIAN_HIP_ERR_NULL;
  for(const float* p : {n->add, n->gamma, n->beta, static_cast<const float*>(n->out)})
    if(reinterpret_cast<uintptr_t>(p) % 16 != 0) return MARIAN_HIP_ERR_ALIGN;
  const uintptr_t out = reinterpret_cast<uintptr_t>(n->out), bytes = (uintptr_t)M * (uintptr_t)K * sizeof(float);
  for(const float* p : {A, n->add}) {
    const uintptr_t in = reinterpret_cast<uintptr_t>(p);
    if(in < out + bytes && out < in + bytes) return MARIAN_HIP_ERR_ALIAS;
  }
  return MARIAN_HIP_OK;
}

// Compute units of the current device (looked up once per device; 256 if the query fails).
inline int compute_units() {
  static std::atomic<int> cus[kMaxDevices];
  int dev = 0;
  if(hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return 256;
  int n = cus[dev].load(std::memory_order_relaxed);
  if(n > 0) return n;
  if(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
    n = 256;
  cus[dev].store(n, std::memory_order_relaxed);
  return n;
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
