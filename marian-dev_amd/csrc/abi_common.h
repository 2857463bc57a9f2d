// Shared by the translation units of the library: the per-thread HIP error behind
// marian_hip_last_hip_error(), and what launchers keep per device.
#pragma once

#include <hip/hip_runtime.h>

#include <array>
#include <atomic>
#include <cstdint>
#include <initializer_list>
#include <tuple>
#include <utility>

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

// Whether there is only one device: then nobody has to be asked which one a stream is of, or is current.
inline bool one_device() {
  static std::atomic<int> devices{0};
  int n = devices.load(std::memory_order_relaxed);
  if(n == 0 && hipGetDeviceCount(&n) == hipSuccess) devices.store(n, std::memory_order_relaxed);
  return n == 1;
}

// The device that work on `stream` runs on: of the default streams the current one.
inline int stream_device(hipStream_t stream, int* dev) {
  if(one_device()) {
    *dev = 0;
    return MARIAN_HIP_OK;
  }
  if(!stream || stream == hipStreamLegacy || stream == hipStreamPerThread) return current_device(dev);
  hipDevice_t d = 0;
  const hipError_t e = hipStreamGetDevice(stream, &d);
  if(e != hipSuccess) return record_hip_error((int)e);
  if(d < 0 || d >= kMaxDevices) return MARIAN_HIP_ERR_RANGE;
  *dev = d;
  return MARIAN_HIP_OK;
}

// Makes `dev` the thread's device until the end of the scope, if it is another one.
class OnDevice {
 public:
  explicit OnDevice(int dev) : status(MARIAN_HIP_OK) {
    if(one_device()) return;
    status = current_device(&before_);
    if(status != MARIAN_HIP_OK || before_ == dev) return;
    const hipError_t e = hipSetDevice(dev);
    if(e != hipSuccess) status = record_hip_error((int)e);
    else moved_ = true;
  }
  ~OnDevice() { if(moved_) (void)hipSetDevice(before_); }
  OnDevice(const OnDevice&) = delete;
  OnDevice& operator=(const OnDevice&) = delete;
  int status;

 private:
  int before_ = 0;
  bool moved_ = false;
};

// The status of a launch that the runtime refused: the error is this call's, and not left for the next one that asks for the last.
inline int refused_launch(hipError_t e) {
  (void)hipGetLastError();
  return record_hip_error((int)e);
}

// Launches KERNEL: its function on the stream's device is looked up once and kept, which spares the host 0.17 us
// of 2.51 a launch (the runtime's table of kernels, and the launch configuration that <<<>>> hands over by a stack; eight arguments, batches
// of 24 launches).  Asking for the stream's device takes 0.07.
// What is kept belongs to the kernel itself, so that no place can find the function of another one.
template <auto KERNEL>
class Launcher;
template <typename... P, void (*KERNEL)(P...)>
class Launcher<KERNEL> {
 public:
  template <typename... A>
  static int launch(dim3 grid, dim3 block, size_t lds, hipStream_t st, const A&... given) {
    int dev = 0;
    const int status = stream_device(st, &dev);
    if(status != MARIAN_HIP_OK) return status;
    const OnDevice on(dev);   // (a symbol's function is that of the thread's device)
    if(on.status != MARIAN_HIP_OK) return on.status;
    hipFunction_t f = function_[dev].load(std::memory_order_acquire);
    if(!f) {
      const hipError_t e = hipGetFuncBySymbol(&f, reinterpret_cast<const void*>(KERNEL));
      if(e != hipSuccess) return refused_launch(e);
      function_[dev].store(f, std::memory_order_release);   // (every thread finds the same function)
    }
    std::tuple<P...> values(static_cast<P>(given)...);
    return launch(f, grid, block, lds, st, values, std::index_sequence_for<P...>());
  }

 private:
  template <typename Values, size_t... I>
  static int launch(hipFunction_t f, dim3 grid, dim3 block, size_t lds, hipStream_t st, Values& values, std::index_sequence<I...>) {
    void* arguments[] = {&std::get<I>(values)...};
    const hipError_t e = hipModuleLaunchKernel(f, grid.x, grid.y, grid.z, block.x, block.y, block.z, (unsigned)lds, st, arguments, nullptr);
    return e == hipSuccess ? MARIAN_HIP_OK : refused_launch(e);
  }
  inline static std::array<std::atomic<hipFunction_t>, kMaxDevices> function_{};
};
// Leaves the calling function with the status of a launch that failed.  (KERNEL: a constant; of several template arguments: in parentheses)
#define MH_LAUNCH(KERNEL, ...)                                                       \
  do {                                                                               \
    const int launch_status_ = marian_hip::Launcher<KERNEL>::launch(__VA_ARGS__);    \
    if(launch_status_ != MARIAN_HIP_OK) return launch_status_;                       \
  } while(0)

// A piece of device memory (p null: none).
struct Span {
  const void* p;
  int64_t bytes;
};

// Every workgroup of a launch that joins several steps reads the inputs of the first one, and the workgroups
// write the outputs of the last one as they finish: where the two share memory the launch races, though the
// steps on their own, one after the other on a stream, do not.
inline int apart(std::initializer_list<Span> written, std::initializer_list<Span> read) {
  for(const Span& w : written)
    for(const Span& r : read) {
      const uintptr_t a = reinterpret_cast<uintptr_t>(w.p), b = reinterpret_cast<uintptr_t>(r.p);
      if(w.p && r.p && a < b + (uintptr_t)r.bytes && b < a + (uintptr_t)w.bytes) return MARIAN_HIP_ERR_ALIAS;
    }
  return MARIAN_HIP_OK;
}

// What the kernels that normalize their input ask of it: few, short rows, whole vectors, an output that no
// workgroup still reads.  (A: the M x K values the norm starts from.)
inline int norm_input_check(const marian_hip_norm_input* n, const float* A, int64_t M, int64_t K) {
  if(M > MARIAN_HIP_NORM_MAX_ROWS || K > MARIAN_HIP_NORM_MAX_COLS || K % 64 != 0) return MARIAN_HIP_ERR_SHAPE;
  if(!n->add || !n->gamma || !n->beta || !n->out) return MARIAN_HIP_ERR_NULL;
  for(const float* p : {n->add, n->gamma, n->beta, static_cast<const float*>(n->out)})
    if(reinterpret_cast<uintptr_t>(p) % 16 != 0) return MARIAN_HIP_ERR_ALIGN;
  const int64_t bytes = M * K * (int64_t)sizeof(float), row = K * (int64_t)sizeof(float);
  return apart({{n->out, bytes}}, {{A, bytes}, {n->add, bytes}, {n->gamma, row}, {n->beta, row}});
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
