// How the library launches kernels (marian-dev_amd/csrc/abi_common.h), against a runtime of this program's own: it has two
// devices, hands out a function per kernel and device, and notes what is launched.  Built and run by tests/test_launcher.py.
#include <cstdio>
#include <vector>

#include "abi_common.h"

using namespace marian_hip;

namespace {
struct Function {
  const void* kernel;
  int device;
};
struct Launch {
  const Function* function;
  int argument, current;   // current: the device the launch was made on
};
int g_current = 0, g_devices = 2, g_recorded = 0;
hipError_t g_refuse = hipSuccess, g_last = hipSuccess;
const hipStream_t kStreamOfOne = reinterpret_cast<hipStream_t>(0x1000);   // a stream of device 1 (the others: of device 0)
std::vector<Function*> g_functions;
std::vector<Launch> g_launches;
int g_failures = 0;

void expect(bool ok, const char* what) {
  if(ok) return;
  std::printf("FAIL: %s\n", what);
  ++g_failures;
}
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* dev) { *dev = g_current; return hipSuccess; }
hipError_t hipSetDevice(int dev) { g_current = dev; return hipSuccess; }
hipError_t hipGetDeviceCount(int* n) { *n = g_devices; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t st, hipDevice_t* dev) {
  if(!st || st == hipStreamLegacy || st == hipStreamPerThread) return hipErrorInvalidHandle;   // (of no device of their own)
  *dev = st == kStreamOfOne ? 1 : 0;
  return hipSuccess;
}
hipError_t hipGetFuncBySymbol(hipFunction_t* f, const void* symbol) {
  for(Function* known : g_functions)
    if(known->kernel == symbol && known->device == g_current) { *f = reinterpret_cast<hipFunction_t>(known); return hipSuccess; }
  g_functions.push_back(new Function{symbol, g_current});
  *f = reinterpret_cast<hipFunction_t>(g_functions.back());
  return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t,
                                 void** arguments, void**) {
  if(g_refuse != hipSuccess) {
    g_last = g_refuse;
    return g_refuse;
  }
  g_launches.push_back(Launch{reinterpret_cast<Function*>(f), *static_cast<int*>(arguments[0]), g_current});
  return hipSuccess;
}
hipError_t hipGetLastError() {   // the last error since it was asked for
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
hipError_t hipDeviceGetAttribute(int*, hipDeviceAttribute_t, int) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
}

namespace marian_hip {
int record_hip_error(int e) {
  g_recorded = e;
  return MARIAN_HIP_ERR_HIP;
}
}

namespace {
// two kernels of one type
template <bool NT>
void kernel(int) { g_failures += NT ? 100 : 200; }

template <auto KERNEL>
int launch_one(int argument, hipStream_t st) {
  MH_LAUNCH(KERNEL, dim3(1), dim3(64), 0, st, argument);
  return MARIAN_HIP_OK;
}
#ifdef KERNEL_BY_POINTER
// a place that launches whatever it is given: one kernel's function would be kept for the other
int launch_given(void (*given)(int), int argument, hipStream_t st) {
  MH_LAUNCH(given, dim3(1), dim3(64), 0, st, argument);
  return MARIAN_HIP_OK;
}
int launch(bool nt, int argument, hipStream_t st) { return nt ? launch_given(kernel<true>, argument, st) : launch_given(kernel<false>, argument, st); }
#else
int launch(bool nt, int argument, hipStream_t st) { return nt ? launch_one<kernel<true>>(argument, st) : launch_one<kernel<false>>(argument, st); }
#endif

void each_kernel_its_own() {
  g_launches.clear();
  for(int i = 0; i < 4; ++i) launch(i % 2 == 0, i, nullptr);
  expect(g_launches.size() == 4, "four launches");
  for(int i = 0; i < (int)g_launches.size(); ++i) {
    expect(g_launches[i].argument == i, "argument");
    expect(g_launches[i].function->kernel == reinterpret_cast<const void*>(i % 2 == 0 ? kernel<true> : kernel<false>), "kernel that was asked for");
  }
}

// The function is the one of the stream's device, whichever device is the thread's when it is looked up; the thread's stays.
template <int N>
void other(int) { g_failures += N; }
template <int N>
void device_of_the_stream(int first_current) {
  g_launches.clear();
  for(int current : {first_current, 1 - first_current})
    for(hipStream_t st : {kStreamOfOne, reinterpret_cast<hipStream_t>(0x2000)}) {
      g_current = current;
      expect(launch_one<other<N>>(0, st) == MARIAN_HIP_OK, "launch on a stream of a device");
      const int device = st == kStreamOfOne ? 1 : 0;
      expect(g_launches.back().function->device == device, "function of the stream's device");
      expect(g_launches.back().current == device, "launched with the stream's device current");
      expect(g_current == current, "the thread's device as it was");
    }
  // the default streams are of the device that is current
  for(int current : {0, 1})
    for(hipStream_t st : {hipStream_t(nullptr), hipStreamLegacy, hipStreamPerThread}) {
      g_current = current;
      expect(launch_one<other<N>>(0, st) == MARIAN_HIP_OK, "launch on a default stream");
      expect(g_launches.back().function->device == current && g_current == current, "function of the current device");
    }
  g_current = 0;
}

// A launch that the runtime refuses is reported by its own call, and by no later one.
template <int N>
void third(int) { g_failures += N; }
void refused_once() {
  g_refuse = hipErrorInvalidConfiguration;
  expect(launch_one<third<3>>(0, nullptr) == MARIAN_HIP_ERR_HIP && g_recorded == hipErrorInvalidConfiguration, "a refused launch is reported");
  g_refuse = hipSuccess;
  expect(launch_one<third<3>>(0, nullptr) == MARIAN_HIP_OK, "the next launch");
  expect(hipGetLastError() == hipSuccess, "no error left for the next call");
}
}  // namespace

int main() {
  each_kernel_its_own();
  device_of_the_stream<1>(0);
  device_of_the_stream<2>(1);
  refused_once();
  if(g_failures) return 1;
  std::printf("ok\n");
  return 0;
}
