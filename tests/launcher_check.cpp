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
  int argument;
};
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
hipError_t hipGetDevice(int* dev) { *dev = 0; return hipSuccess; }
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* dev) { *dev = 0; return hipSuccess; }
hipError_t hipGetFuncBySymbol(hipFunction_t* f, const void* symbol) {
  for(Function* known : g_functions)
    if(known->kernel == symbol) { *f = reinterpret_cast<hipFunction_t>(known); return hipSuccess; }
  g_functions.push_back(new Function{symbol, 0});
  *f = reinterpret_cast<hipFunction_t>(g_functions.back());
  return hipSuccess;
}
hipError_t hipModuleLaunchKernel(hipFunction_t f, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, unsigned, hipStream_t,
                                 void** arguments, void**) {
  g_launches.push_back(Launch{reinterpret_cast<Function*>(f), *static_cast<int*>(arguments[0])});
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipDeviceGetAttribute(int*, hipDeviceAttribute_t, int) { return hipSuccess; }
hipError_t hipFuncSetAttribute(const void*, hipFuncAttribute, int) { return hipSuccess; }
}

namespace marian_hip {
int record_hip_error(int) { return MARIAN_HIP_ERR_HIP; }
}

namespace {
// two kernels of one type
template <bool NT>
void kernel(int) { g_failures += NT ? 100 : 200; }

#ifdef KERNEL_BY_POINTER
// a place that launches whatever it is given: one kernel's function would be kept for the other
int launch_given(void (*given)(int), int argument, hipStream_t st) {
  MH_LAUNCH(given, dim3(1), dim3(64), 0, st, argument);
  return MARIAN_HIP_OK;
}
int launch(bool nt, int argument, hipStream_t st) { return nt ? launch_given(kernel<true>, argument, st) : launch_given(kernel<false>, argument, st); }
#else
template <auto KERNEL>
int launch_one(int argument, hipStream_t st) {
  MH_LAUNCH(KERNEL, dim3(1), dim3(64), 0, st, argument);
  return MARIAN_HIP_OK;
}
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
}  // namespace

int main() {
  each_kernel_its_own();
  if(g_failures) return 1;
  std::printf("ok\n");
  return 0;
}
