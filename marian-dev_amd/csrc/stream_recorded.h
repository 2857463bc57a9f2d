// Whether calls on a stream are recorded into a graph; plain host code, also for compilers other than hipcc.
#pragma once

#include <hip/hip_runtime_api.h>

namespace marian_hip {

// (A query that fails - of the default stream while a stream that waits for it is recorded, for one - leaves no error for a later
// launch to report: the call's own launch will tell.)
inline bool recorded(hipStream_t st) {
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if(hipStreamIsCapturing(st, &status) == hipSuccess) return status == hipStreamCaptureStatusActive;
  (void)hipGetLastError();
  return false;
}

}  // namespace marian_hip
