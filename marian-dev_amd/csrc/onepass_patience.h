// How long the workgroups of a launch wait for one another (onepass_exchange.h); plain functions, so that a CPU program can call them.
#pragma once

#include <stddef.h>

#if !defined(__HIPCC__)
#define __host__
#define __device__
#define __forceinline__ inline
#endif

namespace marian_hip {

// A workgroup's waits draw on one budget of polls.
__host__ __device__ __forceinline__ bool onepass_patience(int polls_left) { return polls_left > 0; }
__host__ __device__ __forceinline__ void onepass_polled(int& polls_left) { --polls_left; }

// Polls of a workgroup before it helps itself, each a memory round trip of about half a microsecond.  A launch that has the chip
// waits for 1.2 us.  Where its last workgroups have to wait for compute units that work on another stream holds - which may itself
// be waiting for compute units held here -, nobody knows how long that takes, so a workgroup waits for about as long as the way out
// takes, every workgroup reading the whole input at 6 TB/s between them: 32 us, and 0.12 us more for every thousand values.
// Two streams with 40 calls each behind an event, us a call of both: prepareA of 1024 x 1024 4.4, 2050 x 4096 42, 4096 x 4096 88 (up to 4 Mi values two
// launches fit a compute unit; with an exchange in four trips 5.0, 63 and 125), an affine call of 200 x 2048 x 1048 20 (19).  The patience was
// chosen with that older exchange and turns of 40 calls that did not start together, means: 2050 x 4096 28, with 20000 polls for every size
// 63; 4096 x 4096 47, with 64 to 1000 polls 77 - 111 and single turns of 90 ms.  On a stream that has half of the CUs prepareA of 2050 x 4096,
// which there waits in vain, takes 1.05 ms, 1.0 of it patience.
__host__ __device__ __forceinline__ int onepass_polls(size_t values) { return 64 + (int)(values / 4096); }

}  // namespace marian_hip
