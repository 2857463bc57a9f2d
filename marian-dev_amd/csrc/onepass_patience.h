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
// waits for 2 us.  Where its last workgroups have to wait for compute units that work on another stream holds - which may itself
// be waiting for compute units held here -, nobody knows how long that takes, so a workgroup waits for about as long as the way out
// takes, every workgroup reading the whole input at 6 TB/s between them: 32 us, and 0.12 us more for every thousand values.
// Two streams of 40 calls each at a time, us a call of both, median and mean: prepareA of 1024 x 1024 6.8 and 6.8 whatever the patience (up to 4 Mi
// values two launches fit a compute unit), 2050 x 4096 16.7 and 28 (with 20000 polls for every size 63), 4096 x 4096
// 33 and 47 (with 64 to 1000 polls 77 - 111, single turns of 40 calls 90 ms: the way out costs 3 ms there); an affine call of
// 200 x 2048 x 1048 16.8 and 17.7 (with 4000 polls 21).
__host__ __device__ __forceinline__ int onepass_polls(size_t values) { return 64 + (int)(values / 4096); }

}  // namespace marian_hip
