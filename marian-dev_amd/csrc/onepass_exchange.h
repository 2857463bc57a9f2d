// The abs-max of a tensor, from that of every workgroup's share of it, within a launch.
#pragma once

#include "int8_common.h"
#include "onepass_patience.h"
#include "quantize_common.h"

namespace marian_hip {

// The workgroups of a launch exchange their abs-max through the workspace, in groups of 16:
//   * every workgroup stores (tag, abs-max bits) into its arrival slot - one 8-byte store at device
//     scope, so tag and value arrive together;
//   * the first workgroup of a group polls its group's slots (one line), takes the maximum and publishes (tag, max) to its
//     word of every one of 16 boards (a line each);
//   * every workgroup polls the words of all groups on one board (16 pollers a board) and takes their maximum;
//   * nothing but these 8-byte words is handed over, so no fence is needed.
// (One workgroup that polls all slots and answers all made the launch 0.9 us longer: 4096 x 1024 8.1 against 7.25 us.)
// The tag is a host nonce plus a generation word that lives in the workspace and that workgroup 0
// advances at the end of every launch: words left by an earlier launch - or by an earlier replay of
// a recorded graph, which repeats the nonce - never match, whatever the workspace held before its
// first use.  Every wait is bounded, and a workgroup's waits together are (onepass_patience.h): one that runs out of patience (the
// device was shared and not all workgroups were resident) takes the abs-max over the whole input itself - the
// result is the same - clears its slot, and the launch still ends.
__device__ __forceinline__ unsigned long long onepass_word(unsigned tag, float v) {
  return ((unsigned long long)tag << 32) | (unsigned long long)__float_as_uint(v);
}
// g: this workgroup of G <= 256, m: the abs-max of its values (in every thread), tag: this launch's (in wave 0), gen: the generation
// word as it was (in thread 0).  scan: the abs-max of the whole input, by this workgroup alone.
template <int THREADS, class Scan>
__device__ __forceinline__ float onepass_exchange(int g, float m, unsigned gen, unsigned tag, unsigned long long* slots,
                                                  unsigned long long* gen_word, unsigned long long* boards, int polls,
                                                  int G, float* red, float* shared_max, Scan scan) {
  const int tid = threadIdx.x;
  static_assert(kOnePassMaxGroups == kOnePassBoards * kOnePassBoards, "a group's slots and a board's words are polled by the same lanes");
  int polls_left = polls;   // (of the whole workgroup: only its first wave waits)
  // n words from p with this launch's tag, polled by the first lanes of wave 0: their maximum, in *found whether all came
  auto collect = [&](const unsigned long long* p, int n, bool* found) {
    float v = 0.0f;
    *found = false;
    for(; onepass_patience(polls_left); onepass_polled(polls_left)) {
      const unsigned long long w = __hip_atomic_load(p + min(tid, n - 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      v = __uint_as_float((unsigned)w);
      *found = __all((unsigned)(w >> 32) == tag);
      if(*found) break;
      __builtin_amdgcn_s_sleep(1);
    }
    return wave_max(v);
  };
  if(tid < kWave) {
    bool found = true;
    if(tid == 0) __hip_atomic_store(&slots[g], onepass_word(tag, m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool leads = g % kOnePassBoards == 0;
    if(leads) {
      const float v = collect(slots + g, min(kOnePassBoards, G - g), &found);
      if(found && tid < kOnePassBoards)
        __hip_atomic_store(&boards[tid * kOnePassBoardWords + g / kOnePassBoards], onepass_word(tag, v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    float v = 0.0f;
    if(found) {
      v = collect(boards + (g % kOnePassBoards) * kOnePassBoardWords, (G + kOnePassBoards - 1) / kOnePassBoards, &found);
      // A group's words that went out behind the generation's end (below) carry the next launch's tag; the words of
      // workgroup 0's group then never match, so they are taken back here.
      if(leads && !found && tid < kOnePassBoards)
        __hip_atomic_store(&boards[tid * kOnePassBoardWords + g / kOnePassBoards], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if(tid == 0) {
      // answered or not, this launch is done with the slot
      __hip_atomic_store(&slots[g], 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      // the next launch (or replay) expects another tag; every workgroup of this launch has read
      // the generation by now, or will find its words unanswered and help itself
      if(g == 0) __hip_atomic_store(gen_word, (unsigned long long)(gen + 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      *shared_max = found ? v : -1.0f;
    }
  }
  __syncthreads();
  const float all = *shared_max;
  return all >= 0.0f ? all : scan();
}
// Abs-max of n4 vectors by one workgroup (the way out of a wait that ran out).
template <int THREADS>
__device__ __forceinline__ float onepass_scan(const float* x, size_t n4, float* red) {
  const v4f* x4 = reinterpret_cast<const v4f*>(x);
  float m = 0.0f;
  for(size_t i = threadIdx.x; i < n4; i += THREADS) m = abs4max(x4[i], m);
  return block_max<THREADS / kWave>(m, red);
}

}  // namespace marian_hip
