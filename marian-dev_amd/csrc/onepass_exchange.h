// The abs-max of a tensor, from that of every workgroup's share of it, within a launch.
#pragma once

#include "int8_common.h"
#include "onepass_patience.h"
#include "quantize_common.h"

namespace marian_hip {

// The workgroups of a launch exchange their abs-max through the workspace, in one step:
//   * every workgroup stores (tag, abs-max bits) into its word of each of four copies - one instruction, 8 bytes at device
//     scope a lane, so tag and value arrive together;
//   * every workgroup polls all words of one copy (2 KB for 256 workgroups, four loads in flight a lane) and takes their maximum;
//     workgroups that start together have their words in different lines (0.1 us);
//   * nothing but these 8-byte words is handed over, so no fence is needed.
// Bound by trips to the memory side, the store's and a poll's, 1.2 us.  The first poll waits for a quarter of that: one that comes back
// unanswered costs a trip, and the 4096 lines that 256 workgroups ask for are in the way of the words and of the loads still under way
// (without the pause, with 512, 1024, 1536 and 2048 clocks of it: 64 x 1024 x 1024 through gemm_rows_kernel 5.7, 5.7, 5.4, 5.6, 5.7 us,
// 256 x 1024 x 1000 7.1, 6.9, 6.5, 6.8, 7.0, prepareA of 4096 x 1024 7.2, 7.0, 6.3, 6.2, 6.4; a wave of its own for the polls, without
// loads in front of them, is no better).  The form before had four trips, groups of 16 whose first workgroup answered for them: 6.6, 7.8 and
// 7.5 us.  These are of gemm_rows_kernel as it asked for all its operands first; it asks for their bulk between its words and the first poll now, which
// takes the pause's place (the launches alone, under the profiler: 5.6 and 8.1 us with the pause, 5.4 and 7.1 so).  Copies, a launch that does nothing else,
// without the pause: 1, 2, 4, 8 and 16 of them 3.8, 3.6, 3.4, 3.4 and 3.5 us, 4.5 in four trips.
// The tag is a host nonce, another for every launch; words left by an earlier launch never match, whatever the workspace
// held before its first use.  A launch that is recorded into a graph repeats its nonce with every replay, so there a generation word that
// lives in the workspace and that workgroup 0 advances at the end of every replay is added to it (0.2 us: gen_word is null elsewhere).
// Every wait is bounded, and a workgroup's waits together are (onepass_patience.h): one that runs out of patience (the
// device was shared and not all workgroups were resident) takes the abs-max over the whole input itself - the
// result is the same -, and the launch still ends.
__device__ __forceinline__ unsigned long long onepass_word(unsigned tag, float v) {
  return ((unsigned long long)tag << 32) | (unsigned long long)__float_as_uint(v);
}
// In two parts, between which a workgroup may ask for what it needs next.  g: this workgroup of G <= 256, m: the abs-max of its values (in
// every thread), nonce: this launch's; gen: the generation word as it was (0 without one).
struct OnepassExchange {
  unsigned long long* words;
  unsigned tag;
  int g, G;
  __device__ __forceinline__ OnepassExchange(int g, unsigned nonce, unsigned gen, unsigned long long* words, int G)
      : words(words), tag((nonce + gen) | 0x80000000u), g(g), G(G) {}   // (the tag is never 0: a cleared word does not match)
  __device__ __forceinline__ int shift() const { return G > 16 ? 28 - __builtin_clz(G - 1) : 0; }   // 1 << shift lines of 16 words: the fewest that hold G
  __device__ __forceinline__ unsigned long long* place() const {   // (lanes below kOnePassCopies)
    return words + ((int)threadIdx.x % kOnePassCopies) * kOnePassMaxGroups + ((g & ((1 << shift()) - 1)) * 16 + (g >> shift()));
  }
  __device__ __forceinline__ void publish(float m) const {
    if(threadIdx.x < kOnePassCopies) __hip_atomic_store(place(), onepass_word(tag, m), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  // scan: the abs-max of the whole input, by this workgroup alone.
  template <class Scan>
  __device__ __forceinline__ float collect(float m, unsigned gen, unsigned long long* gen_word, int polls, float* shared_max, Scan scan) const {
    const int tid = threadIdx.x;
    static_assert(kOnePassMaxGroups == 4 * kWave, "four words a lane");
    int polls_left = polls;   // (of the whole workgroup: only its first wave waits)
    if(tid < kWave) {
      const unsigned long long own = onepass_word(tag, m);
      const int lines = shift();
      const unsigned long long* const get = words + (g % kOnePassCopies) * kOnePassMaxGroups;
      auto word = [&](int i) __attribute__((always_inline)) {
        const int at = i * kWave + tid, from = (at % 16 << lines) + at / 16;   // (lanes past the words: one of theirs again)
        return i * kWave < 16 << lines ? __hip_atomic_load(get + (from < G && at < 16 << lines ? at : 0), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) : own;
      };
      auto tag_of = [](unsigned long long w) { return (unsigned)(w >> 32); };
      auto value_of = [](unsigned long long w) { return __uint_as_float((unsigned)w); };
      float v = 0.0f;
      bool found = false;
      for(; onepass_patience(polls_left); onepass_polled(polls_left)) {
        const unsigned long long w0 = word(0), w1 = word(1), w2 = word(2), w3 = word(3);
        v = fmaxf(fmaxf(value_of(w0), value_of(w1)), fmaxf(value_of(w2), value_of(w3)));
        found = __all(tag_of(w0) == tag && tag_of(w1) == tag && tag_of(w2) == tag && tag_of(w3) == tag);
        if(found) break;
        __builtin_amdgcn_s_sleep(1);
      }
      v = wave_max(v);
      if(gen_word) {
        // Words that went out behind the generation's end carry the next replay's tag.  Their workgroup never finds those of
        // workgroup 0, which ended before it read the generation, so it comes here without an answer and takes them back.
        if(!found && tid < kOnePassCopies) __hip_atomic_store(place(), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the next replay expects another tag; every workgroup of this one has read the generation by now, or will find its
        // words unanswered and help itself
        if(g == 0 && tid == 0) __hip_atomic_store(gen_word, (unsigned long long)(gen + 1u), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      if(tid == 0) *shared_max = found ? v : -1.0f;
    }
    __syncthreads();
    const float all = *shared_max;
    return all >= 0.0f ? all : scan();
  }
};
// Both, with the pause between them.
template <class Scan>
__device__ __forceinline__ float onepass_exchange(int g, float m, unsigned nonce, unsigned gen, unsigned long long* words,
                                                  unsigned long long* gen_word, int polls, int G, float* shared_max, Scan scan) {
  const OnepassExchange exchange(g, nonce, gen, words, G);
  exchange.publish(m);
  if(threadIdx.x < kWave) __builtin_amdgcn_s_sleep(16);   // (1024 clocks, see above)
  return exchange.collect(m, gen, gen_word, polls, shared_max, scan);
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
