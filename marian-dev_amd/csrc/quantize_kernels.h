// abs-max + int8 quantize kernels (activation prepareA and offline weight prepareB).
#pragma once

#include "int8_common.h"
#include "onepass_exchange.h"
#include "quantize_common.h"

namespace marian_hip {

// Pass 1: per-workgroup abs-max of n floats (n % 4 == 0) -> partials[blockIdx.x].
__global__ __launch_bounds__(kQuantThreads) void absmax_partial_kernel(
    const float* __restrict__ x, size_t n4, float* __restrict__ partials, int blocks) {
  __shared__ float red[kQuantThreads / kWave];
  const v4f* x4 = reinterpret_cast<const v4f*>(x);
  float m = 0.0f;
  size_t stride = (size_t)blocks * kQuantThreads;
  size_t i = (size_t)blockIdx.x * kQuantThreads + threadIdx.x;
  // four independent loads in flight per thread
  for(; i + 3 * stride < n4; i += 4 * stride) {
    v4f a = x4[i], b = x4[i + stride], c = x4[i + 2 * stride], d = x4[i + 3 * stride];
    m = abs4max(a, m); m = abs4max(b, m); m = abs4max(c, m); m = abs4max(d, m);
  }
  for(; i < n4; i += stride) m = abs4max(x4[i], m);
  m = block_max<kQuantThreads / kWave>(m, red);
  if(threadIdx.x == 0) partials[blockIdx.x] = m;
}

// Clears n floats (a kernel rather than a memset node, so callers may capture the call in a graph).
__global__ __launch_bounds__(kQuantThreads) void zero_floats_kernel(float* __restrict__ p, int n, int blocks) {
  for(int i = blockIdx.x * kQuantThreads + threadIdx.x; i < n; i += blocks * kQuantThreads) p[i] = 0.0f;
}

// Small activations: one workgroup computes abs-max and quantizes (one launch instead of two).
__global__ __launch_bounds__(kSingleBlockThreads) void prepare_a_single_block_kernel(
    const float* __restrict__ x, int n16, int8_t* __restrict__ out) {
  __shared__ float red[kSingleBlockThreads / kWave];
  const v4f* x4 = reinterpret_cast<const v4f*>(x);
  float m = 0.0f;
  // (eight loads in flight per thread; positions past the end are clamped - a repeated value does
  // not change a maximum)
  const int n4 = n16 * 4;
  for(int i = threadIdx.x; i < n4; i += 8 * kSingleBlockThreads) {
    v4f v[8];
#pragma unroll
    for(int u = 0; u < 8; ++u) v[u] = x4[min(i + u * kSingleBlockThreads, n4 - 1)];
#pragma unroll
    for(int u = 0; u < 8; ++u) m = abs4max(v[u], m);
  }
  m = block_max<kSingleBlockThreads / kWave>(m, red);
  const float qm = quant_mult_from_maxabs(m), by = quantizer(qm);
  uint4* o16 = reinterpret_cast<uint4*>(out);
  for(int i = threadIdx.x; i < n16; i += kSingleBlockThreads) {
    v4f a = x4[4 * i], b = x4[4 * i + 1], c = x4[4 * i + 2], d = x4[4 * i + 3];
    uint4 q;
    q.x = quantize_pack4(a, by);
    q.y = quantize_pack4(b, by);
    q.z = quantize_pack4(c, by);
    q.w = quantize_pack4(d, by);
    o16[i] = q;
  }
  if(threadIdx.x == 0) *reinterpret_cast<float*>(out + (size_t)n16 * 16) = qm;
}

// ---- prepareA in one pass over the input ----------------------------------------------------
// The two-pass form reads the fp32 input twice (abs-max, then quantize); at encoder sizes the
// second read costs as much as the first (67 MB: 14 us each, the memory-side cache does not help).
// Here the input stays in registers between the two steps: at most one workgroup of 1024 threads
// per CU, each thread holding SETS x 16 values, so 256 CUs hold up to 16.7 M values (4096 x 4096).
// In between, the workgroups exchange their abs-max (onepass_exchange.h).
template <int SETS>
__global__ __launch_bounds__(1024) void prepare_a_onepass_kernel(const float* __restrict__ x, unsigned n16,
                                                                 int8_t* __restrict__ out,
                                                                 unsigned long long* words,
                                                                 unsigned long long* gen_word,
                                                                 unsigned nonce, int polls, int groups) {
  __shared__ float red[1024 / kWave];
  __shared__ float shared_max;
  __shared__ __attribute__((aligned(16))) uint32_t turn[1024 * 4];   // 16 bytes per thread
  const int tid = threadIdx.x, quad = tid / 4, qlane = tid % 4;
  const int G = groups, g = blockIdx.x;
  // (one wave per workgroup asks for the generation: every access to the word is served by the
  // same memory channel, one after the other)
  unsigned gen = 0;
  if(tid < kWave && gen_word) gen = (unsigned)__hip_atomic_load(gen_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  // set j of this workgroup: quads (g * SETS + j) * 256 .. + 255, a quad = four consecutive 16-value
  // groups (256 contiguous bytes); load e brings lane i of the quad the i-th four values of group e
  v4f vals[SETS][4];
  bool live[SETS];
  float m = 0.0f;
#pragma unroll
  for(int j = 0; j < SETS; ++j) {
    const unsigned q = (unsigned)(g * SETS + j) * 256u + (unsigned)quad;
    live[j] = 4u * q < n16;   // (n16 is a multiple of four: K % 64 == 0)
    const unsigned qc = live[j] ? q : 0u;
    const char* src = reinterpret_cast<const char*>(x) + (size_t)qc * 256 + qlane * 16;
#pragma unroll
    for(int e = 0; e < 4; ++e) vals[j][e] = *reinterpret_cast<const v4f*>(src + e * 64);
  }
#pragma unroll
  for(int j = 0; j < SETS; ++j)
    if(live[j]) {
#pragma unroll
      for(int e = 0; e < 4; ++e) m = abs4max(vals[j][e], m);
    }
  m = block_max<1024 / kWave>(m, red);
  float amax = m;
  if(G > 1)
    amax = onepass_exchange((int)blockIdx.x, m, nonce, gen, words, gen_word, polls, G, &shared_max,
                                  [&] { return onepass_scan<1024>(x, (size_t)n16 * 4, red); });
  const float qm = quant_mult_from_maxabs(amax), by = quantizer(qm);
#pragma unroll
  for(int j = 0; j < SETS; ++j) {
    if(!live[j]) continue;
    const unsigned q = (unsigned)(g * SETS + j) * 256u + (unsigned)quad;
    // Lane i of the quad holds dword i of the quad's four 16-byte outputs; through LDS (the four
    // lanes sit in one wave, whose LDS operations execute in order) it picks up the four dwords of
    // output i, so that a wave stores 1 KB of contiguous bytes, 16 per lane.
#pragma unroll
    for(int e = 0; e < 4; ++e)
      turn[(quad * 4 + e) * 4 + qlane] = quantize_pack4(vals[j][e], by);
    const uint4 w = *reinterpret_cast<const uint4*>(&turn[(quad * 4 + qlane) * 4]);
    *reinterpret_cast<uint4*>(reinterpret_cast<char*>(out) + (size_t)q * 64 + qlane * 16) = w;
  }
  if(g == 0 && tid == 0) *reinterpret_cast<float*>(out + (size_t)n16 * 16) = qm;
}

// Pass 2 of prepareA, and quantization alone where the abs-max is known (left in `partials` by the kernel that
// produced x): the memory access pattern of the one-pass kernel above - a quad of lanes reads 64
// contiguous bytes per load, four loads in flight per thread (eight while the next set is on its
// way), the packed bytes take a turn through LDS so that a wave stores 1 KB of contiguous output -
// without its exchange.  A set = THREADS / 4 quads = 64 THREADS bytes of input per workgroup and step.
// n_partials: 1 .. kAbsmaxSlots, all requested at once, behind the first values.
template <int THREADS>
__global__ __launch_bounds__(THREADS) void quantize_a_wide_kernel(const float* __restrict__ x, unsigned n16,
                                                                  const float* __restrict__ partials, int n_partials,
                                                                  int8_t* __restrict__ out, unsigned blocks) {
  __shared__ float red[THREADS / kWave];
  __shared__ __attribute__((aligned(16))) uint32_t turn[THREADS * 4];   // 16 bytes per thread
  const int tid = threadIdx.x, quad = tid / 4, qlane = tid % 4;
  constexpr unsigned kQuads = THREADS / 4;
  const unsigned n_sets = (n16 / 4 + kQuads - 1) / kQuads;
  auto load_set = [&](unsigned set, v4f (&v)[4]) {
    const unsigned q = set * kQuads + (unsigned)quad;
    const unsigned qc = 4u * q < n16 ? q : 0u;   // (n16 is a multiple of four: whole quads)
    const char* src = reinterpret_cast<const char*>(x) + (size_t)qc * 256 + qlane * 16;
#pragma unroll
    for(int e = 0; e < 4; ++e) v[e] = *reinterpret_cast<const v4f*>(src + e * 64);
  };
  // the first loads are on their way while the partials are reduced
  unsigned set = blockIdx.x;
  v4f vals[4];
  if(set < n_sets) load_set(set, vals);
  float pm[kAbsmaxSlots / THREADS], m = 0.0f;
#pragma unroll
  for(int i = 0; i < kAbsmaxSlots / THREADS; ++i) pm[i] = partials[min(tid + i * THREADS, n_partials - 1)];
#pragma unroll
  for(int i = 0; i < kAbsmaxSlots / THREADS; ++i) m = fmaxf(m, pm[i]);
  m = block_max<THREADS / kWave>(m, red);
  const float qm = quant_mult_from_maxabs(m), by = quantizer(qm);
  for(; set < n_sets; set += blocks) {
    v4f cur[4];
#pragma unroll
    for(int e = 0; e < 4; ++e) cur[e] = vals[e];
    if(set + blocks < n_sets) load_set(set + blocks, vals);
    const unsigned q = set * kQuads + (unsigned)quad;
    if(4u * q < n16) {
      // (the four lanes of a quad sit in one wave, whose LDS operations execute in order)
#pragma unroll
      for(int e = 0; e < 4; ++e)
        turn[(quad * 4 + e) * 4 + qlane] = quantize_pack4(cur[e], by);
      const uint4 w = *reinterpret_cast<const uint4*>(&turn[(quad * 4 + qlane) * 4]);
      *reinterpret_cast<uint4*>(reinterpret_cast<char*>(out) + (size_t)q * 64 + qlane * 16) = w;
    }
  }
  if(blockIdx.x == 0 && tid == 0) *reinterpret_cast<float*>(out + (size_t)n16 * 16) = qm;
}

// prepareB: W fp32 [K x N] -> K-blocked int8 payload of the quantized transpose + tail, in two parts that the kernels below
// share.  256 threads transpose a 64(k) x 64(n) tile through LDS: a thread reads four columns of four k rows, sixteen threads 256 bytes of a
// row (a load takes the CU's address unit sixteen clocks whatever its width: a column of sixteen rows to a thread, four times the loads,
// made 1024 x 1024 take 4.35 us, now 4.07; 1024 x 4096 7.7 and 7.75), writes are 16-byte chunks of K values, the columns of a K sub-step side by side.
// thread: 0 .. 255 of them.
__device__ __forceinline__ void load_b_tile(const float* __restrict__ W, int K, int N, int n0, int k0, int thread, v4f (&v)[4]) {
  // (K % 64 == 0: the k rows of a tile are all inside; columns past N read the last four, N % 8 == 0, and are not written)
  const float* w = W + (size_t)(k0 + thread / 16 * 4) * N + min(n0 + thread % 16 * 4, N - 4);
#pragma unroll
  for(int k = 0; k < 4; ++k) v[k] = *reinterpret_cast<const v4f*>(w + (size_t)k * N);
}
// tile: [n][k / 4] as packed dwords, 17 dwords per row: the 64 lanes of a wave hit every bank
// twice, the minimum for 64 lanes on 32 banks.  Holds a barrier: every thread of the workgroup calls it.
__device__ __forceinline__ void store_b_tile(const v4f (&v)[4], float qm, uint32_t (*tile)[17], int K, int N, int n0, int k0,
                                             int thread, bool live, int8_t* __restrict__ out) {
  const float by = quantizer(qm);
#pragma unroll
  for(int e = 0; e < 4; ++e)   // four consecutive k of a column: one packed dword
    tile[thread % 16 * 4 + e][thread / 16] = quantize_pack4(v4f{v[0][e], v[1][e], v[2][e], v[3][e]}, by);
  __syncthreads();
  // 64 columns (n) x four 16-byte chunks (k): two neighbouring threads write the two halves of a
  // column's sub-step, a wave 32 columns of one sub-step (1 KB of consecutive memory)
  const int rn = (thread / 2) % 64, ck = (thread / 128) * 32 + (thread % 2) * 16;
  const int n = n0 + rn, k = k0 + ck;
  if(live && n < N) {
    uint4 q;
    q.x = tile[rn][ck / 4]; q.y = tile[rn][ck / 4 + 1]; q.z = tile[rn][ck / 4 + 2]; q.w = tile[rn][ck / 4 + 3];
    *reinterpret_cast<uint4*>(out + b_chunk_offset(n, k / 16, N)) = q;
  }
}

// Pass 2 of prepareB (the abs-max is that of `partials`), one tile to a workgroup.
__global__ __launch_bounds__(256) void quantize_b_transpose_kernel(
    const float* __restrict__ W, int K, int N, const float* __restrict__ partials,
    int n_partials, int8_t* __restrict__ out) {
  __shared__ float red[256 / kWave];
  __shared__ uint32_t tile[64][17];
  const int n0 = blockIdx.x * 64, k0 = blockIdx.y * 64;
  // the tile and the partials are requested together
  v4f v[4];
  float pm[(kMaxPartials + 255) / 256];
  load_b_tile(W, K, N, n0, k0, threadIdx.x, v);
#pragma unroll
  for(int i = 0; i < (kMaxPartials + 255) / 256; ++i) pm[i] = partials[min((int)threadIdx.x + i * 256, n_partials - 1)];
  float m = 0.0f;
#pragma unroll
  for(int i = 0; i < (kMaxPartials + 255) / 256; ++i) m = fmaxf(m, pm[i]);
  m = block_max<256 / kWave>(m, red);
  const float qm = quant_mult_from_maxabs(m);
  store_b_tile(v, qm, tile, K, N, n0, k0, threadIdx.x, true, out);
  if(blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0)
    *reinterpret_cast<float*>(out + (size_t)K * N) = qm;
}

// prepareB in one launch, for matrices of up to four tiles a CU: TILES tiles to a workgroup of TILES x 256 threads, held in
// registers while the workgroups exchange their abs-max (as the one-pass form of prepareA).  The call is bound by its launches
// on the host: 1024 x 1024 in two of them 7.9 us, in one 5.7.
template <int TILES>
__global__ __launch_bounds__(TILES * 256) void prepare_b_onepass_kernel(const float* __restrict__ W, int K, int N,
                                                                        int8_t* __restrict__ out, unsigned long long* words,
                                                                        unsigned long long* gen_word, unsigned nonce,
                                                                        int polls, int groups, int tiles_n, int tiles) {
  __shared__ float red[TILES * 256 / kWave];
  __shared__ float shared_max;
  __shared__ uint32_t turn[TILES][64][17];
  const int tid = threadIdx.x, sub = tid / 256, thread = tid % 256;
  unsigned gen = 0;
  if(tid < kWave && gen_word) gen = (unsigned)__hip_atomic_load(gen_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const int wanted = __builtin_amdgcn_readfirstlane((int)blockIdx.x * TILES + sub);
  const bool live = wanted < tiles;
  const int t = live ? wanted : 0;   // (read again and not written: a repeated value does not change a maximum)
  const int n0 = (t % tiles_n) * 64, k0 = (t / tiles_n) * 64;
  v4f v[4];
  float m = 0.0f;
  load_b_tile(W, K, N, n0, k0, thread, v);
#pragma unroll
  for(int k = 0; k < 4; ++k) m = abs4max(v[k], m);
  m = block_max<TILES * 256 / kWave>(m, red);
  float amax = m;
  if(groups > 1)
    amax = onepass_exchange((int)blockIdx.x, m, nonce, gen, words, gen_word, polls, groups, &shared_max,
                            [&] { return onepass_scan<TILES * 256>(W, (size_t)K * N / 4, red); });
  const float qm = quant_mult_from_maxabs(amax);
  store_b_tile(v, qm, turn[sub], K, N, n0, k0, thread, live, out);
  if(blockIdx.x == 0 && tid == 0) *reinterpret_cast<float*>(out + (size_t)K * N) = qm;
}

// prepareBQuantizedTransposed: int8 W^T as plain rows [N x K] (the payload of a model file) -> the
// K-blocked layout.  One 16-byte chunk per thread, in output order (writes are consecutive).
__global__ __launch_bounds__(256) void retile_b_kernel(const int8_t* __restrict__ in, int K, int N,
                                                       int8_t* __restrict__ out) {
  const size_t chunks = (size_t)K * (size_t)N / 16;
  const size_t o = (size_t)blockIdx.x * 256 + threadIdx.x;
  if(o < chunks) {
    // chunk o of the output: sub-step o / (2 N), then column, half
    const int s = (int)(o / (2 * (size_t)N)), rem = (int)(o % (2 * (size_t)N));
    const int n = rem / 2, half = rem % 2;
    const uint4 v = *reinterpret_cast<const uint4*>(in + (size_t)n * K + (size_t)(2 * s + half) * 16);
    *reinterpret_cast<uint4*>(out + o * 16) = v;
  }
  if(o == 0) *reinterpret_cast<float*>(out + (size_t)K * N) = *reinterpret_cast<const float*>(in + (size_t)K * N);
}

}  // namespace marian_hip
