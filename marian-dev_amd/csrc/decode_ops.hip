// Float32 operators between the int8 GEMMs of a transformer decode step: layer normalization
// (with the skip connection in front of it), softmax (with the attention mask in front of it),
// log-softmax, the 0213 transpose of the head split/join, and the batched attention products.
// Declarations and the reference code each entry point replaces: include/marian_hip_ops.h
//
// All of them are memory- or latency-bound at decode sizes (a few hundred KB per call), so the
// kernels are single-pass where the row fits in registers and use 64-lane wave reductions;
// nothing here needs LDS tiling or MFMA.
#include "../../include/marian_hip_ops.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <type_traits>

#include "../../include/marian_hip_int8.h"
#include "abi_common.h"
#include "attention_plan.h"
#include "attention_rows_kernel.h"
#include "int8_common.h"
#include "layer_norm_row.h"
#include "nbest_plan.h"
#include "quantize_common.h"

using namespace marian_hip;

namespace {

constexpr int64_t kMaxElemsOps = 2147483647LL;

// Maximum over the wave, the same value in all lanes (`t > v ? t : v` at every step): the same
// steps.
__device__ __forceinline__ float wave_maxf(float v) {
  auto pick = [](float t, float v) { return t > v ? t : v; };
  v = pick(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false)), v);
  v = pick(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false)), v);
  v = pick(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false)), v);
  v = pick(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, false)), v);
  v = pick(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false)), v);   // row_bcast:15
  v = pick(__builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, v), __builtin_bit_cast(int, v), 0x143, 0xC, 0xF, false)), v);   // row_bcast:31
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

// Reduction over the THREADS threads that share a row (64: one wave, no LDS; more: through LDS).
// red: one float per wave of the workgroup.
template <int THREADS, bool MAX>
__device__ __forceinline__ float row_reduce(float v, float* red) {
  v = MAX ? wave_maxf(v) : wave_sum(v);
  if(THREADS > 64) {
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    __syncthreads();
    if(lane == 0) red[wave] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for(int w = 1; w < THREADS / 64; ++w) r = MAX ? (red[w] > r ? red[w] : r) : r + red[w];
    v = r;
  }
  return v;
}

// The same for a `red` that nothing has read or written since the last workgroup barrier (a
// fresh array per reduction): no barrier in front.
template <int THREADS, bool MAX>
__device__ __forceinline__ float row_reduce_fresh(float v, float* red) {
  v = MAX ? wave_maxf(v) : wave_sum(v);
  if(THREADS > 64) {
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    if(lane == 0) red[wave] = v;
    __syncthreads();
    float r = red[0];
#pragma unroll
    for(int w = 1; w < THREADS / 64; ++w) r = MAX ? (red[w] > r ? red[w] : r) : r + red[w];
    v = r;
  }
  return v;
}

// ---------------------------------------------------------------- layer normalization
// One workgroup of 256 threads per row.  CACHE float4 vectors per thread hold the row in
// registers (cols <= 1024 * CACHE, cols % 4 == 0, 16-byte aligned rows); CACHE == 0 is the
// general form, which re-reads the row (it stays in L2).
template <int CACHE>
__global__ __launch_bounds__(256) void layer_norm_kernel(const float* in,
                                                         const float* __restrict__ add,
                                                         const float* __restrict__ gamma, int gamma_stride,
                                                         const float* __restrict__ beta, int beta_stride,
                                                         float* out, int cols, float eps,
                                                         float* __restrict__ absmax_out, int absmax_wrap, int rows) {
  __shared__ float red[4];
  float omax = 0.0f;   // max |y| over what this thread writes
  const size_t row = blockIdx.x;
  const float* x = in + row * cols;
  const float* a = add ? add + row * cols : nullptr;
  float* y = out + row * cols;
  const int tid = threadIdx.x;
  if(CACHE > 0) {
    const int cols4 = cols / 4;
    v4f v[CACHE > 0 ? CACHE : 1];
    // scale and shift are requested together with the row: read where they are used, behind the two
    // reductions, they would cost the kernel another memory round trip
    float gm[CACHE > 0 ? CACHE : 1][4], bt[CACHE > 0 ? CACHE : 1][4];
    float sum = 0.0f;
#pragma unroll
    for(int j = 0; j < CACHE; ++j) {
      const int i = j * 256 + tid;
      v[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      if(i < cols4) {
        v[j] = reinterpret_cast<const v4f*>(x)[i];
        v4f t = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        if(a) t = reinterpret_cast<const v4f*>(a)[i];
#pragma unroll
        for(int e = 0; e < 4; ++e) {
          gm[j][e] = gamma[gamma_stride * (4 * i + e)];
          bt[j][e] = beta ? beta[beta_stride * (4 * i + e)] : 0.0f;
        }
        if(a) {
          v[j].x = v[j].x + t.x; v[j].y = v[j].y + t.y; v[j].z = v[j].z + t.z; v[j].w = v[j].w + t.w;
        }
        sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
      }
    }
    const float mean = row_reduce<256, false>(sum, red) / (float)cols;
    float sq = 0.0f;
#pragma unroll
    for(int j = 0; j < CACHE; ++j) {
      if(j * 256 + tid < cols4) {
        const float d0 = v[j].x - mean, d1 = v[j].y - mean, d2 = v[j].z - mean, d3 = v[j].w - mean;
        sq += (d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3);
      }
    }
    const float sigma = sqrtf(row_reduce<256, false>(sq, red) / (float)cols + eps);
#pragma unroll
    for(int j = 0; j < CACHE; ++j) {
      const int i = j * 256 + tid;
      if(i < cols4) {
        float r[4] = {v[j].x, v[j].y, v[j].z, v[j].w};
#pragma unroll
        for(int e = 0; e < 4; ++e) {
          float t = gm[j][e] * ((r[e] - mean) / sigma);
          if(beta) t = t + bt[j][e];
          r[e] = t;
          omax = fmaxf(omax, fabsf(t));
        }
        reinterpret_cast<v4f*>(y)[i] = v4f{r[0], r[1], r[2], r[3]};
      }
    }
  } else {
    float sum = 0.0f;
    for(int i = tid; i < cols; i += 256) sum += a ? x[i] + a[i] : x[i];
    const float mean = row_reduce<256, false>(sum, red) / (float)cols;
    float sq = 0.0f;
    for(int i = tid; i < cols; i += 256) {
      const float d = (a ? x[i] + a[i] : x[i]) - mean;
      sq += d * d;
    }
    const float sigma = sqrtf(row_reduce<256, false>(sq, red) / (float)cols + eps);
    for(int i = tid; i < cols; i += 256) {
      float t = gamma[gamma_stride * i] * (((a ? x[i] + a[i] : x[i]) - mean) / sigma);
      if(beta) t = t + beta[beta_stride * i];
      y[i] = t;
      omax = fmaxf(omax, fabsf(t));
    }
  }
  if(absmax_out) {   // slot `row`; workgroup 0 zeroes the slots past the last row
    omax = row_reduce<256, true>(omax, red);
    if(absmax_wrap) {
      // more rows than slots: the rows share the slots (cleared by the launcher) through an integer
      // maximum on the bits, which orders non-negative floats as the floats themselves
      if(tid == 0) atomicMax(reinterpret_cast<int*>(absmax_out) + (int)(row % kAbsmaxSlots), __float_as_int(omax));
    } else {
      if(tid == 0) absmax_out[row] = omax;
      if(row == 0)
        for(int sl = rows + tid; sl < kAbsmaxSlots; sl += 256) absmax_out[sl] = 0.0f;
    }
  }
}

// Rows of up to 1024 values: one wave per row and per workgroup, four float4 per lane.  The three reductions stay
// inside the wave, so the kernel has no workgroup barrier and no LDS traffic between its load and its
// store; scale and shift come as 16-byte loads (gamma_stride / beta_stride 1, 16-byte aligned) or as one
// broadcast value (0).
// MANY: more rows than abs-max slots.  Four waves to a workgroup, each takes every 4 blocks-th row, and the workgroup
// leaves the maximum of all of them in its slot (one row to a workgroup and shared slots took a launch that clears
// them and atomic maxima: 4.5 + 10.4 us for 4096 x 1024, now 10.4 us; one wave to a workgroup and two rows to a
// wave 12.0).
// PLAIN: a skip input, a scale and a shift vector, as all layer norms of a model have them.  No branch and no address of its own for any load -
// rows are buffers that end behind their last value, past which loads give zeros and stores nothing - and none around the additions.
// Bound by its own instructions, one wave to a SIMD: 128 x 1024 3.38 -> 3.14 us, 65 x 512 3.40 -> 3.14, of which 2.6 are the launch and the first
// loads (steps of 6 layers 360.0 -> 354.4 and 294.1 -> 287.2); 4096 x 1024 10.3 -> 10.1, the copy rate.
template <bool MANY, bool PLAIN>
__global__ __launch_bounds__(MANY ? 256 : 64) void layer_norm_wave_kernel(const float* in, const float* __restrict__ add,
                                                             const float* __restrict__ gamma, int gamma_stride,
                                                             const float* __restrict__ beta, int beta_stride,
                                                             float* out, int cols, float eps,
                                                             float* __restrict__ absmax_out, int blocks, int rows) {
  constexpr int VPL = kNormVecs, WAVES = MANY ? 4 : 1;
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), cols4 = cols / 4;
  const v4f zero = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  v4f v[VPL], t[VPL], gm[VPL], bt[VPL];
  auto load_buffer = [&](const float* p, v4f (&r)[VPL]) __attribute__((always_inline)) {   // (p: a scalar)
    const auto buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, cols * 4, kRawBuffer);
#pragma unroll
    for(int j = 0; j < VPL; ++j) r[j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(buf, lane * 16 + j * 1024, 0, 0));
  };
  // all loads at once; positions past the row (zeros of a buffer, or the last values again) are dropped afterwards
  auto load_row = [&](size_t row, v4f (&v)[VPL], v4f (&t)[VPL]) __attribute__((always_inline)) {
    if constexpr(PLAIN) {
      load_buffer(in + row * cols, v);
      load_buffer(add + row * cols, t);
      return;
    }
    const v4f* x = reinterpret_cast<const v4f*>(in + row * cols);
    const v4f* a = add ? reinterpret_cast<const v4f*>(add + row * cols) : nullptr;
#pragma unroll
    for(int j = 0; j < VPL; ++j) {
      const int i = min(j * 64 + lane, cols4 - 1);
      v[j] = x[i];
      t[j] = a ? a[i] : zero;
    }
  };
  load_row((size_t)min((int)blockIdx.x * WAVES + wave, rows - 1), v, t);
  if constexpr(PLAIN) {
    load_buffer(gamma, gm);
    load_buffer(beta, bt);
  } else {
#pragma unroll
    for(int j = 0; j < VPL; ++j) {
      const int i = min(j * 64 + lane, cols4 - 1);
      if(gamma_stride) gm[j] = reinterpret_cast<const v4f*>(gamma)[i];
      if(beta && beta_stride) bt[j] = reinterpret_cast<const v4f*>(beta)[i];
    }
    if(!gamma_stride) {
      const float g0 = gamma[0];
#pragma unroll
      for(int j = 0; j < VPL; ++j) gm[j] = v4f{g0, g0, g0, g0};
    }
    if(!(beta && beta_stride)) {
      const float b0 = beta ? beta[0] : 0.0f;
#pragma unroll
      for(int j = 0; j < VPL; ++j) bt[j] = v4f{b0, b0, b0, b0};
    }
  }
  float omax = 0.0f;
  for(int row = (int)blockIdx.x * WAVES + wave; row < rows; row += blocks * WAVES) {
    omax = fmaxf(omax, normalize_row(v, t, PLAIN || add != nullptr, gm, bt, PLAIN || beta != nullptr, cols, eps));
    if constexpr(PLAIN) {
      const auto y = __builtin_amdgcn_make_buffer_rsrc(out + (size_t)row * cols, 0, cols * 4, kRawBuffer);
#pragma unroll
      for(int j = 0; j < VPL; ++j) __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u_raw, v[j]), y, lane * 16 + j * 1024, 0, 0);
    } else {
      v4f* y = reinterpret_cast<v4f*>(out + (size_t)row * cols);
#pragma unroll
      for(int j = 0; j < VPL; ++j)
        if(j * 64 + lane < cols4) y[j * 64 + lane] = v[j];
    }
    if constexpr(MANY) {
      if(row + blocks * WAVES < rows) load_row((size_t)(row + blocks * WAVES), v, t);
    } else {
      break;
    }
  }
  if(absmax_out) {   // a slot per workgroup; the slots past the last one are zeroed by all workgroups together
    omax = wave_maxf(omax);
    if constexpr(MANY) {
      __shared__ float top[WAVES];
      if(lane == 0) top[wave] = omax;
      __syncthreads();
      omax = fmaxf(fmaxf(top[0], top[1]), fmaxf(top[2], top[3]));
    }
    if(threadIdx.x == 0) absmax_out[blockIdx.x] = omax;
    if(wave == 0)
      for(int sl = blocks + (int)blockIdx.x * 64 + lane; sl < kAbsmaxSlots; sl += blocks * 64) absmax_out[sl] = 0.0f;
  }
}

// ---------------------------------------------------------------- softmax / log-softmax
// THREADS threads per row, 256 / THREADS... rows per workgroup: 64 (a wave per row, four rows
// per workgroup: attention scores) or 1024 (vocabulary-size rows).  Three passes over the row:
// max, sum of exponentials, result; the row stays in L1/L2 between them.
template <int THREADS, bool LOG>
__global__ __launch_bounds__(THREADS < 256 ? 256 : THREADS) void softmax_kernel(
    const float* in, const float* __restrict__ mask, long long n_masks,
    long long rows_per_mask, float* out, long long rows, int cols) {
  __shared__ float red[THREADS > 64 ? THREADS / 64 : 1];
  constexpr int kRowsPerBlock = THREADS < 256 ? 256 / THREADS : 1;
  const long long row = (long long)blockIdx.x * kRowsPerBlock + (THREADS < 256 ? threadIdx.x / THREADS : 0);
  const int t = threadIdx.x % THREADS;
  if(THREADS <= 64 && row >= rows) return;   // whole waves leave; no workgroup barrier is used
  const float* x = in + (size_t)row * cols;
  const float* m = mask ? mask + (size_t)((row / rows_per_mask) % n_masks) * cols : nullptr;
  float* y = out + (size_t)row * cols;
  float mx = -__builtin_inff();
  for(int i = t; i < cols; i += THREADS) {
    const float v = m ? x[i] + m[i] : x[i];
    mx = v > mx ? v : mx;
  }
  mx = row_reduce<THREADS, true>(mx, red);
  float sum = 0.0f;
  for(int i = t; i < cols; i += THREADS) sum += expf((m ? x[i] + m[i] : x[i]) - mx);
  sum = row_reduce<THREADS, false>(sum, red);
  if(LOG) {
    const float log_sum = logf(sum);
    for(int i = t; i < cols; i += THREADS) y[i] = ((m ? x[i] + m[i] : x[i]) - mx) - log_sum;
  } else {
    for(int i = t; i < cols; i += THREADS) y[i] = expf((m ? x[i] + m[i] : x[i]) - mx) / sum;
  }
}

// Rows kept in registers (cols % 4 == 0, 16-byte aligned rows and mask), so that they are read
// once: 256 threads with four float4 each for rows up to 4096 values, 1024 threads with eight or
// sixteen for vocabulary-size rows (up to 32768 / 65536).  Same
// operations per element as softmax_kernel.
// softmax_wide_row leaves in v (vector j of thread t = elements 4 * (j * THREADS + t) .. + 3 of the
// row, where they exist): LOG: x - max, and returns log(sum of exp(x - max)); otherwise exp(x - max),
// and returns their sum.  red: 2 * THREADS / 64 floats that nothing else uses meanwhile (the wave
// maxima, then the wave sums: no barrier in front of either reduction).  after_max(max, wave maxima)
// runs between the two reductions, when the THREADS / 64 wave maxima are in red[0 ...]; they stay
// there.
struct NoAfterMax {
  __device__ void operator()(float, const float*, float) const {}
};
template <bool LOG, int THREADS, int VPT, typename AfterMax = NoAfterMax>
__device__ __forceinline__ float softmax_wide_row(const v4f* x, const v4f* mk, int cols4, v4f (&v)[VPT], float* red,
                                                  AfterMax after_max = AfterMax()) {
  const int t = threadIdx.x;
  float mx = -__builtin_inff();
  // (all loads at once, positions past the row clamped and dropped afterwards: a load behind a
  // range check is waited for inside its branch, one memory latency per load)
#pragma unroll
  for(int j = 0; j < VPT; ++j) v[j] = x[min(j * THREADS + t, cols4 - 1)];
  if(mk) {   // (wave-uniform: the whole row has a mask or none)
    v4f mv[VPT];
#pragma unroll
    for(int j = 0; j < VPT; ++j) mv[j] = mk[min(j * THREADS + t, cols4 - 1)];
#pragma unroll
    for(int j = 0; j < VPT; ++j) {
      v[j].x = v[j].x + mv[j].x; v[j].y = v[j].y + mv[j].y; v[j].z = v[j].z + mv[j].z; v[j].w = v[j].w + mv[j].w;
    }
  }
#pragma unroll
  for(int j = 0; j < VPT; ++j) {
    const int i = j * THREADS + t;
    if(i < cols4) {
      // (one instruction for two values; a NaN, which it lets through, makes all results NaN by way of the sum as well)
      mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, v[j].x), v[j].y);
      mx = __builtin_elementwise_maximum(__builtin_elementwise_maximum(mx, v[j].z), v[j].w);
    }
  }
  const float own = mx;
  mx = row_reduce_fresh<THREADS, true>(mx, red);
  after_max(mx, red, own);
  float sum = 0.0f;
#pragma unroll
  for(int j = 0; j < VPT; ++j) {
    if(j * THREADS + t < cols4) {
      if(LOG) {
        v[j].x = v[j].x - mx; v[j].y = v[j].y - mx; v[j].z = v[j].z - mx; v[j].w = v[j].w - mx;
        // (the exponentials only enter the logarithm of their sum: the hardware exp2 form, about
        // 1e-6 relative, moves log(sum) by 1e-6 absolute, and it is a fifth of the instructions of
        // this kernel's busiest loop)
        sum += (__expf(v[j].x) + __expf(v[j].y)) + (__expf(v[j].z) + __expf(v[j].w));
      } else {
        v[j].x = expf(v[j].x - mx); v[j].y = expf(v[j].y - mx);
        v[j].z = expf(v[j].z - mx); v[j].w = expf(v[j].w - mx);
        sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
      }
    }
  }
  sum = row_reduce_fresh<THREADS, false>(sum, red + THREADS / 64);
  return LOG ? logf(sum) : sum;
}

template <bool LOG, int THREADS, int VPT>
__global__ __launch_bounds__(THREADS) void softmax_wide_kernel(const float* in, const float* __restrict__ mask,
                                                                long long n_masks, long long rows_per_mask,
                                                                float* out, int cols) {
  __shared__ float red[2 * THREADS / 64];
  const size_t row = blockIdx.x;
  const v4f* x = reinterpret_cast<const v4f*>(in + row * cols);
  const v4f* mk = mask ? reinterpret_cast<const v4f*>(mask + (size_t)((row / rows_per_mask) % n_masks) * cols) : nullptr;
  v4f* y = reinterpret_cast<v4f*>(out + row * cols);
  const int cols4 = cols / 4, t = threadIdx.x;
  v4f v[VPT];
  const float s = softmax_wide_row<LOG, THREADS, VPT>(x, mk, cols4, v, red);   // log(sum) or sum
#pragma unroll
  for(int j = 0; j < VPT; ++j) {
    const int i = j * THREADS + t;
    if(i < cols4) {
      if(LOG) y[i] = v4f{v[j].x - s, v[j].y - s, v[j].z - s, v[j].w - s};
      else y[i] = v4f{v[j].x / s, v[j].y / s, v[j].z / s, v[j].w / s};
    }
  }
}

// ---------------------------------------------------------------- transpose 0213
// One element (VEC floats of the innermost dimension) per thread, indexed by the output.
template <int VEC>
__global__ __launch_bounds__(256) void transpose0213_kernel(const float* in,
                                                            float* __restrict__ out, long long total,
                                                            int d1, int d2, int d3v, int blocks) {
  const long long stride = (long long)blocks * 256;
  for(long long o = (long long)blockIdx.x * 256 + threadIdx.x; o < total; o += stride) {
    const int i3 = (int)(o % d3v);
    long long r = o / d3v;
    const int i1 = (int)(r % d1);
    r /= d1;
    const int i2 = (int)(r % d2);
    const long long i0 = r / d2;
    const long long src = ((i0 * d1 + i1) * d2 + i2) * d3v + i3;
    if(VEC == 4) reinterpret_cast<v4f*>(out)[o] = reinterpret_cast<const v4f*>(in)[src];
    else out[o] = in[src];
  }
}

// ---------------------------------------------------------------- batched product
// One wave per output row (batch i, row r): lanes walk the n columns, every lane runs over k.
// At decode sizes (m = 1, k or n = 64, a few thousand batch entries) a product is a matrix-vector
// product of a few KB; the operands of a wave stay in L1 while it walks k.
__global__ __launch_bounds__(256) void bdot_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                   float* __restrict__ C, long long batchA,
                                                   long long batchB, long long rows_total, int m, int n,
                                                   int k, int transA, int transB, float scalar) {
  const long long wr = (long long)blockIdx.x * 4 + threadIdx.x / 64;   // output row of this wave
  if(wr >= rows_total) return;
  const int lane = threadIdx.x % 64;
  const long long i = wr / m;
  const int r = (int)(wr % m);
  const float* a = A + (size_t)(i % batchA) * m * k;
  const float* b = B + (size_t)(i % batchB) * n * k;
  float* c = C + (size_t)wr * n;
  const int lda = transA ? m : k, ldb = transB ? k : n;
  for(int q = lane; q < n; q += 64) {
    float s = 0.0f;
    if(!transA && transB && (k % 4) == 0 && ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) % 16) == 0) {
      const v4f* ar = reinterpret_cast<const v4f*>(a + (size_t)r * lda);
      const v4f* br = reinterpret_cast<const v4f*>(b + (size_t)q * ldb);
      for(int p = 0; p < k / 4; ++p) {
        const v4f av = ar[p], bv = br[p];
        s = fmaf(av.x, bv.x, s);
        s = fmaf(av.y, bv.y, s);
        s = fmaf(av.z, bv.z, s);
        s = fmaf(av.w, bv.w, s);
      }
    } else {
      for(int p = 0; p < k; ++p) {
        const float av = transA ? a[(size_t)p * lda + r] : a[(size_t)r * lda + p];
        const float bv = transB ? b[(size_t)q * ldb + p] : b[(size_t)p * ldb + q];
        s = fmaf(av, bv, s);
      }
    }
    c[q] = scalar * s;
  }
}

// The same products for matrices with many rows (encoder-size attention: m = n = 64 per head):
// a workgroup takes a 64 x 64 tile of one batch entry, K in chunks of 32 through LDS, a thread a
// 4 x 4 patch.  Every output is still summed over p = 0 .. k-1 in ascending order with one fma per
// term, so the result equals bdot_kernel's bit for bit.  A not transposed, k % 4 == 0 (TRANSB:
// B is [n x k]) or n % 4 == 0 (B is [k x n]), 16-byte aligned matrices.
template <bool TRANSB>
__global__ __launch_bounds__(256) void bdot_tile_kernel(const float* __restrict__ A, const float* __restrict__ B,
                                                        float* __restrict__ C, long long batchA,
                                                        long long batchB, int m, int n, int k, float scalar) {
  constexpr int KC = 32, LD = 64 + 4;
  __shared__ __attribute__((aligned(16))) float As[KC][LD];   // [p][row]
  __shared__ __attribute__((aligned(16))) float Bs[KC][LD];   // [p][col]
  const long long i = blockIdx.z;
  const float* a = A + (size_t)(i % batchA) * m * k;
  const float* b = B + (size_t)(i % batchB) * n * k;
  float* c = C + (size_t)i * m * n;
  const int r0 = blockIdx.y * 64, c0 = blockIdx.x * 64;
  const int tid = threadIdx.x, ty = tid / 16, tx = tid % 16;
  float acc[4][4];
#pragma unroll
  for(int y = 0; y < 4; ++y)
#pragma unroll
    for(int x = 0; x < 4; ++x) acc[y][x] = 0.0f;
  for(int p0 = 0; p0 < k; p0 += KC) {
    const int pc = min(KC, k - p0);   // a multiple of four
    __syncthreads();                  // the previous chunk has been read
    // rows of A (and of a transposed B): lane = row, so that the transposing LDS writes of a wave
    // fall into consecutive banks; four consecutive p per load
#pragma unroll
    for(int h = 0; h < 2; ++h) {
      const int idx = h * 256 + tid, row = idx % 64, p4 = idx / 64;   // p4 = 0 .. 7
      if(p4 * 4 < pc) {
        const v4f v = *reinterpret_cast<const v4f*>(a + (size_t)min(r0 + row, m - 1) * k + p0 + p4 * 4);
        As[p4 * 4][row] = v.x; As[p4 * 4 + 1][row] = v.y; As[p4 * 4 + 2][row] = v.z; As[p4 * 4 + 3][row] = v.w;
        if(TRANSB) {
          const v4f w = *reinterpret_cast<const v4f*>(b + (size_t)min(c0 + row, n - 1) * k + p0 + p4 * 4);
          Bs[p4 * 4][row] = w.x; Bs[p4 * 4 + 1][row] = w.y; Bs[p4 * 4 + 2][row] = w.z; Bs[p4 * 4 + 3][row] = w.w;
        }
      }
    }
    if(!TRANSB) {   // B is [k x n]: rows p, four consecutive columns per load
#pragma unroll
      for(int h = 0; h < 2; ++h) {
        const int idx = h * 256 + tid, col4 = idx % 16, p = idx / 16;   // p = 0 .. 31
        if(p < pc) {
          const int col = min(c0 + col4 * 4, n - 4);   // (n % 4 == 0; columns past n are never stored)
          *reinterpret_cast<v4f*>(&Bs[p][col4 * 4]) = *reinterpret_cast<const v4f*>(b + (size_t)(p0 + p) * n + col);
        }
      }
    }
    __syncthreads();
    for(int p = 0; p < pc; ++p) {
      const v4f av = *reinterpret_cast<const v4f*>(&As[p][ty * 4]);
      const v4f bv = *reinterpret_cast<const v4f*>(&Bs[p][tx * 4]);
      const float ar[4] = {av.x, av.y, av.z, av.w}, br[4] = {bv.x, bv.y, bv.z, bv.w};
#pragma unroll
      for(int y = 0; y < 4; ++y)
#pragma unroll
        for(int x = 0; x < 4; ++x) acc[y][x] = fmaf(ar[y], br[x], acc[y][x]);
    }
  }
#pragma unroll
  for(int y = 0; y < 4; ++y) {
    const int r = r0 + ty * 4 + y;
    if(r >= m) continue;
#pragma unroll
    for(int x = 0; x < 4; ++x) {
      const int q = c0 + tx * 4 + x;
      if(q < n) c[(size_t)r * n + q] = scalar * acc[y][x];
    }
  }
}

// ---------------------------------------------------------------- one-launch attention
// One wave per query row (entry i, row r): scores over the key positions (a lane per position,
// the query row and a key row are walked with the same fused multiply-adds, in the same order,
// as bdot_kernel walks them), softmax over them exactly as softmax_kernel<64> computes it, then
// the weighted sum of the value rows (a lane per output column, positions in ascending order,
// as bdot_kernel does).  The scores of a row live in LDS: `len` floats per wave.
// ANC (m == 1, dk == 64, one cache entry per query row, entry = hypothesis * heads + head): cached
// position p of hypothesis h is read from the entry of hypothesis anc[h * kv_cap + p] - the caches
// of a beam search stay where they were written and the table of ancestors says whose row a
// position of a hypothesis's history is; the newest position comes from k_new / v_new and goes into
// the hypothesis's own entry.
// STRIDED (no k_new): q, k, v and out have the strides of `hs` instead of lying head by head.
struct AttentionStrides {
  HeadStrides q, k, v, out;
};
template <bool ANC, bool STRIDED>
__global__ __launch_bounds__(256) void attention_kernel(const float* __restrict__ Q, float* Kt, float* V,
                                                        const float* __restrict__ k_new,
                                                        const float* __restrict__ v_new,
                                                        const float* __restrict__ mask,
                                                        unsigned n_masks, unsigned rows_per_mask,
                                                        float* __restrict__ out, unsigned rows_total,
                                                        unsigned batchKV, int m, int len, int kv_cap, int dk,
                                                        float scale, float* __restrict__ absmax_out,
                                                        const uint32_t* __restrict__ anc, unsigned heads, AttentionStrides hs) {
  // kv_cap: positions a cache entry has room for (its stride, in rows of dk values); len of them are in use
  // (row counts are below 2^31, checked by the launcher: 32-bit divisions, a tenth of the
  // instructions of 64-bit ones, and this kernel is a chain of short phases)
  extern __shared__ __attribute__((aligned(16))) float att_lds[];
  const unsigned wr = blockIdx.x * 4 + threadIdx.x / 64;
  if(absmax_out && blockIdx.x == 0)   // slots past the last query row
    for(int sl = (int)rows_total + threadIdx.x; sl < kAbsmaxSlots; sl += 256) absmax_out[sl] = 0.0f;
  if(wr >= rows_total) return;   // whole waves leave; no workgroup barrier is used
  // per wave: the scores (rounded up to whole 16-byte units, so that the partial outputs behind
  // them are 16-byte aligned for the v4f stores), then 4 x 64 partial outputs
  const int len4 = (len + 3) & ~3;
  float* sc = att_lds + (threadIdx.x / 64) * (len4 + 256);
  float* part = sc + len4;
  const int lane = threadIdx.x % 64;
  // (no division in the usual cases: one position per entry, as many cache entries as entries)
  const unsigned i = m == 1 ? wr : wr / (unsigned)m;
  const unsigned entry = i < batchKV ? i : i % batchKV;
  const size_t k_row = STRIDED ? (size_t)hs.k.row : (size_t)dk, v_row = STRIDED ? (size_t)hs.v.row : (size_t)dk;
  const float* q = STRIDED ? Q + hs.q.entry(i, heads) + (size_t)(wr - i * (unsigned)m) * hs.q.row : Q + (size_t)wr * dk;
  float* kb = Kt + (STRIDED ? hs.k.entry(entry, heads) : (size_t)entry * kv_cap * dk);
  float* vb = V + (STRIDED ? hs.v.entry(entry, heads) : (size_t)entry * kv_cap * dk);
  float* y = out + (STRIDED ? hs.out.entry(i, heads) + (size_t)(wr - i * (unsigned)m) * hs.out.row : (size_t)wr * dk);
  // Newest position (m == 1, one wave per cache entry): its key and value rows go into the cache
  // for the following steps; this step reads them from k_new / v_new directly.  Up to 64 values per
  // row they are requested here and stored at the end of the kernel (nothing in this call waits
  // for the copy, and a store right here would hold the wave for a memory round trip first).
  float k_app = 0.0f, v_app = 0.0f;
  const bool append_late = k_new && dk <= 64;
  if(append_late && lane < dk) {
    k_app = k_new[(size_t)wr * dk + lane];
    v_app = v_new[(size_t)wr * dk + lane];
  }
  if(k_new && !append_late) {
    for(int d = lane; d < dk; d += 64) {
      kb[(size_t)(len - 1) * dk + d] = k_new[(size_t)wr * dk + d];
      vb[(size_t)(len - 1) * dk + d] = v_new[(size_t)wr * dk + d];
    }
  }
  const float* k_last = k_new ? k_new + (size_t)wr * dk : kb + (size_t)(len - 1) * k_row;
  const float* v_last = v_new ? v_new + (size_t)wr * dk : vb + (size_t)(len - 1) * v_row;
  unsigned mask_row = 0;
  if(mask) {
    mask_row = rows_per_mask == 1 ? wr : wr / rows_per_mask;
    if(mask_row >= n_masks) mask_row %= n_masks;
  }
  const float* mk = mask ? mask + (size_t)mask_row * len : nullptr;
  const bool vec = (dk % 4) == 0 && ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(kb) |
                                     reinterpret_cast<uintptr_t>(k_last)) % 16) == 0;
  float mx = -__builtin_inff();
  float omax = 0.0f;   // max |out| of this query row
  const bool fast = vec && dk == 64 && ((reinterpret_cast<uintptr_t>(vb) | reinterpret_cast<uintptr_t>(v_last)) % 16) == 0;
  // The usual head size.  Sixteen lanes cover the 64 values of a key or value row with 16 bytes each
  // and the four groups of sixteen take four consecutive positions, so one load of the wave moves
  // 1 KB of contiguous cache.  Up to sixteen loads, 64 positions, are in flight at a time, and the
  // first 64 value rows are requested together with the first 64 key rows, so up to 64 positions
  // the call is one memory round trip.  Loads and products stop at the last group of four that
  // holds a position (the CU's address unit takes 16 clocks per load whether or not the row is a
  // duplicate, and eight waves share it).  The mask joins the scores afterwards, a lane per
  // position: one load for the first 64 positions, requested ahead of the key rows (inside the
  // score loop it was a dependent load per group of four).
  constexpr int kAttU = 16;
  v4f vr[kAttU];
  const int g = lane / 16, c = lane % 16;
  // Group of four positions U = (base + 4 u) / 4: this lane's position is 4 U + g, its row 4 U dk
  // floats behind the lane's first row; from group u_last on the lane's position is the last one
  // or past it, and it reads the last row (given separately: it may not be in the cache yet).
  const int u_last = (len + 2 - g) / 4;   // = ceil((len - 1 - g) / 4)
  auto load_rows = [&](const float* rows, size_t row, const float* last, int base, v4f (&r)[kAttU]) __attribute__((always_inline)) {
    const float* first = rows + (size_t)g * row + 4 * c;
    const float* last_c = last + 4 * c;
#pragma unroll
    for(int u = 0; u < kAttU; ++u) {
      if(base + 4 * u < len) {   // (the same for the whole wave)
        const int U = base / 4 + u;
        const float* p = U >= u_last ? last_c : first + (size_t)U * 4 * row;
        r[u] = *reinterpret_cast<const v4f*>(p);
      } else if(base + 4 * (u & ~3) < len) {   // (read with its group of sixteen positions below)
        r[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
  };
  // ANC: the entry a cached position is read from differs from position to position.  The lane's
  // (up to sixteen) ancestors of a batch of 64 positions are requested together, one round trip
  // ahead of the key and value rows.
  unsigned au[ANC ? kAttU : 1];
  const unsigned hyp = ANC ? wr / heads : 0u, head = ANC ? wr % heads : 0u;
  auto load_ancestors = [&](int base) __attribute__((always_inline)) {
    if(ANC) {
      const uint32_t* row = anc + (size_t)hyp * kv_cap;
      const unsigned n_hyp = rows_total / heads;
#pragma unroll
      for(int u = 0; u < kAttU; ++u)
        if(base + 4 * u < len) au[u] = min(row[min(base + 4 * u + g, len - 1)], n_hyp - 1u);
    }
  };
  auto load_rows_anc = [&](const float* tensor, const float* last, int base, v4f (&r)[kAttU]) __attribute__((always_inline)) {
    const float* last_c = last + 4 * c;
#pragma unroll
    for(int u = 0; u < kAttU; ++u) {
      if(base + 4 * u < len) {   // (the same for the whole wave)
        const int U = base / 4 + u;
        const float* p = U >= u_last ? last_c
                                     : tensor + ((size_t)(au[ANC ? u : 0] * heads + head) * kv_cap + (size_t)(4 * U + g)) * dk + 4 * c;
        r[u] = *reinterpret_cast<const v4f*>(p);
      } else if(base + 4 * (u & ~3) < len) {
        r[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
  };
  auto load_k = [&](int base, v4f (&r)[kAttU]) __attribute__((always_inline)) {
    if(ANC) load_rows_anc(Kt, k_last, base, r);
    else load_rows(kb, k_row, k_last, base, r);
  };
  auto load_v = [&](int base, v4f (&r)[kAttU]) __attribute__((always_inline)) {
    if(ANC) load_rows_anc(V, v_last, base, r);
    else load_rows(vb, v_row, v_last, base, r);
  };
  if(fast) {
    float mk0 = 0.0f;
    if(mk) mk0 = mk[min(lane, len - 1)];
    const v4f q4 = reinterpret_cast<const v4f*>(q)[c];
    v4f kr[kAttU];
    load_ancestors(0);
    load_k(0, kr);
    load_v(0, vr);
    // (sixteen positions at a time without a branch between them: the four products and the four
    // exchange steps of a group of four positions depend on one another, and only independent
    // groups side by side keep the wave issuing; rows that were not loaded are zeros here and their
    // results are dropped)
    for(int base = 0;;) {
#pragma unroll
      for(int u0 = 0; u0 < kAttU; u0 += 4) {
        if(base + 4 * u0 < len) {
          float s[4];
#pragma unroll
          for(int u = u0; u < u0 + 4; ++u) {
            float t = q4.x * kr[u].x;
            t = fmaf(q4.y, kr[u].y, t);
            t = fmaf(q4.z, kr[u].z, t);
            s[u - u0] = fmaf(q4.w, kr[u].w, t);
          }
#pragma unroll
          for(int u = 0; u < 4; ++u) s[u] = row16_sum(s[u]);
#pragma unroll
          for(int u = u0; u < u0 + 4; ++u) {
            const int pos = base + 4 * u + g;
            if(c == 0 && pos < len) sc[pos] = scale * s[u - u0];
          }
        }
      }
      base += 4 * kAttU;
      if(base >= len) break;
      load_ancestors(base);
      load_k(base, kr);
    }
    for(int pos = lane; pos < len; pos += 64) {
      float z = sc[pos];
      if(mk) {
        z = z + (pos < 64 ? mk0 : mk[pos]);
        sc[pos] = z;
      }
      mx = fmaxf(mx, z);
    }
  }
  for(int pos = lane; pos < len && !fast; pos += 64) {
    float s = 0.0f;
    const float* krow = pos == len - 1 ? k_last : kb + (size_t)pos * k_row;
    if(vec && dk == 64) {   // the usual head size: all sixteen loads of the key row in flight at once
      const v4f* ar = reinterpret_cast<const v4f*>(q);
      const v4f* br = reinterpret_cast<const v4f*>(krow);
      v4f kr[16];
#pragma unroll
      for(int p = 0; p < 16; ++p) kr[p] = br[p];
#pragma unroll
      for(int p = 0; p < 16; ++p) {
        const v4f av = ar[p];
        s = fmaf(av.x, kr[p].x, s);
        s = fmaf(av.y, kr[p].y, s);
        s = fmaf(av.z, kr[p].z, s);
        s = fmaf(av.w, kr[p].w, s);
      }
    } else if(vec) {
      const v4f* ar = reinterpret_cast<const v4f*>(q);
      const v4f* br = reinterpret_cast<const v4f*>(krow);
      for(int p = 0; p < dk / 4; ++p) {
        const v4f av = ar[p], bv = br[p];
        s = fmaf(av.x, bv.x, s);
        s = fmaf(av.y, bv.y, s);
        s = fmaf(av.z, bv.z, s);
        s = fmaf(av.w, bv.w, s);
      }
    } else {
      for(int p = 0; p < dk; ++p) s = fmaf(q[p], krow[p], s);
    }
    float z = scale * s;
    if(mk) z = z + mk[pos];
    sc[pos] = z;
    mx = z > mx ? z : mx;
  }
  mx = wave_maxf(mx);
  float sum = 0.0f;
  float e_first = 0.0f;   // exp of this lane's first position, kept for the division below
  for(int pos = lane; pos < len; pos += 64) {
    const float e = expf(sc[pos] - mx);
    if(pos == lane) e_first = e;
    sum += e;
  }
  sum = wave_sum(sum);
  for(int pos = lane; pos < len; pos += 64) sc[pos] = (pos == lane ? e_first : expf(sc[pos] - mx)) / sum;
  // (a wave's LDS writes are visible to its own later reads: same wave, program order)
  if(fast) {
    v4f o4 = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for(int base = 0; base < len; base += 4 * kAttU) {
      if(base > 0) {
        load_ancestors(base);
        load_v(base, vr);
      }
#pragma unroll
      for(int u0 = 0; u0 < kAttU; u0 += 4) {
        if(base + 4 * u0 < len) {
          // the four weights first (reads inside this wave's score area: a position past the row
          // reads a stale value there, which is replaced by zero)
          float w[4];
#pragma unroll
          for(int u = u0; u < u0 + 4; ++u) w[u - u0] = sc[min(base + 4 * u + g, len4 + 255)];
#pragma unroll
          for(int u = u0; u < u0 + 4; ++u) {
            const float wu = base + 4 * u + g < len ? w[u - u0] : 0.0f;
            o4.x = fmaf(wu, vr[u].x, o4.x);
            o4.y = fmaf(wu, vr[u].y, o4.y);
            o4.z = fmaf(wu, vr[u].z, o4.z);
            o4.w = fmaf(wu, vr[u].w, o4.w);
          }
        }
      }
    }
    reinterpret_cast<v4f*>(part)[g * 16 + c] = o4;   // partial sums of the positions g, g + 4, ...
    const float o = ((part[lane] + part[64 + lane]) + part[128 + lane]) + part[192 + lane];
    y[lane] = o;
    omax = fabsf(o);
  }
  for(int d = lane; d < dk && !fast; d += 64) {
    float o = 0.0f;
    int pos = 0;
    for(; pos + 8 <= len; pos += 8) {   // eight value loads in flight, same summation order
      float vr[8];
#pragma unroll
      for(int u = 0; u < 8; ++u) vr[u] = pos + u == len - 1 ? v_last[d] : vb[(size_t)(pos + u) * v_row + d];
#pragma unroll
      for(int u = 0; u < 8; ++u) o = fmaf(sc[pos + u], vr[u], o);
    }
    for(; pos < len; ++pos) o = fmaf(sc[pos], pos == len - 1 ? v_last[d] : vb[(size_t)pos * v_row + d], o);
    y[d] = 1.0f * o;
    omax = fmaxf(omax, fabsf(1.0f * o));
  }
  if(absmax_out) {   // slot = query row
    omax = wave_maxf(omax);
    if(lane == 0) absmax_out[wr] = omax;
  }
  if(append_late && lane < dk) {
    kb[(size_t)(len - 1) * dk + lane] = k_app;
    vb[(size_t)(len - 1) * dk + lane] = v_app;
  }
}

// ---------------------------------------------------------------- projection + attention in one launch
// The projections in front of an attention and the attention itself for one new target position
// (reference src/models/transformer.h:279-348: q = affine(input, Wq, bq), for self-attention also
// k, v = affine(input, Wk / Wv, ..), split into heads, then Attention()): a workgroup owns the 64
// columns of ONE head in every projection for R rows of the input, so it has everything that
// head's attention needs for its rows and runs it before it exits - one launch instead of two, and
// q (k, v) never travel through memory.
//   1. the abs-max of the input comes from the slots its producer left (or an abs-max launch);
//   2. the workgroup quantizes its R rows of the float32 input into LDS in matrix-operand order
//      (exactly the quantize-on-stage form of the decode GEMM: same quantizer, same layout); the
//      workgroups of head 0 also write them out, so the prepareA node's tensor still exists;
//   3. eight waves = 2 column tiles x 4 ranges of K; every wave requests its weights of all
//      projections at kernel start (up to 24 loads of 1 KB in flight), multiplies, and drops its
//      partial tiles into LDS;
//   4. the partial tiles are added (exact), dequantized with bias exactly like the GEMM epilogues
//      (two roundings) and kept in LDS as q[R][64] (k_new, v_new); k_new and v_new also go into
//      the caches at position len - 1, and all three into proj_out where a caller asks for them;
//   5. wave w runs the attention of row w: the code of attention_kernel's 64-wide path, operation
//      for operation, with q and the newest key/value row read from LDS.
// Where the caches are complete and shared - the encoder's keys and values, which every hypothesis
// of a sentence attends to (row m reads sentence m % sentences) - a workgroup takes hypotheses of
// the same one or two sentences instead of eight consecutive rows (ProjRowPlan in
// operand_addressing.h: as many hypotheses of a sentence as a workgroup has rows for, the rest in
// further workgroups; rows without a hypothesis idle), reads these sentences' keys and
// values once (asked for as soon as the abs-max is known, stored to LDS in step 4) and its waves
// take them from LDS: a quarter of the bytes through the CU's memory path with four hypotheses a
// sentence (60 positions: 60 KB instead of 240 KB per workgroup).
// Requirements (checked by the launcher): head size 64, K % 128 == 0, K <= 1024, len <= 512.
// Measured (transformer-big step, 128 rows, 16 heads): 13.5 us against 8.2 + 8.4 us for q, k, v and
// the self-attention over 21 positions, 13.9 against 5.3 + 8.4 us for Wq and the context attention over
// 60 positions with every wave reading its own keys and values; staging the shared ones takes the
// whole step from 0.437 to 0.425 ms.  The self-attention form is bound by what a CU can fetch: 310 KB per workgroup
// (192 KB of weights, 32 KB of input, 86 KB of keys and values), the latter from HBM.  Clocks inside the kernel: the
// cached rows came only when the projections were there, 10 800 of 26 100; asked for behind the weights into registers (HELD)
// the attention takes 3 400, the wait for the abs-max 4 400 more (a wave's requests are accepted as fast as the CU fetches),
// and the whole 24 100.  In the smaller forms K = 512 asks for the sub-steps it has (PW: eight with repeats before), and rows are worked
// out without a division (the launch has a dimension for sentence groups and one for hypothesis chunks): 6 rows x 8 heads over 12
// positions 19 800 -> 15 600 clocks, their context over 23 positions 18 100 -> 14 100; 65 rows over 34 positions 19 300 -> 17 900.
// Then (attention_row64_short, the input quantized behind half of the weights' loads, requests and code that are not needed left out) launches of 6 rows
// 8.9 -> 7.6 us and 8.1 -> 6.2 (context), of 65 rows over 34 positions 10.5 -> 8.9 and over 47 of the source 7.6 -> 6.3, of 128 rows 13.4 -> 12.4 and 11.5 -> 9.6.
// Tried and dropped: barriers that put every wave's small requests in front of any wave's large ones; the
// workgroups of a head starting at different sub-steps of K, so that they would not all miss L2 on
// the same lines of the weights at the same time (+5 us per step).
constexpr int kProjThreads = 512, kProjMaxK = 1024, kProjMaxLen = 512;
// keys and values shared by the rows of a workgroup are staged in LDS up to this many positions
constexpr int kProjStageLen = 96;
constexpr int kProjMaxLds = 160 * 1024 - 256;   // dynamic LDS of a workgroup (a few bytes are static)

struct ProjAttentionArgs {
  const float* A;           // [M, K] float32
  int8_t* aq_out;           // [M, K] int8 + quantMult tail
  const float* partials;    // abs-max slots of A
  int n_partials;
  const int8_t* Bq[3];      // prepared weights [K, heads * 64]
  const float* bias[3];     // or null
  float* proj_out[3];       // [M, heads * 64] or null: the projections themselves, for callers that want them
  int M, K, heads;
  float* k_cache;           // [batchKV, kv_cap, 64]
  float* v_cache;
  unsigned batchKV;
  int len, kv_cap;
  const float* mask;        // [n_masks, len] or null, one row per (query row / heads) % n_masks
  unsigned n_masks;
  float att_scale;
  float* out;               // [M * heads, 64]
  float* absmax_out;        // slots or null
  // Which input rows a workgroup takes (ProjRowPlan).  share_shift < 0: eight consecutive ones.
  // Otherwise the caches hold `share_nb` sentences that share_hyps hypotheses each attend to (row m
  // reads sentence m % share_nb), and a workgroup takes share_per of them for 1 << share_shift
  // neighbouring sentences, so that the waves that read the same keys and values sit on one CU.
  int share_shift, share_nb, share_hyps, share_per;
  // With it (and sentences two or one to a workgroup, len <= kProjStageLen): the keys and values of
  // the workgroup's sentences are read once, into LDS, and every hypothesis' wave takes them from there.
  int stage_kv;
  const uint32_t* anc;      // (ANC) [M, kv_cap]: the hypothesis in whose entry a cached position lies
  NormInput norm;           // (NORM) A is what the layer norm in front of the projections reads
};

// Entry g of one of the argument arrays, g differing between the threads: selected from the three
// values in scalar registers.  (Indexed by a thread-dependent g the compiler reads the entry from
// the kernel-argument memory with a vector load, and the wait for it - loads complete in order -
// is a wait for every load the thread has issued before: the weights.)
template <typename T>
__device__ __forceinline__ T pick3(const T (&a)[3], int g) {
  const T a0 = a[0], a1 = a[1], a2 = a[2];   // (values: a conditional between the elements themselves selects an address)
  return g == 0 ? a0 : (g == 1 ? a1 : a2);
}

// the row permutation of the staged activations (gemm_stream32_kernel.h: stream32_row_key)
__device__ __forceinline__ int proj_row_key(int c16) { return (c16 ^ (c16 >> 2)) & 7; }

// One query row of 64 values by one wave: attention_kernel's path for that head size (sixteen lanes
// cover a key or value row, four consecutive positions per load, up to 64 positions in flight), the
// same operations in the same order, so the result has the same bits.  q, k_last, v_last may lie
// in LDS.  sc: len4 floats of this wave (len rounded up to four), part: the 256 floats behind them.  Returns |out| of this lane.
// ANC: kb and vb are the whole caches, and cached position p lies in the entry of hypothesis anc.row[p], as in
// attention_kernel's form of that name; anc.first: row[4 u + lane / 16], requested by the caller (past the newest position: not looked at).
constexpr int kAttU = 16;
struct Ancestors {
  const uint32_t* row;
  unsigned n_hyp, heads, head;
  int kv_cap;
  unsigned first[kAttU];
};
// The cached rows of up to 4 HELD positions in registers: position 4 u + lane / 16 in k[u] and v[u] but for the newest.
template <int HELD>
struct HeldRows {
  v4f k[HELD], v[HELD];
};
template <>
struct HeldRows<0> {};
template <bool ANC = false>
__device__ __forceinline__ float attention_row64(const float* q, const float* kb, const float* vb, const float* k_last,
                                                 const float* v_last, const float* mk, float mk0, int len, float scale, float* sc,
                                                 float* part, float* out_row, int lane, const Ancestors* anc = nullptr) {
  constexpr int dk = 64;
  const int len4 = (len + 3) & ~3;
  const int g = lane / 16, c = lane % 16;
  const int u_last = (len + 2 - g) / 4;
  auto load_rows = [&](const float* rows, const float* last, int base, v4f (&r)[kAttU]) __attribute__((always_inline)) {
    const float* first = rows + (size_t)g * dk + 4 * c;
    const float* last_c = last + 4 * c;
#pragma unroll
    for(int u = 0; u < kAttU; ++u) {
      if(base + 4 * u < len) {
        const int U = base / 4 + u;
        if constexpr(ANC) {
          unsigned from = base == 0 ? anc->first[u] : anc->row[min(4 * U + g, len - 1)];
          from = min(from, anc->n_hyp - 1u);
          const float* at = rows + ((size_t)(from * anc->heads + anc->head) * anc->kv_cap + (size_t)(4 * U + g)) * dk + 4 * c;
          r[u] = *reinterpret_cast<const v4f*>(U >= u_last ? last_c : at);
        } else if(U >= u_last) r[u] = *reinterpret_cast<const v4f*>(last_c);
        else r[u] = *reinterpret_cast<const v4f*>(first + (size_t)U * 4 * dk);
      } else if(base + 4 * (u & ~3) < len) {
        r[u] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
  };
  const v4f q4 = reinterpret_cast<const v4f*>(q)[c];
  v4f kr[kAttU], vr[kAttU];
  load_rows(kb, k_last, 0, kr);
  load_rows(vb, v_last, 0, vr);
  for(int base = 0;;) {
#pragma unroll
    for(int u0 = 0; u0 < kAttU; u0 += 4) {
      if(base + 4 * u0 < len) {
        float s[4];
#pragma unroll
        for(int u = u0; u < u0 + 4; ++u) {
          float t = q4.x * kr[u].x;
          t = fmaf(q4.y, kr[u].y, t);
          t = fmaf(q4.z, kr[u].z, t);
          s[u - u0] = fmaf(q4.w, kr[u].w, t);
        }
#pragma unroll
        for(int u = 0; u < 4; ++u) s[u] = row16_sum(s[u]);
#pragma unroll
        for(int u = u0; u < u0 + 4; ++u) {
          const int pos = base + 4 * u + g;
          if(c == 0 && pos < len) sc[pos] = scale * s[u - u0];
        }
      }
    }
    base += 4 * kAttU;
    if(base >= len) break;
    load_rows(kb, k_last, base, kr);
  }
  float mx = -__builtin_inff();
  for(int pos = lane; pos < len; pos += 64) {
    float z = sc[pos];
    if(mk) {
      z = z + (pos < 64 ? mk0 : mk[pos]);
      sc[pos] = z;
    }
    mx = fmaxf(mx, z);
  }
  mx = wave_maxf(mx);
  float sum = 0.0f;
  float e_first = 0.0f;
  for(int pos = lane; pos < len; pos += 64) {
    const float e = expf(sc[pos] - mx);
    if(pos == lane) e_first = e;
    sum += e;
  }
  sum = wave_sum(sum);
  for(int pos = lane; pos < len; pos += 64) sc[pos] = (pos == lane ? e_first : expf(sc[pos] - mx)) / sum;
  v4f o4 = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  for(int base = 0; base < len; base += 4 * kAttU) {
    if(base > 0) load_rows(vb, v_last, base, vr);
#pragma unroll
    for(int u0 = 0; u0 < kAttU; u0 += 4) {
      if(base + 4 * u0 < len) {
        float w[4];
#pragma unroll
        for(int u = u0; u < u0 + 4; ++u) w[u - u0] = sc[min(base + 4 * u + g, len4 + 255)];
#pragma unroll
        for(int u = u0; u < u0 + 4; ++u) {
          const float wu = base + 4 * u + g < len ? w[u - u0] : 0.0f;
          o4.x = fmaf(wu, vr[u].x, o4.x);
          o4.y = fmaf(wu, vr[u].y, o4.y);
          o4.z = fmaf(wu, vr[u].z, o4.z);
          o4.w = fmaf(wu, vr[u].w, o4.w);
        }
      }
    }
  }
  reinterpret_cast<v4f*>(part)[g * 16 + c] = o4;
  const float o = ((part[lane] + part[64 + lane]) + part[128 + lane]) + part[192 + lane];
  out_row[lane] = o;
  return fabsf(o);
}

// attention_row64 where all rows are at hand, in LDS or in registers, and no more than 16 BLOCKS: no pass after another, no
// address of its own for every row and no loop over positions - 64 of them are the lanes of the wave.  The same operations in the same
// order.  Bound by its own instructions, one wave to a row and two to a SIMD: the general form took 5200 - 6500 clocks of a launch's 15 000 - 20 000
// with staged rows (a branch around every LDS load, 2200 of them), 3000 - 4600 with held ones.  Steps of 6 layers, with it, weights asked for
// without vector arithmetic and one copy of the quantization instead of eight: 6 x 512 over 12 and 23 positions 208.7 -> 196.8 us, 65 x 512 over
// 34 and 47 315.9 -> 307.7, 128 x 1024 over 21 and 60 392.0 -> 378.4.
// keys(r), values(r): rows 4 u + lane / 16 (those past the last one: it again), four values from 4 (lane % 16) on.
// Positions past len within four weigh nothing, fours past it are not added.
// sc and part lie one behind the other (len4 + 256 floats in all, 16 BLOCKS or more): scores and weights of all 16 BLOCKS positions, zeros past len, fill sc and
// the beginning of part, which is written when the weights have been read.
template <int BLOCKS, class Keys, class Values>
__device__ __forceinline__ float attention_row64_short(const float* q, Keys keys, Values values, const float* mk, float mk0, int len,
                                                       float scale, float* sc, float* part, float* out_row, int lane) {
  static_assert(BLOCKS <= 8, "two positions a lane");
  const int g = lane / 16, c = lane % 16;
  const v4f q4 = reinterpret_cast<const v4f*>(q)[c];
  v4f r[4 * BLOCKS];
  keys(r);
  [[maybe_unused]] float mk1 = 0.0f;
  if constexpr(BLOCKS > 4) {
    if(mk) mk1 = mk[min(64 + lane, len - 1)];
  }
#pragma unroll
  for(int b = 0; b < BLOCKS; ++b) {
    if(b == 0 || 16 * b < len) {
      float s[4];
#pragma unroll
      for(int u = 0; u < 4; ++u) {
        float t = q4.x * r[4 * b + u].x;
        t = fmaf(q4.y, r[4 * b + u].y, t);
        t = fmaf(q4.z, r[4 * b + u].z, t);
        s[u] = fmaf(q4.w, r[4 * b + u].w, t);
      }
#pragma unroll
      for(int u = 0; u < 4; ++u) s[u] = row16_sum(s[u]);
      if(c == 0) {   // (past len: not looked at)
#pragma unroll
        for(int u = 0; u < 4; ++u) sc[16 * b + 4 * u + g] = scale * s[u];
      }
    }
  }
  values(r);
  const bool here = lane < len;
  [[maybe_unused]] const bool here1 = 64 + lane < len;
  [[maybe_unused]] float z1 = 0.0f, e1 = 0.0f;
  float z = sc[lane];
  if(mk) z = z + mk0;
  float mx = here ? fmaxf(-__builtin_inff(), z) : -__builtin_inff();
  if constexpr(BLOCKS > 4) {
    z1 = sc[64 + lane];
    if(mk) z1 = z1 + mk1;
    mx = here1 ? fmaxf(mx, z1) : mx;
  }
  mx = wave_maxf(mx);
  const float e = here ? expf(z - mx) : 0.0f;
  float sum = 0.0f + e;
  if constexpr(BLOCKS > 4) {
    e1 = here1 ? expf(z1 - mx) : 0.0f;
    sum += e1;
  }
  sum = wave_sum(sum);
  sc[lane] = here ? e / sum : 0.0f;
  if constexpr(BLOCKS > 4) sc[64 + lane] = here1 ? e1 / sum : 0.0f;
  float w[4 * BLOCKS];
#pragma unroll
  for(int u = 0; u < 4 * BLOCKS; ++u) w[u] = sc[4 * u + g];
  v4f o4 = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for(int b = 0; b < BLOCKS; ++b) {
    if(b == 0 || 16 * b < len) {
#pragma unroll
      for(int u = 4 * b; u < 4 * b + 4; ++u) {
        const bool there = u % 4 == 0 || 4 * u < len;   // (rows that are not there may be infinite)
        o4.x = fmaf(w[u], there ? r[u].x : 0.0f, o4.x);
        o4.y = fmaf(w[u], there ? r[u].y : 0.0f, o4.y);
        o4.z = fmaf(w[u], there ? r[u].z : 0.0f, o4.z);
        o4.w = fmaf(w[u], there ? r[u].w : 0.0f, o4.w);
      }
    }
  }
  reinterpret_cast<v4f*>(part)[g * 16 + c] = o4;   // partial sums of the positions g, g + 4, ...
  const float o = ((part[lane] + part[64 + lane]) + part[128 + lane]) + part[192 + lane];
  out_row[lane] = o;
  return fabsf(o);
}
// Rows of 64 values one after the other in LDS.
template <int BLOCKS>
struct StagedRows {
  const float* rows;
  int len, lane;
  __device__ __forceinline__ void operator()(v4f (&r)[4 * BLOCKS]) const {
    const unsigned first = (unsigned)(lane / 16) * 256u, last = (unsigned)(len - 1) * 256u;
#pragma unroll
    for(int u = 0; u < 4 * BLOCKS; ++u)
      r[u] = *reinterpret_cast<const v4f*>(reinterpret_cast<const char*>(rows) + min(first + 1024u * u, last) + (lane % 16) * 16);
  }
};

// Attention over caches that several query rows share (the encoder's keys and values: query row
// r reads cache entry r % batchKV, so rows e, e + batchKV, e + 2 batchKV, .. - the hypotheses of a
// sentence, for one head - read the same entry).  Workgroup (e, y) takes rows e + (4 y + w) batchKV
// for its waves w = 0 .. 3, reads entry e's keys and values once (sixteen threads per position,
// PASSES passes of sixteen positions; positions past the end repeat the last one) into LDS, and each
// wave then runs attention_row64_short on them: the operations of attention_kernel's 64-wide path in the
// same order, so the same bits, with a quarter (for four hypotheses) of the bytes through the
// CU's memory path and out of L2.  One position per query row, head size 64, len <= 16 * PASSES.
constexpr int kSharedAttLen = 96;
template <int PASSES>
__global__ __launch_bounds__(256) void attention_shared_kernel(const float* __restrict__ Q, const float* __restrict__ Kt,
                                                               const float* __restrict__ V, const float* __restrict__ mask,
                                                               unsigned n_masks, unsigned rows_per_mask,
                                                               float* __restrict__ out, unsigned rows_total,
                                                               unsigned batchKV, int len, int kv_cap, float scale,
                                                               float* __restrict__ absmax_out) {
  static_assert(PASSES * 16 <= kSharedAttLen, "sixteen positions per pass");
  extern __shared__ __attribute__((aligned(16))) float satt_lds[];
  const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
  const unsigned entry = blockIdx.x;
  const unsigned wr = entry + (blockIdx.y * 4u + (unsigned)wave) * batchKV;
  const bool valid = wr < rows_total;
  if(absmax_out && blockIdx.x == 0 && blockIdx.y == 0)   // slots past the last query row
    for(int sl = (int)rows_total + tid; sl < kAbsmaxSlots; sl += 256) absmax_out[sl] = 0.0f;
  // everything is requested before anything is used: keys, values, the mask value of this lane
  v4f kst[PASSES], vst[PASSES];
  {
    const float* ksrc = Kt + (size_t)entry * kv_cap * 64 + (tid % 16) * 4;
    const float* vsrc = V + (size_t)entry * kv_cap * 64 + (tid % 16) * 4;
#pragma unroll
    for(int j = 0; j < PASSES; ++j) kst[j] = *reinterpret_cast<const v4f*>(ksrc + (size_t)min(tid / 16 + 16 * j, len - 1) * 64);
#pragma unroll
    for(int j = 0; j < PASSES; ++j) vst[j] = *reinterpret_cast<const v4f*>(vsrc + (size_t)min(tid / 16 + 16 * j, len - 1) * 64);
  }
  const float* mk = nullptr;
  if(mask && valid) {
    unsigned mask_row = rows_per_mask == 1 ? wr : wr / rows_per_mask;
    if(mask_row >= n_masks) mask_row %= n_masks;
    mk = mask + (size_t)mask_row * len;
  }
  const float mk0 = *(mk ? mk + min(lane, len - 1) : Q);   // (the latter not looked at)
  const int len4 = (len + 3) & ~3;
  float* ks = satt_lds;                       // [len][64]
  float* vs = ks + (size_t)len * 64;          // [len][64]
  float* sc = vs + (size_t)len * 64 + wave * (len4 + 256);   // per wave: scores + 256 partial outputs
#pragma unroll
  for(int j = 0; j < PASSES; ++j) {
    const int pos = tid / 16 + 16 * j;
    if(pos < len) {
      *reinterpret_cast<v4f*>(ks + (size_t)pos * 64 + (tid % 16) * 4) = kst[j];
      *reinterpret_cast<v4f*>(vs + (size_t)pos * 64 + (tid % 16) * 4) = vst[j];
    }
  }
  __syncthreads();
  if(valid) {   // (whole waves)
    float omax = attention_row64_short<PASSES>(Q + (size_t)wr * 64, StagedRows<PASSES>{ks, len, lane}, StagedRows<PASSES>{vs, len, lane}, mk,
                                               mk0, len, scale, sc, sc + len4, out + (size_t)wr * 64, lane);
    if(absmax_out) {
      omax = wave_maxf(omax);
      if(lane == 0) absmax_out[wr] = omax;
    }
  }
}

// NPROJ: 3 (q, k_new, v_new: self-attention, the new key/value row is appended to the caches) or
// 1 (q only: attention over caches that are complete, e.g. the encoder's).  R: input rows per
// workgroup, 8 (a wave per row in the attention) or 4 (without staging: half of the waves attend).
// NORM: the projections' input is the layer norm of A + norm.add, up to kNormMaxRows rows: every workgroup
// normalizes all of them, a wave each, while its weights are on their way (a launch of its own for the norm
// took 3.5 us of GPU and 4 of host time).
// ANC: the self-attention's cached positions are read through the table of ancestors (attention_kernel's ANC).
// aux: the abs-max partials, or (NORM) what is added to A.
// PW: K sub-steps of 32 a wave loads, K / 128 rounded up to 4 or 8.
// HELD: (self-attention) cached keys and values of up to 4 HELD positions are asked for behind the weights, so that they arrive
// during quantization and products; 0: longer histories, asked for when the projections are there.
template <int NPROJ, int R, int SEGS, int PASSES, int PW, int HELD, bool NORM = false, bool ANC = false>
__global__ __launch_bounds__(kProjThreads) void proj_attention_kernel(const float* A, const float* aux, const int8_t* Bq0, const int8_t* Bq1,
                                                                      const int8_t* Bq2, int M, int K, int heads, int n_partials,
                                                                      ProjAttentionArgs p) {
  p.A = A; p.Bq[0] = Bq0; p.Bq[1] = Bq1; p.Bq[2] = Bq2;   // (what is needed first comes in registers, see the Makefile)
  p.M = M; p.K = K; p.heads = heads; p.n_partials = n_partials; p.partials = aux;
  static_assert(HELD == 0 || NPROJ == 3, "the newest key and value come from the projections");
  static_assert(R == 8 || (R == 4 && !(SEGS > 0)), "a wave per row in the attention");
  constexpr bool STAGED = SEGS > 0;
  static_assert(!STAGED || NPROJ == 1, "keys and values are shared only where the caches are complete");
  static_assert(SEGS == 0 || SEGS == 2 || SEGS == 4, "keys and values of one or two sentences");
  static_assert(PASSES * 32 <= kProjStageLen, "32 positions per pass");
  typedef int v16i_p __attribute__((ext_vector_type(16)));
  extern __shared__ __attribute__((aligned(16))) int8_t plds[];
  __shared__ float red[kProjThreads / 64];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;   // (a scalar: what follows from it is too)
  const int wn = wave % 2, kw = wave / 2, li = lane % 32, lg = lane / 32;
  const int h = blockIdx.x;
  // input row r of this workgroup (rows past the end: M or more)
  const int sent_base = p.share_shift < 0 ? 0 : proj_first_sentence(p.share_shift, (int)blockIdx.y);
  auto row_of = [&](int r) -> int {
    return proj_row_of(p.share_shift, p.share_nb, p.share_hyps, p.share_per, (int)blockIdx.y, (int)blockIdx.z, r);
  };
  const bool first_rows = blockIdx.y == 0 && blockIdx.z == 0;
  const int S = K / 32, steps = S / 4, N = p.heads * 64;   // steps: sub-steps of a wave, at most PW
  int8_t* a_lds = plds;                                   // 32 rows x K bytes, operand order
  int8_t* part_lds = a_lds + 32 * K;                      // NPROJ x 2 x 4 partial tiles of R rows x 128 bytes
  float* proj_lds = reinterpret_cast<float*>(part_lds + NPROJ * 8 * R * 128);   // [NPROJ][R][64]
  float* att_lds = proj_lds + NPROJ * R * 64;             // per wave: scores + 256 partial outputs
  const int len4s = (p.len + 3) & ~3;
  float* kv_lds = att_lds + R * (len4s + 256);            // staged keys and values: [sentence][k, v][len][64]

  const int m_wave = row_of(min(wave, R - 1));   // the row this wave attends for
  Ancestors anc;
  auto load_ancestors = [&]() __attribute__((always_inline)) {   // (unconditional: waits count)
    static_assert(!ANC || (NPROJ == 3 && !STAGED), "self-attention");
    anc.row = p.anc + (size_t)min(m_wave, M - 1) * p.kv_cap;
    anc.n_hyp = (unsigned)M; anc.heads = (unsigned)p.heads; anc.head = (unsigned)h; anc.kv_cap = p.kv_cap;
    const auto row_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(anc.row), 0, p.len * 4, kRawBuffer);
#pragma unroll
    for(int u = 0; u < (HELD > 0 ? HELD : kAttU); ++u)   // (past the end: hypothesis 0, not looked at)
      anc.first[u] = __builtin_amdgcn_raw_buffer_load_b32(row_buf, (unsigned)lane / 16 * 4u, 16u * u, 0);
  };
  if constexpr(ANC && HELD > 0) {   // (they are addresses)
    load_ancestors();
    __builtin_amdgcn_sched_barrier(0);
  }

  // ---- everything this workgroup will need is requested now, in the order of its use (a wave's
  //      loads complete in the order of their issue): abs-max slots, the input rows, weights, the
  //      mask value, the quantization multipliers of the weights, bias ----
  [[maybe_unused]] PartialMaxima<kProjThreads> pm;
  // a quad of lanes takes four consecutive 16-value groups of one row: 64 contiguous bytes per load
  const int grp = (tid / 4) * 4, qlane = tid % 4;
  const int r_in = grp / (2 * S), c16 = grp % (2 * S);
  const bool has_in = !NORM && r_in < R;
  v4f in[4];
  NormRow<PW == 4 ? kNormVecs / 2 : kNormVecs> nr;
  if constexpr(NORM) {
    nr.load(p.A, aux, p.norm, M, K);
    __builtin_amdgcn_sched_barrier(0);
  } else {
    pm.load(p.partials, p.n_partials);
    const int m = min(row_of(min(r_in, R - 1)), M - 1);
    const float* src = p.A + (size_t)m * (size_t)K + (size_t)c16 * 16 + qlane * 4;
#pragma unroll
    for(int e = 0; e < 4; ++e) in[e] = *reinterpret_cast<const v4f*>(src + e * 16);
  }
  v4i w[NPROJ][PW];
  const unsigned w_off = stream32_lane_offset(h * 64 + wn * 32 + li, lg), w_step = 32u * (unsigned)N;
  // (asked for in the order the multiplication takes them: sub-step by sub-step, all projections; as buffers: no vector arithmetic)
  auto load_weights = [&](int from, int to) __attribute__((always_inline)) {
#pragma unroll
    for(int pp = from; pp < to; ++pp) {
      const unsigned at = (unsigned)stream32_clamped_substep(kw * steps + pp, S) * w_step;
#pragma unroll
      for(int g = 0; g < NPROJ; ++g) {
        const auto w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(p.Bq[g]), 0, (int)((unsigned)K * (unsigned)N), kRawBuffer);
        w[g][pp] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w_buf, w_off, at, 0));
      }
    }
  };
  float aqm = 0.0f;
  constexpr int kFirstSubsteps = NORM ? PW : PW / 2;
  load_weights(0, kFirstSubsteps);
  if constexpr(!NORM) {
    // ---- 1, 2: abs-max, quantize into LDS, behind half of the weights' loads: a wave goes on only when its loads have been accepted, and behind
    //      all of them that was 5000 - 9000 clocks after the input had come (a step of 65 x 512 298.9 -> 293.2 us; 128 x 1024, which is bound by what a
    //      CU can fetch, the same with half or a quarter) ----
    __builtin_amdgcn_sched_barrier(0);
    aqm = quant_mult_from_maxabs(block_max<kProjThreads / 64>(pm.max(), red));
    const float by = quantizer(aqm);
    if(has_in) {
      uint32_t q[4];
#pragma unroll
      for(int e = 0; e < 4; ++e) q[e] = quantize_pack4(in[e], by);
      const int slot0 = (c16 / 2) * 64, x = r_in ^ proj_row_key(c16);
      const int m = row_of(min(r_in, R - 1));
#pragma unroll
      for(int e = 0; e < 4; ++e) {
        const int sw = slot0 + (e / 2) * 64 + (e % 2) * 32 + (x ^ e);
        *reinterpret_cast<uint32_t*>(a_lds + sw * 16 + qlane * 4) = q[e];
        if(p.aq_out && h == 0 && m < M)
          *reinterpret_cast<uint32_t*>(p.aq_out + (size_t)m * (size_t)K + (size_t)(c16 + e) * 16 + qlane * 4) = q[e];
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    load_weights(kFirstSubsteps, PW);
  }
  // keys and values of the workgroup's sentences: sixteen threads per position, 32 positions per pass
  constexpr int kStageSegs = STAGED ? SEGS : 1, kStagePasses = STAGED ? PASSES : 1;
  v4f stage[kStageSegs][kStagePasses];
  // the mask value of this wave's row for position `lane`
  const float* mk = nullptr;
  if(p.mask && m_wave < M) {
    unsigned mask_row = (unsigned)m_wave;
    if(mask_row >= p.n_masks) mask_row %= p.n_masks;
    mk = p.mask + (size_t)mask_row * p.len;
  }
  const float mk0 = *(mk ? mk + min(lane, p.len - 1) : p.A);   // (the latter not looked at)
  if constexpr(ANC && HELD == 0) load_ancestors();
  float bqm[NPROJ];
#pragma unroll
  for(int g = 0; g < NPROJ; ++g) bqm[g] = tail_quant_mult(p.Bq[g], (size_t)K * (size_t)N);
  // the (up to two) pieces of four outputs this thread finishes in step 4, and their bias
  constexpr int kItems = NPROJ * 2 * R * 8;
  v4f bias4[2];
#pragma unroll
  for(int it = 0; it < 2; ++it) {
    const int item = min(it * kProjThreads + tid, kItems - 1);
    const int tg = item / (R * 8), pc = item % 8;
    const float* b = pick3(p.bias, tg / 2);
    // (no bias: sixteen bytes of the weights instead, not looked at)
    bias4[it] = *reinterpret_cast<const v4f*>(b ? b + h * 64 + (tg % 2) * 32 + pc * 4 : reinterpret_cast<const float*>(p.Bq[0]));
  }

  // NORM: as which row this workgroup multiplies the one that this wave normalizes (found while the loads are under way)
  [[maybe_unused]] int norm_at = -1;
  if constexpr(NORM) {
    norm_at = __builtin_amdgcn_readfirstlane(proj_place_of(p.share_shift, p.share_nb, p.share_hyps, p.share_per, (int)blockIdx.y, (int)blockIdx.z, wave));
    if(norm_at >= R) norm_at = -1;
  }

  // The keys and values are asked for last - a wave's loads complete in the order of their issue, and they are needed
  // last.  No branches around them (positions past the end repeat the last one; the number of loads is the kernel's), so that the
  // waits in front of the earlier loads' uses count exactly.  Behind a layer norm, whose reductions they would come in
  // between, only when the abs-max is there (65 x 512 over 47 source positions 7.8 -> 7.5 us with them here, 128 x 1024 over 60 11.4 and 11.4).
  auto load_stage = [&]() __attribute__((always_inline)) {
#pragma unroll
    for(int seg = 0; seg < SEGS; ++seg) {
      const unsigned entry = (unsigned)(sent_base + (seg >> 1)) * (unsigned)p.heads + (unsigned)h;
      const float* src = ((seg & 1) ? p.v_cache : p.k_cache) + (size_t)entry * p.kv_cap * 64 + (tid % 16) * 4;
#pragma unroll
      for(int j = 0; j < PASSES; ++j)
        stage[seg][j] = *reinterpret_cast<const v4f*>(src + (size_t)min(tid / 16 + 32 * j, p.len - 1) * 64);
    }
  };
  if constexpr(STAGED && !NORM) {
    __builtin_amdgcn_sched_barrier(0);
    load_stage();
    __builtin_amdgcn_sched_barrier(0);
  }

  HeldRows<HELD> held;
  if constexpr(HELD > 0) {   // (as buffers: a wave without a row asks for nothing, and the waits still count)
    __builtin_amdgcn_sched_barrier(0);
    const bool mine = wave < R && m_wave < M;
    const size_t entry = ANC ? 0 : (size_t)min(m_wave, M - 1) * p.heads + h;
    const unsigned bytes = mine ? (ANC ? (unsigned)M * (unsigned)p.heads : 1u) * (unsigned)p.kv_cap * 256u : 0u;
    const auto k_buf = __builtin_amdgcn_make_buffer_rsrc(p.k_cache + entry * p.kv_cap * 64, 0, (int)bytes, kRawBuffer);
    const auto v_buf = __builtin_amdgcn_make_buffer_rsrc(p.v_cache + entry * p.kv_cap * 64, 0, (int)bytes, kRawBuffer);
    unsigned at[HELD];
    const unsigned rows_of_one = (unsigned)p.heads * (unsigned)p.kv_cap, first = (unsigned)h * (unsigned)p.kv_cap + (unsigned)lane / 16;
#pragma unroll
    for(int u = 0; u < HELD; ++u) {
      const unsigned pos = (unsigned)(4 * u + lane / 16);
      // (both below 2^24, see the launcher: a full-rate multiplication)
      if(ANC) at[u] = (__umul24(min(anc.first[u], anc.n_hyp - 1u), rows_of_one) + (first + 4u * u)) * 256u + (lane % 16) * 16u;
      else at[u] = pos * 256u + (lane % 16) * 16u;
      if((int)pos >= p.len - 1) at[u] = 0xFFFFFFF0u;   // (past the cached ones: past the buffer, nothing is fetched)
    }
#pragma unroll
    for(int u = 0; u < HELD; ++u) held.k[u] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(k_buf, at[u], 0, 0));
#pragma unroll
    for(int u = 0; u < HELD; ++u) held.v[u] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(v_buf, at[u], 0, 0));
    __builtin_amdgcn_sched_barrier(0);
  }

  if constexpr(NORM) {   // 1, 2: wave w holds row w, quantized where this workgroup multiplies it, written out by one workgroup
    const float amax = block_max<kProjThreads / 64>(nr.normalize(p.norm, K), red);
    if constexpr(STAGED) load_stage();
    aqm = quant_mult_from_maxabs(amax);
    const int row = wave;
    if(row < M) {
      if(norm_at >= 0) nr.quantize(a_lds, norm_at, K, aqm, proj_row_key);
      if(h == 0 && first_rows) nr.store(p.norm, row, K);
    }
  }
  if(p.aq_out && h == 0 && first_rows && tid == 0) *reinterpret_cast<float*>(p.aq_out + (size_t)M * K) = aqm;
  __syncthreads();

  // ---- 3: multiply (rows R .. 31 of the operand are whatever LDS held: they only feed output rows
  //      that are never looked at) ----
  v16i_p acc[NPROJ];
#pragma unroll
  for(int g = 0; g < NPROJ; ++g)
#pragma unroll
    for(int v = 0; v < 16; ++v) acc[g][v] = 0;
#pragma unroll
  for(int pp = 0; pp < PW; ++pp) {
    if(pp < steps) {   // (the same for the whole workgroup)
      const int s = kw * steps + pp;
      const v4i a = *reinterpret_cast<const v4i*>(a_lds + s * 1024 + (lg * 32 + (li ^ proj_row_key(2 * s + lg))) * 16);
#pragma unroll
      for(int g = 0; g < NPROJ; ++g) acc[g] = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[g][pp], a, acc[g], 0, 0, 0);
    }
  }
  float unquant[NPROJ];   // (while the products are made)
#pragma unroll
  for(int g = 0; g < NPROJ; ++g) unquant[g] = unquant_mult(aqm, bqm[g], 1.0f);
  // accumulator value v of lane (li, lg): input row li, column 8 * (v / 4) + 4 * lg + v % 4 of the
  // wave's 32; a tile row is 128 bytes, its eight 16-byte pieces XOR-permuted by the row number
  if(li < R) {
#pragma unroll
    for(int g = 0; g < NPROJ; ++g) {
      int8_t* mine = part_lds + ((g * 2 + wn) * 4 + kw) * (R * 128);
#pragma unroll
      for(int q = 0; q < 4; ++q)
        *reinterpret_cast<v4i*>(mine + li * 128 + (((2 * q + lg) ^ (li & 7)) * 16)) =
            v4i{acc[g][4 * q], acc[g][4 * q + 1], acc[g][4 * q + 2], acc[g][4 * q + 3]};
    }
  }
  __syncthreads();

  // ---- 4: add the four K ranges, dequantize, keep in LDS, append k_new / v_new to the caches ----
#pragma unroll
  for(int it = 0; it < 2; ++it) {
    const int item = it * kProjThreads + tid;
    if(item < kItems) {
      const int tg = item / (R * 8), r = (item / 8) % R, pc = item % 8;
      const int g = tg / 2, col = (tg % 2) * 32 + pc * 4;
      const int8_t* src = part_lds + (tg * 4) * (R * 128) + r * 128 + ((pc ^ (r & 7)) * 16);
      v4i sum = *reinterpret_cast<const v4i*>(src);
#pragma unroll
      for(int t = 1; t < 4; ++t) sum += *reinterpret_cast<const v4i*>(src + t * (R * 128));
      float uq = unquant[0];
      if constexpr(NPROJ == 3) uq = g == 0 ? unquant[0] : (g == 1 ? unquant[1] : unquant[2]);
      const bool has_bias = pick3(p.bias, g) != nullptr;
      const float b[4] = {bias4[it].x, bias4[it].y, bias4[it].z, bias4[it].w};
      float y[4];
#pragma unroll
      for(int e = 0; e < 4; ++e) {
        y[e] = (float)sum[e] * uq;
        if(has_bias) y[e] = y[e] + b[e];
      }
      const v4f yv = v4f{y[0], y[1], y[2], y[3]};
      *reinterpret_cast<v4f*>(proj_lds + (g * R + r) * 64 + col) = yv;
      const int m = row_of(r);
      if(m < M) {
        float* const po = pick3(p.proj_out, g);
        if(po) *reinterpret_cast<v4f*>(po + (size_t)m * (size_t)N + h * 64 + col) = yv;
        if(NPROJ == 3 && g > 0) {
          float* cache = g == 1 ? p.k_cache : p.v_cache;
          const size_t entry = (size_t)m * (size_t)p.heads + (size_t)h;
          *reinterpret_cast<v4f*>(cache + (entry * (size_t)p.kv_cap + (size_t)(p.len - 1)) * 64 + col) = yv;
        }
      }
    }
  }
  if constexpr(STAGED) {
#pragma unroll
    for(int seg = 0; seg < SEGS; ++seg) {
#pragma unroll
      for(int j = 0; j < PASSES; ++j) {
        const int pos = tid / 16 + 32 * j;
        if(pos < p.len) *reinterpret_cast<v4f*>(kv_lds + ((size_t)(seg * p.len + pos) * 64 + (tid % 16) * 4)) = stage[seg][j];
      }
    }
  }
  __syncthreads();

  // ---- 5: the attention of row `wave` ----
  const int rows_total = M * p.heads;
  if(p.absmax_out && h == 0 && first_rows)   // slots past the last query row
    for(int sl = rows_total + tid; sl < kAbsmaxSlots; sl += kProjThreads) p.absmax_out[sl] = 0.0f;
  const int m = m_wave;
  if(wave < R && m < M) {   // (whole waves)
    const unsigned wr = (unsigned)m * (unsigned)p.heads + (unsigned)h;
    const unsigned entry = wr < p.batchKV ? wr : wr % p.batchKV;
    const float* kb = p.k_cache + (size_t)entry * p.kv_cap * 64;
    const float* vb = p.v_cache + (size_t)entry * p.kv_cap * 64;
    const float* q = proj_lds + wave * 64;
    const float* k_last = NPROJ == 3 ? proj_lds + (R + wave) * 64 : kb + (size_t)(p.len - 1) * 64;
    const float* v_last = NPROJ == 3 ? proj_lds + (2 * R + wave) * 64 : vb + (size_t)(p.len - 1) * 64;
    const int len4 = (p.len + 3) & ~3;
    float* sc = att_lds + wave * (len4 + 256);
    float omax;
    if constexpr(STAGED) {
      const float* ks = kv_lds + (size_t)(2 * (wave & ((1 << p.share_shift) - 1))) * p.len * 64;
      const float* vs = ks + (size_t)p.len * 64;
      using Rows = StagedRows<2 * PASSES>;
      omax = attention_row64_short<2 * PASSES>(q, Rows{ks, p.len, lane}, Rows{vs, p.len, lane}, mk, mk0, p.len, p.att_scale, sc, sc + len4,
                                               p.out + (size_t)wr * 64, lane);
    } else if constexpr(HELD > 0) {
      // (positions past the last one: it again, dropped by their weight)
      struct WithNewest {
        const v4f (&rows)[HELD];
        const float* newest;
        int len, lane;
        __device__ __forceinline__ void operator()(v4f (&r)[HELD]) const {
          const v4f last = reinterpret_cast<const v4f*>(newest)[lane % 16];
#pragma unroll
          for(int u = 0; u < HELD; ++u) r[u] = 4 * u + lane / 16 >= len - 1 ? last : rows[u];
        }
      };
      omax = attention_row64_short<HELD / 4>(q, WithNewest{held.k, k_last, p.len, lane}, WithNewest{held.v, v_last, p.len, lane}, mk, mk0, p.len, p.att_scale, sc,
                                             sc + len4, p.out + (size_t)wr * 64, lane);
    } else if constexpr(ANC) {
      omax = attention_row64<true>(q, p.k_cache, p.v_cache, k_last, v_last, mk, mk0, p.len, p.att_scale, sc, sc + len4,
                                          p.out + (size_t)wr * 64, lane, &anc);
    } else {
      omax = attention_row64(q, kb, vb, k_last, v_last, mk, mk0, p.len, p.att_scale, sc, sc + len4,
                             p.out + (size_t)wr * 64, lane);
    }
    if(p.absmax_out) {
      omax = wave_maxf(omax);
      if(lane == 0) p.absmax_out[wr] = omax;
    }
  }
}

// ---------------------------------------------------------------- n-best
// One workgroup of 1024 threads per row; a thread looks at every 1024th element (or group of
// four).  Scores are ordered by (value descending, index ascending).
//   1. every thread finds the largest of its scores, every wave the largest of its threads'; the
//      N-th largest of these 16 is a bound T: at least N elements of the row are >= T, so nothing
//      below T can be among the N best;
//   2. the row is read again (from cache) and the elements >= T - usually little more than N of
//      them - are collected in LDS with their positions;
//   3. the N best of the collected ones are found by rank (each candidate counts the candidates
//      before it), or drawn one at a time when there are more than 256.
// If more than 1024 elements pass the bound (large values concentrated in a few threads, or
// massive ties) every thread instead keeps the KEEP >= N best of its elements in registers and
// the draw pops them one by one.
constexpr int kNbestMax = 16;
constexpr int kNbestWaveCols = 2048;   // rows up to this length: a wave each (32 values a lane)
constexpr long long kNbestMaxBatch = 4096;     // batch entries of the beam-major form
// Its counters, 256 bytes apart: atomics on one cache line are served one after the other
// (measured: the 256 arrivals of 32 entries on one line cost 7 us).
constexpr int kNbestCounterStride = 64;
constexpr size_t kNbestCounterBytes = kNbestMaxBatch * kNbestCounterStride * 4;

__device__ __forceinline__ bool nbest_before(float v, unsigned i, float w, unsigned j) {
  return v > w || (v == w && i < j);
}

struct NbestShared {
  alignas(16) float val[16];
  unsigned idx[16];
  int who[16];
  int winner;
  int count;
  float cand_val[1024];
  unsigned cand_idx[1024];
};

// Workgroup-wide best of one (value, index) per thread; every thread gets the result and the id of
// the thread that held it.
__device__ __forceinline__ void nbest_arg_best(float v, unsigned i, NbestShared& sh, float& gv, unsigned& gi,
                                               int& gw) {
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
  float bv = v;
  unsigned bi = i;
  int bw = tid;
#pragma unroll
  for(int o = 32; o > 0; o >>= 1) {
    const float ov = __shfl_xor(bv, o, 64);
    const unsigned oi = (unsigned)__shfl_xor((int)bi, o, 64);
    const int ow = __shfl_xor(bw, o, 64);
    if(nbest_before(ov, oi, bv, bi)) {
      bv = ov; bi = oi; bw = ow;
    }
  }
  __syncthreads();   // the previous round's results have been read
  if(lane == 0) {
    sh.val[wave] = bv; sh.idx[wave] = bi; sh.who[wave] = bw;
  }
  __syncthreads();
  gv = sh.val[0]; gi = sh.idx[0]; gw = sh.who[0];
#pragma unroll
  for(int w = 1; w < 16; ++w)
    if(nbest_before(sh.val[w], sh.idx[w], gv, gi)) {
      gv = sh.val[w]; gi = sh.idx[w]; gw = sh.who[w];
    }
}

// One wave: the n best of `count` <= 64 (value, index) pairs, lane l's the l-th (lanes past them: any).
// A lane counts the pairs that come before its own, which it gets from registers: log-softmax and n-best of 13 x 5 hypotheses, 25 pairs
// each, 12.0 -> 11.4 us with these reads and without LDS in front of them, of 32 x 4 hypotheses 11.7 before and now.  The lanes of rank < n
// call emit(rank, ...) themselves, and ranks that no pair fills (count < n) are emitted as (-inf, none) by lane 0.
template <typename Emit>
__device__ __forceinline__ void nbest_small_draw(float v, unsigned ix, int count, int n, Emit emit) {
  const int lane = threadIdx.x % 64;
  int rank = 0;
  for(int c = 0; c < count; ++c) {   // (equal pairs - fillers (-inf, none) - rank in lane order)
    const float ov = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), c));
    const unsigned oi = (unsigned)__builtin_amdgcn_readlane((int)ix, c);
    rank += (nbest_before(ov, oi, v, ix) || (ov == v && oi == ix && c < lane)) ? 1 : 0;
  }
  if(lane < count && rank < n) emit(rank, v, ix);
  if(lane == 0)
    for(int r = count; r < n; ++r) emit(r, -__builtin_inff(), 0xFFFFFFFFu);
}

// Wave 0 only: draws the n best of the `count` <= 1024 (value, index) pairs in lv/li (LDS),
// sixteen per lane, without workgroup barriers.  emit(n, value, index) is called by lane 0.
template <typename Emit>
__device__ __forceinline__ void nbest_wave_draw(const float* lv, const unsigned* li, int count, int n,
                                                Emit emit) {
  const int lane = threadIdx.x % 64;
  const float ninf = -__builtin_inff();
  const unsigned none = 0xFFFFFFFFu;
  float v[16];
  unsigned ix[16];
#pragma unroll
  for(int j = 0; j < 16; ++j) {   // (clamped positions, dropped afterwards: all 32 loads in flight at once)
    const int e = min(j * 64 + lane, count - 1);
    v[j] = lv[e];
    ix[j] = li[e];
  }
#pragma unroll
  for(int j = 0; j < 16; ++j)
    if(j * 64 + lane >= count) {
      v[j] = ninf; ix[j] = none;
    }
  for(int r = 0; r < n; ++r) {
    float bv = v[0];
    unsigned bi = ix[0];
#pragma unroll
    for(int j = 1; j < 16; ++j)
      if(nbest_before(v[j], ix[j], bv, bi)) {
        bv = v[j]; bi = ix[j];
      }
    float gv = bv;
    unsigned gi = bi;
#pragma unroll
    for(int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(gv, o, 64);
      const unsigned oi = (unsigned)__shfl_xor((int)gi, o, 64);
      if(nbest_before(ov, oi, gv, gi)) {
        gv = ov; gi = oi;
      }
    }
    if(lane == 0) emit(r, gv, gi);
    // the holder drops it (indices are unique, so at most one entry matches)
#pragma unroll
    for(int j = 0; j < 16; ++j)
      if(ix[j] == gi && gi != none) {
        v[j] = ninf; ix[j] = none;
      }
  }
}

// The N best of x[0 .. rowLen), by the whole workgroup (1024 threads).  emit(r, value, index) is
// called once for r = 0 .. N-1 (best first) by one thread each; index is the position within x.
// scan(f) calls f(value, index) for every element this thread owns (each element of the row is
// owned by exactly one thread of the workgroup; the order does not matter).
// The N-th largest of 16 values in LDS (equal values in index order), the same in every thread: the four lanes l % 16 = c of a wave
// compare value c with four of them each, the lane whose rank is N - 1 has it (the cost does not grow with N; every wave of a
// workgroup of sixteen does this, and a lane to all sixteen comparisons took 1200 clocks of the launch more).
__device__ __forceinline__ float nth_largest_of_16(const float* w16, int N) {
  const int c = threadIdx.x % 16, row = threadIdx.x % 64 / 16;
  const float cvv = w16[c];
  const v4f four = reinterpret_cast<const v4f*>(w16)[row];
  unsigned rank = 0;
#pragma unroll
  for(int w = 0; w < 4; ++w) rank += (four[w] > cvv || (four[w] == cvv && 4 * row + w < c)) ? 1u : 0u;
  v2u_rows s = __builtin_amdgcn_permlane16_swap(rank, rank, false, false);   // (the sum over the four rows of sixteen lanes)
  s = __builtin_amdgcn_permlane32_swap(s.x + s.y, s.x + s.y, false, false);
  rank = s.x + s.y;
  const unsigned long long holders = __ballot(rank == (unsigned)(N - 1)) & 0xFFFFull;
  const int holder = holders ? __builtin_ctzll(holders) : 0;   // (ranks 0 .. 15 are all taken, but for NaN among the values)
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)__float_as_uint(cvv), holder));
}

// Step 3, all threads: the N best of what has been collected, or of all that scan goes over where that was too much.
template <int KEEP, typename Scan, typename Emit>
__device__ __forceinline__ void nbest_of_collected(Scan scan, int N, NbestShared& sh, Emit emit) {
  const int tid = threadIdx.x;
  const float ninf = -__builtin_inff();
  const unsigned none = 0xFFFFFFFFu;
  __syncthreads();
  const int count = sh.count;

  if(__builtin_expect(count <= 1024, 1)) {   // (the draws stand here, what follows them behind: a launch fetches its code)
    // 3. the N best of the collected elements, drawn by wave 0: up to 64, one per lane; more,
    //    sixteen per lane
    if(__builtin_expect(count <= 64, 1)) {
      if(tid < 64) {   // (no candidates - a row of NaN -: lane 0 emits fillers)
        const int e = max(min(tid, count - 1), 0);
        nbest_small_draw(sh.cand_val[e], sh.cand_idx[e], count, N, emit);
      }
    } else if(count <= 256) {
      // up to 256 (long lists): thread t ranks candidate t among all of them (distinct elements)
      if(tid < count) {
        const float v = sh.cand_val[tid];
        const unsigned ix = sh.cand_idx[tid];
        int rank = 0;
        for(int c = 0; c < count; ++c) rank += nbest_before(sh.cand_val[c], sh.cand_idx[c], v, ix) ? 1 : 0;
        if(rank < N) emit(rank, v, ix);
      }
    } else if(tid < 64) {
      nbest_wave_draw(sh.cand_val, sh.cand_idx, count, N, emit);
    }
    return;
  }

  // too many at or before the bound: per-thread sorted lists of the KEEP best, popped by the draw
  float val[KEEP];
  unsigned idx[KEEP];
#pragma unroll
  for(int j = 0; j < KEEP; ++j) {
    val[j] = ninf;
    idx[j] = none;
  }
  scan([&](float v, unsigned i) {
    if(nbest_before(v, i, val[KEEP - 1], idx[KEEP - 1])) {
      val[KEEP - 1] = v;
      idx[KEEP - 1] = i;
#pragma unroll
      for(int j = KEEP - 1; j > 0; --j) {
        if(nbest_before(val[j], idx[j], val[j - 1], idx[j - 1])) {
          const float sv = val[j]; val[j] = val[j - 1]; val[j - 1] = sv;
          const unsigned si = idx[j]; idx[j] = idx[j - 1]; idx[j - 1] = si;
        }
      }
    }
  });
  for(int n = 0; n < N; ++n) {
    float gv; unsigned gi; int who;
    nbest_arg_best(val[0], idx[0], sh, gv, gi, who);
    if(tid == 0) emit(n, gv, gi);
    if(tid == who) {   // pop the head
#pragma unroll
      for(int j = 0; j < KEEP - 1; ++j) {
        val[j] = val[j + 1];
        idx[j] = idx[j + 1];
      }
      val[KEEP - 1] = ninf;
      idx[KEEP - 1] = none;
    }
  }
}

// Step 2: what reaches tv, a bound that at least N elements of the row reach (or -inf).  sh.count has been zero since a workgroup barrier.
template <typename Scan>
__device__ __forceinline__ void nbest_collect(Scan scan, NbestShared& sh, float tv) {
  scan([&](float v, unsigned i) {
    if(v >= tv) {
      const int slot = atomicAdd(&sh.count, 1);
      if(slot < 1024) {
        sh.cand_val[slot] = v; sh.cand_idx[slot] = i;
      }
    }
  });
}

// Steps 2 and 3.
template <int KEEP, typename Scan, typename Emit>
__device__ __forceinline__ void nbest_from_bound(Scan scan, int N, NbestShared& sh, Emit emit, float tv) {
  if(threadIdx.x == 0) sh.count = 0;
  __syncthreads();
  nbest_collect(scan, sh, tv);
  nbest_of_collected<KEEP>(scan, N, sh, emit);
}

template <int KEEP, typename Scan, typename Emit>
__device__ __forceinline__ void nbest_core(Scan scan, int N, NbestShared& sh, Emit emit) {
  const int tid = threadIdx.x;
  // 1. largest score of this thread, of its wave, and the N-th largest of the 16 wave maxima: the
  //    bound T.  The maxima belong to 16 distinct elements and N <= 16, so at least N elements of the
  //    row are >= T; for N = 16 and scores without structure some 50 are.  (A wave without elements
  //    contributes -inf; with fewer than N waves that hold elements the bound is -inf and
  //    everything passes.)
  float mv = -__builtin_inff();
  scan([&](float v, unsigned) { mv = fmaxf(mv, v); });
  const float wv = wave_maxf(mv);
  if(tid % 64 == 0) sh.val[tid / 64] = wv;
  __syncthreads();
  const float tv = nth_largest_of_16(sh.val, N);
  nbest_from_bound<KEEP>(scan, N, sh, emit, tv);
}

// The row in memory.  (Every scan keeps eight 16-byte loads in flight per thread; the last round
// reads clamped positions unconditionally and drops them afterwards, because loads behind a range
// check would be waited for one by one.)
template <int KEEP, typename Emit>
__device__ __forceinline__ void nbest_of_row(const float* __restrict__ x, long long rowLen, int N,
                                             NbestShared& sh, Emit emit) {
  const int tid = threadIdx.x;
  const bool vec = (rowLen % 4) == 0 && (reinterpret_cast<uintptr_t>(x) % 16) == 0;
  const long long n4 = rowLen / 4;
  auto scan = [&](auto f) __attribute__((always_inline)) {
    if(vec) {   // elements 4 * (t + 1024 * j) .. + 3
      const v4f* x4 = reinterpret_cast<const v4f*>(x);
      for(long long i = tid; i < n4; i += 8 * 1024) {
        v4f v[8];
#pragma unroll
        for(int u = 0; u < 8; ++u) v[u] = x4[min(i + u * 1024, n4 - 1)];
#pragma unroll
        for(int u = 0; u < 8; ++u) {
          if(i + u * 1024 >= n4) break;
          const unsigned b = (unsigned)(4 * (i + u * 1024));
          f(v[u].x, b); f(v[u].y, b + 1); f(v[u].z, b + 2); f(v[u].w, b + 3);
        }
      }
    } else {
      for(long long i = tid; i < rowLen; i += 16 * 1024) {
        float v[16];
#pragma unroll
        for(int u = 0; u < 16; ++u) v[u] = x[min(i + u * 1024, rowLen - 1)];
#pragma unroll
        for(int u = 0; u < 16; ++u)
          if(i + u * 1024 < rowLen) f(v[u], (unsigned)(i + u * 1024));
      }
    }
  };
  nbest_core<KEEP>(scan, N, sh, emit);
}

// Where the winners of a row go: keys = absolute positions (uint32), or words = the positions within the
// row, taken through ids where a shortlist gave the columns (a filler's position -1 is then the last
// column, as an index counted from the end).
struct NbestOut {
  float* scores;
  unsigned* keys;        // one of the two is set
  long long* words;
  const uint32_t* ids;   // or null
  __device__ __forceinline__ void put(long long row, long long rowLen, int N, int r, float v, unsigned i) const {
    scores[row * N + r] = v;
    if(keys) {
      keys[row * N + r] = (unsigned)(row * rowLen) + i;
    } else {
      const long long at = (int)i == -1 ? -1 : (long long)i;
      words[row * N + r] = ids ? (long long)(int)ids[at < 0 ? rowLen - 1 : at] : at;
    }
  }
};

template <int KEEP>
__global__ __launch_bounds__(1024) void nbest_kernel(const float* __restrict__ scores, long long rowLen, int N, NbestOut out) {
  __shared__ NbestShared sh;
  const long long row = blockIdx.x;
  nbest_of_row<KEEP>(scores + row * rowLen, rowLen, N, sh, [&](int r, float v, unsigned i) { out.put(row, rowLen, N, r, v, i); });
}

// Short rows (a shortlist's columns): one wave to a row, 64 * VPT elements in registers, no workgroup
// barrier.  What bounds the launch is its chain - load, bound, collection, draw - and not the bytes.
// The bound is the N-th largest of the 64 lane maxima (N elements reach it); what reaches it is
// collected by ballots, normally N to 2 N elements, and ranked one to a lane.  More than 64 (rows of
// equal or infinite values): drawn one by one, each the best element behind the one before.
template <int VPT>
__global__ __launch_bounds__(64) void nbest_wave_kernel(const float* __restrict__ scores, int rowLen, int N, NbestOut out) {
  __shared__ float cand_val[64];
  __shared__ unsigned cand_idx[64];
  const int lane = threadIdx.x;
  const long long row = blockIdx.x;
  const float* x = scores + row * rowLen;
  const float ninf = -__builtin_inff();
  const unsigned none = 0xFFFFFFFFu;
  float v[VPT];
#pragma unroll
  for(int j = 0; j < VPT; ++j) v[j] = x[min(j * 64 + lane, rowLen - 1)];
#pragma unroll
  for(int j = 0; j < VPT; ++j)
    if(j * 64 + lane >= rowLen) v[j] = __builtin_nanf("");   // (reaches no bound and comes before nothing)
  float mv = ninf;
#pragma unroll
  for(int j = 0; j < VPT; ++j) mv = fmaxf(mv, v[j]);
  float tv = ninf;
  for(int r = 0; r < N; ++r) {
    tv = wave_maxf(mv);
    const unsigned long long holders = __ballot(mv == tv);
    if(lane == __ffsll((long long)holders) - 1) mv = ninf;
  }
  int count = 0;
#pragma unroll
  for(int j = 0; j < VPT; ++j) {
    const unsigned long long m = __ballot(v[j] >= tv);
    if(m) {
      const int at = count + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
      if(v[j] >= tv && at < 64) {
        cand_val[at] = v[j]; cand_idx[at] = (unsigned)(j * 64 + lane);
      }
      count += __popcll(m);
    }
  }
  if(count <= 64) {
    __syncthreads();   // (one wave: orders the LDS accesses)
    const float cv = lane < count ? cand_val[lane] : ninf;
    const unsigned ci = lane < count ? cand_idx[lane] : none;
    int rank = 0;
    for(int c = 0; c < count; ++c) {
      const float ov = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(cv), c));
      rank += nbest_before(ov, (unsigned)__builtin_amdgcn_readlane((int)ci, c), cv, ci) ? 1 : 0;
    }
    if(lane < count && rank < N) out.put(row, rowLen, N, rank, cv, ci);
    if(lane >= count && lane < N) out.put(row, rowLen, N, lane, ninf, none);   // (NaN in the row: fewer than N candidates)
    return;
  }
  float pv = __builtin_inff();
  unsigned pi = 0;
  for(int r = 0; r < N; ++r) {
    float bv = ninf;
    unsigned bi = none;
#pragma unroll
    for(int j = 0; j < VPT; ++j) {
      const unsigned i = (unsigned)(j * 64 + lane);
      if((r == 0 || nbest_before(pv, pi, v[j], i)) && nbest_before(v[j], i, bv, bi)) {
        bv = v[j]; bi = i;
      }
    }
#pragma unroll
    for(int o = 32; o > 0; o >>= 1) {
      const float ov = __shfl_xor(bv, o, 64);
      const unsigned oi = (unsigned)__shfl_xor((int)bi, o, 64);
      if(nbest_before(ov, oi, bv, bi)) {
        bv = ov; bi = oi;
      }
    }
    if(lane == 0) out.put(row, rowLen, N, r, bv, bi);
    pv = bv;
    pi = bi;
  }
}

// Hand-over of per-part candidates to the workgroup that finishes an entry last, without fences.
// What it relies on (gfx942/gfx950 memory model as the AMDGPU backend documents it): an agent-scope
// store or atomic bypasses the XCD-local L2 and is performed at the memory side, where all XCDs see
// it; a wave's vmcnt reaches zero only once each of its stores has been acknowledged from there; an
// agent-scope load reads from there too.  So: candidates stored (agent scope) -> vmcnt(0) in every
// wave -> workgroup barrier -> counter incremented; the workgroup that reads parts - 1 from the
// counter then loads (agent scope) candidates that are all in memory already.  FENCED makes the
// counter update an acquire-release operation instead (the compiler then adds the cache write-back /
// invalidate the language-level memory model asks for; ~8 us slower).  The tuning build holds both
// forms (marian_hip_nbest_set_fenced) and a GPU test compares them: if results ever differ, the
// hand-over is at fault and not the selection.  rowLen: length of an entry's whole row (keys are
// b * rowLen + position).
template <bool FENCED>
__device__ __forceinline__ void nbest_hand_over(NbestShared& sh, int* is_last, long long b, int parts, int N,
                                                long long rowLen, float* candVal, unsigned* candIdx,
                                                unsigned* counters, float* __restrict__ outScores,
                                                unsigned* __restrict__ outKeys) {
  constexpr int kCounterOrder = FENCED ? __ATOMIC_ACQ_REL : __ATOMIC_RELAXED;
  const int total = parts * N;
  auto arrive = [&]() __attribute__((always_inline)) {
    return __hip_atomic_fetch_add(&counters[b * kNbestCounterStride], 1u, kCounterOrder, __HIP_MEMORY_SCOPE_AGENT) == (unsigned)(parts - 1);
  };
  auto result = [&](int r, float v, unsigned i) __attribute__((always_inline)) {
    outScores[b * N + r] = v;
    outKeys[b * N + r] = (unsigned)(b * rowLen) + i;
  };
  // an entry's candidate, read past this XCD's caches
  auto value_at = [&](int e) __attribute__((always_inline)) {
    return __hip_atomic_load(candVal + (size_t)b * total + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto index_at = [&](int e) __attribute__((always_inline)) {
    return __hip_atomic_load(candIdx + (size_t)b * total + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  auto reset = [&]() __attribute__((always_inline)) {   // for the next call (every part of this entry has arrived: nobody else touches it)
    __hip_atomic_store(&counters[b * kNbestCounterStride], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // every wave's stores have reached memory ...
  __syncthreads();                                   // ... before the count goes up
  if(total <= 64) {   // few candidates: one wave, without LDS and barriers in between
    if(threadIdx.x >= 64) return;
    int last = 0;
    if(threadIdx.x == 0) last = arrive();
    if(!__builtin_amdgcn_readfirstlane(last)) return;
    asm volatile("" ::: "memory");   // (the candidates are asked for behind the answer)
    const int e = min((int)threadIdx.x, total - 1);
    nbest_small_draw(value_at(e), index_at(e), total, N, result);
    if(threadIdx.x == 0) reset();
    return;
  }
  if(threadIdx.x == 0) *is_last = arrive();
  __syncthreads();
  if(!*is_last) return;
  for(int e = threadIdx.x; e < total; e += 1024) {   // (at most 1024)
    sh.cand_val[e] = value_at(e);
    sh.cand_idx[e] = index_at(e);
  }
  __syncthreads();
  if(threadIdx.x < 64) {
    nbest_wave_draw(sh.cand_val, sh.cand_idx, total, N, result);
    if(threadIdx.x == 0) reset();
  }
}

// Beam-major scores [beam, dimBatch, vocab]; the row of batch entry b is the beam's `beam` segments
// of `vocab` scores, element (k, v) at logical position k * vocab + v.  Workgroup (part, b) takes
// slice part % perSeg of segment part / perSeg and leaves the N best of it, with their logical
// positions, in cand*[(b * parts + part) * N ..]; a slice shorter than N fills up with
// (-inf, none), which sorts last.  The workgroup that finishes last for a batch entry (a counter per
// entry, zero between calls) draws the N best of all the entry's candidates.  No workgroup waits
// for another.
template <int KEEP, bool FENCED = false>
__global__ __launch_bounds__(1024) void nbest_part_kernel(const float* __restrict__ scores, long long dimBatch,
                                                          long long vocab, int perSeg, long long sliceLen,
                                                          int N, int parts, float* candVal, unsigned* candIdx,
                                                          unsigned* counters, float* __restrict__ outScores,
                                                          unsigned* __restrict__ outKeys) {
  __shared__ NbestShared sh;
  __shared__ int is_last;
  const int part = blockIdx.x;
  const long long b = blockIdx.y;
  const long long k = part / perSeg, v0 = (long long)(part % perSeg) * sliceLen;
  const long long len = min(sliceLen, vocab - v0);
  float* cv = candVal + ((size_t)b * parts + part) * N;
  unsigned* ci = candIdx + ((size_t)b * parts + part) * N;
  // Every path below publishes the candidates with stores that go through to memory
  // (device scope), so that whichever workgroup turns out to be the last can read them without a
  // cache write-back and invalidation around the counter (a fence pair costs ~8 us here).
  auto publish = [&](int r, float v, unsigned i) {
    __hip_atomic_store(cv + r, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ci + r, i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  };
  if(len < N) {   // (only a ragged last slice can be this short: one thread sorts it)
    if(threadIdx.x == 0) {
      const float* x = scores + ((size_t)k * dimBatch + b) * vocab + v0;
      float pv = __builtin_inff();
      long long pi = -1;
      for(int r = 0; r < N; ++r) {
        float bv = -__builtin_inff();
        long long bi = -1;
        for(long long c = 0; c < len; ++c) {
          const float v = x[c];
          const bool after_prev = r == 0 || v < pv || (v == pv && c > pi);
          if(after_prev && (bi < 0 || v > bv)) {
            bv = v; bi = c;
          }
        }
        publish(r, bi < 0 ? -__builtin_inff() : bv, bi < 0 ? 0xFFFFFFFFu : (unsigned)(k * vocab + v0 + bi));
        if(bi >= 0) { pv = bv; pi = bi; }
      }
    }
  } else {
    const unsigned base = (unsigned)(k * vocab + v0);
    nbest_of_row<KEEP>(scores + ((size_t)k * dimBatch + b) * vocab + v0, len, N, sh,
                       [&](int r, float v, unsigned i) { publish(r, v, base + i); });
  }
  nbest_hand_over<FENCED>(sh, &is_last, b, parts, N, (long long)(parts / perSeg) * vocab, candVal, candIdx, counters,
                  outScores, outKeys);
}

// Log-softmax of the rows of beam-major logits [beam, dimBatch, vocab] and the N best of every
// batch entry's beam * vocab log-probabilities in one launch: workgroup (k, b) keeps row (k, b) in
// registers (read once), computes the log-probabilities exactly as softmax_wide_kernel<true> does
// (optionally adds the row's path score and optionally writes them out), selects the N best of the
// row from the registers and leaves them as part k of entry b; the workgroup that finishes an
// entry last draws the N best of its beam * N candidates.
template <int VPT, int KEEP, bool FENCED = false>
__global__ __launch_bounds__(1024) void logsoftmax_nbest_kernel(const float* __restrict__ in,
                                                                const float* __restrict__ rowAdd,
                                                                float* __restrict__ lpOut, long long dimBatch,
                                                                int vocab, int N, int parts, float* candVal,
                                                                unsigned* candIdx, unsigned* counters,
                                                                float* __restrict__ outScores,
                                                                unsigned* __restrict__ outKeys) {
  __shared__ NbestShared sh;
  __shared__ int is_last;
  __shared__ __attribute__((aligned(16))) float red[32];
  const int k = blockIdx.x, t = threadIdx.x;
  const long long b = blockIdx.y;
  const size_t row = (size_t)k * dimBatch + b;
  const int cols4 = vocab / 4;
  v4f v[VPT];
  if(t == 0) sh.count = 0;   // (the selection starts behind the barriers of the two reductions)
  // The selection's bound comes out of the softmax's own maximum: the N-th largest of the 16 wave
  // maxima of the logits (at least N logits reach it), taken through the same operations as every
  // element below, which are monotonic, so at least N scores reach the result.
  float bound_logit = -__builtin_inff(), row_max = 0.0f, own_max = 0.0f;
  const float log_sum = softmax_wide_row<true, 1024, VPT>(
      reinterpret_cast<const v4f*>(in + row * vocab), nullptr, cols4, v, red, [&](float mx, const float* wave_max, float own) {
        row_max = mx;
        own_max = own;
        bound_logit = nth_largest_of_16(wave_max, N);
      });
  const float add = rowAdd ? rowAdd[row] : -0.0f;   // (the number that changes none)
  auto score = [&](float x) __attribute__((always_inline)) { return (x - log_sum) + add; };
  const float tv = score(bound_logit - row_max);
  if(lpOut) {
#pragma unroll
    for(int j = 0; j < VPT; ++j)
      if(j * 1024 + t < cols4)
        reinterpret_cast<v4f*>(lpOut + row * vocab)[j * 1024 + t] = v4f{v[j].x - log_sum, v[j].y - log_sum, v[j].z - log_sum, v[j].w - log_sum};
  }
  auto scan = [&](auto f) __attribute__((always_inline)) {
#pragma unroll
    for(int j = 0; j < VPT; ++j) {
      const int i4 = j * 1024 + t;
      if(i4 < cols4) {
        const unsigned e = 4u * (unsigned)i4;
        f(score(v[j].x), e); f(score(v[j].y), e + 1); f(score(v[j].z), e + 2); f(score(v[j].w), e + 3);
      }
    }
  };
  // What reaches the bound lies in few threads, those whose largest score does (of N waves, but for equal scores).  Where it is one or two of a
  // wave, each one's values take a turn through LDS to a lane each, which appends those that reach it; of more, every thread goes through its own.
  // (Times of recorded launches, N best of so many rows and words: every thread of all waves through its own, a turn for each of a wave's threads, and
  // so: 128 x 32000, N = 1 8.7, 7.1, 7.1 us; 4 8.7, 7.7, 7.8; 6 9.0, 8.3, 8.2; 12 10.4, 11.0, 9.8; 16 19.3, 23.9, 18.5.  6 x 32000, N = 1 8.2, 6.7, 6.7; 16 15.0, 17.2, 14.1.  65 x 8000 with every eighth
  // word the best, N = 1 8.8, 37.4, 7.9; 6 13.5, 42.7, 12.7: turns follow one another, 2000 clocks each where all sixteen waves have some.  One turn at the most is 0 - 3 % ahead of
  // two there and behind them where other launches ran before and the code is cold: in a step of 6 hypotheses 10.5 and 9.5 us, of 65 11.1 and 10.3.)
  __shared__ __attribute__((aligned(16))) float turn[16][4 * VPT];
  static_assert(4 * VPT <= 64, "a lane for each of a thread's values");
  const unsigned long long reaching = __ballot(score(own_max - row_max) >= tv);   // (whole waves)
  if(__builtin_expect(__popcll(reaching) > 2, 0)) {
    nbest_collect(scan, sh, tv);
  } else {
    for(unsigned long long todo = reaching; todo; todo &= todo - 1) {
      const int from = __builtin_ctzll(todo), lane = t % 64, i = min(lane, 4 * VPT - 1);
      if(lane == from) {
#pragma unroll
        for(int j = 0; j < VPT; ++j) reinterpret_cast<v4f*>(turn[t / 64])[j] = v[j];
      }
      // (a wave's LDS operations keep their order)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const float sv = score(turn[t / 64][i]);
      const int i4 = i / 4 * 1024 + t - lane + from;
      const unsigned long long reached = __ballot(lane == i && i4 < cols4 && sv >= tv);
      int slot = 0;
      if(lane == 0) slot = atomicAdd(&sh.count, (int)__popcll(reached));
      slot = __builtin_amdgcn_readfirstlane(slot) + (int)__builtin_amdgcn_mbcnt_hi((unsigned)(reached >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)reached, 0u));
      if((reached >> lane & 1) && slot < 1024) {
        sh.cand_val[slot] = sv; sh.cand_idx[slot] = 4u * (unsigned)i4 + (unsigned)i % 4u;
      }
      __builtin_amdgcn_wave_barrier();
    }
  }
  float* cv = candVal + ((size_t)b * parts + k) * N;
  unsigned* ci = candIdx + ((size_t)b * parts + k) * N;
  const unsigned base = (unsigned)k * (unsigned)vocab;
  nbest_of_collected<KEEP>(scan, N, sh, [&](int r, float val, unsigned i) {
    __hip_atomic_store(cv + r, val, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __hip_atomic_store(ci + r, base + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  });
  nbest_hand_over<FENCED>(sh, &is_last, b, parts, N, (long long)parts * vocab, candVal, candIdx, counters, outScores, outKeys);
}

// Fill: the 16-byte aligned middle of the range with 16-byte stores of the repeated pattern, the
// bytes before and after it one by one (byte i of the range holds byte i % elem_bytes of the
// pattern; the middle starts on an element boundary because the range does).
__global__ __launch_bounds__(256) void fill_kernel(unsigned char* __restrict__ p, long long bytes, long long head,
                                                   long long vecs, int elem_bytes, unsigned long long pattern, int blocks) {
  const long long tid = (long long)blockIdx.x * 256 + threadIdx.x, nthreads = (long long)blocks * 256;
  unsigned long long rep = pattern;
  if(elem_bytes == 1) rep = (pattern & 0xFFull) * 0x0101010101010101ull;
  else if(elem_bytes == 2) rep = (pattern & 0xFFFFull) * 0x0001000100010001ull;
  else if(elem_bytes == 4) rep = (pattern & 0xFFFFFFFFull) * 0x0000000100000001ull;
  typedef unsigned long long v2u64 __attribute__((ext_vector_type(2)));
  v2u64* mid = reinterpret_cast<v2u64*>(p + head);
  for(long long i = tid; i < vecs; i += nthreads) mid[i] = v2u64{rep, rep};
  const long long tail0 = head + vecs * 16;
  for(long long i = tid; i < head + (bytes - tail0); i += nthreads) {
    const long long at = i < head ? i : tail0 + (i - head);
    p[at] = (unsigned char)(pattern >> (8 * (at % elem_bytes)));
  }
}

// ---------------------------------------------------------------- embedding step
// Workgroup (r, chunk) takes kEmbedChunk values of output row r: out[r, :] = scale * E[ids[r], :]
// (+ signal[(r / rows_per_signal) % n_signals, :]); rows of an embedding table are one chunk, the
// long rows of a decoder state (all cached positions of a hypothesis) many, so that such a gather
// fills the chip.  The product and the sum round separately.  An id at or past the table's end
// reads the table's last row.
constexpr int kEmbedChunk = 4096;
template <bool VEC>
__global__ __launch_bounds__(256) void embed_kernel(const float* __restrict__ E, const uint32_t* __restrict__ ids,
                                                    unsigned vocab, int dimEmb, float scale,
                                                    const float* __restrict__ signal, unsigned rows_per_signal,
                                                    unsigned n_signals, float* __restrict__ out,
                                                    float* __restrict__ absmax_out, unsigned rows, unsigned chunks) {
  __shared__ float red[4];
  const unsigned row = blockIdx.x, chunk = blockIdx.y;
  const int tid = threadIdx.x;
  unsigned id = ids[row];
  id = id < vocab ? id : vocab - 1u;
  const int c0 = (int)chunk * kEmbedChunk, c1 = min(c0 + kEmbedChunk, dimEmb);
  const float* src = E + (size_t)id * dimEmb;
  const float* sg = signal ? signal + (size_t)((row / rows_per_signal) % n_signals) * dimEmb : nullptr;
  float* y = out + (size_t)row * dimEmb;
  float omax = 0.0f;
  if(VEC) {   // (four 16-byte loads per thread and operand, all requested before the first is used)
    constexpr int kV = kEmbedChunk / 4 / 256;
    const int last = c1 / 4 - 1;
    v4f e[kV], s[kV];
#pragma unroll
    for(int j = 0; j < kV; ++j) {
      const int i = min(c0 / 4 + j * 256 + tid, last);
      e[j] = reinterpret_cast<const v4f*>(src)[i];
      s[j] = sg ? reinterpret_cast<const v4f*>(sg)[i] : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    }
#pragma unroll
    for(int j = 0; j < kV; ++j) {
      const int i = c0 / 4 + j * 256 + tid;
      if(i <= last) {
        v4f r = v4f{scale * e[j].x, scale * e[j].y, scale * e[j].z, scale * e[j].w};
        if(sg) r = v4f{r.x + s[j].x, r.y + s[j].y, r.z + s[j].z, r.w + s[j].w};
        omax = fmaxf(fmaxf(omax, fmaxf(fabsf(r.x), fabsf(r.y))), fmaxf(fabsf(r.z), fabsf(r.w)));
        reinterpret_cast<v4f*>(y)[i] = r;
      }
    }
  } else {
    for(int i = c0 + tid; i < c1; i += 256) {
      float r = scale * src[i];
      if(sg) r = r + sg[i];
      omax = fmaxf(omax, fabsf(r));
      y[i] = r;
    }
  }
  if(absmax_out) {   // a slot per workgroup; the first workgroup zeroes the slots past the last one
    const unsigned slot = row * chunks + chunk, slots = rows * chunks;
    omax = row_reduce<256, true>(omax, red);
    if(tid == 0) absmax_out[slot] = omax;
    if(slot == 0)
      for(int sl = (int)slots + tid; sl < kAbsmaxSlots; sl += 256) absmax_out[sl] = 0.0f;
  }
}

// The selection of decoder states whose entries are `segs` segments of seg_cap values of which the
// first seg_len are in use (cached positions of the heads of a hypothesis): workgroup (r * segs + s,
// chunk) copies kEmbedChunk values of segment s of entry ids[r]; what lies behind seg_len is neither
// read nor written.
template <bool VEC>
__global__ __launch_bounds__(256) void select_state_kernel(const float* __restrict__ in, const uint32_t* __restrict__ ids,
                                                           unsigned entries, unsigned segs, long long seg_cap,
                                                           int seg_len, float* __restrict__ out) {
  const unsigned row = blockIdx.x / segs, seg = blockIdx.x % segs, chunk = blockIdx.y;
  const int tid = threadIdx.x;
  unsigned id = ids[row];
  id = id < entries ? id : entries - 1u;
  const int c0 = (int)chunk * kEmbedChunk, c1 = min(c0 + kEmbedChunk, seg_len);
  const float* src = in + ((size_t)id * segs + seg) * (size_t)seg_cap;
  float* dst = out + ((size_t)row * segs + seg) * (size_t)seg_cap;
  if(VEC) {
    constexpr int kV = kEmbedChunk / 4 / 256;
    const int last = c1 / 4 - 1;
    v4f e[kV];
#pragma unroll
    for(int j = 0; j < kV; ++j) e[j] = reinterpret_cast<const v4f*>(src)[min(c0 / 4 + j * 256 + tid, last)];
#pragma unroll
    for(int j = 0; j < kV; ++j) {
      const int i = c0 / 4 + j * 256 + tid;
      if(i <= last) reinterpret_cast<v4f*>(dst)[i] = e[j];
    }
  } else {
    for(int i = c0 + tid; i < c1; i += 256) dst[i] = src[i];
  }
}

__global__ __launch_bounds__(256) void zero_words_kernel(unsigned* __restrict__ p, long long n, int blocks) {
  for(long long i = (long long)blockIdx.x * 256 + threadIdx.x; i < n; i += (long long)blocks * 256)
    p[i] = 0u;
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) % 16) == 0; }
inline bool aligned4(const void* p) { return (reinterpret_cast<uintptr_t>(p) % 4) == 0; }

#define MH_HIP(expr)                                      \
  do {                                                    \
    hipError_t e_ = (expr);                               \
    if(e_ != hipSuccess) return record_hip_error((int)e_); \
  } while(0)

// Which form of the n-best hand-over the launchers take: the shipped library has the unfenced one
// only; the tuning build holds both behind a process-wide switch.
#ifdef MARIAN_HIP_TUNING
std::atomic<int> g_nbest_fenced{0};
inline bool nbest_fenced() { return g_nbest_fenced.load(std::memory_order_relaxed) != 0; }
#else
constexpr bool nbest_fenced() { return false; }
#endif

}  // namespace

extern "C" {

#ifdef MARIAN_HIP_TUNING
int marian_hip_nbest_set_fenced(int on) { return g_nbest_fenced.exchange(on ? 1 : 0); }
#endif

int marian_hip_layer_norm(const float* in, const float* add, const float* gamma, int64_t gamma_cols,
                          const float* beta, int64_t beta_cols, float* out, int64_t rows,
                          int64_t cols, float eps, float* absmax_out, void* stream) {
  if(absmax_out && !aligned4(absmax_out)) return MARIAN_HIP_ERR_ALIGN;
  if(rows < 0 || cols <= 0) return MARIAN_HIP_ERR_SHAPE;
  if((gamma_cols != cols && gamma_cols != 1) || (beta && beta_cols != cols && beta_cols != 1))
    return MARIAN_HIP_ERR_SHAPE;
  if(rows == 0) return MARIAN_HIP_OK;
  if(!in || !gamma || !out) return MARIAN_HIP_ERR_NULL;
  if(rows * cols > kMaxElemsOps) return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(in) || !aligned4(out) || !aligned4(gamma) || (add && !aligned4(add)) || (beta && !aligned4(beta)))
    return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const int gs = gamma_cols > 1 ? 1 : 0, bs = (beta && beta_cols > 1) ? 1 : 0;
  const bool vec = cols % 4 == 0 && aligned16(in) && aligned16(out) && (!add || aligned16(add));
  const bool wave_form = vec && cols <= 1024 && (gs == 0 || aligned16(gamma)) &&
                         (!beta || bs == 0 || aligned16(beta));
  // more rows than abs-max slots (an encoder's sentence batch): the wave form deals the rows out over as many
  // workgroups as there are slots; the others share the slots, which are cleared first (a kernel, so that
  // the call may sit in a recorded graph)
  const int wrap = absmax_out && rows > kAbsmaxSlots ? 1 : 0;
  if(wave_form) {
    const int blocks = wrap ? (rows + 3 < 4 * (int64_t)kAbsmaxSlots ? (int)((rows + 3) / 4) : kAbsmaxSlots) : (int)rows;
#define MH_NORM(MANY, PLAIN)                                                                                                       \
  MH_LAUNCH((layer_norm_wave_kernel<MANY, PLAIN>), dim3((unsigned)blocks), dim3(MANY ? 256 : 64), 0, st, in, add, gamma, gs, beta, bs, out, \
            (int)cols, eps, absmax_out, blocks, (int)rows)
    const bool plain = add && gs && beta && bs;
    if(wrap && plain) MH_NORM(true, true);
    else if(wrap) MH_NORM(true, false);
    else if(plain) MH_NORM(false, true);
    else MH_NORM(false, false);
#undef MH_NORM
    MH_HIP(hipGetLastError());
    return MARIAN_HIP_OK;
  }
  if(wrap) {
    MH_LAUNCH(zero_words_kernel, dim3(kAbsmaxSlots / 256), dim3(256), 0, st, reinterpret_cast<unsigned*>(absmax_out),
                       (long long)kAbsmaxSlots, kAbsmaxSlots / 256);
    MH_HIP(hipGetLastError());
  }
  if(vec && cols <= 1024)
    MH_LAUNCH(layer_norm_kernel<1>, dim3((unsigned)rows), dim3(256), 0, st, in, add, gamma, gs, beta, bs, out, (int)cols, eps, absmax_out, wrap, (int)rows);
  else if(vec && cols <= 4096)
    MH_LAUNCH(layer_norm_kernel<4>, dim3((unsigned)rows), dim3(256), 0, st, in, add, gamma, gs, beta, bs, out, (int)cols, eps, absmax_out, wrap, (int)rows);
  else if(vec && cols <= 8192)
    MH_LAUNCH(layer_norm_kernel<8>, dim3((unsigned)rows), dim3(256), 0, st, in, add, gamma, gs, beta, bs, out, (int)cols, eps, absmax_out, wrap, (int)rows);
  else
    MH_LAUNCH(layer_norm_kernel<0>, dim3((unsigned)rows), dim3(256), 0, st, in, add, gamma, gs, beta, bs, out, (int)cols, eps, absmax_out, wrap, (int)rows);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_embed(const float* E, const uint32_t* ids, int64_t rows, int64_t vocab, int64_t dimEmb,
                     float scale, const float* signal, int64_t rows_per_signal, int64_t n_signals,
                     float* out, float* absmax_out, void* stream) {
  if(rows < 0 || vocab <= 0 || dimEmb <= 0) return MARIAN_HIP_ERR_SHAPE;
  const int64_t chunks = (dimEmb + kEmbedChunk - 1) / kEmbedChunk;
  if(absmax_out && rows * chunks > kAbsmaxSlots) return MARIAN_HIP_ERR_RANGE;
  if(absmax_out && !aligned4(absmax_out)) return MARIAN_HIP_ERR_ALIGN;
  if(signal && (rows_per_signal <= 0 || n_signals <= 0)) return MARIAN_HIP_ERR_SHAPE;
  if(rows == 0) return MARIAN_HIP_OK;
  if(!E || !ids || !out) return MARIAN_HIP_ERR_NULL;
  if(chunks > 65535 || rows * dimEmb > kMaxElemsOps || vocab > 0xFFFFFFFFLL || rows_per_signal > 0x7FFFFFFFLL ||
     n_signals > 0x7FFFFFFFLL || (signal && n_signals * dimEmb > kMaxElemsOps))
    return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(E) || !aligned4(ids) || !aligned4(out) || (signal && !aligned4(signal))) return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool vec = dimEmb % 4 == 0 && aligned16(E) && aligned16(out) && (!signal || aligned16(signal));
  const unsigned rps = signal ? (unsigned)rows_per_signal : 1u, ns = signal ? (unsigned)n_signals : 1u;
  if(vec)
    MH_LAUNCH(embed_kernel<true>, dim3((unsigned)rows, (unsigned)chunks), dim3(256), 0, st, E, ids,
                       (unsigned)vocab, (int)dimEmb, scale, signal, rps, ns, out, absmax_out, (unsigned)rows, (unsigned)chunks);
  else
    MH_LAUNCH(embed_kernel<false>, dim3((unsigned)rows, (unsigned)chunks), dim3(256), 0, st, E, ids,
                       (unsigned)vocab, (int)dimEmb, scale, signal, rps, ns, out, absmax_out, (unsigned)rows, (unsigned)chunks);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_select_state(const float* state, const uint32_t* ids, int64_t rows, int64_t entries,
                            int64_t segments, int64_t seg_capacity, int64_t seg_len, float* out, void* stream) {
  if(rows < 0 || entries <= 0 || segments <= 0 || seg_capacity <= 0 || seg_len < 0 || seg_len > seg_capacity)
    return MARIAN_HIP_ERR_SHAPE;
  if(rows == 0 || seg_len == 0) return MARIAN_HIP_OK;
  if(!state || !ids || !out) return MARIAN_HIP_ERR_NULL;
  const int64_t chunks = (seg_len + kEmbedChunk - 1) / kEmbedChunk;
  if(entries > 0xFFFFFFFFLL || segments > 65535 || rows > kMaxElemsOps / segments || chunks > 65535 ||
     seg_len > kMaxElemsOps ||
     entries * segments > kMaxElemsOps / seg_capacity || rows * segments > kMaxElemsOps / seg_capacity)
    return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(state) || !aligned4(ids) || !aligned4(out)) return MARIAN_HIP_ERR_ALIGN;
  // not in place: an entry may be read after the row of the same number has been written
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(state), a1 = a0 + (uintptr_t)(entries * segments * seg_capacity) * 4;
  const uintptr_t b0 = reinterpret_cast<uintptr_t>(out), b1 = b0 + (uintptr_t)(rows * segments * seg_capacity) * 4;
  if(a0 < b1 && b0 < a1) return MARIAN_HIP_ERR_ALIAS;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool vec = seg_len % 4 == 0 && seg_capacity % 4 == 0 && aligned16(state) && aligned16(out);
  const dim3 grid((unsigned)(rows * segments), (unsigned)chunks);
  if(vec)
    MH_LAUNCH(select_state_kernel<true>, grid, dim3(256), 0, st, state, ids, (unsigned)entries, (unsigned)segments,
                       (long long)seg_capacity, (int)seg_len, out);
  else
    MH_LAUNCH(select_state_kernel<false>, grid, dim3(256), 0, st, state, ids, (unsigned)entries, (unsigned)segments,
                       (long long)seg_capacity, (int)seg_len, out);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_sinusoidal_position_embeddings(float* host_out, int64_t dimWords, int64_t dimEmb, int64_t start) {
  if(dimWords < 0 || dimEmb < 4) return MARIAN_HIP_ERR_SHAPE;   // (one timescale: the increment divides by zero)
  if(dimWords == 0) return MARIAN_HIP_OK;
  if(!host_out) return MARIAN_HIP_ERR_NULL;
  if(dimWords * dimEmb > kMaxElemsOps || start < 0 || start + dimWords > 0x7FFFFFFFLL) return MARIAN_HIP_ERR_RANGE;
  const float numTimescales = (float)dimEmb / 2;
  const int half = (int)numTimescales;
  const float logTimescaleIncrement = std::log(10000.f) / (numTimescales - 1.f);
  for(int64_t j = 0; j < dimWords; ++j) {
    const int position = (int)(j + start);
    float* row = host_out + j * dimEmb;
    for(int i = 0; i < (int)dimEmb; ++i) {
      const float v = (float)position * std::exp((float)(i % half) * -logTimescaleIncrement);
      row[i] = i < half ? std::sin(v) : std::cos(v);
    }
  }
  return MARIAN_HIP_OK;
}

static int softmax_common(const float* in, const float* mask, int64_t n_masks, int64_t rows_per_mask,
                          float* out, int64_t rows, int64_t cols, bool log, void* stream) {
  if(rows < 0 || cols <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(mask && (n_masks <= 0 || rows_per_mask <= 0)) return MARIAN_HIP_ERR_SHAPE;
  if(rows == 0) return MARIAN_HIP_OK;
  if(!in || !out) return MARIAN_HIP_ERR_NULL;
  if(rows * cols > kMaxElemsOps) return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(in) || !aligned4(out) || (mask && !aligned4(mask))) return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if(!mask) { n_masks = 1; rows_per_mask = 1; }
  // rows of more than 256 values that fit the registers of one workgroup: read once (a wave per row
  // walks a 1024-value row in 16 dependent steps per pass: 10 us for 128 rows against 4)
  const bool wide_ok = cols % 4 == 0 && cols <= 65536 && aligned16(in) && aligned16(out) && (!mask || aligned16(mask));
  if(cols <= 2048 && !(wide_ok && cols > 256)) {
    const unsigned blocks = (unsigned)((rows + 3) / 4);
    if(log) MH_LAUNCH((softmax_kernel<64, true>), dim3(blocks), dim3(256), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (long long)rows, (int)cols);
    else MH_LAUNCH((softmax_kernel<64, false>), dim3(blocks), dim3(256), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (long long)rows, (int)cols);
  } else if(wide_ok && cols <= 4096) {
    if(log) MH_LAUNCH((softmax_wide_kernel<true, 256, 4>), dim3((unsigned)rows), dim3(256), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (int)cols);
    else MH_LAUNCH((softmax_wide_kernel<false, 256, 4>), dim3((unsigned)rows), dim3(256), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (int)cols);
  } else if(wide_ok && cols <= 32768) {
    if(log) MH_LAUNCH((softmax_wide_kernel<true, 1024, 8>), dim3((unsigned)rows), dim3(1024), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (int)cols);
    else MH_LAUNCH((softmax_wide_kernel<false, 1024, 8>), dim3((unsigned)rows), dim3(1024), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (int)cols);
  } else if(wide_ok) {
    if(log) MH_LAUNCH((softmax_wide_kernel<true, 1024, 16>), dim3((unsigned)rows), dim3(1024), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (int)cols);
    else MH_LAUNCH((softmax_wide_kernel<false, 1024, 16>), dim3((unsigned)rows), dim3(1024), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (int)cols);
  } else {
    if(log) MH_LAUNCH((softmax_kernel<1024, true>), dim3((unsigned)rows), dim3(1024), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (long long)rows, (int)cols);
    else MH_LAUNCH((softmax_kernel<1024, false>), dim3((unsigned)rows), dim3(1024), 0, st, in, mask, (long long)n_masks, (long long)rows_per_mask, out, (long long)rows, (int)cols);
  }
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_softmax(const float* in, const float* mask, int64_t n_masks, int64_t rows_per_mask,
                       float* out, int64_t rows, int64_t cols, void* stream) {
  return softmax_common(in, mask, n_masks, rows_per_mask, out, rows, cols, false, stream);
}

int marian_hip_logsoftmax(const float* in, float* out, int64_t rows, int64_t cols, void* stream) {
  return softmax_common(in, nullptr, 1, 1, out, rows, cols, true, stream);
}

int marian_hip_transpose0213(const float* in, float* out, int64_t d0, int64_t d1, int64_t d2,
                             int64_t d3, void* stream) {
  if(d0 < 0 || d1 <= 0 || d2 <= 0 || d3 <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(d0 == 0) return MARIAN_HIP_OK;
  if(!in || !out) return MARIAN_HIP_ERR_NULL;
  if(in == out) return MARIAN_HIP_ERR_SHAPE;
  if(d0 * d1 * d2 * d3 > kMaxElemsOps) return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(in) || !aligned4(out)) return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const bool vec = d3 % 4 == 0 && aligned16(in) && aligned16(out);
  const long long total = d0 * d1 * d2 * (vec ? d3 / 4 : d3);
  long long blocks = (total + 255) / 256;
  if(blocks > 8192) blocks = 8192;
  if(vec) MH_LAUNCH(transpose0213_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, st, in, out, total, (int)d1, (int)d2, (int)(d3 / 4), (int)blocks);
  else MH_LAUNCH(transpose0213_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, st, in, out, total, (int)d1, (int)d2, (int)d3, (int)blocks);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_bdot_legacy(const float* A, const float* B, float* C, int64_t batchA, int64_t batchB,
                           int64_t m, int64_t n, int64_t k, int transA, int transB, float scalar,
                           void* stream) {
  if(batchA < 0 || batchB < 0 || m <= 0 || n <= 0 || k <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(batchA == 0 || batchB == 0) return MARIAN_HIP_OK;
  if(!A || !B || !C) return MARIAN_HIP_ERR_NULL;
  const int64_t batchC = batchA > batchB ? batchA : batchB;
  if(batchA * m * k > kMaxElemsOps || batchB * n * k > kMaxElemsOps || batchC * m * n > kMaxElemsOps)
    return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(A) || !aligned4(B) || !aligned4(C)) return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const long long rows_total = batchC * m;
  const bool tile_ok = !transA && m >= 8 && batchC <= 65535 && aligned16(A) && aligned16(B) &&
                       (transB ? k % 4 == 0 : (k % 4 == 0 && n % 4 == 0));
  if(tile_ok) {
    const dim3 grid((unsigned)((n + 63) / 64), (unsigned)((m + 63) / 64), (unsigned)batchC);
    if(transB)
      MH_LAUNCH(bdot_tile_kernel<true>, grid, dim3(256), 0, st, A, B, C, (long long)batchA,
                         (long long)batchB, (int)m, (int)n, (int)k, scalar);
    else
      MH_LAUNCH(bdot_tile_kernel<false>, grid, dim3(256), 0, st, A, B, C, (long long)batchA,
                         (long long)batchB, (int)m, (int)n, (int)k, scalar);
    MH_HIP(hipGetLastError());
    return MARIAN_HIP_OK;
  }
  MH_LAUNCH(bdot_kernel, dim3((unsigned)((rows_total + 3) / 4)), dim3(256), 0, st, A, B, C,
                     (long long)batchA, (long long)batchB, rows_total, (int)m, (int)n, (int)k,
                     transA ? 1 : 0, transB ? 1 : 0, scalar);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_attention(const float* q, float* k, float* v, const float* mask, int64_t n_masks,
                         int64_t rows_per_mask, float* out, int64_t batchQ, int64_t batchKV,
                         int64_t m, int64_t len, int64_t dk, float scale, float* absmax_out,
                         const float* k_new, const float* v_new, void* stream) {
  return marian_hip_attention_cached(q, k, v, mask, n_masks, rows_per_mask, out, batchQ, batchKV, m, len, len, dk,
                                     scale, absmax_out, k_new, v_new, stream);
}

int marian_hip_attention_rows(const float* q, const int64_t* q_strides, const float* k, const int64_t* k_strides,
                              const float* v, const int64_t* v_strides, const float* mask, int64_t n_masks,
                              int64_t rows_per_mask, float* out, const int64_t* out_strides, int64_t batchQ,
                              int64_t batchKV, int64_t heads, int64_t m, int64_t len, int64_t dk, float scale,
                              float* absmax_out, void* stream) {
  if(batchQ < 0 || batchKV <= 0 || heads <= 0 || m <= 0 || len <= 0 || dk <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(mask && (n_masks <= 0 || rows_per_mask <= 0)) return MARIAN_HIP_ERR_SHAPE;
  const bool blocks = dk == 64 && m >= MARIAN_HIP_ATTENTION_ROWS_MIN && len <= MARIAN_HIP_ATTENTION_ROWS_MAX_LEN;
  if(!blocks && m >= MARIAN_HIP_ATTENTION_ROWS_MIN) return MARIAN_HIP_ERR_SHAPE;
  if(!q_strides || !k_strides || !v_strides || !out_strides) return MARIAN_HIP_ERR_NULL;
  if(batchQ == 0) return MARIAN_HIP_OK;
  if(!q || !k || !v || !out) return MARIAN_HIP_ERR_NULL;
  if(mask && (n_masks > 2147483647LL || rows_per_mask > 2147483647LL)) return MARIAN_HIP_ERR_RANGE;
  if(heads > kMaxElemsOps || dk > kMaxElemsOps || m > kMaxElemsOps / dk || len > 4096 || batchQ > kMaxElemsOps / (m * dk) ||
     batchKV > kMaxElemsOps / (len * dk))
    return MARIAN_HIP_ERR_RANGE;
  AttentionStrides hs;
  HeadStrides* const to[4] = {&hs.q, &hs.k, &hs.v, &hs.out};
  const int64_t* const given[4] = {q_strides, k_strides, v_strides, out_strides};
  for(int i = 0; i < 4; ++i) {
    for(int j = 0; j < 3; ++j)
      if(given[i][j] < 0 || given[i][j] % 4 != 0) return MARIAN_HIP_ERR_ALIGN;
    *to[i] = HeadStrides{given[i][0], given[i][1], given[i][2]};
  }
  // (positions within a sentence are reached with 32-bit offsets)
  if(q_strides[2] > kMaxElemsOps / m || out_strides[2] > kMaxElemsOps / m || k_strides[2] > kMaxElemsOps / len || v_strides[2] > kMaxElemsOps / len)
    return MARIAN_HIP_ERR_RANGE;
  if(!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(out) || (mask && !aligned4(mask)) || (absmax_out && !aligned4(absmax_out)))
    return MARIAN_HIP_ERR_ALIGN;
  if(!mask) { n_masks = 1; rows_per_mask = 1; }
  hipStream_t hst = reinterpret_cast<hipStream_t>(stream);
  if(!blocks) {   // (a wave per query row)
    if(absmax_out && batchQ * m > kAbsmaxSlots) return MARIAN_HIP_ERR_RANGE;
    static std::atomic<uint64_t> lds_done{0};
    const int lds_status = allow_lds(attention_kernel<false, true>, 72 * 1024, lds_done);
    if(lds_status != MARIAN_HIP_OK) return lds_status;
    const size_t lds = (size_t)4 * (size_t)(((len + 3) & ~(int64_t)3) + 256) * sizeof(float);
    MH_LAUNCH((attention_kernel<false, true>), dim3((unsigned)((batchQ * m + 3) / 4)), dim3(256), lds, hst, q, const_cast<float*>(k),
                       const_cast<float*>(v), nullptr, nullptr, mask, (unsigned)n_masks, (unsigned)rows_per_mask, out, (unsigned)(batchQ * m),
                       (unsigned)batchKV, (int)m, (int)len, (int)len, (int)dk, scale, absmax_out, nullptr, (unsigned)heads, hs);
    MH_HIP(hipGetLastError());
    return MARIAN_HIP_OK;
  }
  // One workgroup to a head reads its keys and values once; several where the heads are fewer than CUs, and at most
  // four blocks of rows to a workgroup, one after the other (128 heads of 64 x 64: 9.0, 6.2, 7.5 us with 1, 2, 4
  // workgroups a head; 384 of 128 x 128: 36.0, 29.5, 31.6; 1024 of 64 x 64: 23.1, 24.3, 28.9).
  const int64_t row_blocks = (m + 15) / 16;
  int64_t groups = batchQ >= 256 ? 1 : (256 + batchQ - 1) / batchQ;
  if(groups < (row_blocks + 3) / 4) groups = (row_blocks + 3) / 4;
  if(groups > row_blocks) groups = row_blocks;
  if(batchQ * groups > kMaxElemsOps / 256) return MARIAN_HIP_ERR_RANGE;
  if(absmax_out && batchQ * groups * 4 > kAbsmaxSlots) return MARIAN_HIP_ERR_RANGE;
  const AttentionHeadsPlan plan = attention_heads_plan(batchQ, groups, row_blocks, len);
  if(plan.workgroups) {   // a wave to 16 query rows
    const int tiles = plan.tiles, waves = plan.waves;
    const int64_t wgs = plan.workgroups;   // of a head
    // (its buffers hold a head each, offsets past the last row included, and end behind the last row of 64 values)
    auto fits = [](int64_t row, int64_t positions) { return row <= (1 << 29) / (positions + 128); };
    if(fits(q_strides[2], m) && fits(k_strides[2], len) && fits(v_strides[2], len) && fits(out_strides[2], m) && k_strides[2] >= 64 && v_strides[2] >= 64 &&
       (!mask || n_masks <= (1 << 29) / (len + 128)) && (!absmax_out || batchQ * wgs * waves <= kAbsmaxSlots)) {
      AttentionRowsArgs a{q, k, v, mask, out, absmax_out, hs.q, hs.k, hs.v, hs.out, (unsigned)batchQ, (unsigned)batchKV, (unsigned)heads,
                          (unsigned)n_masks, (unsigned)rows_per_mask, (int)m, (int)len, (int)row_blocks, (int)wgs, scale,
                          mask && rows_per_mask % m == 0};
      const dim3 grid((unsigned)(batchQ * wgs)), block((unsigned)waves * 64);
#define MH_HEADS(TILES, WAVES) MH_LAUNCH((attention_heads_kernel<TILES, WAVES>), grid, block, 0, hst, a)
      if(tiles == 2) MH_HEADS(2, 2);
      else if(tiles == 3) MH_HEADS(3, 3);
      else if(tiles == 4) MH_HEADS(4, 4);
      else if(tiles == 5) MH_HEADS(5, 3);
      else if(tiles == 6) MH_HEADS(6, 3);
      else MH_HEADS(8, 4);
#undef MH_HEADS
      MH_HIP(hipGetLastError());
      return MARIAN_HIP_OK;
    }
  }
  AttentionRowsArgs a{q, k, v, mask, out, absmax_out, hs.q, hs.k, hs.v, hs.out, (unsigned)batchQ, (unsigned)batchKV, (unsigned)heads,
                      (unsigned)n_masks, (unsigned)rows_per_mask, (int)m, (int)len, (int)row_blocks, (int)groups, scale,
                      mask && rows_per_mask % m == 0};
  const dim3 grid((unsigned)(batchQ * groups));
#define MH_ROWS(NB) MH_LAUNCH(attention_rows_kernel<NB>, grid, dim3(256), 0, hst, a)
  if(len <= 64) MH_ROWS(1);
  else if(len <= 128) MH_ROWS(2);
  else if(len <= 192) MH_ROWS(3);
  else MH_ROWS(4);
#undef MH_ROWS
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

static int attention_impl(const float* q, float* k, float* v, const float* mask, int64_t n_masks,
                          int64_t rows_per_mask, float* out, int64_t batchQ, int64_t batchKV, int64_t m,
                          int64_t len, int64_t kv_capacity, int64_t dk, float scale, float* absmax_out,
                          const float* k_new, const float* v_new, const uint32_t* ancestors, int64_t heads,
                          void* stream);

int marian_hip_attention_cached(const float* q, float* k, float* v, const float* mask, int64_t n_masks,
                                int64_t rows_per_mask, float* out, int64_t batchQ, int64_t batchKV,
                                int64_t m, int64_t len, int64_t kv_capacity, int64_t dk, float scale,
                                float* absmax_out, const float* k_new, const float* v_new, void* stream) {
  return attention_impl(q, k, v, mask, n_masks, rows_per_mask, out, batchQ, batchKV, m, len, kv_capacity, dk, scale,
                        absmax_out, k_new, v_new, nullptr, 1, stream);
}

int marian_hip_attention_ancestors(const float* q, float* k, float* v, float* out, int64_t n_hyp, int64_t heads,
                                   int64_t len, int64_t kv_capacity, int64_t dk, float scale, float* absmax_out,
                                   const float* k_new, const float* v_new, const uint32_t* ancestors,
                                   void* stream) {
  if(n_hyp < 0 || heads <= 0 || dk != 64) return MARIAN_HIP_ERR_SHAPE;
  if(n_hyp == 0) return MARIAN_HIP_OK;
  if(!ancestors || !k_new || !v_new) return MARIAN_HIP_ERR_NULL;
  if(n_hyp > kMaxElemsOps / heads) return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(ancestors)) return MARIAN_HIP_ERR_ALIGN;
  if(q && k && v && (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(k_new) || !aligned16(v_new)))
    return MARIAN_HIP_ERR_ALIGN;
  return attention_impl(q, k, v, nullptr, 0, 0, out, n_hyp * heads, n_hyp * heads, 1, len, kv_capacity, dk, scale,
                        absmax_out, k_new, v_new, ancestors, heads, stream);
}

// next[h, p] = prev[parents[h], p] for the len_prev positions cached so far, next[h, len_prev] = h:
// the position the coming step appends lies in the hypothesis's own entry.
__global__ __launch_bounds__(256) void ancestors_advance_kernel(const uint32_t* __restrict__ prev,
                                                                const uint32_t* __restrict__ parents, unsigned n_hyp,
                                                                unsigned kv_cap, unsigned len_prev,
                                                                uint32_t* __restrict__ next) {
  const unsigned i = blockIdx.x * 256 + threadIdx.x;
  if(i >= n_hyp * (len_prev + 1)) return;
  const unsigned h = i / (len_prev + 1), p = i % (len_prev + 1);
  const unsigned from = min(parents[h], n_hyp - 1u);
  next[(size_t)h * kv_cap + p] = p < len_prev ? prev[(size_t)from * kv_cap + p] : h;
}

int marian_hip_ancestors_advance(const uint32_t* prev, const uint32_t* parents, int64_t n_hyp, int64_t kv_capacity,
                                 int64_t len_prev, uint32_t* next, void* stream) {
  if(n_hyp < 0 || kv_capacity <= 0 || len_prev < 0 || len_prev >= kv_capacity) return MARIAN_HIP_ERR_SHAPE;
  if(n_hyp == 0) return MARIAN_HIP_OK;
  if(!prev || !parents || !next) return MARIAN_HIP_ERR_NULL;
  if(n_hyp > kMaxElemsOps / kv_capacity) return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(prev) || !aligned4(parents) || !aligned4(next)) return MARIAN_HIP_ERR_ALIGN;
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(prev), b0 = reinterpret_cast<uintptr_t>(next);
  const uintptr_t bytes = (uintptr_t)(n_hyp * kv_capacity) * 4;
  if(a0 < b0 + bytes && b0 < a0 + bytes) return MARIAN_HIP_ERR_ALIAS;   // (a row may be read after the row of the same number has been written)
  const int64_t n = n_hyp * (len_prev + 1);
  MH_LAUNCH(ancestors_advance_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                     reinterpret_cast<hipStream_t>(stream), prev, parents, (unsigned)n_hyp, (unsigned)kv_capacity,
                     (unsigned)len_prev, next);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

static int attention_impl(const float* q, float* k, float* v, const float* mask, int64_t n_masks,
                          int64_t rows_per_mask, float* out, int64_t batchQ, int64_t batchKV, int64_t m,
                          int64_t len, int64_t kv_capacity, int64_t dk, float scale, float* absmax_out,
                          const float* k_new, const float* v_new, const uint32_t* ancestors, int64_t heads,
                          void* stream) {
  if((k_new != nullptr) != (v_new != nullptr)) return MARIAN_HIP_ERR_NULL;
  if(kv_capacity < len) return MARIAN_HIP_ERR_SHAPE;
  if(k_new && (m != 1 || batchKV != batchQ)) return MARIAN_HIP_ERR_SHAPE;
  if(k_new && (!aligned4(k_new) || !aligned4(v_new))) return MARIAN_HIP_ERR_ALIGN;
  if(absmax_out && batchQ * m > kAbsmaxSlots) return MARIAN_HIP_ERR_RANGE;
  if(absmax_out && !aligned4(absmax_out)) return MARIAN_HIP_ERR_ALIGN;
  if(batchQ < 0 || batchKV <= 0 || m <= 0 || len <= 0 || dk <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(mask && (n_masks <= 0 || rows_per_mask <= 0)) return MARIAN_HIP_ERR_SHAPE;
  if(mask && (n_masks > 2147483647LL || rows_per_mask > 2147483647LL)) return MARIAN_HIP_ERR_RANGE;
  if(len > 4096) return MARIAN_HIP_ERR_RANGE;
  if(batchQ == 0) return MARIAN_HIP_OK;
  if(!q || !k || !v || !out) return MARIAN_HIP_ERR_NULL;
  if(kv_capacity > kMaxElemsOps || batchQ * m * dk > kMaxElemsOps || batchKV * kv_capacity * dk > kMaxElemsOps)
    return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(q) || !aligned4(k) || !aligned4(v) || !aligned4(out) || (mask && !aligned4(mask)))
    return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if(!mask) { n_masks = 1; rows_per_mask = 1; }
  const long long rows_total = batchQ * m;
  const size_t lds = (size_t)4 * (size_t)(((len + 3) & ~(int64_t)3) + 256) * sizeof(float);   // per wave: scores (whole 16-byte units) + partial outputs
  {   // the kernel's dynamic LDS limit, raised once per device (one bit per device)
    static std::atomic<uint64_t> lds_done{0};
    int dev = 0;
    MH_HIP(hipGetDevice(&dev));
    if(dev < 0 || dev >= 64) return MARIAN_HIP_ERR_RANGE;
    if(!(lds_done.load(std::memory_order_acquire) & (1ull << dev))) {
      MH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(attention_kernel<false, false>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, 72 * 1024));
      MH_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(attention_kernel<true, false>),
                                 hipFuncAttributeMaxDynamicSharedMemorySize, 72 * 1024));
      lds_done.fetch_or(1ull << dev, std::memory_order_release);
    }
  }
  // Complete caches that several query rows share, head size 64, one position per row, everything
  // aligned for 16-byte loads: the rows of a cache entry in one workgroup, the entry read once.
  if(!ancestors && !k_new && dk == 64 && m == 1 && len <= kSharedAttLen && batchKV < rows_total && rows_total % batchKV == 0 &&
     rows_total / batchKV <= 4 * 65535 && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out)) {
    const long long hyps = rows_total / batchKV;
    const dim3 grid((unsigned)batchKV, (unsigned)((hyps + 3) / 4));
    const size_t slds = (size_t)2 * (size_t)len * 256 + lds;
#define MH_SATT(PASSES) \
    MH_LAUNCH(attention_shared_kernel<PASSES>, grid, dim3(256), slds, st, q, k, v, mask, (unsigned)n_masks, \
                       (unsigned)rows_per_mask, out, (unsigned)rows_total, (unsigned)batchKV, (int)len, (int)kv_capacity, \
                       scale, absmax_out)
    if(len <= 32) MH_SATT(2);
    else if(len <= 64) MH_SATT(4);
    else MH_SATT(6);
#undef MH_SATT
    MH_HIP(hipGetLastError());
    return MARIAN_HIP_OK;
  }
  if(ancestors)
    MH_LAUNCH((attention_kernel<true, false>), dim3((unsigned)((rows_total + 3) / 4)), dim3(256), lds, st, q, k, v,
                       k_new, v_new, mask, (unsigned)n_masks, (unsigned)rows_per_mask, out, (unsigned)rows_total,
                       (unsigned)batchKV, (int)m, (int)len, (int)kv_capacity, (int)dk, scale, absmax_out, ancestors,
                       (unsigned)heads, AttentionStrides());
  else
    MH_LAUNCH((attention_kernel<false, false>), dim3((unsigned)((rows_total + 3) / 4)), dim3(256), lds, st, q, k, v,
                       k_new, v_new, mask, (unsigned)n_masks, (unsigned)rows_per_mask, out, (unsigned)rows_total,
                       (unsigned)batchKV, (int)m, (int)len, (int)kv_capacity, (int)dk, scale, absmax_out, ancestors,
                       1u, AttentionStrides());
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

}  // extern "C"
template <int NPROJ, int R, int SEGS, int PASSES, int PW, int HELD, bool NORM, bool ANC>
static int launch_proj(const ProjAttentionArgs& p, dim3 grid, size_t lds, hipStream_t st) {
  constexpr auto kernel = proj_attention_kernel<NPROJ, R, SEGS, PASSES, PW, HELD, NORM, ANC>;
  static std::atomic<uint64_t> lds_done{0};
  const int lst = allow_lds(kernel, SEGS > 0 ? kProjMaxLds : 96 * 1024, lds_done);
  if(lst != MARIAN_HIP_OK) return lst;
  MH_LAUNCH(kernel, grid, dim3(kProjThreads), lds, st, p.A, NORM ? p.norm.add : p.partials, p.Bq[0], p.Bq[1], p.Bq[2], p.M, p.K, p.heads,
                     p.n_partials, p);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

extern "C" {
static int proj_attention(const float* A, const marian_hip_norm_input* norm, const uint32_t* anc, int8_t* Aq, int64_t n_proj, const int8_t* const* Bq,
                          const float* const* bias, float* const* proj_out, int64_t M, int64_t K,
                          int64_t heads, float* k_cache, float* v_cache, int64_t batchKV, int64_t len,
                          int64_t kv_capacity, const float* mask, int64_t n_masks, float att_scale,
                          float* out, const float* absmax_in, float* absmax_out, void* workspace,
                          size_t workspace_bytes, void* stream) {
  if(n_proj != 1 && n_proj != 3) return MARIAN_HIP_ERR_SHAPE;
  if(M < 0 || K <= 0 || heads <= 0 || (K % 128) != 0 || K > kProjMaxK) return MARIAN_HIP_ERR_SHAPE;
  if(len <= 0 || len > kProjMaxLen || kv_capacity < len || batchKV <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(mask && n_masks <= 0) return MARIAN_HIP_ERR_SHAPE;
  if(M == 0) return MARIAN_HIP_OK;
  if(!A || (!Aq && !norm) || !Bq || !k_cache || !v_cache || !out) return MARIAN_HIP_ERR_NULL;
  if(M * heads > kMaxElemsOps / 64 || batchKV * kv_capacity > kMaxElemsOps / 64 || M * K > kMaxElemsOps ||
     K * heads * 64 > kMaxElemsOps || n_masks > 2147483647LL)
    return MARIAN_HIP_ERR_RANGE;
  // the self-attention form appends to the caches: every query row needs an entry of its own
  if(n_proj == 3 && batchKV != M * heads) return MARIAN_HIP_ERR_SHAPE;
  if(absmax_out && M * heads > kAbsmaxSlots) return MARIAN_HIP_ERR_RANGE;
  if(!aligned16(A) || (Aq && !aligned16(Aq)) || !aligned16(k_cache) || !aligned16(v_cache) || !aligned16(out))
    return MARIAN_HIP_ERR_ALIGN;
  if((mask && !aligned4(mask)) || (absmax_in && !aligned4(absmax_in)) || (absmax_out && !aligned4(absmax_out)))
    return MARIAN_HIP_ERR_ALIGN;
  ProjAttentionArgs p;
  for(int g = 0; g < 3; ++g) {
    p.Bq[g] = nullptr; p.bias[g] = nullptr; p.proj_out[g] = nullptr;
  }
  for(int64_t g = 0; g < n_proj; ++g) {
    if(!Bq[g]) return MARIAN_HIP_ERR_NULL;
    p.Bq[g] = Bq[g];
    p.bias[g] = bias ? bias[g] : nullptr;
    p.proj_out[g] = proj_out ? proj_out[g] : nullptr;
    if(!aligned16(p.Bq[g]) || (p.bias[g] && !aligned16(p.bias[g])) || (p.proj_out[g] && !aligned16(p.proj_out[g])))
      return MARIAN_HIP_ERR_ALIGN;
  }
  {
    const int64_t f = sizeof(float), values = M * heads * 64 * f, cached = batchKV * kv_capacity * 64 * f, slots = kAbsmaxSlots * f;
    const Span a{A, M * K * f}, add{norm ? norm->add : nullptr, M * K * f}, x{norm ? norm->out : nullptr, M * K * f};
    const Span gamma{norm ? norm->gamma : nullptr, K * f}, beta{norm ? norm->beta : nullptr, K * f};
    const Span known{norm ? nullptr : absmax_in, slots}, k{k_cache, cached}, v{v_cache, cached};
    int ast = apart({{out, values}, {p.proj_out[0], values}, {p.proj_out[1], values}, {p.proj_out[2], values}, {absmax_out, slots},
                     {norm ? nullptr : Aq, M * K + f}}, {a, add, x, gamma, beta, known, k, v});
    if(ast == MARIAN_HIP_OK) ast = apart({k, v}, {a, add, x, gamma, beta, known});   // (appended to, or read beside x)
    if(ast != MARIAN_HIP_OK) return ast;
  }
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  p.A = A; p.aq_out = Aq;
  p.norm = NormInput{nullptr, nullptr, nullptr, nullptr, 0.0f};
  p.anc = anc;
  p.partials = nullptr;
  p.n_partials = 0;
  if(norm) {
    static_assert(MARIAN_HIP_NORM_MAX_ROWS == kNormMaxRows && MARIAN_HIP_NORM_MAX_COLS == kNormMaxCols, "limits");
    const int nst = norm_input_check(norm, A, M, K);
    if(nst != MARIAN_HIP_OK) return nst;
    p.norm = NormInput{norm->add, norm->gamma, norm->beta, norm->out, norm->eps};
  } else if(absmax_in) {
    p.partials = absmax_in;
    p.n_partials = kAbsmaxSlots;
  } else {   // nobody left the abs-max of the input: a launch for it
    if(!workspace) return MARIAN_HIP_ERR_NULL;
    if(workspace_bytes < kWorkspaceBytes) return MARIAN_HIP_ERR_WORKSPACE;
    if(!aligned4(workspace)) return MARIAN_HIP_ERR_ALIGN;
    float* partials = reinterpret_cast<float*>(workspace);
    int n_partials = 0;
    const int pst = launch_absmax_partials(A, (size_t)M * (size_t)K, partials, &n_partials, stream);
    if(pst != MARIAN_HIP_OK) return pst;
    p.partials = partials;
    p.n_partials = n_partials;
  }
  p.M = (int)M; p.K = (int)K; p.heads = (int)heads;
  p.k_cache = k_cache; p.v_cache = v_cache; p.batchKV = (unsigned)batchKV;
  p.len = (int)len; p.kv_cap = (int)kv_capacity;
  p.mask = mask; p.n_masks = mask ? (unsigned)n_masks : 1u;
  p.att_scale = att_scale; p.out = out; p.absmax_out = absmax_out;
  constexpr int R = 8;
  const int len4 = ((int)len + 3) & ~3;
  // Self-attention, every row its own caches: four rows to a workgroup where eight leave half of the CUs idle
  // (what a workgroup fetches bounds it: 96 KB of weights and 17 KB a row for 65 rows of 8 heads over 34 positions).
  const bool four = n_proj == 3 && 2 * heads * ((M + 7) / 8) <= compute_units();
  const int rows = four ? 4 : R;
  size_t lds = (size_t)32 * (size_t)K + (size_t)n_proj * 8 * rows * 128 + (size_t)n_proj * rows * 64 * 4 +
               (size_t)rows * (size_t)(len4 + 256) * 4;
  ProjRowPlan plan = proj_row_plan(n_proj, M, heads, batchKV, len, kProjStageLen, lds, (size_t)kProjMaxLds);
  if(four) {
    plan.per_wg = 4;
    plan.blocks_y = (M + 3) / 4;
  }
  p.share_shift = plan.shift;
  p.share_nb = plan.sentences;
  p.share_hyps = plan.hyps;
  p.share_per = plan.per_wg;
  p.stage_kv = plan.stage;
  if(plan.blocks_y > 65535) return MARIAN_HIP_ERR_RANGE;
  if(plan.stage) lds += (size_t)(2 << plan.shift) * (size_t)len * 256;
  const unsigned groups = plan.shift < 0 ? (unsigned)plan.blocks_y : (unsigned)proj_groups(plan.shift, plan.sentences);
  const dim3 grid((unsigned)heads, groups, (unsigned)plan.blocks_y / groups);
  // The cached rows are asked for behind the weights where they and the weights fit the registers: 64 positions beside 4 sub-steps of
  // three matrices, 32 beside 8 (an ancestor's row by a 32-bit offset into the caches).
  const int most_held = K <= 512 ? 16 : 8;
  const int held = n_proj != 3 || len > 4 * most_held || (anc && M * heads * kv_capacity >= (1 << 24)) || kv_capacity >= (1 << 24)
                       ? 0 : (len <= 32 ? 8 : 16);
  const int passes = ((int)len + 31) / 32;   // of the staged context's positions, 1 .. 3
  auto launch = [&](auto pw) {
    constexpr int PW = decltype(pw)::value;
    auto rows_held = [&](auto rows, auto held_tag) {
      constexpr int ROWS = decltype(rows)::value, HELD = decltype(held_tag)::value;
      if(anc && norm) return launch_proj<3, ROWS, 0, 0, PW, HELD, true, true>(p, grid, lds, st);
      if(anc) return launch_proj<3, ROWS, 0, 0, PW, HELD, false, true>(p, grid, lds, st);
      if(norm) return launch_proj<3, ROWS, 0, 0, PW, HELD, true, false>(p, grid, lds, st);
      return launch_proj<3, ROWS, 0, 0, PW, HELD, false, false>(p, grid, lds, st);
    };
    auto self = [&](auto rows) {
      if constexpr(PW == 4) {
        if(held == 16) return rows_held(rows, std::integral_constant<int, 16>());
      }
      if(held == 8) return rows_held(rows, std::integral_constant<int, 8>());
      return rows_held(rows, std::integral_constant<int, 0>());
    };
    auto context = [&](auto segs, auto pass) {
      constexpr int SEGS = decltype(segs)::value, PASSES = decltype(pass)::value;
      if(norm) return launch_proj<1, R, SEGS, PASSES, PW, 0, true, false>(p, grid, lds, st);
      return launch_proj<1, R, SEGS, PASSES, PW, 0, false, false>(p, grid, lds, st);
    };
    auto staged = [&](auto segs) {
      if(passes == 1) return context(segs, std::integral_constant<int, 1>());
      if(passes == 2) return context(segs, std::integral_constant<int, 2>());
      return context(segs, std::integral_constant<int, 3>());
    };
    if(four) return self(std::integral_constant<int, 4>());
    if(n_proj == 3) return self(std::integral_constant<int, R>());
    if(!p.stage_kv) return context(std::integral_constant<int, 0>(), std::integral_constant<int, 0>());
    return p.share_shift == 0 ? staged(std::integral_constant<int, 2>()) : staged(std::integral_constant<int, 4>());   // one sentence or two
  };
  return K <= 512 ? launch(std::integral_constant<int, 4>()) : launch(std::integral_constant<int, 8>());
}

int marian_hip_int8_proj_attention(const float* A, int8_t* Aq, int64_t n_proj, const int8_t* const* Bq,
                                   const float* const* bias, float* const* proj_out, int64_t M, int64_t K,
                                   int64_t heads, float* k_cache, float* v_cache, int64_t batchKV, int64_t len,
                                   int64_t kv_capacity, const float* mask, int64_t n_masks, float att_scale,
                                   float* out, const float* absmax_in, float* absmax_out, void* workspace,
                                   size_t workspace_bytes, void* stream) {
  return proj_attention(A, nullptr, nullptr, Aq, n_proj, Bq, bias, proj_out, M, K, heads, k_cache, v_cache, batchKV, len, kv_capacity, mask,
                        n_masks, att_scale, out, absmax_in, absmax_out, workspace, workspace_bytes, stream);
}

int marian_hip_int8_proj_attention_ancestors(const float* A, const marian_hip_norm_input* norm, int8_t* Aq, const int8_t* const* Bq,
                                             const float* const* bias, float* const* proj_out, int64_t M, int64_t K, int64_t heads,
                                             float* k_cache, float* v_cache, int64_t len, int64_t kv_capacity,
                                             const uint32_t* ancestors, float att_scale, float* out, const float* absmax_in,
                                             float* absmax_out, void* workspace, size_t workspace_bytes, void* stream) {
  if(!ancestors) return MARIAN_HIP_ERR_NULL;
  if(!aligned4(ancestors)) return MARIAN_HIP_ERR_ALIGN;
  if(M < 0 || heads <= 0 || M > kMaxElemsOps / heads) return MARIAN_HIP_ERR_SHAPE;
  return proj_attention(A, norm, ancestors, Aq, 3, Bq, bias, proj_out, M, K, heads, k_cache, v_cache, M ? M * heads : 1, len, kv_capacity,
                        nullptr, 0, att_scale, out, absmax_in, absmax_out, workspace, workspace_bytes, stream);
}

int marian_hip_int8_proj_attention_normed(const float* A, const marian_hip_norm_input* norm, int64_t n_proj, const int8_t* const* Bq,
                                          const float* const* bias, float* const* proj_out, int64_t M, int64_t K,
                                          int64_t heads, float* k_cache, float* v_cache, int64_t batchKV, int64_t len,
                                          int64_t kv_capacity, const float* mask, int64_t n_masks, float att_scale,
                                          float* out, float* absmax_out, void* stream) {
  if(!norm) return MARIAN_HIP_ERR_NULL;
  return proj_attention(A, norm, nullptr, nullptr, n_proj, Bq, bias, proj_out, M, K, heads, k_cache, v_cache, batchKV, len, kv_capacity, mask,
                        n_masks, att_scale, out, nullptr, absmax_out, nullptr, 0, stream);
}

// Rows of up to kNbestWaveCols values: a wave each; longer ones: 1024 threads each.
static int nbest_rows(const float* scores, int64_t rows, int64_t rowLen, int64_t N, const NbestOut& out, void* stream) {
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
#define MH_NBW(VPT) MH_LAUNCH(nbest_wave_kernel<VPT>, dim3((unsigned)rows), dim3(64), 0, st, scores, (int)rowLen, (int)N, out)
#define MH_NBK(KEEP) MH_LAUNCH(nbest_kernel<KEEP>, dim3((unsigned)rows), dim3(1024), 0, st, scores, (long long)rowLen, (int)N, out)
  if(rowLen <= kNbestWaveCols / 2) MH_NBW(kNbestWaveCols / 128);
  else if(rowLen <= kNbestWaveCols) MH_NBW(kNbestWaveCols / 64);
  else if(N <= 4) MH_NBK(4);
  else if(N <= 8) MH_NBK(8);
  else MH_NBK(16);
#undef MH_NBW
#undef MH_NBK
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_nbest(const float* scores, int64_t dimBatch, int64_t rowLen, int64_t N,
                     float* outScores, uint32_t* outKeys, void* stream) {
  if(dimBatch < 0 || rowLen <= 0 || N <= 0 || N > kNbestMax || N > rowLen) return MARIAN_HIP_ERR_SHAPE;
  if(dimBatch == 0) return MARIAN_HIP_OK;
  if(!scores || !outScores || !outKeys) return MARIAN_HIP_ERR_NULL;
  if(dimBatch * rowLen > 4294967295LL) return MARIAN_HIP_ERR_RANGE;   // keys are uint32
  if(!aligned4(scores) || !aligned4(outScores) || !aligned4(outKeys)) return MARIAN_HIP_ERR_ALIGN;
  return nbest_rows(scores, dimBatch, rowLen, N, NbestOut{outScores, outKeys, nullptr, nullptr}, stream);
}

int marian_hip_nbest_words(const float* scores, int64_t rows, int64_t rowLen, int64_t N, const uint32_t* ids,
                           float* outScores, int64_t* outWords, void* stream) {
  if(rows < 0 || rowLen <= 0 || N <= 0 || N > kNbestMax || N > rowLen) return MARIAN_HIP_ERR_SHAPE;
  if(rows == 0) return MARIAN_HIP_OK;
  if(!scores || !outScores || !outWords) return MARIAN_HIP_ERR_NULL;
  if(rows * rowLen > 4294967295LL) return MARIAN_HIP_ERR_RANGE;
  if(!aligned4(scores) || !aligned4(outScores) || reinterpret_cast<uintptr_t>(outWords) % 8 != 0 || (ids && !aligned4(ids)))
    return MARIAN_HIP_ERR_ALIGN;
  return nbest_rows(scores, rows, rowLen, N, NbestOut{outScores, nullptr, reinterpret_cast<long long*>(outWords), ids}, stream);
}

int marian_hip_fill(void* begin, int64_t count, int elem_bytes, uint64_t pattern, void* stream) {
  if(count < 0 || (elem_bytes != 1 && elem_bytes != 2 && elem_bytes != 4 && elem_bytes != 8))
    return MARIAN_HIP_ERR_SHAPE;
  if(count == 0) return MARIAN_HIP_OK;
  if(!begin) return MARIAN_HIP_ERR_NULL;
  if(reinterpret_cast<uintptr_t>(begin) % (uintptr_t)elem_bytes != 0) return MARIAN_HIP_ERR_ALIGN;
  if(count > (int64_t)(0x7FFFFFFFFFFFFFFFll / 8)) return MARIAN_HIP_ERR_RANGE;
  const long long bytes = (long long)count * elem_bytes;
  long long head = (long long)((16 - reinterpret_cast<uintptr_t>(begin) % 16) % 16);
  if(head > bytes) head = bytes;
  const long long vecs = (bytes - head) / 16;
  long long blocks = (vecs + 255) / 256;
  if(blocks < 1) blocks = 1;
  if(blocks > 4096) blocks = 4096;
  MH_LAUNCH(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                     reinterpret_cast<unsigned char*>(begin), bytes, head, vecs, elem_bytes,
                     (unsigned long long)pattern, (int)blocks);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

size_t marian_hip_nbest_beams_workspace_bytes(int64_t beam, int64_t dimBatch, int64_t vocab, int64_t N) {
  if(beam <= 0 || dimBatch <= 0 || vocab <= 0 || N <= 0 || N > kNbestMax) return 0;
  const NbestPlan plan = nbest_plan(beam, dimBatch, vocab, N);
  return kNbestCounterBytes + (size_t)dimBatch * plan.parts * N * 8;
}

int marian_hip_nbest_beams_workspace_init(void* workspace, size_t workspace_bytes, void* stream) {
  if(workspace_bytes == 0) return MARIAN_HIP_OK;
  if(!workspace) return MARIAN_HIP_ERR_NULL;
  if(!aligned4(workspace)) return MARIAN_HIP_ERR_ALIGN;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const long long words = (long long)(workspace_bytes / 4);
  const unsigned blocks = (unsigned)((words + 255) / 256 < 1024 ? (words + 255) / 256 : 1024);
  if(words > 0)
    MH_LAUNCH(zero_words_kernel, dim3(blocks), dim3(256), 0, st, reinterpret_cast<unsigned*>(workspace), words, (int)blocks);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_nbest_beams(const float* scores, int64_t beam, int64_t dimBatch, int64_t vocab, int64_t N,
                           float* outScores, uint32_t* outKeys, void* workspace, size_t workspace_bytes,
                           void* stream) {
  if(beam <= 0 || dimBatch < 0 || vocab <= 0 || N <= 0 || N > kNbestMax || N > beam * vocab)
    return MARIAN_HIP_ERR_SHAPE;
  if(beam * N > 1024) return MARIAN_HIP_ERR_SHAPE;
  if(dimBatch == 0) return MARIAN_HIP_OK;
  if(!scores || !outScores || !outKeys || !workspace) return MARIAN_HIP_ERR_NULL;
  if(dimBatch * beam * vocab > 4294967295LL || dimBatch > kNbestMaxBatch) return MARIAN_HIP_ERR_RANGE;   // keys are uint32
  if(!aligned4(scores) || !aligned4(outScores) || !aligned4(outKeys) || !aligned4(workspace))
    return MARIAN_HIP_ERR_ALIGN;
  const NbestPlan plan = nbest_plan(beam, dimBatch, vocab, N);
  const size_t entries = (size_t)dimBatch * plan.parts * N;
  if(workspace_bytes < kNbestCounterBytes + entries * 8) return MARIAN_HIP_ERR_WORKSPACE;
  // layout: the counters (one per batch entry, zero between calls) in a region of fixed size, so
  // that no call's candidates ever land on another call's counters; then candidate scores and
  // candidate positions
  unsigned* counters = reinterpret_cast<unsigned*>(workspace);
  float* candVal = reinterpret_cast<float*>(counters + kNbestMaxBatch * kNbestCounterStride);
  unsigned* candIdx = reinterpret_cast<unsigned*>(candVal + entries);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)plan.parts, (unsigned)dimBatch);
#define MH_NBP(KEEP, FENCED)                                                                                   \
  MH_LAUNCH((nbest_part_kernel<KEEP, FENCED>), grid, dim3(1024), 0, st, scores, (long long)dimBatch, \
                     (long long)vocab, plan.perSeg, plan.sliceLen, (int)N, (int)plan.parts, candVal, candIdx, counters,         \
                     outScores, outKeys)
  if(nbest_fenced()) {
#ifdef MARIAN_HIP_TUNING
    if(N <= 4) MH_NBP(4, true);
    else if(N <= 8) MH_NBP(8, true);
    else MH_NBP(16, true);
#endif
  } else {
    if(N <= 4) MH_NBP(4, false);
    else if(N <= 8) MH_NBP(8, false);
    else MH_NBP(16, false);
  }
#undef MH_NBP
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_logsoftmax_nbest_beams(const float* logits, const float* rowAdd, float* logProbs, int64_t beam,
                                      int64_t dimBatch, int64_t vocab, int64_t N, float* outScores,
                                      uint32_t* outKeys, void* workspace, size_t workspace_bytes, void* stream) {
  if(beam <= 0 || dimBatch < 0 || vocab <= 0 || N <= 0 || N > kNbestMax || N > vocab) return MARIAN_HIP_ERR_SHAPE;
  // (a row in the registers of one workgroup, and the sizes for which marian_hip_logsoftmax takes the
  // same row computation, softmax_wide_kernel<true, 1024, 8>: the results are to be the same bits)
  if(beam * N > 1024 || (vocab % 4) != 0 || vocab <= 4096 || vocab > 32768) return MARIAN_HIP_ERR_SHAPE;
  if(dimBatch == 0) return MARIAN_HIP_OK;
  if(!logits || !outScores || !outKeys || !workspace) return MARIAN_HIP_ERR_NULL;
  if(dimBatch * beam * vocab > 4294967295LL || dimBatch > kNbestMaxBatch) return MARIAN_HIP_ERR_RANGE;   // keys are uint32
  if(!aligned16(logits) || (logProbs && !aligned16(logProbs)) || (rowAdd && !aligned4(rowAdd)) ||
     !aligned4(outScores) || !aligned4(outKeys) || !aligned4(workspace))
    return MARIAN_HIP_ERR_ALIGN;
  const size_t entries = (size_t)dimBatch * beam * N;
  if(workspace_bytes < kNbestCounterBytes + entries * 8) return MARIAN_HIP_ERR_WORKSPACE;
  // (the layout of marian_hip_nbest_beams with one part per beam entry)
  unsigned* counters = reinterpret_cast<unsigned*>(workspace);
  float* candVal = reinterpret_cast<float*>(counters + kNbestMaxBatch * kNbestCounterStride);
  unsigned* candIdx = reinterpret_cast<unsigned*>(candVal + entries);
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)beam, (unsigned)dimBatch);
#define MH_LSNB(VPT, KEEP, FENCED)                                                                                   \
  MH_LAUNCH((logsoftmax_nbest_kernel<VPT, KEEP, FENCED>), grid, dim3(1024), 0, st, logits, rowAdd, logProbs, \
                     (long long)dimBatch, (int)vocab, (int)N, (int)beam, candVal, candIdx, counters, outScores, outKeys)
  if(nbest_fenced()) {
#ifdef MARIAN_HIP_TUNING
    if(N <= 4) MH_LSNB(8, 4, true);
    else if(N <= 8) MH_LSNB(8, 8, true);
    else MH_LSNB(8, 16, true);
#endif
  } else {
    if(N <= 4) MH_LSNB(8, 4, false);
    else if(N <= 8) MH_LSNB(8, 8, false);
    else MH_LSNB(8, 16, false);
  }
#undef MH_LSNB
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

}  // extern "C"
