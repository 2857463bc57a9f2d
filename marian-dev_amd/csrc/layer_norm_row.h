// Layer normalization of a row of up to 1024 values by one wave, four float4 per lane: the row computation
// of the layer-norm launch and of the kernels that normalize their input themselves.  The same operations
// in the same order everywhere, so the results have the same bits.
#pragma once

#include "int8_common.h"
#include "quantize_common.h"

namespace marian_hip {

// Sum over each group of 16 consecutive lanes, left in all 16 of them (four DPP steps: the two
// lane swaps within a quad, then the mirror within half a row and within the row).
__device__ __forceinline__ float row16_sum(float v) {
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0xB1, 0xF, 0xF, false));   // quad_perm [1,0,3,2]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x4E, 0xF, 0xF, false));   // quad_perm [2,3,0,1]
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x141, 0xF, 0xF, false));  // row_half_mirror
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x140, 0xF, 0xF, false));  // row_mirror
  return v;
}
// Sum over the wave, the same value in all lanes: within the rows of 16 lanes, then across them
// with the two row-broadcast DPP steps (rows 1 and 3 take in the last lane of the row before them,
// then rows 2 and 3 the last lane of row 1), which leaves the total in lane 63, read from there as
// a scalar.  No step goes through the LDS crossbar (a lane exchange there costs ten times a DPP
// step).  All lanes of the wave must be active.
__device__ __forceinline__ float wave_sum(float v) {
  v = row16_sum(v);
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x142, 0xA, 0xF, false));   // row_bcast:15
  v += __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x143, 0xC, 0xF, false));   // row_bcast:31
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}

constexpr int kNormVecs = 4;   // float4 per lane: rows of up to 1024 values, cols % 4 == 0 (half as many: up to 512)

// Value j of a lane is float4 number j * 64 + lane of the row; positions past the row hold whatever the loader gives there (zeros of a
// buffer, or the row's last values again) and are dropped here.  v: the row, becomes its normalization (those positions: anything); t: what is added to
// it first (has_add).  Returns the largest magnitude of this lane's values.
template <int VECS>
__device__ __forceinline__ float normalize_row(v4f (&v)[VECS], const v4f (&t)[VECS], bool has_add, const v4f (&gm)[VECS],
                                               const v4f (&bt)[VECS], bool has_beta, int cols, float eps) {
  const int lane = threadIdx.x % kWave, cols4 = cols / 4;
  float sum = 0.0f;
#pragma unroll
  for(int j = 0; j < VECS; ++j) {
    if(has_add) v[j] = v4f{v[j].x + t[j].x, v[j].y + t[j].y, v[j].z + t[j].z, v[j].w + t[j].w};
    if(j * kWave + lane < cols4) sum += (v[j].x + v[j].y) + (v[j].z + v[j].w);
  }
  const float mean = wave_sum(sum) / (float)cols;
  float sq = 0.0f, least = kQuotientMost;
#pragma unroll
  for(int j = 0; j < VECS; ++j) {
    v[j] = v4f{v[j].x - mean, v[j].y - mean, v[j].z - mean, v[j].w - mean};
    if(j * kWave + lane < cols4) {
      sq += (v[j].x * v[j].x + v[j].y * v[j].y) + (v[j].z * v[j].z + v[j].w * v[j].w);
      least = fminf(fminf(fminf(least, fabsf(v[j].x)), fminf(fabsf(v[j].y), fabsf(v[j].z))), fabsf(v[j].w));
    }
  }
  const float sigma = sqrtf(wave_sum(sq) / (float)cols + eps);
  // Quotients by a shared reciprocal, a few operations each where a division takes eleven, unless a step could under- or overflow (no
  // quotient is above sqrt(cols)).  The division stands in a loop, not unrolled: what a launch runs once it also fetches, and with a second copy of
  // the code steps of 6 layers were no faster (128 x 1024 374.5 us before, 368.9 so; 64 x 64 words through an encoder of 1024 957 and 951).
  // Values equal to the mean (rows of padding) are zeros here, for which the reciprocal will do as well; a wave that has some finds that out off the
  // others' way (a launch of 6 x 512 zeros 3.2 us by division, 4.1 in the loop, 3.0 so, of 4096 x 1024 9.7, 11.5 and 9.8, without a skip input 7.7, 9.9
  // and 7.4; other rows the same.  With one copy of the quotients behind the second look a step of 6 hypotheses took 0.9 % longer).
  const bool in_range = sigma >= kDivisorLeast && sigma <= kDivisorMost;
  auto by_reciprocal = [&](float sigma) __attribute__((always_inline)) {
    const float reciprocal = 1.0f / sigma;
#pragma unroll
    for(int j = 0; j < VECS; ++j)
#pragma unroll
      for(int e = 0; e < 4; ++e) v[j][e] = shared_quotient(v[j][e], sigma, reciprocal);
  };
  if(__builtin_expect(__all(least >= kQuotientLeast) && in_range, 1)) {
    by_reciprocal(sigma);
  } else {
    unsigned order = ~0u;
#pragma unroll
    for(int j = 0; j < VECS; ++j)
      if(j * kWave + lane < cols4)
#pragma unroll
        for(int e = 0; e < 4; ++e) order = min(order, dividend_order(v[j][e]));
    if(__all(order >= kDividendLeast) && in_range) {
      float same = sigma;
      asm volatile("" : "+v"(same));   // (or else the compiler has one copy of this for both, behind everything)
      by_reciprocal(same);
    } else {
#pragma unroll 1
      for(int i = 0; i < 4 * VECS; ++i) {   // (the first value is divided and goes to the end)
        const float q = v[0][0] / sigma;
#pragma unroll
        for(int k = 0; k < 4 * VECS - 1; ++k) v[k / 4][k % 4] = v[(k + 1) / 4][(k + 1) % 4];
        v[VECS - 1][3] = q;
      }
    }
  }
  float omax = 0.0f;
#pragma unroll
  for(int j = 0; j < VECS; ++j) {
    if(j * kWave + lane < cols4) {
      const float g[4] = {gm[j].x, gm[j].y, gm[j].z, gm[j].w}, b[4] = {bt[j].x, bt[j].y, bt[j].z, bt[j].w};
#pragma unroll
      for(int e = 0; e < 4; ++e) {
        float o = g[e] * v[j][e];
        if(has_beta) o = o + b[e];
        v[j][e] = o;
        omax = fmaxf(omax, fabsf(o));
      }
    }
  }
  return omax;
}

// A decoding step's few hypotheses: the kernel that multiplies the normalized rows normalizes them itself -
// every workgroup all of them, a wave to a row - instead of reading what a launch of its own has left.
constexpr int kNormMaxRows = 8, kNormMaxCols = 256 * kNormVecs;
struct NormInput {
  const float* add;     // [M x K]: the skip connection
  const float* gamma;   // [K]
  const float* beta;    // [K]
  float* out;           // [M x K]: the normalized rows, written by one workgroup
  float eps;
};
// The same with the vectors a lane takes of a row, as a kernel argument.
template <int VECS>
struct NormInputOf : NormInput {
  static constexpr int kVecs = VECS;
};
template <int VECS>
struct NormRow {
  v4f v[VECS], t[VECS], gm[VECS], bt[VECS];
  // Wave w loads row w (rows past M: a copy of the last one).  All loads unconditional, so that waits count them exactly.
  __device__ __forceinline__ void load(const float* A, const float* add, const NormInput& n, int M, int K) {
    const int lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const size_t row = (size_t)min(wave, M - 1) * K;
    auto load_buffer = [&](const float* p, int j) __attribute__((always_inline)) {   // (past the row: zeros)
      return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(
                                         __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p), 0, K * 4, kRawBuffer), lane * 16 + j * 1024, 0, 0));
    };
#pragma unroll
    for(int j = 0; j < VECS; ++j) {
      v[j] = load_buffer(A + row, j);
      t[j] = load_buffer(add + row, j);
    }
#pragma unroll
    for(int j = 0; j < VECS; ++j) {
      gm[j] = load_buffer(n.gamma, j);
      bt[j] = load_buffer(n.beta, j);
    }
  }
  __device__ __forceinline__ float normalize(const NormInput& n, int K) {
    return normalize_row(v, t, true, gm, bt, true, K, n.eps);
  }
  // The row's quantized values into LDS in operand order: slot (c16 / 2, c16 % 2, row) of 16 bytes holds 16-byte
  // chunk c16 of the row, rows XOR-permuted by the key of the chunk.
  template <typename KEY>
  __device__ __forceinline__ void quantize(int8_t* lds, int row, int K, float qm, KEY key) const {
    const int lane = threadIdx.x % kWave;
    const float by = quantizer(qm);
#pragma unroll
    for(int j = 0; j < VECS; ++j) {
      const int i = j * kWave + lane, c16 = i / 4;
      if(i < K / 4)
        *reinterpret_cast<uint32_t*>(lds + ((c16 / 2) * 64 + (c16 % 2) * 32 + (row ^ key(c16))) * 16 + (i % 4) * 4) = quantize_pack4(v[j], by);
    }
  }
  __device__ __forceinline__ void store(const NormInput& n, int row, int K) const {
    const int lane = threadIdx.x % kWave;
#pragma unroll
    for(int j = 0; j < VECS; ++j)
      if(j * kWave + lane < K / 4) reinterpret_cast<v4f*>(n.out + (size_t)row * K)[j * kWave + lane] = v[j];
  }
};

}  // namespace marian_hip
