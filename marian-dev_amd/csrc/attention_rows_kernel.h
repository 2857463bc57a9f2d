// Attention with several query positions per head (encoder layers, whole target sentences), head size 64:
// softmax(scale * q k^T + mask) v in one launch on the float32 matrix instruction, over heads that lie
// side by side in a row (the affine call's output as it is) or apart.
#pragma once

#include "int8_common.h"
#include "quantize_common.h"

namespace marian_hip {

// A tensor [batch, heads, positions, dk]: floats from one sentence, head and position to the next.
struct HeadStrides {
  long long batch, head, row;
  __host__ __device__ size_t entry(unsigned e, unsigned heads) const { return (size_t)(e / heads) * batch + (size_t)(e % heads) * head; }
};

struct AttentionRowsArgs {
  const float *q, *k, *v, *mask;
  float* out;
  float* absmax_out;   // kAbsmaxSlots values whose maximum is max|out| (a slot per wave), or null
  HeadStrides qs, ks, vs, os;
  unsigned batchQ, batchKV, heads, n_masks, rows_per_mask;
  int m, len, row_blocks;
  float scale;
};

typedef v4f v4f_any __attribute__((aligned(4)));   // sixteen bytes at any float's address

// Four registers of the four rows of sixteen lanes, transposed: register x of row g becomes register g of row x.
__device__ __forceinline__ v4f rows_to_registers(v4f m) {
  typedef unsigned v2u __attribute__((ext_vector_type(2)));
  unsigned r[4];
#pragma unroll
  for(int e = 0; e < 4; ++e) r[e] = __float_as_uint(m[e]);
#pragma unroll
  for(int e = 0; e < 2; ++e) {   // lanes 32 .. 63 of one against lanes 0 .. 31 of the other
    const v2u s = __builtin_amdgcn_permlane32_swap(r[e], r[e + 2], false, false);
    r[e] = s.x;
    r[e + 2] = s.y;
  }
#pragma unroll
  for(int e = 0; e < 4; e += 2) {   // rows 1 and 3 of one against rows 0 and 2 of the other
    const v2u s = __builtin_amdgcn_permlane16_swap(r[e], r[e + 1], false, false);
    r[e] = s.x;
    r[e + 1] = s.y;
  }
  return v4f{__uint_as_float(r[0]), __uint_as_float(r[1]), __uint_as_float(r[2]), __uint_as_float(r[3])};
}

// A wave makes 16 R query rows of one head over len <= 64 NB keys; waves share nothing, so there is no LDS and no
// barrier.  Scores come as S^T = K Q^T: lane (c = lane % 16, g = lane / 16) then holds, for query row c, the scores of
// keys 16 t + 4 g + r (t, r = 0 .. 3) of each block of 64, so a row's maximum and sum need two lane exchanges, and
// O^T = V^T P^T takes the weights as its second operand, transposed within four lanes.  Every load is sixteen
// bytes a lane and a wave's lanes cover whole lines: four dimensions of key or query row c (transposed within
// four lanes as well), four of value row 16 t + 4 r + g.
// The results are those of bdot_legacy, softmax and bdot_legacy bit for bit: the matrix instruction adds its four
// products to the accumulator in order of k, each with one rounding, exactly as a chain of fmaf does (checked
// over normal and denormal numbers), so with k-steps in ascending order every product sums as bdot_kernel sums;
// exponentials, their sum (elements 64 apart first, then the tree of wave_sum) and the division are
// softmax_kernel's.  A rounding that moves here moves an 8-bit quantization further down the network.
// Bound by the float32 matrix rate (16 x 16 x 4 in 32 clocks: 1024 heads of 64 x 64 take 6.8 us at 2.4 GHz) and, with
// R = 1, by the loads (keys and values again for every sixteen rows).  The three operators it replaces took 59 us
// there, and the transpositions to and from heads 32 us.
template <int R, int NB>
__global__ __launch_bounds__(256, 2) void attention_rows_kernel(AttentionRowsArgs p) {
  const unsigned w = blockIdx.x * 4u + threadIdx.x / 64u;
  if(p.absmax_out && blockIdx.x == 0)   // slots past the last wave
    for(unsigned sl = p.batchQ * (unsigned)p.row_blocks + threadIdx.x; sl < (unsigned)kAbsmaxSlots; sl += 256) p.absmax_out[sl] = 0.0f;
  const unsigned entry = w / (unsigned)p.row_blocks;
  if(entry >= p.batchQ) return;   // (whole waves)
  const int row0 = (int)(w % (unsigned)p.row_blocks) * (16 * R);
  const int lane = threadIdx.x % 64, c = lane % 16, g = lane / 16;
  const unsigned ekv = entry < p.batchKV ? entry : entry % p.batchKV;
  const float* kb = p.k + p.ks.entry(ekv, p.heads) + 4 * g;
  const float* vb = p.v + p.vs.entry(ekv, p.heads) + 4 * c;
  const float* qb = p.q + p.qs.entry(entry, p.heads) + 4 * g;

  v4f q[R][4];
  const float* mask[R];
#pragma unroll
  for(int rt = 0; rt < R; ++rt) {
    const int row = min(row0 + 16 * rt + c, p.m - 1);   // (rows past the end: the last one again, not stored)
#pragma unroll
    for(int s = 0; s < 4; ++s) q[rt][s] = *reinterpret_cast<const v4f*>(qb + (size_t)row * p.qs.row + 16 * s);
    unsigned mr = (entry * (unsigned)p.m + (unsigned)row) / p.rows_per_mask;
    if(mr >= p.n_masks) mr %= p.n_masks;
    mask[rt] = p.mask ? p.mask + (size_t)mr * p.len : nullptr;
  }
  v4f k[4][4], v[4][4], z[R][NB][4];
  auto load_k = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for(int t = 0; t < 4; ++t) {
      const float* src = kb + (size_t)min(64 * b + 16 * t + c, p.len - 1) * p.ks.row;
#pragma unroll
      for(int s = 0; s < 4; ++s) k[t][s] = *reinterpret_cast<const v4f*>(src + 16 * s);
    }
  };
  auto load_v = [&](int b) __attribute__((always_inline)) {
#pragma unroll
    for(int t = 0; t < 4; ++t)
#pragma unroll
      for(int r = 0; r < 4; ++r) v[t][r] = *reinterpret_cast<const v4f*>(vb + (size_t)min(64 * b + 16 * t + 4 * r + g, p.len - 1) * p.vs.row);
  };
  load_k(0);
#pragma unroll
  for(int rt = 0; rt < R; ++rt)
#pragma unroll
    for(int s = 0; s < 4; ++s) q[rt][s] = rows_to_registers(q[rt][s]);

  // ---- scores ----
#pragma unroll
  for(int b = 0; b < NB; ++b) {
#pragma unroll
    for(int rt = 0; rt < R; ++rt)
#pragma unroll
      for(int t = 0; t < 4; ++t) z[rt][b][t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for(int t = 0; t < 4; ++t)
#pragma unroll
      for(int s = 0; s < 4; ++s) {
        const v4f kt = rows_to_registers(k[t][s]);
#pragma unroll
        for(int x = 0; x < 4; ++x)
#pragma unroll
          for(int rt = 0; rt < R; ++rt) z[rt][b][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(kt[x], q[rt][s][x], z[rt][b][t], 0, 0, 0);
      }
    if(b + 1 < NB) load_k(b + 1);
    else load_v(0);
  }

  // ---- weights ----
#pragma unroll
  for(int rt = 0; rt < R; ++rt) {
    float mx = -__builtin_inff();
#pragma unroll
    for(int b = 0; b < NB; ++b) {
      const bool whole = b + 1 < NB || 64 * NB == p.len;   // (the same for every wave)
#pragma unroll
      for(int t = 0; t < 4; ++t) {
        const int key = 64 * b + 16 * t + 4 * g;
        v4f mk = v4f{0.0f, 0.0f, 0.0f, 0.0f};
        if(p.mask) {
          if(whole) mk = *reinterpret_cast<const v4f_any*>(mask[rt] + key);
          else {
#pragma unroll
            for(int r = 0; r < 4; ++r) mk[r] = mask[rt][min(key + r, p.len - 1)];
          }
        }
#pragma unroll
        for(int r = 0; r < 4; ++r) {
          float x = p.scale * z[rt][b][t][r];
          if(p.mask) x = x + mk[r];
          if(!whole && key + r >= p.len) x = -__builtin_inff();
          z[rt][b][t][r] = x;
          mx = fmaxf(mx, x);
        }
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    // (a column past the end of the row adds nothing, also where the whole row is -inf and its sum NaN)
    float at[4][4];   // the sums of elements 64 apart
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int t = 0; t < 4; ++t)
#pragma unroll
        for(int r = 0; r < 4; ++r) {
          float e = expf(z[rt][b][t][r] - mx);
          if(b + 1 == NB && 64 * b + 16 * t + 4 * g + r >= p.len) e = 0.0f;
          z[rt][b][t][r] = e;
          at[t][r] = b == 0 ? e : at[t][r] + e;
        }
    float row[4];
#pragma unroll
    for(int t = 0; t < 4; ++t) {
      float s = (at[t][0] + at[t][1]) + (at[t][2] + at[t][3]);
      s += __shfl_xor(s, 16);
      row[t] = s + __shfl_xor(s, 32);
    }
    const float sum = (row[0] + row[1]) + (row[2] + row[3]);
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int t = 0; t < 4; ++t) {
#pragma unroll
        for(int r = 0; r < 4; ++r) z[rt][b][t][r] = z[rt][b][t][r] / sum;
        z[rt][b][t] = rows_to_registers(z[rt][b][t]);   // weight of key 16 t + 4 x + g in register x
      }
  }

  // ---- weighted values ----
  v4f o[R][4];
#pragma unroll
  for(int rt = 0; rt < R; ++rt)
#pragma unroll
    for(int j = 0; j < 4; ++j) o[rt][j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for(int b = 0; b < NB; ++b) {
    if(b + 1 == NB) {   // past the last key: nothing, whatever the last value row holds
#pragma unroll
      for(int t = 0; t < 4; ++t)
#pragma unroll
        for(int x = 0; x < 4; ++x)
          if(64 * b + 16 * t + 4 * x + g >= p.len) {
            v[t][x] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for(int rt = 0; rt < R; ++rt) z[rt][b][t][x] = 0.0f;
          }
    }
#pragma unroll
    for(int t = 0; t < 4; ++t)
#pragma unroll
      for(int x = 0; x < 4; ++x)
#pragma unroll
        for(int j = 0; j < 4; ++j)
#pragma unroll
          for(int rt = 0; rt < R; ++rt) o[rt][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[t][x][j], z[rt][b][t][x], o[rt][j], 0, 0, 0);
    if(b + 1 < NB) load_v(b + 1);
  }
  // lane (c, g): row c, d = 16 g + 4 r + j
  float omax = 0.0f;
#pragma unroll
  for(int rt = 0; rt < R; ++rt) {
    const int row = row0 + 16 * rt + c;
    if(row < p.m) {
      float* dst = p.out + p.os.entry(entry, p.heads) + (size_t)row * p.os.row + 16 * g;
#pragma unroll
      for(int r = 0; r < 4; ++r) {
        const v4f y = v4f{o[rt][0][r], o[rt][1][r], o[rt][2][r], o[rt][3][r]};
        *reinterpret_cast<v4f*>(dst + 4 * r) = y;
        omax = abs4max(y, omax);
      }
    }
  }
  if(p.absmax_out) {
    omax = wave_max(omax);
    if(lane == 0) p.absmax_out[w] = omax;
  }
}

}  // namespace marian_hip
