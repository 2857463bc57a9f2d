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
  int m, len, row_blocks, row_groups;   // blocks of 16 query rows, and over how many workgroups a head's are dealt out
  float scale;
  int head_mask;   // all query rows of a head have the same mask row: it is looked up and loaded once
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

// A workgroup of four waves takes one head and every row_groups-th block of 16 query rows, len <= 64 NB keys.
// Wave w multiplies keys 16 w .. 16 w + 15 of each block of 64 and makes outputs 16 w .. 16 w + 15, so that its share of
// keys and values (16 NB registers each) is read once for all rows; the scores' maxima, the sums and the weights
// (4 NB KB) change hands in LDS.
// Scores come as S^T = K Q^T: lane (c = lane % 16, g = lane / 16) holds, for query row c, the scores of keys 16 w +
// 4 g + r (r = 0 .. 3) of each block, so a row's maximum and sum need two lane exchanges within the wave, and
// O^T = V^T P^T takes the weights of row c as its second operand.  Rows of K are loaded four dimensions a lane, whole
// lines a wave, and transposed within four lanes; rows of Q once for the four waves, through LDS.
// The results are those of bdot_legacy, softmax and bdot_legacy bit for bit: the matrix instruction adds its four
// products to the accumulator in order of k, each with one rounding, exactly as a chain of fmaf does (checked
// over normal and denormal numbers), so with k-steps in ascending order every product sums as bdot_kernel sums;
// exponentials, their sum (elements 64 apart first, then the tree of wave_sum) and the division are
// softmax_kernel's.  A rounding that moves here moves an 8-bit quantization further down the network.
// Bound by its chains for a few heads, by the float32 matrix rate (16 x 16 x 4 in 32 clocks: 1024 heads of 64 x 64 take
// 6.8 us at 2.4 GHz) and the traffic (67 MB there) for many.
// Measured (in a graph, masks included): 8 heads of 23 x 23 4.1 us, 128 of 64 x 64 6.2, 1024 of 64 x 64 22.0, 384 of 128 x 128
// 28.1 (23.1 and 29.4 with a mask row looked up and loaded per block of query rows; fewer resident workgroups or staggered starts
// change nothing).  Before, 1024 heads took three operators of 59 us and four transpositions of 32 us, one sentence 8.7 us with
// a wave to 16 rows and all keys (no LDS, the same bits).
template <int NB>
__global__ __launch_bounds__(256, NB == 1 ? 4 : (NB == 2 ? 3 : 2)) void attention_rows_kernel(AttentionRowsArgs p) {
  constexpr int kPitch = 64 * NB + 4;   // floats of a weight row
  __shared__ float top_lds[2][4][16], sum_lds[2][4][16];
  __shared__ __attribute__((aligned(16))) float weight_lds[2][16][kPitch];
  __shared__ __attribute__((aligned(16))) float q_lds[2][16][64 + 4];   // d = 16 s + 4 x + y of a row at 16 s + 4 y + x
  const unsigned entry = blockIdx.x / (unsigned)p.row_groups;
  const int group = (int)(blockIdx.x % (unsigned)p.row_groups);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, c = lane % 16, g = lane / 16;
  if(p.absmax_out && blockIdx.x == 0)   // slots past the last wave
    for(unsigned sl = p.batchQ * (unsigned)p.row_groups * 4u + threadIdx.x; sl < (unsigned)kAbsmaxSlots; sl += 256) p.absmax_out[sl] = 0.0f;
  const unsigned ekv = entry < p.batchKV ? entry : entry % p.batchKV;
  // (offsets within a tensor fit 32 bits: checked by the launcher)
  const float* kb = p.k + p.ks.entry(ekv, p.heads);
  const float* vb = p.v + p.vs.entry(ekv, p.heads);
  const float* qb = p.q + p.qs.entry(entry, p.heads);
  float* ob = p.out + p.os.entry(entry, p.heads);
  const int k_row = (int)p.ks.row, v_row = (int)p.vs.row, q_row = (int)p.qs.row, o_row = (int)p.os.row;

  v4f k[NB][4], q_next;
  float v[NB][4][4], mask_next[NB][4];
  // a block of query rows: sixteen bytes a thread; and the mask values of this lane's scores
  const int q_in = threadIdx.x / 16, q_at = threadIdx.x % 16;
  auto load_q = [&](int block) __attribute__((always_inline)) {   // (rows past the end: the last one again, not stored)
    q_next = *reinterpret_cast<const v4f*>(qb + min(block * 16 + q_in, p.m - 1) * q_row + 4 * q_at);
  };
  auto load_mask = [&](int block) __attribute__((always_inline)) {
    unsigned mr = (entry * (unsigned)p.m + (unsigned)min(block * 16 + c, p.m - 1)) / p.rows_per_mask;
    if(mr >= p.n_masks) mr %= p.n_masks;
    const float* m = p.mask + (size_t)mr * p.len;
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int r = 0; r < 4; ++r) mask_next[b][r] = m[min(64 * b + 16 * wave + 4 * g + r, p.len - 1)];
  };
  auto keep_q = [&](int turn) __attribute__((always_inline)) {
#pragma unroll
    for(int y = 0; y < 4; ++y) q_lds[turn][q_in][16 * (q_at / 4) + 4 * y + q_at % 4] = q_next[y];
  };
  load_q(group);
  if(p.mask) load_mask(group);
#pragma unroll
  for(int b = 0; b < NB; ++b) {
    const float* src = kb + min(64 * b + 16 * wave + c, p.len - 1) * k_row + 4 * g;
#pragma unroll
    for(int s = 0; s < 4; ++s) k[b][s] = *reinterpret_cast<const v4f*>(src + 16 * s);
  }
#pragma unroll
  for(int b = 0; b < NB; ++b)
#pragma unroll
    for(int t = 0; t < 4; ++t)
#pragma unroll
      for(int x = 0; x < 4; ++x) v[b][t][x] = vb[min(64 * b + 16 * t + 4 * x + g, p.len - 1) * v_row + 16 * wave + c];
#pragma unroll
  for(int b = 0; b < NB; ++b)
#pragma unroll
    for(int s = 0; s < 4; ++s) k[b][s] = rows_to_registers(k[b][s]);
  const int tiles = (p.len + 15) / 16;   // blocks of 16 keys
  if(p.len % 16 != 0) {   // past the last key: nothing, whatever the last value row holds
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int t = 0; t < 4; ++t)
        if(4 * b + t == tiles - 1) {
#pragma unroll
          for(int x = 0; x < 4; ++x)
            if(64 * b + 16 * t + 4 * x + g >= p.len) v[b][t][x] = 0.0f;
        }
  }

  keep_q(0);
  __syncthreads();
  float omax = 0.0f;
  int turn = 0;   // (a wave may still read one turn's values in LDS while another writes the next's)
  for(int block = group; block < p.row_blocks; block += p.row_groups, turn ^= 1) {
    const int row = block * 16 + c;
    v4f q[4];
#pragma unroll
    for(int s = 0; s < 4; ++s) q[s] = *reinterpret_cast<const v4f*>(&q_lds[turn][c][16 * s + 4 * g]);
    float mask[NB][4];
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int r = 0; r < 4; ++r) mask[b][r] = mask_next[b][r];
    load_q(min(block + p.row_groups, p.row_blocks - 1));
    if(p.mask && !p.head_mask) load_mask(min(block + p.row_groups, p.row_blocks - 1));
    // ---- scores ----
    v4f z[NB];
#pragma unroll
    for(int b = 0; b < NB; ++b) {
      z[b] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
      if(4 * b + wave < tiles) {
#pragma unroll
        for(int s = 0; s < 4; ++s)
#pragma unroll
          for(int x = 0; x < 4; ++x) z[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[b][s][x], q[s][x], z[b], 0, 0, 0);
      }
    }
    float mx = -__builtin_inff();
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int r = 0; r < 4; ++r) {
        const int key = 64 * b + 16 * wave + 4 * g + r;
        float x = p.scale * z[b][r];
        if(p.mask) x = x + mask[b][r];
        z[b][r] = key < p.len ? x : -__builtin_inff();
        mx = fmaxf(mx, z[b][r]);
      }
    mx = fmaxf(mx, __shfl_xor(mx, 16));
    mx = fmaxf(mx, __shfl_xor(mx, 32));
    if(g == 0) top_lds[turn][wave][c] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(top_lds[turn][0][c], top_lds[turn][1][c]), fmaxf(top_lds[turn][2][c], top_lds[turn][3][c]));
    // ---- weights ----
    float at[4];   // the sums of elements 64 apart
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int r = 0; r < 4; ++r) {
        float e = expf(z[b][r] - mx);
        if(64 * b + 16 * wave + 4 * g + r >= p.len) e = 0.0f;   // (also where the whole row is -inf and its sum NaN)
        z[b][r] = e;
        at[r] = b == 0 ? e : at[r] + e;
      }
    float part = (at[0] + at[1]) + (at[2] + at[3]);
    part += __shfl_xor(part, 16);
    part += __shfl_xor(part, 32);
    if(g == 0) sum_lds[turn][wave][c] = part;
    __syncthreads();
    const float sum = (sum_lds[turn][0][c] + sum_lds[turn][1][c]) + (sum_lds[turn][2][c] + sum_lds[turn][3][c]);
    // (key 16 t + 4 x + y of a block at 16 t + 4 y + x: what a lane of the next product needs lies together)
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int r = 0; r < 4; ++r) {
        const float w = z[b][r] / sum;
        weight_lds[turn][c][64 * b + 16 * wave + 4 * r + g] = 64 * b + 16 * wave + 4 * g + r < p.len ? w : 0.0f;
      }
    keep_q(turn ^ 1);
    __syncthreads();
    // ---- weighted values ----
    v4f o = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for(int b = 0; b < NB; ++b)
#pragma unroll
      for(int t = 0; t < 4; ++t)
        if(4 * b + t < tiles) {
          const v4f w = *reinterpret_cast<const v4f*>(&weight_lds[turn][c][64 * b + 16 * t + 4 * g]);
#pragma unroll
          for(int x = 0; x < 4; ++x) o = __builtin_amdgcn_mfma_f32_16x16x4f32(v[b][t][x], w[x], o, 0, 0, 0);
        }
    if(row < p.m) {
      *reinterpret_cast<v4f*>(ob + row * o_row + 16 * wave + 4 * g) = o;
      omax = abs4max(o, omax);
    }
  }
  if(p.absmax_out) {
    omax = wave_max(omax);
    if(lane == 0) p.absmax_out[blockIdx.x * 4u + wave] = omax;
  }
}

// Max and sum over the four rows of sixteen lanes, in all of them: two swaps of register halves, nothing through LDS.
typedef unsigned v2u_rows __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float rows4_max(float v) {
  v2u_rows s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(s.x), __uint_as_float(s.y));
  s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(s.x), __uint_as_float(s.y));
}
__device__ __forceinline__ float rows4_sum(float v) {
  v2u_rows s = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(s.x) + __uint_as_float(s.y);
  s = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(s.x) + __uint_as_float(s.y);
}

// As attention_rows_kernel, for heads that fill the chip: a wave takes 16 query rows and all keys, so nothing changes hands
// between the waves but the keys and values, which they lay out in LDS in matrix-operand order once.  The weights of a row
// stay in registers (a transposition over the rows of sixteen lanes makes them operands).
// Bound by the float32 pipes: a float32 matrix instruction holds up the SIMD's other float32 instructions, of other waves
// too (32 of them and 128 fmaf take 0.45 and 0.23 us by themselves, 0.67 together), so the 128 products of 32 clocks and some 450
// vector instructions of a wave of 64 keys add up; the form above has 890 of the latter, a division and three barriers of
// four waves to every 16 x 64 scores.  Loads run past the ends into nothing (buffers) instead of having their rows clamped, divisions share
// their divisor's reciprocal.
// Measured (masks included, the form above and this): 1024 heads of 64 x 64 21.8 -> 18.8 us, 256 of them 9.2 -> 7.1; 1024 of 23 x 23 10.0 -> 7.6;
// 512 of 48 x 48 9.6 -> 8.6; 512 of 70 x 70 23.0 -> 20.0; 384 of 128 x 128 28.5 -> 26.0.  Which heads take it:
// attention_plan.h.  The least number of blocks of keys is a kernel of its own (four for 37 keys 14.8 us, three 12.7), but for seven, which run as eight
// without the products of the last block's values.
// TILES: blocks of 16 keys; WAVES: 16-row blocks of queries of a workgroup.
template <int TILES, int WAVES>
__global__ __launch_bounds__(WAVES * 64, 4) void attention_heads_kernel(AttentionRowsArgs p) {
  constexpr int kTiles = TILES, kWaves = WAVES, kStage = (TILES + WAVES - 1) / WAVES;
  __shared__ v4f k_lds[kTiles][4][kWave], v_lds[kTiles][4][kWave];
  const unsigned entry = blockIdx.x / (unsigned)p.row_groups;
  const int group = (int)(blockIdx.x % (unsigned)p.row_groups);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64, c = lane % 16, g = lane / 16;
  if(p.absmax_out && blockIdx.x == 0)   // slots past the last wave
    for(unsigned sl = p.batchQ * (unsigned)p.row_groups * kWaves + threadIdx.x; sl < (unsigned)kAbsmaxSlots; sl += 64 * kWaves) p.absmax_out[sl] = 0.0f;
  const unsigned ekv = entry < p.batchKV ? entry : entry % p.batchKV;
  const unsigned k_row = (unsigned)p.ks.row * 4u, v_row = (unsigned)p.vs.row * 4u, q_row = (unsigned)p.qs.row * 4u;   // bytes
  const int row0 = (group * kWaves + wave) * 16, row = row0 + c;
  // (as buffers that end behind their last row: rows past it read as zeros, without a check.  The hardware holds the sum of the lane's and the scalar
  // offset against the buffer's end, also where the latter alone lies behind it: looked at for 45 of both, within an allocation that goes on)
  const auto k_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.k + p.ks.entry(ekv, p.heads)), 0, (int)((unsigned)(p.len - 1) * k_row + 256u), kRawBuffer);
  const auto v_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.v + p.vs.entry(ekv, p.heads)), 0, (int)((unsigned)(p.len - 1) * v_row + 256u), kRawBuffer);
  const auto q_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.q + p.qs.entry(entry, p.heads)), 0, (int)((unsigned)(p.m - 1) * q_row + 256u), kRawBuffer);
  auto load = [](auto buf, unsigned lane_at, unsigned at) __attribute__((always_inline)) { return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(buf, lane_at, at, 0)); };

  // ---- keys and values of the wave's block of sixteen, its query rows, their mask values ----
  v4f kr[kStage][4], vr[kStage][4], q[4], mask[kTiles];
  const unsigned k_at = (unsigned)(16 * wave + c) * k_row + 16u * g, v_at = (unsigned)(16 * wave + g) * v_row + 16u * c, q_at = (unsigned)row * q_row + 16u * g;
#pragma unroll
  for(int i = 0; i < kStage; ++i)
#pragma unroll
    for(int s = 0; s < 4; ++s) kr[i][s] = load(k_buf, k_at, 16u * kWaves * i * k_row + 64u * s);
#pragma unroll
  for(int i = 0; i < kStage; ++i)
#pragma unroll
    for(int x = 0; x < 4; ++x) vr[i][x] = load(v_buf, v_at, (16u * kWaves * i + 4u * x) * v_row);
#pragma unroll
  for(int s = 0; s < 4; ++s) q[s] = load(q_buf, q_at, 64u * s);
  if(p.mask) {   // (values past a mask row's end: of the next row or none, not looked at)
    unsigned mr = entry * (unsigned)p.m;
    if(p.head_mask) {
      mr /= p.rows_per_mask;
      if(mr >= p.n_masks) mr %= p.n_masks;
    } else {
      mr = (mr + (unsigned)min(row, p.m - 1)) / p.rows_per_mask;
      if(mr >= p.n_masks) mr %= p.n_masks;
    }
    const auto m_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(p.mask), 0, (int)(p.n_masks * (unsigned)p.len * 4u), kRawBuffer);
    const unsigned m_at = mr * (unsigned)p.len * 4u + 16u * g;
#pragma unroll
    for(int t = 0; t < kTiles; ++t) mask[t] = load(m_buf, m_at, 64u * t);
  }
#pragma unroll
  for(int i = 0; i < kStage; ++i) {
    const int t = wave + kWaves * i;
    if(kTiles % kWaves == 0 || t < kTiles) {
#pragma unroll
      for(int s = 0; s < 4; ++s) k_lds[t][s][lane] = rows_to_registers(kr[i][s]);
#pragma unroll
      for(int e = 0; e < 4; ++e) v_lds[t][c / 4][16 * g + 4 * (c % 4) + e] = v4f{vr[i][0][e], vr[i][1][e], vr[i][2][e], vr[i][3][e]};
    }
  }
  __syncthreads();
  [[maybe_unused]] const int tiles = (p.len + 15) / 16;
  float omax = 0.0f;
  if(row0 < p.m) {   // (whole waves)
#pragma unroll
    for(int s = 0; s < 4; ++s) q[s] = rows_to_registers(q[s]);
    // ---- scores ----
    v4f z[kTiles];
#pragma unroll
    for(int t = 0; t < kTiles; ++t) z[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for(int t = 0; t < kTiles; t += 2) {   // (two at a time: a product waits for the one before it into the same scores)
#pragma unroll
      for(int s = 0; s < 4; ++s) {
        const v4f k0 = k_lds[t][s][lane], k1 = k_lds[t + 1 < kTiles ? t + 1 : t][s][lane];
#pragma unroll
        for(int x = 0; x < 4; ++x) {
          z[t] = __builtin_amdgcn_mfma_f32_16x16x4f32(k0[x], q[s][x], z[t], 0, 0, 0);
          if(t + 1 < kTiles) z[t + 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k1[x], q[s][x], z[t + 1], 0, 0, 0);
        }
      }
    }
#pragma unroll
    for(int t = 0; t < kTiles; ++t)
#pragma unroll
      for(int r = 0; r < 4; ++r) z[t][r] = p.scale * z[t][r];
    if(p.mask) {
#pragma unroll
      for(int t = 0; t < kTiles; ++t)
#pragma unroll
        for(int r = 0; r < 4; ++r) z[t][r] = z[t][r] + mask[t][r];
    }
    if(p.len < 16 * kTiles) {
#pragma unroll
      for(int t = 0; t < kTiles; ++t)
#pragma unroll
        for(int r = 0; r < 4; ++r) z[t][r] = 16 * t + 4 * g + r < p.len ? z[t][r] : -__builtin_inff();
    }
    float mx = -__builtin_inff();
#pragma unroll
    for(int t = 0; t < kTiles; ++t)
#pragma unroll
      for(int r = 0; r < 4; ++r) mx = fmaxf(mx, z[t][r]);
    mx = rows4_max(mx);
    // ---- weights (past the last key: exp(-inf) = 0, or NaN in a row whose sum is NaN anyway) ----
    v4f part;
    unsigned least = ~0u;
#pragma unroll
    for(int t = 0; t < 4; ++t) {
      float at[4] = {0.0f, 0.0f, 0.0f, 0.0f};   // the sums of elements 64 apart
#pragma unroll
      for(int b = t; b < kTiles; b += 4)
#pragma unroll
        for(int r = 0; r < 4; ++r) {
          const float e = expf(z[b][r] - mx);
          z[b][r] = e;
          least = min(least, __float_as_uint(e) - 1u);   // (zeros pass)
          at[r] = b == t ? e : at[r] + e;
        }
      part[t] = (at[0] + at[1]) + (at[2] + at[3]);
    }
    part = rows_to_registers(part);   // row t: block t's four rows
    const float sum = rows4_sum((part.x + part.y) + (part.z + part.w));   // (1 .. 16 TILES, or NaN)
    if(__all(least >= __float_as_uint(kQuotientLeast) - 1u)) {
      const float r1 = 1.0f / sum;
#pragma unroll
      for(int t = 0; t < kTiles; ++t)
#pragma unroll
        for(int r = 0; r < 4; ++r) z[t][r] = shared_quotient(z[t][r], sum, r1);
    } else {
#pragma unroll
      for(int t = 0; t < kTiles; ++t)
#pragma unroll
        for(int r = 0; r < 4; ++r) z[t][r] = z[t][r] / sum;
    }
#pragma unroll
    for(int t = 0; t < kTiles; ++t) z[t] = rows_to_registers(z[t]);
    // ---- weighted values ----
    v4f o[4];
#pragma unroll
    for(int j = 0; j < 4; ++j) o[j] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for(int t = 0; t < kTiles; ++t)
      if(TILES < 7 || t < tiles) {
        v4f v[4];
#pragma unroll
        for(int j = 0; j < 4; ++j) v[j] = v_lds[t][j][lane];
#pragma unroll
        for(int x = 0; x < 4; ++x)
#pragma unroll
          for(int j = 0; j < 4; ++j) o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[j][x], z[t][x], o[j], 0, 0, 0);
      }
    if(row < p.m) {
      float* ob = p.out + p.os.entry(entry, p.heads) + (unsigned)row * (unsigned)p.os.row + 4 * g;
#pragma unroll
      for(int j = 0; j < 4; ++j) {
        *reinterpret_cast<v4f*>(ob + 16 * j) = o[j];
        omax = abs4max(o[j], omax);
      }
    }
  }
  if(p.absmax_out) {
    omax = wave_max(omax);
    if(lane == 0) p.absmax_out[blockIdx.x * (unsigned)kWaves + wave] = omax;
  }
}

}  // namespace marian_hip
