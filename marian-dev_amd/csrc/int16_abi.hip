// The 16-bit intgemm path (Type::intgemm16): quantizers, GEMMs on the 8-bit matrix instructions and its C ABI.
// Declarations and the reference call sites each entry point replaces: include/marian_hip_int16.h
#include "../../include/marian_hip_int16.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>

#include "../../include/marian_hip_int8.h"
#include "abi_common.h"
#include "int8_common.h"

using namespace marian_hip;

namespace {

typedef short v2s __attribute__((ext_vector_type(2)));

constexpr int64_t kMaxElems16 = 2147483647LL;
constexpr float kQuantMult16 = 1024.0f;   // reference src/tensors/cpu/integer_common.h:174-175

#define MH_HIP(expr)                                       \
  do {                                                     \
    hipError_t e_ = (expr);                                \
    if(e_ != hipSuccess) return record_hip_error((int)e_); \
  } while(0)

inline bool aligned(const void* p, size_t a) { return (reinterpret_cast<uintptr_t>(p) % a) == 0; }

// q = saturate_int16(rne(fl32(x * qm))); a product that is NaN or not below 2^31 gives -32768
// (x86 cvtps2dq "integer indefinite" INT_MIN, then packssdw); products at or below -2^31 saturate
// to -32768 anyway.  med3 returns the smallest operand when one is NaN.
__device__ __forceinline__ int quantize16_one(float x, float qm) {
  const float v = x * qm;
  const float c = __builtin_amdgcn_fmed3f(v, -32768.0f, 32767.0f);
  return (int)__builtin_rintf(v >= 2147483648.0f ? -32768.0f : c);
}
__device__ __forceinline__ uint32_t quantize16_pair(float x0, float x1, float qm) {
  return ((uint32_t)quantize16_one(x0, qm) & 0xFFFFu) | ((uint32_t)quantize16_one(x1, qm) << 16);
}

// prepareA: elementwise, eight values (two 16-byte loads, one 16-byte store) per thread and step
__global__ __launch_bounds__(256) void quantize16_a_kernel(const float* __restrict__ x, size_t n8,
                                                           int16_t* __restrict__ out, int blocks) {
  const v4f* x4 = reinterpret_cast<const v4f*>(x);
  uint4* o = reinterpret_cast<uint4*>(out);
  const size_t stride = (size_t)blocks * 256;
  for(size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += stride) {
    const v4f a = x4[2 * i], b = x4[2 * i + 1];
    uint4 q;
    q.x = quantize16_pair(a.x, a.y, kQuantMult16);
    q.y = quantize16_pair(a.z, a.w, kQuantMult16);
    q.z = quantize16_pair(b.x, b.y, kQuantMult16);
    q.w = quantize16_pair(b.z, b.w, kQuantMult16);
    o[i] = q;
  }
  if(blockIdx.x == 0 && threadIdx.x == 0) *reinterpret_cast<float*>(out + n8 * 8) = kQuantMult16;
}

// prepareB: W fp32 [K x N] -> payload int16 [N x K].  A workgroup transposes a 32(k) x 64(n) tile
// through LDS: reads coalesced along n, writes 16-byte runs along k (K % 32 == 0).
__global__ __launch_bounds__(256) void quantize16_b_transpose_kernel(const float* __restrict__ W, int K, int N,
                                                                      int16_t* __restrict__ out) {
  __shared__ uint32_t tile[64][17];   // [n][k / 2] packed pairs, 17 dwords per row
  const int n0 = blockIdx.x * 64, k0 = blockIdx.y * 32;
  const int tn = threadIdx.x % 64, tk = threadIdx.x / 64;   // wave tk takes k rows 8*tk .. 8*tk+7
  const int n_in = n0 + tn;
#pragma unroll
  for(int g = 0; g < 4; ++g) {
    const int kk = tk * 8 + g * 2;
    float w0 = 0.0f, w1 = 0.0f;
    if(n_in < N) {
      w0 = W[(size_t)(k0 + kk) * N + n_in];
      w1 = W[(size_t)(k0 + kk + 1) * N + n_in];
    }
    tile[tn][kk / 2] = quantize16_pair(w0, w1, kQuantMult16);
  }
  __syncthreads();
  // 64 rows (n) x 64 bytes (32 k): 4 threads per row, 16 bytes each
  const int rn = threadIdx.x / 4, c4 = (threadIdx.x % 4) * 4;
  const int n = n0 + rn;
  if(n < N) {
    uint4 v;
    v.x = tile[rn][c4]; v.y = tile[rn][c4 + 1]; v.z = tile[rn][c4 + 2]; v.w = tile[rn][c4 + 3];
    *reinterpret_cast<uint4*>(out + (size_t)n * K + k0 + c4 * 2) = v;
  }
  if(blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0)
    *reinterpret_cast<float*>(out + (size_t)K * N) = kQuantMult16;
}

// ---- multiplication --------------------------------------------------------------------------
// C[m, n] = sum_k A[m, k] * B[n, k] mod 2^32 over int16 operands, both K-contiguous, on the 8-bit matrix
// instructions.  A value is taken apart into bytes, v = 256 h + l + 128 with h = v >> 8 and l = (v & 255) - 128,
// both in int8, so with v' = v - 128 = 256 h + l
//     sum a b = sum a' b' + 128 (sum a + sum b) - 16384 K,
//     sum a' b' = 65536 sum ha hb + 256 sum (ha lb + la hb) + sum la lb :
// four 16x16x64 byte products per 64 values of k and two row sums.  Every identity holds mod 2^32, so sums
// that leave int32 wrap as they do on the CPU.  The products with v_dot2_i32_i16 that this replaces had
// an eighth of the rate (509 x 512 x 2048 and back: 25.2 and 79.8 us).
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// 16 values of k of one row as two matrix operands (hi and lo bytes), and their sum
struct Planes {
  v4i h, l;
  int sum;
};

__device__ __forceinline__ void split_words(unsigned d0, unsigned d1, int& h, int& l) {   // four int16 in two words
  h = (int)__builtin_amdgcn_perm(d1, d0, 0x07050301u);
  l = (int)(__builtin_amdgcn_perm(d1, d0, 0x06040200u) ^ 0x80808080u);
}

// The 16 values of a block of 64 k that lane group lk (0 .. 3) supplies: k = 8 lk .. 8 lk + 7 and 32 + 8 lk ..
// 32 + 8 lk + 7 (the same for both operands, so any order does), which makes the four lanes of a row read
// 64 contiguous bytes.  Loaded first, taken apart later, so that loads are in flight in between.  Where K ends
// in half a block (K % 32 == 0) the second run of A is zeros and that of B a copy of other values: the identity
// above holds for any pair, also with a = 0.
template <typename T>
struct Raw;
template <>
struct Raw<int16_t> {
  v4u w[2];
  __device__ __forceinline__ void load(const int16_t* p, int second) {
    w[0] = *reinterpret_cast<const v4u*>(p);
    w[1] = *reinterpret_cast<const v4u*>(p + second);
  }
  __device__ __forceinline__ void clear_second() { w[1] = v4u{0, 0, 0, 0}; }
  __device__ __forceinline__ Planes planes() const {
    Planes r;
    r.sum = 0;
    const unsigned d[8] = {w[0].x, w[0].y, w[0].z, w[0].w, w[1].x, w[1].y, w[1].z, w[1].w};
    int h[4], l[4];
#pragma unroll
    for(int i = 0; i < 4; ++i) split_words(d[2 * i], d[2 * i + 1], h[i], l[i]);
#pragma unroll
    for(int i = 0; i < 8; ++i) r.sum = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, d[i]), v2s{1, 1}, r.sum, false);
    r.h = v4i{h[0], h[1], h[2], h[3]};
    r.l = v4i{l[0], l[1], l[2], l[3]};
    return r;
  }
};
// float32 activations, quantized on the way.  x * 1024 is exact, so one fused multiply-add with 1.5 * 2^23
// rounds to nearest-even and leaves the integer in the low bytes of the sum, once x is clamped to int16's
// range (med3: NaN to the lower end); products of 2^31 and more give -32768 (quantize16_one).
template <>
struct Raw<float> {
  v4f w[4];
  __device__ __forceinline__ void load(const float* p, int second) {
    w[0] = reinterpret_cast<const v4f*>(p)[0];
    w[1] = reinterpret_cast<const v4f*>(p)[1];
    w[2] = reinterpret_cast<const v4f*>(p + second)[0];
    w[3] = reinterpret_cast<const v4f*>(p + second)[1];
  }
  __device__ __forceinline__ void clear_second() { w[2] = w[3] = v4f{0.0f, 0.0f, 0.0f, 0.0f}; }
  __device__ __forceinline__ Planes planes() const {
    constexpr unsigned kMagicBits = 0x4B400000u;
    float x[16];
#pragma unroll
    for(int i = 0; i < 4; ++i) { x[4 * i] = w[i].x; x[4 * i + 1] = w[i].y; x[4 * i + 2] = w[i].z; x[4 * i + 3] = w[i].w; }
    float top = x[0];
#pragma unroll
    for(int i = 1; i < 16; ++i) top = fmaxf(top, x[i]);
    if(top >= 2097152.0f) {   // (rare: x * 1024 >= 2^31)
#pragma unroll
      for(int i = 0; i < 16; ++i) x[i] = x[i] >= 2097152.0f ? -32.0f : x[i];
    }
    unsigned b[16], sum = 0;
#pragma unroll
    for(int i = 0; i < 16; ++i) {
      const float c = __builtin_amdgcn_fmed3f(x[i], -32.0f, 32767.0f / 1024.0f);
      b[i] = __float_as_uint(fmaf(c, kQuantMult16, 12582912.0f));
      sum += b[i];
    }
    Planes r;
    r.sum = (int)(sum - 16u * kMagicBits);
    int h[4], l[4];
#pragma unroll
    for(int i = 0; i < 4; ++i) {
      const unsigned p = __builtin_amdgcn_perm(b[4 * i + 1], b[4 * i], 0x05010400u);       // h1 h0 l1 l0
      const unsigned q = __builtin_amdgcn_perm(b[4 * i + 3], b[4 * i + 2], 0x05010400u);   // h3 h2 l3 l2
      h[i] = (int)__builtin_amdgcn_perm(q, p, 0x07060302u);
      l[i] = (int)(__builtin_amdgcn_perm(q, p, 0x05040100u) ^ 0x80808080u);
    }
    r.h = v4i{h[0], h[1], h[2], h[3]};
    r.l = v4i{l[0], l[1], l[2], l[3]};
    return r;
  }
};
// the three accumulators of one 16 x 16 tile (rows: columns of the output, see mfma_i8_16x16x64)
struct Acc16 {
  v4i hh, mid, ll;
  __device__ __forceinline__ void clear() { hh = mid = ll = v4i{0, 0, 0, 0}; }
  __device__ __forceinline__ void add(v4i bh, v4i bl, v4i ah, v4i al) {
    hh = mfma_i8_16x16x64(bh, ah, hh);
    mid = mfma_i8_16x16x64(bh, al, mid);
    ll = mfma_i8_16x16x64(bl, al, ll);
    mid = mfma_i8_16x16x64(bl, ah, mid);
  }
  __device__ __forceinline__ v4i sum() const {   // mod 2^32
    v4i r;
#pragma unroll
    for(int e = 0; e < 4; ++e) r[e] = (int)(((unsigned)hh[e] << 16) + ((unsigned)mid[e] << 8) + (unsigned)ll[e]);
    return r;
  }
};

struct Gemm16Args {
  const void* A;
  const int16_t* Bq;
  const float* bias;
  void* out;
  int M, K, N;
  float scale;
  int relu;
};

// four neighbouring columns n .. n + 3 of output row m: y = float(acc) * unquant (+ bias); relu: y > 0 ? y : 0;
// multiply and add round separately
template <bool DUMP>
__device__ __forceinline__ void store16(const Gemm16Args& g, v4i acc, int m, int n, float unquant) {
  if(m >= g.M || n >= g.N) return;   // (N % 8 == 0: four columns are inside or outside together)
  const size_t off = (size_t)m * g.N + n;
  if(DUMP) {
    *reinterpret_cast<v4i*>(reinterpret_cast<int32_t*>(g.out) + off) = acc;
    return;
  }
  v4f y;
#pragma unroll
  for(int e = 0; e < 4; ++e) {
    float v = (float)acc[e] * unquant;
    if(g.bias) v = v + g.bias[n + e];
    if(g.relu) v = v > 0.0f ? v : 0.0f;
    y[e] = v;
  }
  *reinterpret_cast<v4f*>(reinterpret_cast<float*>(g.out) + off) = y;
}

template <typename AT>
__device__ __forceinline__ float unquant16(const Gemm16Args& g) {
  float aqm = kQuantMult16;
  if constexpr(sizeof(AT) == 2) aqm = *reinterpret_cast<const float*>(reinterpret_cast<const int16_t*>(g.A) + (size_t)g.M * g.K);
  return unquant_mult(aqm, *reinterpret_cast<const float*>(g.Bq + (size_t)g.K * g.N), g.scale);
}

// Few tiles: the eight waves of a workgroup split K between them, operands go from memory straight into
// registers (a lane takes 16 consecutive k of its row, four lanes a 128-byte line) and the partial sums meet
// in LDS.  A workgroup makes (16 MT) x (16 NT) outputs.  Bound by what a CU can fetch: the activations of
// 16 MT rows are read again for every 16 NT columns.
constexpr int kStream16Waves = 8;
template <typename AT, int MT, int NT, bool DUMP>
__global__ __launch_bounds__(64 * kStream16Waves) void gemm16_stream_kernel(Gemm16Args g) {
  constexpr int KW = kStream16Waves, TILES = MT * NT;
  __shared__ __attribute__((aligned(16))) int part[KW][TILES][64][4];
  const int lane = threadIdx.x % 64, wave = threadIdx.x / 64, lr = lane % 16, lk = lane / 16;
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const AT* arow[MT];
  const int16_t* brow[NT];
#pragma unroll
  for(int i = 0; i < MT; ++i) arow[i] = reinterpret_cast<const AT*>(g.A) + (size_t)min(m0 + 16 * i + lr, g.M - 1) * g.K;
#pragma unroll
  for(int j = 0; j < NT; ++j) brow[j] = g.Bq + (size_t)min(n0 + 16 * j + lr, g.N - 1) * g.K;
  Acc16 acc[MT][NT];
  int asum[MT], bsum[NT], taken = 0;
#pragma unroll
  for(int i = 0; i < MT; ++i) {
    asum[i] = 0;
#pragma unroll
    for(int j = 0; j < NT; ++j) acc[i][j].clear();
  }
#pragma unroll
  for(int j = 0; j < NT; ++j) bsum[j] = 0;
  const int S = (g.K + 63) / 64;
  const bool half = g.K % 64 != 0;
  Raw<AT> ra[MT];
  Raw<int16_t> rb[NT];
  auto load = [&](int s) __attribute__((always_inline)) {
    const int k = s * 64 + lk * 8, second = half && s == S - 1 ? 0 : 32;
#pragma unroll
    for(int j = 0; j < NT; ++j) rb[j].load(brow[j] + k, second);
#pragma unroll
    for(int i = 0; i < MT; ++i) ra[i].load(arow[i] + k, second);
  };
  // one step: its operands are taken apart, the next step's loads take their place, then the products
  auto step = [&](int s, bool more) __attribute__((always_inline)) {
    Planes a[MT], b[NT];
    if(!more && half && s == S - 1) {
#pragma unroll
      for(int i = 0; i < MT; ++i) ra[i].clear_second();
    }
#pragma unroll
    for(int j = 0; j < NT; ++j) b[j] = rb[j].planes();
#pragma unroll
    for(int i = 0; i < MT; ++i) a[i] = ra[i].planes();
    if(more) load(s + KW);
#pragma unroll
    for(int i = 0; i < MT; ++i) {
      asum[i] += a[i].sum;
#pragma unroll
      for(int j = 0; j < NT; ++j) acc[i][j].add(b[j].h, b[j].l, a[i].h, a[i].l);
    }
#pragma unroll
    for(int j = 0; j < NT; ++j) bsum[j] += b[j].sum;
    taken += 64;
  };
  int s = wave;
  if(s < S) {
    load(s);
    // (the load of the next step stands behind no branch: the compiler would wait for it at once)
    for(; s + KW < S; s += KW) step(s, true);
    step(s, false);
  }
  // row sums over the four lane groups; lane (lr, lk) holds outputs row lr, columns 4 lk .. 4 lk + 3
#pragma unroll
  for(int i = 0; i < MT; ++i) {
    asum[i] += __shfl_xor(asum[i], 16);
    asum[i] += __shfl_xor(asum[i], 32);
  }
#pragma unroll
  for(int j = 0; j < NT; ++j) {
    bsum[j] += __shfl_xor(bsum[j], 16);
    bsum[j] += __shfl_xor(bsum[j], 32);
    int bs[4];
#pragma unroll
    for(int e = 0; e < 4; ++e) bs[e] = __shfl(bsum[j], 4 * lk + e);
#pragma unroll
    for(int i = 0; i < MT; ++i) {
      v4i t = acc[i][j].sum();
#pragma unroll
      for(int e = 0; e < 4; ++e) t[e] = (int)((unsigned)t[e] + 128u * (unsigned)(asum[i] + bs[e]) - 16384u * (unsigned)taken);
      *reinterpret_cast<v4i*>(part[wave][i * NT + j][lane]) = t;
    }
  }
  float unquant = 0.0f;
  if(!DUMP) unquant = unquant16<AT>(g);
  __syncthreads();
  for(int t = threadIdx.x; t < TILES * 64; t += 64 * KW) {
    const int tile = t / 64, l = t % 64;
    v4i sum = *reinterpret_cast<const v4i*>(part[0][tile][l]);
#pragma unroll
    for(int w = 1; w < KW; ++w) {
      const v4i p = *reinterpret_cast<const v4i*>(part[w][tile][l]);
#pragma unroll
      for(int e = 0; e < 4; ++e) sum[e] = (int)((unsigned)sum[e] + (unsigned)p[e]);
    }
    store16<DUMP>(g, sum, m0 + 16 * (tile / NT) + l % 16, n0 + 16 * (tile % NT) + 4 * (l / 16), unquant);
  }
}

// Many tiles: a workgroup of eight waves makes a BM x BN tile, both operands of a block of 64 k go through
// registers (taken apart there, once per workgroup) into LDS, two blocks in turn: while one is multiplied the
// next is on its way.  LDS rows are 64 bytes,
// their four pieces permuted by the row number so that reads of neighbouring rows fall on different banks.
constexpr int kPitch16 = 64, kTile16Depth = 2;
__device__ __forceinline__ int piece16(int row, int c) { return (c ^ ((row >> 1) & 3)) * 16; }
template <int BM, int BN>
constexpr int tile16_lds() { return 2 * 2 * (BM + BN) * kPitch16; }
template <typename AT, int BM, int BN, int WM, int WN, bool DUMP>
__global__ __launch_bounds__(64 * WM * WN) void gemm16_tile_kernel(Gemm16Args g, int tiles_n) {
  constexpr int T = 64 * WM * WN, FM = BM / WM / 16, FN = BN / WN / 16;
  constexpr int UA = BM * 4 / T, UB = BN * 4 / T;   // pieces of 16 k a thread stages per block
  static_assert(UA * T == BM * 4 && UB * T == BN * 4 && (T / 4) % 8 == 0, "whole pieces per thread");
  extern __shared__ __attribute__((aligned(16))) int8_t lds16[];
  int* const sums = reinterpret_cast<int*>(lds16);   // [BM + BN], at the end
  const int tid = threadIdx.x, lane = tid % 64, wave = tid / 64, lr = lane % 16, lk = lane / 16;
  const int wm = wave / WN, wn = wave % WN;
  const int m0 = (int)(blockIdx.x / tiles_n) * BM, n0 = (int)(blockIdx.x % tiles_n) * BN;
  const int srow = tid / 4, sk = (tid % 4) * 8, spiece = piece16(srow, tid % 4);   // staging: four threads a row, T / 4 rows at a time
  const AT* asrc[UA];
  const int16_t* bsrc[UB];
#pragma unroll
  for(int u = 0; u < UA; ++u) asrc[u] = reinterpret_cast<const AT*>(g.A) + (size_t)min(m0 + srow + u * (T / 4), g.M - 1) * g.K;
#pragma unroll
  for(int u = 0; u < UB; ++u) bsrc[u] = g.Bq + (size_t)min(n0 + srow + u * (T / 4), g.N - 1) * g.K;
  constexpr int D = kTile16Depth;   // blocks of K on their way
  Raw<AT> ra[D][UA];
  Raw<int16_t> rb[D][UB];
  int asum[UA], bsum[UB];
#pragma unroll
  for(int u = 0; u < UA; ++u) asum[u] = 0;
#pragma unroll
  for(int u = 0; u < UB; ++u) bsum[u] = 0;
  Acc16 acc[FM][FN];
#pragma unroll
  for(int i = 0; i < FM; ++i)
#pragma unroll
    for(int j = 0; j < FN; ++j) acc[i][j].clear();
  const int blocks = (g.K + 63) / 64;
  const bool half = g.K % 64 != 0;
  auto load = [&](int kb, Raw<AT> (&ra)[UA], Raw<int16_t> (&rb)[UB]) __attribute__((always_inline)) {
    kb = min(kb, blocks - 1);
    const int k = kb * 64 + sk, second = half && kb == blocks - 1 ? 0 : 32;
#pragma unroll
    for(int u = 0; u < UA; ++u) ra[u].load(asrc[u] + k, second);
#pragma unroll
    for(int u = 0; u < UB; ++u) rb[u].load(bsrc[u] + k, second);
  };
  // planes of stage t: A hi, A lo, B hi, B lo
  auto plane = [&](int t, int which, int row) {
    return lds16 + (size_t)t * (2 * (BM + BN) * kPitch16) + (which < 2 ? which * BM : 2 * BM + (which - 2) * BN) * kPitch16 + row * kPitch16;
  };
  auto stage = [&](int t, int kb, Raw<AT> (&ra)[UA], Raw<int16_t> (&rb)[UB]) __attribute__((always_inline)) {
    if(half && kb == blocks - 1) {   // (the same for the whole workgroup)
#pragma unroll
      for(int u = 0; u < UA; ++u) ra[u].clear_second();
    }
#pragma unroll
    for(int u = 0; u < UA; ++u) {
      const Planes p = ra[u].planes();
      asum[u] += p.sum;
      *reinterpret_cast<v4i*>(plane(t, 0, srow + u * (T / 4)) + spiece) = p.h;
      *reinterpret_cast<v4i*>(plane(t, 1, srow + u * (T / 4)) + spiece) = p.l;
    }
#pragma unroll
    for(int u = 0; u < UB; ++u) {
      const Planes p = rb[u].planes();
      bsum[u] += p.sum;
      *reinterpret_cast<v4i*>(plane(t, 2, srow + u * (T / 4)) + spiece) = p.h;
      *reinterpret_cast<v4i*>(plane(t, 3, srow + u * (T / 4)) + spiece) = p.l;
    }
  };
  auto multiply = [&](int t) __attribute__((always_inline)) {
    v4i bh[FN], bl[FN];
#pragma unroll
    for(int j = 0; j < FN; ++j) {
      const int row = (wn * FN + j) * 16 + lr;
      bh[j] = *reinterpret_cast<const v4i*>(plane(t, 2, row) + piece16(row, lk));
      bl[j] = *reinterpret_cast<const v4i*>(plane(t, 3, row) + piece16(row, lk));
    }
#pragma unroll
    for(int i = 0; i < FM; ++i) {
      const int row = (wm * FM + i) * 16 + lr;
      const v4i ah = *reinterpret_cast<const v4i*>(plane(t, 0, row) + piece16(row, lk));
      const v4i al = *reinterpret_cast<const v4i*>(plane(t, 1, row) + piece16(row, lk));
#pragma unroll
      for(int j = 0; j < FN; ++j) acc[i][j].add(bh[j], bl[j], ah, al);
    }
  };
#pragma unroll
  for(int d = 0; d < D; ++d) load(d, ra[d], rb[d]);
  stage(0, 0, ra[0], rb[0]);
  load(D, ra[0], rb[0]);
  __syncthreads();
  int kb = 0;
  // (the loads inside the loop stand behind no branch: the compiler would wait for them at once)
  for(; kb + 2 * D < blocks; kb += D) {
#pragma unroll
    for(int d = 0; d < D; ++d) {
      const int t = (kb + d) & 1, next = (d + 1) % D;
      multiply(t);
      stage(t ^ 1, kb + d + 1, ra[next], rb[next]);   // (the other stage was read before the last barrier)
      load(kb + d + 1 + D, ra[next], rb[next]);
      __syncthreads();
    }
  }
#pragma unroll
  for(int d = 0; d < 2 * D; ++d) {
    if(kb + d < blocks) {   // (the same for the whole workgroup)
      const int t = (kb + d) & 1, next = (d + 1) % D;
      multiply(t);
      if(kb + d + 1 < blocks) stage(t ^ 1, kb + d + 1, ra[next], rb[next]);
      if(d + 1 < D && kb + d + 1 + D < blocks) load(kb + d + 1 + D, ra[next], rb[next]);
      __syncthreads();
    }
  }
  // row sums: the four threads of a row sit side by side
#pragma unroll
  for(int u = 0; u < UA; ++u) {
    asum[u] += __shfl_xor(asum[u], 1);
    asum[u] += __shfl_xor(asum[u], 2);
    if(tid % 4 == 0) sums[srow + u * (T / 4)] = asum[u];
  }
#pragma unroll
  for(int u = 0; u < UB; ++u) {
    bsum[u] += __shfl_xor(bsum[u], 1);
    bsum[u] += __shfl_xor(bsum[u], 2);
    if(tid % 4 == 0) sums[BM + srow + u * (T / 4)] = bsum[u];
  }
  float unquant = 0.0f;
  if(!DUMP) unquant = unquant16<AT>(g);
  __syncthreads();
#pragma unroll
  for(int i = 0; i < FM; ++i) {
    const int r = (wm * FM + i) * 16 + lr;
    const int as = sums[r];
#pragma unroll
    for(int j = 0; j < FN; ++j) {
      const int c = (wn * FN + j) * 16 + 4 * lk;
      v4i v = acc[i][j].sum();
#pragma unroll
      for(int e = 0; e < 4; ++e) v[e] = (int)((unsigned)v[e] + 128u * (unsigned)(as + sums[BM + c + e]) - 16384u * 64u * (unsigned)blocks);
      store16<DUMP>(g, v, m0 + r, n0 + c, unquant);
    }
  }
}

int check16(const void* Aq, const void* Bq, const void* out, const float* bias, int64_t M, int64_t K, int64_t N) {
  if(M < 0 || K <= 0 || N < 0 || (K % 32) != 0 || (N % 8) != 0) return MARIAN_HIP_ERR_SHAPE;
  if(M == 0 || N == 0) return MARIAN_HIP_OK;
  if(!Aq || !Bq || !out) return MARIAN_HIP_ERR_NULL;
  if(M * K > kMaxElems16 || K * N > kMaxElems16 || M * N > kMaxElems16) return MARIAN_HIP_ERR_RANGE;
  if(!aligned(Aq, 16) || !aligned(Bq, 16) || !aligned(out, 16) || (bias && !aligned(bias, 4))) return MARIAN_HIP_ERR_ALIGN;
  return MARIAN_HIP_OK;
}

template <typename AT, int MT, int NT, bool DUMP>
int launch_stream16(const Gemm16Args& g, hipStream_t st) {
  const dim3 grid((unsigned)((g.N + 16 * NT - 1) / (16 * NT)), (unsigned)((g.M + 16 * MT - 1) / (16 * MT)));
  hipLaunchKernelGGL((gemm16_stream_kernel<AT, MT, NT, DUMP>), grid, dim3(64 * kStream16Waves), 0, st, g);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

template <typename AT, int BM, int BN, int WM, int WN, bool DUMP>
int launch_tile16(const Gemm16Args& g, hipStream_t st) {
  const int tiles_n = (g.N + BN - 1) / BN, tiles_m = (g.M + BM - 1) / BM;
  constexpr int lds = tile16_lds<BM, BN>();
  auto kernel = gemm16_tile_kernel<AT, BM, BN, WM, WN, DUMP>;
  static std::atomic<uint64_t> lds_done{0};
  const int lds_status = allow_lds(kernel, lds, lds_done);
  if(lds_status != MARIAN_HIP_OK) return lds_status;
  hipLaunchKernelGGL(kernel, dim3((unsigned)tiles_n * (unsigned)tiles_m), dim3(64 * WM * WN), lds, st, g, tiles_n);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

// Which form a call takes: the one whose busiest CU takes in the fewest bytes per step of k - its workgroups per CU
// (at least one) times the bytes a workgroup loads, converts and multiplies for each k; the 128 x 128 tiles count half
// again (one workgroup to a CU: products, conversion and LDS traffic overlap less).  Measured at 99 sizes (K, N = 256 ..
// 4096, M = 1 .. 4096, launches in a graph), the form taken was never more than 6 % behind the best with int16
// activations, 10 % with float32 ones (profiles/int16_forms.txt: every form, both kinds).  us, int16 activations:
//   1 x 512 x 512 3.0 (stream 16 x 16), 64 x 512 x 2048 4.2 (16 x 32), 509 x 2048 x 512 10.4 (32 x 32), 509 x 512 x 2048
//   8.6 (64 x 64), 4096 x 4096 x 4096 263 (128 x 128: 523 TOPS of 16-bit products).
// What a call takes is another matter: each form has a start of its own and its own price of a byte (least squares over
// the same measurements where the form is near the best: -29 .. +19 %); a CU holds one 128 x 128 tile at a time.
struct Form16 {
  enum Name { kStream16, kStream16x32, kStream32x32, kTile64, kTile128 };
  Name form;
  double cost;   // bytes per k through the busiest CU
  double ns;     // of the call
};
inline Form16 plan16(int M, int K, int N, int a_bytes) {
  struct Shape { Form16::Name form; int rows, cols; double factor, start_ns, a_byte_ns, b_byte_ns; };
  constexpr Shape shapes[] = {{Form16::kStream16, 16, 16, 1.0, 2600.0, 0.025, 0.033}, {Form16::kStream16x32, 16, 32, 1.0, 2900.0, 0.028, 0.030},
                              {Form16::kStream32x32, 32, 32, 1.0, 3400.0, 0.033, 0.022}, {Form16::kTile64, 64, 64, 1.0, 5400.0, 0.019, 0.032},
                              {Form16::kTile128, 128, 128, 1.5, 10000.0, 0.0155, 0.035}};
  Form16 best{Form16::kTile128, 1e30, 0.0};
  for(const Shape& s : shapes) {
    if(s.form < Form16::kTile64 && (M + s.rows - 1) / s.rows > 65535) continue;   // (row tiles are the grid's second dimension)
    const double workgroups = (double)((M + s.rows - 1) / s.rows) * ((N + s.cols - 1) / s.cols) / 256.0;
    const double per_cu = workgroups > 1.0 ? workgroups : 1.0;
    const double cost = per_cu * s.factor * (s.rows * a_bytes + s.cols * 2);
    if(cost >= best.cost) continue;
    const int rows = M < s.rows ? M : s.rows;   // (rows past the end repeat the last one, which is in the cache)
    const double tile = K * (s.a_byte_ns * rows * a_bytes + s.b_byte_ns * s.cols * 2);
    best = Form16{s.form, cost, s.form == Form16::kTile128 ? std::ceil(per_cu) * (s.start_ns + tile) : s.start_ns + per_cu * tile};
  }
  return best;
}

// Whether float32 activations are quantized by a launch of their own first: where the multiplication then saves more
// than the launch costs: 2 us, and 2.5 ns per thousand values up to 1.2 million and half of one beyond (the pass over
// them, and the multiplication's wait for values that were just written).  At the 99 sizes the choice is at most 3 %
// behind the better one but for 256 rows of 512 and of 704 values, which two 32 x 32 workgroups a CU quantize on the way (10
// and 18 %); with one price for all forms (30 ps a byte) it was 4 .. 18 % behind at nine.
inline bool quantize_first16(int64_t M, int64_t K, int64_t N) {
  const double saved = plan16((int)M, (int)K, (int)N, 4).ns - plan16((int)M, (int)K, (int)N, 2).ns;
  const double values = (double)M * (double)K, near = values < 1.2e6 ? values : 1.2e6;
  return saved > 2000.0 + 0.002 * near + 0.00055 * values;
}

template <typename AT, bool DUMP>
int run16(const AT* A, const int16_t* Bq, const float* bias, void* out, int64_t M, int64_t K, int64_t N,
          float scale, int relu, void* stream) {
  int status = check16(A, Bq, out, bias, M, K, N);
  if(status != MARIAN_HIP_OK) return status;
  if(M == 0 || N == 0) return MARIAN_HIP_OK;
  Gemm16Args g{A, Bq, bias, out, (int)M, (int)K, (int)N, scale, relu ? 1 : 0};
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  switch(plan16((int)M, (int)K, (int)N, (int)sizeof(AT)).form) {
    case Form16::kStream16: return launch_stream16<AT, 1, 1, DUMP>(g, st);
    case Form16::kStream16x32: return launch_stream16<AT, 1, 2, DUMP>(g, st);
    case Form16::kStream32x32: return launch_stream16<AT, 2, 2, DUMP>(g, st);
    case Form16::kTile64: return launch_tile16<AT, 64, 64, 2, 2, DUMP>(g, st);
    default: return launch_tile16<AT, 128, 128, 2, 4, DUMP>(g, st);
  }
}

}  // namespace

extern "C" {

int marian_hip_int16_prepare_a(const float* A, int16_t* Aq, int64_t M, int64_t K, void* stream) {
  if(M < 0 || K <= 0 || (K % 32) != 0) return MARIAN_HIP_ERR_SHAPE;
  if(M == 0) return MARIAN_HIP_OK;
  if(!A || !Aq) return MARIAN_HIP_ERR_NULL;
  if(M * K > kMaxElems16) return MARIAN_HIP_ERR_RANGE;
  if(!aligned(A, 16) || !aligned(Aq, 16)) return MARIAN_HIP_ERR_ALIGN;
  const size_t n8 = (size_t)M * (size_t)K / 8;
  size_t blocks = (n8 + 255) / 256;
  if(blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(quantize16_a_kernel, dim3((unsigned)blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), A, n8, Aq, (int)blocks);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_int16_prepare_b(const float* W, int16_t* Bq, int64_t K, int64_t N, void* stream) {
  if(K <= 0 || N <= 0 || (K % 32) != 0 || (N % 8) != 0) return MARIAN_HIP_ERR_SHAPE;
  if(!W || !Bq) return MARIAN_HIP_ERR_NULL;
  if(K * N > kMaxElems16) return MARIAN_HIP_ERR_RANGE;
  if(!aligned(W, 4) || !aligned(Bq, 16)) return MARIAN_HIP_ERR_ALIGN;
  const dim3 grid((unsigned)((N + 63) / 64), (unsigned)(K / 32));
  if(grid.y > 65535) return MARIAN_HIP_ERR_RANGE;
  hipLaunchKernelGGL(quantize16_b_transpose_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), W, (int)K, (int)N, Bq);
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

int marian_hip_int16_prepare_b_quantized_transposed(const int16_t* in, int16_t* out, int64_t K, int64_t N, void* stream) {
  if(!in || !out) return MARIAN_HIP_ERR_NULL;
  if(K <= 0 || N <= 0 || (K % 32) != 0 || (N % 8) != 0) return MARIAN_HIP_ERR_SHAPE;
  if(K * N > 2147483647LL) return MARIAN_HIP_ERR_RANGE;
  if(in == out) return MARIAN_HIP_OK;   // the two orders are the same for 16-bit tensors: nothing to do in place
  // a copy between buffers that overlap only in part has no defined result
  const uintptr_t a0 = reinterpret_cast<uintptr_t>(in), b0 = reinterpret_cast<uintptr_t>(out);
  const uintptr_t bytes = 2 * (uintptr_t)K * (uintptr_t)N + sizeof(float);
  if(a0 < b0 + bytes && b0 < a0 + bytes) return MARIAN_HIP_ERR_ALIAS;
  MH_HIP(hipMemcpyAsync(out, in, 2 * (size_t)K * (size_t)N + sizeof(float), hipMemcpyDeviceToDevice,
                        reinterpret_cast<hipStream_t>(stream)));
  return MARIAN_HIP_OK;
}

int marian_hip_int16_affine(const int16_t* Aq, const int16_t* Bq, const float* bias, float* out, int64_t M, int64_t K,
                            int64_t N, float scale, int relu, void* stream) {
  return run16<int16_t, false>(Aq, Bq, bias, out, M, K, N, scale, relu, stream);
}

int marian_hip_int16_multiply_i32(const int16_t* Aq, const int16_t* Bq, int32_t* acc, int64_t M, int64_t K, int64_t N,
                                  void* stream) {
  return run16<int16_t, true>(Aq, Bq, nullptr, acc, M, K, N, 1.0f, 0, stream);
}

size_t marian_hip_int16_scratch_bytes(int64_t M, int64_t K, int64_t N) {
  if(M <= 0 || K <= 0 || N <= 0 || M * K > kMaxElems16) return 0;
  return quantize_first16(M, K, N) ? 2 * (size_t)M * (size_t)K + sizeof(float) : 0;
}

int marian_hip_int16_affine_f32(const float* A, int16_t* Aq, const int16_t* Bq, const float* bias, float* out, int64_t M, int64_t K,
                                int64_t N, float scale, int relu, void* stream) {
  if(Aq && M > 0 && N > 0 && marian_hip_int16_scratch_bytes(M, K, N)) {
    const int status = check16(A, Bq, out, bias, M, K, N);   // (nothing is launched for a call that is refused)
    if(status != MARIAN_HIP_OK) return status;
    const int quantized = marian_hip_int16_prepare_a(A, Aq, M, K, stream);
    if(quantized != MARIAN_HIP_OK) return quantized;
    return marian_hip_int16_affine(Aq, Bq, bias, out, M, K, N, scale, relu, stream);
  }
  return run16<float, false>(A, Bq, bias, out, M, K, N, scale, relu, stream);
}

}  // extern "C"
