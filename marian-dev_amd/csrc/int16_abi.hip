// The 16-bit intgemm path (Type::intgemm16): quantizers, GEMMs on the 8-bit matrix instructions and its C ABI.
// Declarations and the reference call sites each entry point replaces: include/marian_hip_int16.h
#include "../../include/marian_hip_int16.h"

#include <hip/hip_runtime.h>

#include <atomic>
#include <cmath>
#include <type_traits>

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

__device__ __forceinline__ Planes planes_of_words(const unsigned (&d)[8]) {   // 16 int16
  Planes r;
  r.sum = 0;
  int h[4], l[4];
#pragma unroll
  for(int i = 0; i < 4; ++i) split_words(d[2 * i], d[2 * i + 1], h[i], l[i]);
#pragma unroll
  for(int i = 0; i < 8; ++i) r.sum = __builtin_amdgcn_sdot2(__builtin_bit_cast(v2s, d[i]), v2s{1, 1}, r.sum, false);
  r.h = v4i{h[0], h[1], h[2], h[3]};
  r.l = v4i{l[0], l[1], l[2], l[3]};
  return r;
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
    const unsigned d[8] = {w[0].x, w[0].y, w[0].z, w[0].w, w[1].x, w[1].y, w[1].z, w[1].w};
    return planes_of_words(d);
  }
};
// float32 activations, quantized on the way.  A sum with 12288 = 1.5 * 2^13 has steps of 1/1024, so the addition rounds x * 1024
// to nearest-even and leaves the int16 in the low half of the sum, which it writes to where it belongs, as long as it
// is in range.  A maximum that lets NaN through tells whether all 16 values are; the few that are not are replaced by the
// value they saturate to (quantize16_one: NaN and products of 2^31 and more give -32768).  2.8 vector instructions a value, where a
// clamp of every value and sums of the unpacked integers took 5.
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
    float x[16];
#pragma unroll
    for(int i = 0; i < 4; ++i) { x[4 * i] = w[i].x; x[4 * i + 1] = w[i].y; x[4 * i + 2] = w[i].z; x[4 * i + 3] = w[i].w; }
    float top = 0.0f;
#pragma unroll
    for(int i = 0; i < 16; i += 2)
      top = __builtin_elementwise_maximum(__builtin_elementwise_maximum(top, __builtin_fabsf(x[i])), __builtin_fabsf(x[i + 1]));
    if(!(top <= 31.99f)) {   // (rare)
#pragma unroll
      for(int i = 0; i < 16; ++i)
        x[i] = x[i] >= 2097152.0f ? -32.0f : __builtin_amdgcn_fmed3f(x[i], -32.0f, 32767.0f / 1024.0f);
    }
    unsigned d[8];
#pragma unroll
    for(int i = 0; i < 8; ++i) {
      const float magic = 12288.0f;
      asm("v_add_f32_sdwa %0, %1, %2 dst_sel:WORD_0 dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:DWORD" : "=v"(d[i]) : "v"(x[2 * i]), "v"(magic));
      asm("v_add_f32_sdwa %0, %1, %2 dst_sel:WORD_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD" : "+v"(d[i]) : "v"(x[2 * i + 1]), "v"(magic));
    }
    return planes_of_words(d);
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

// Kernel arguments behind those that come in registers (see the Makefile).  Six of 56 bytes in all: nine of 104, with these and the tile counts
// beside them, made a 6 x 256 x 512 block of two calls take 8.3 us from Python, not 7.8.
struct Gemm16Rest {
  void* out;
  float scale;
  int relu;
};
__device__ __forceinline__ Gemm16Args gemm16_args(const void* A, const int16_t* Bq, const float* bias, unsigned long long M_K, int N,
                                                  const Gemm16Rest& rest) {
  return Gemm16Args{A, Bq, bias, rest.out, int_pair(M_K).first, int_pair(M_K).second, N, rest.scale, rest.relu};
}

// four neighbouring outputs: y = float(acc) * unquant (+ bias); relu: y > 0 ? y : 0; multiply and add round separately
template <bool DUMP>
__device__ __forceinline__ void store16(const Gemm16Args& g, v4i acc, size_t off, float unquant, const float (&bias)[4]) {
  if(DUMP) {
    *reinterpret_cast<v4i*>(reinterpret_cast<int32_t*>(g.out) + off) = acc;
    return;
  }
  v4f y;
#pragma unroll
  for(int e = 0; e < 4; ++e) {
    float v = (float)acc[e] * unquant;
    if(g.bias) v = v + bias[e];
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

// Sum over the four lanes of a quad, left in all of them (two DPP lane swaps).
__device__ __forceinline__ int quad_sum(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false);   // quad_perm [1,0,3,2]
  v += __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false);   // quad_perm [2,3,0,1]
  return v;
}

// Few tiles: the eight waves of a workgroup split K between them and the partial sums meet in LDS.  A workgroup
// makes (16 MT) x (16 NT) outputs.  Operands do not need LDS to be shared, but a matrix instruction wants neighbouring
// lanes to hold neighbouring rows, and a load of which the four lanes of a quad ask for four lines takes the address unit four
// times as long: that was the bound (16 bytes a clock and CU).  So a quad loads one row's line, takes its values apart,
// and the bytes change lanes through the wave's own LDS; two steps of K are on their way.  509 x 2048 x 512 from float32: 14.6 -> 8.8 us,
// of it 0.4 the order of the tiles over the XCDs; what is left is 384 KB per CU at 64 bytes a clock (2.9 us), beside conversions
// of about as long, and 3.5 us of launch, first loads and write-out.
constexpr int kStream16Waves = 8;
template <int MT, int NT>
constexpr int stream16_lds() { return kStream16Waves * 1024 * (2 * (MT + NT) > MT * NT ? 2 * (MT + NT) : MT * NT); }
template <typename AT, int MT, int NT, int D, bool DUMP>
__global__ __launch_bounds__(64 * kStream16Waves) void gemm16_stream_kernel(const void* A, const int16_t* Bq, const float* bias_in,
                                                                              unsigned long long M_K, int N, Gemm16Rest rest) {
  const Gemm16Args g = gemm16_args(A, Bq, bias_in, M_K, N, rest);
  const int tiles_n = (int)((unsigned)(g.N + 16 * NT - 1) / (16 * NT)), tiles_m = (int)((unsigned)(g.M + 16 * MT - 1) / (16 * MT));
  constexpr int KW = kStream16Waves, TILES = MT * NT, kWaveBytes = stream16_lds<MT, NT>() / KW;
  extern __shared__ __attribute__((aligned(16))) int8_t lds16[];
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int lr = lane % 16, lk = lane / 16;   // the operand row and run of k that a matrix instruction takes from this lane
  const int qr = lane / 4, qk = lane % 4;     // and those that it loads and takes apart
  int tn, tm;
  xcd_order16(tiles_n, tiles_m, blockIdx.x, tn, tm);
  const int n0 = tn * 16 * NT, m0 = tm * 16 * MT;
  // what the write-out needs, requested first: the biases of this thread's four columns (without a bias the weights stand in)
  static_assert(TILES * 64 <= 64 * KW, "a thread finishes four outputs");
  const int wr_n = n0 + 16 * (threadIdx.x / 64 % NT) + 4 * lk, wr_m = m0 + 16 * (threadIdx.x / 64 / NT) + lr;
  float bias[4];
  const float* bias_src = g.bias ? g.bias : reinterpret_cast<const float*>(g.Bq);
#pragma unroll
  for(int e = 0; e < 4; ++e) bias[e] = bias_src[min(wr_n, g.N - 4) + e];
  float unquant = 0.0f;
  if(!DUMP) unquant = unquant16<AT>(g);
  int8_t* const mine = lds16 + wave * kWaveBytes;
  const AT* arow[MT];
  const int16_t* brow[NT];
#pragma unroll
  for(int i = 0; i < MT; ++i) arow[i] = reinterpret_cast<const AT*>(g.A) + row16_offset(m0 + 16 * i + qr, g.M, g.K) + piece16_offset(qk);
#pragma unroll
  for(int j = 0; j < NT; ++j) brow[j] = g.Bq + row16_offset(n0 + 16 * j + qr, g.N, g.K) + piece16_offset(qk);
  Acc16 acc[MT][NT];
  int asum[MT], bsum[NT];
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
  const int steps = wave < S ? (S - wave + KW - 1) / KW : 0;   // of this wave: wave, wave + KW, ..
  Raw<AT> ra[D][MT];
  Raw<int16_t> rb[D][NT];
  auto load = [&](int t, Raw<AT> (&ra)[MT], Raw<int16_t> (&rb)[NT]) __attribute__((always_inline)) {
    const int s = wave + t * KW, k = s * kStep16, second = half && s == S - 1 ? 0 : 32;
#pragma unroll
    for(int i = 0; i < MT; ++i) ra[i].load(arow[i] + k, second);
#pragma unroll
    for(int j = 0; j < NT; ++j) rb[j].load(brow[j] + k, second);
  };
  // operands of a step change lanes through the wave's own LDS (a wave's LDS operations keep their order)
  const int put = (qk * 16 + (qr ^ (2 * qk))) * 16, get = (lk * 16 + (lr ^ (2 * lk))) * 16;
  auto step = [&](int t, int next, Raw<AT> (&ra)[MT], Raw<int16_t> (&rb)[NT]) __attribute__((always_inline)) {
    if(half && wave + t * KW == S - 1) {
#pragma unroll
      for(int i = 0; i < MT; ++i) ra[i].clear_second();
    }
#pragma unroll
    for(int i = 0; i < MT; ++i) {
      const Planes p = ra[i].planes();
      asum[i] += p.sum;
      *reinterpret_cast<v4i*>(mine + (2 * i) * 1024 + put) = p.h;
      *reinterpret_cast<v4i*>(mine + (2 * i + 1) * 1024 + put) = p.l;
    }
#pragma unroll
    for(int j = 0; j < NT; ++j) {
      const Planes p = rb[j].planes();
      bsum[j] += p.sum;
      *reinterpret_cast<v4i*>(mine + (2 * MT + 2 * j) * 1024 + put) = p.h;
      *reinterpret_cast<v4i*>(mine + (2 * MT + 2 * j + 1) * 1024 + put) = p.l;
    }
    if(next >= 0) load(next, ra, rb);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    v4i bh[NT], bl[NT];
#pragma unroll
    for(int j = 0; j < NT; ++j) {
      bh[j] = *reinterpret_cast<const v4i*>(mine + (2 * MT + 2 * j) * 1024 + get);
      bl[j] = *reinterpret_cast<const v4i*>(mine + (2 * MT + 2 * j + 1) * 1024 + get);
    }
#pragma unroll
    for(int i = 0; i < MT; ++i) {
      const v4i ah = *reinterpret_cast<const v4i*>(mine + (2 * i) * 1024 + get);
      const v4i al = *reinterpret_cast<const v4i*>(mine + (2 * i + 1) * 1024 + get);
#pragma unroll
      for(int j = 0; j < NT; ++j) acc[i][j].add(bh[j], bl[j], ah, al);
    }
    __builtin_amdgcn_wave_barrier();
  };
  // (the loads of later steps stand behind no branch of their own: the compiler would wait for them at once)
  if(D == 1 || steps < 2) {
    if(steps > 0) {
      load(0, ra[0], rb[0]);
      int t = 0;
      for(; t + 1 < steps; ++t) step(t, t + 1, ra[0], rb[0]);
      step(t, -1, ra[0], rb[0]);
    }
  } else {
    load(0, ra[0], rb[0]);
    load(1, ra[D - 1], rb[D - 1]);
    int t = 0;
    for(; t + 3 < steps; t += 2) {
      step(t, t + 2, ra[0], rb[0]);
      step(t + 1, t + 3, ra[D - 1], rb[D - 1]);
    }
    if(t + 2 < steps) {
      step(t, t + 2, ra[0], rb[0]);
      step(t + 1, -1, ra[D - 1], rb[D - 1]);
      step(t + 2, -1, ra[0], rb[0]);
    } else {
      step(t, -1, ra[0], rb[0]);
      step(t + 1, -1, ra[D - 1], rb[D - 1]);
    }
  }
  // row sums over the quads; lane (lr, lk) holds outputs row lr, columns 4 lk .. 4 lk + 3
#pragma unroll
  for(int i = 0; i < MT; ++i) asum[i] = __shfl(quad_sum(asum[i]), 4 * lr);
#pragma unroll
  for(int j = 0; j < NT; ++j) {
    bsum[j] = quad_sum(bsum[j]);
    int bs[4];
#pragma unroll
    for(int e = 0; e < 4; ++e) bs[e] = __shfl(bsum[j], 16 * lk + 4 * e);
#pragma unroll
    for(int i = 0; i < MT; ++i) {
      v4i t = acc[i][j].sum();
#pragma unroll
      for(int e = 0; e < 4; ++e)
        t[e] = (int)((unsigned)t[e] + 128u * (unsigned)(asum[i] + bs[e]) - 16384u * 64u * (unsigned)steps);
      *reinterpret_cast<v4i*>(mine + (i * NT + j) * 1024 + lane * 16) = t;
    }
  }
  __syncthreads();
  if(wave < TILES && wr_m < g.M && wr_n < g.N) {   // (N % 8 == 0: four columns are inside or outside together)
    v4i sum = v4i{0, 0, 0, 0};
#pragma unroll
    for(int w = 0; w < KW; ++w) {
      const v4i p = *reinterpret_cast<const v4i*>(lds16 + w * kWaveBytes + wave * 1024 + lane * 16);
#pragma unroll
      for(int e = 0; e < 4; ++e) sum[e] = (int)((unsigned)sum[e] + (unsigned)p[e]);
    }
    store16<DUMP>(g, sum, (size_t)wr_m * g.N + wr_n, unquant, bias);
  }
}

// Many tiles: a workgroup of eight waves makes a BM x BN tile; both operands of a block of 64 k go through registers
// (taken apart there, once per workgroup) into LDS, two stages in turn: while one is multiplied the next is filled.
// Waves 0 .. 3 stage A, waves 4 .. 7 B - a wave of each kind on every SIMD -, and the first multiply before they stage, the
// others after, so that one wave's matrix instructions run under the other's vector instructions.
// LDS rows are 64 bytes, their four pieces permuted by the row number so that reads of neighbouring rows fall on
// different banks.  The sums leave through LDS as whole rows.  Bound by the vector instructions of the conversion (about 560 clocks per
// block of 64 k of a 64 x 64 tile, beside 256 of matrix instructions): 509 x 512 x 2048 from float32 10.2 -> 6.8 us, 4096 x 1024 x 4096
// 106 -> 84 (four waves, or eight that all staged and then all multiplied; a bias load waited for before each store).  32 x 32 x 32
// instructions are slower here (4096 x 4096 x 1024 82.6 against 74.0 us), and so are four blocks on their way or two blocks to a barrier
// (more than 128 registers: one workgroup a CU; 2048 x 1024 x 1024 19.7 and 20.5 against 16.6 us).
constexpr int kPitch16 = 64, kTile16Depth = 2, kTile16Threads = 512;
__device__ __forceinline__ int piece16(int row, int c) { return (c ^ ((row >> 1) & 3)) * 16; }
template <int BM, int BN>
constexpr int tile16_sums() { return 4 * BM * BN > 4 * (BM + BN) * kPitch16 ? 4 * BM * BN : 4 * (BM + BN) * kPitch16; }
template <int BM, int BN>
constexpr int tile16_lds() { return tile16_sums<BM, BN>() + 4 * (BM + BN); }
template <typename AT, int BM, int BN, int WM, int WN, bool DUMP>
__global__ __launch_bounds__(kTile16Threads) void gemm16_tile_kernel(const void* A, const int16_t* Bq, const float* bias_in,
                                                                     unsigned long long M_K, int N, Gemm16Rest rest) {
  const Gemm16Args g = gemm16_args(A, Bq, bias_in, M_K, N, rest);
  const int tiles_n = (int)((unsigned)(g.N + BN - 1) / BN), tiles_m = (int)((unsigned)(g.M + BM - 1) / BM);
  static_assert(WM * WN == 8, "eight waves");
  constexpr int FM = BM / WM / 16, FN = BN / WN / 16, D = kTile16Depth;   // D: blocks of K on their way
  extern __shared__ __attribute__((aligned(16))) int8_t lds16[];
  int* const sums = reinterpret_cast<int*>(lds16 + tile16_sums<BM, BN>());   // [BM + BN]
  const int tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64), lr = lane % 16, lk = lane / 16;
  const int wm = wave / WN, wn = wave % WN;
  int tn, tm;
  xcd_order16(tiles_n, tiles_m, blockIdx.x, tn, tm);
  const int m0 = tm * BM, n0 = tn * BN;
  // what the write-out needs, requested first: this thread's four columns' biases (without a bias the weights stand in)
  constexpr int kRowThreads = BN / 4;
  const int wr_col = 4 * (tid % kRowThreads);
  float bias[4];
  const float* bias_src = g.bias ? g.bias : reinterpret_cast<const float*>(g.Bq);
#pragma unroll
  for(int e = 0; e < 4; ++e) bias[e] = bias_src[min(n0 + wr_col, g.N - 4) + e];
  float unquant = 0.0f;
  if(!DUMP) unquant = unquant16<AT>(g);
  Acc16 acc[FM][FN];
#pragma unroll
  for(int i = 0; i < FM; ++i)
#pragma unroll
    for(int j = 0; j < FN; ++j) acc[i][j].clear();
  const int blocks = (g.K + 63) / 64;
  const bool half = g.K % 64 != 0;
  // planes of stage t: A hi, A lo, B hi, B lo
  auto plane = [&](int t, int which, int row) {
    return lds16 + (size_t)t * (2 * (BM + BN) * kPitch16) + (which < 2 ? which * BM : 2 * BM + (which - 2) * BN) * kPitch16 + row * kPitch16;
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
  auto run = [&](auto operand, auto element) __attribute__((always_inline)) {
    constexpr bool kIsA = decltype(operand)::value;
    using E = decltype(element);
    constexpr int ROWS = kIsA ? BM : BN, U = ROWS * 4 / 256;   // pieces of 16 k a thread stages per block
    static_assert(U * 256 == ROWS * 4, "whole pieces per thread");
    const int st = tid % 256, srow = st / 4, sk = piece16_offset(st % 4), spiece = piece16(srow, st % 4);   // four threads a row, 64 rows at a time
    const E* src[U];
    int sum[U];
    Raw<E> raw[D][U];
#pragma unroll
    for(int u = 0; u < U; ++u) {
      const int row = srow + u * 64;
      if constexpr(kIsA) src[u] = reinterpret_cast<const E*>(g.A) + row16_offset(m0 + row, g.M, g.K);
      else src[u] = g.Bq + row16_offset(n0 + row, g.N, g.K);
      sum[u] = 0;
    }
    auto load = [&](int kb, Raw<E> (&r)[U]) __attribute__((always_inline)) {
      kb = min(kb, blocks - 1);
      const int k = kb * kStep16 + sk, second = half && kb == blocks - 1 ? 0 : 32;
#pragma unroll
      for(int u = 0; u < U; ++u) r[u].load(src[u] + k, second);
    };
    auto stage = [&](int t, int kb, Raw<E> (&r)[U]) __attribute__((always_inline)) {
      if(kIsA && half && kb == blocks - 1) {
#pragma unroll
        for(int u = 0; u < U; ++u) r[u].clear_second();
      }
#pragma unroll
      for(int u = 0; u < U; ++u) {
        const Planes p = r[u].planes();
        sum[u] += p.sum;
        *reinterpret_cast<v4i*>(plane(t, kIsA ? 0 : 2, srow + u * 64) + spiece) = p.h;
        *reinterpret_cast<v4i*>(plane(t, kIsA ? 1 : 3, srow + u * 64) + spiece) = p.l;
      }
    };
    // one block: multiplied from stage t while block kb + 1 goes into the other one (which was read before the last barrier)
    auto block = [&](int kb, Raw<E> (&r)[U], bool fill, bool more) __attribute__((always_inline)) {
      const int t = kb & 1;
      if(kIsA) multiply(t);
      if(fill) stage(t ^ 1, kb + 1, r);
      if(more) load(kb + 1 + D, r);
      if(!kIsA) multiply(t);
      lds_barrier();
    };
#pragma unroll
    for(int d = 0; d < D; ++d) load(d, raw[d]);
    stage(0, 0, raw[0]);
    load(D, raw[0]);
    lds_barrier();
    int kb = 0;
    // (the loads inside the loop stand behind no branch: the compiler would wait for them at once)
    for(; kb + 2 * D < blocks; kb += D) {
#pragma unroll
      for(int d = 0; d < D; ++d) block(kb + d, raw[(d + 1) % D], true, true);
    }
#pragma unroll
    for(int d = 0; d < 2 * D; ++d) {
      if(kb + d < blocks) block(kb + d, raw[(d + 1) % D], kb + d + 1 < blocks, d + 1 < D && kb + d + 1 + D < blocks);
    }
    // row sums: the four threads of a row sit side by side
#pragma unroll
    for(int u = 0; u < U; ++u) {
      const int total = quad_sum(sum[u]);
      if(st % 4 == 0) sums[(kIsA ? 0 : BM) + srow + u * 64] = total;
    }
  };
  // (waves of a workgroup meet at the barriers of different instances: see gemm_rows_kernel)
  if(wave < 4) run(std::true_type(), AT());
  else run(std::false_type(), int16_t());
  // (every wave is past its last read of the stages) the sums as rows of BN, their 16-byte pieces permuted by the row number
  constexpr int kMask = 7;
#pragma unroll
  for(int i = 0; i < FM; ++i) {
    const int r = (wm * FM + i) * 16 + lr;
#pragma unroll
    for(int j = 0; j < FN; ++j) {
      const int p = (wn * FN + j) * 4 + lk;
      *reinterpret_cast<v4i*>(lds16 + (r * (BN / 4) + (p ^ (r & kMask))) * 16) = acc[i][j].sum();
    }
  }
  lds_barrier();
  const int n = n0 + wr_col;
  unsigned bs[4];
#pragma unroll
  for(int e = 0; e < 4; ++e) {
    bs[e] = 128u * (unsigned)sums[BM + wr_col + e] - 16384u * 64u * (unsigned)blocks;
    asm volatile("" ::"v"(bias[e]));   // (the wait for the biases stands here, not among the stores)
  }
#pragma unroll
  for(int i = 0; i < BM * kRowThreads / kTile16Threads; ++i) {
    const int r = i * (kTile16Threads / kRowThreads) + tid / kRowThreads, m = m0 + r;
    v4i v = *reinterpret_cast<const v4i*>(lds16 + (r * (BN / 4) + ((wr_col / 4) ^ (r & kMask))) * 16);
    const unsigned as = 128u * (unsigned)sums[r];
#pragma unroll
    for(int e = 0; e < 4; ++e) v[e] = (int)((unsigned)v[e] + as + bs[e]);
    if(m < g.M && n < g.N) store16<DUMP>(g, v, (size_t)m * g.N + n, unquant, bias);
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
  const int tiles_n = (g.N + 16 * NT - 1) / (16 * NT), tiles_m = (g.M + 16 * MT - 1) / (16 * MT);
  constexpr int lds = stream16_lds<MT, NT>();
  static_assert(lds <= 65536, "no attribute needed");
  MH_LAUNCH((gemm16_stream_kernel<AT, MT, NT, 2, DUMP>), dim3((unsigned)tiles_n * (unsigned)tiles_m), dim3(64 * kStream16Waves), lds, st,
            g.A, g.Bq, g.bias, int_pair(g.M, g.K), g.N, Gemm16Rest{g.out, g.scale, g.relu});
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

template <typename AT, int BM, int BN, int WM, int WN, bool DUMP>
int launch_tile16(const Gemm16Args& g, hipStream_t st) {
  const int tiles_n = (g.N + BN - 1) / BN, tiles_m = (g.M + BM - 1) / BM;
  constexpr int lds = tile16_lds<BM, BN>();
  constexpr auto kernel = gemm16_tile_kernel<AT, BM, BN, WM, WN, DUMP>;
  static std::atomic<uint64_t> lds_done{0};
  const int lds_status = allow_lds(kernel, lds, lds_done);
  if(lds_status != MARIAN_HIP_OK) return lds_status;
  MH_LAUNCH(kernel, dim3((unsigned)tiles_n * (unsigned)tiles_m), dim3(kTile16Threads), lds, st, g.A, g.Bq, g.bias,
            int_pair(g.M, g.K), g.N, Gemm16Rest{g.out, g.scale, g.relu});
  MH_HIP(hipGetLastError());
  return MARIAN_HIP_OK;
}

// Which form a call takes: the one whose time is the least by a model that has three prices for each form - of a
// launch, of a further workgroup per CU, and of a byte of either operand that a workgroup takes in (least squares over measurements
// at 99 sizes where the form is near the best: -26 .. +17 %; K, N = 256 .. 4096, M = 1 .. 4096, launches in a graph; a CU holds one
// 128 x 128 tile at a time).  The form taken is the best or at most 4 % behind it but for 256 rows of 704 values by 1408
// (14 and 17 %, int16 and float32 activations: eleven steps of K over eight waves) and 64 float32 rows of them (7 %;
// profiles/int16_forms.txt: every form, both kinds).  us, int16
// and float32 activations:
//   1 x 512 x 512 2.8 and 3.0 (stream 16 x 16), 64 x 512 x 2048 3.6 and 3.7 (16 x 32), 509 x 2048 x 512 8.1 and 8.8 (32 x 32;
//   10.4 and 14.6 with lanes that loaded the rows they multiply), 509 x 512 x 2048 6.5 and 6.8 (64 x 64; 8.6 and 10.2 with four
//   waves that all staged and then all multiplied), 4096 x 4096 x 4096 259 and 270 (128 x 128).
struct Form16 {
  enum Name { kStream16, kStream16x32, kStream32x32, kTile64, kTile128 };
  Name form;
  double ns;     // of the call
};
inline Form16 plan16(int M, int K, int N, int a_bytes) {
  struct Shape { Form16::Name form; int rows, cols; double launch_ns, workgroup_ns, a_byte_ns, b_byte_ns; };
  constexpr Shape shapes[] = {{Form16::kStream16, 16, 16, 2250.0, 270.0, 0.0057, 0.0257}, {Form16::kStream16x32, 16, 32, 1100.0, 1480.0, 0.0058, 0.0228},
                              {Form16::kStream32x32, 32, 32, 700.0, 2190.0, 0.0098, 0.0249}, {Form16::kTile64, 64, 64, 2750.0, 530.0, 0.0061, 0.0363},
                              {Form16::kTile128, 128, 128, 1500.0, 4400.0, 0.0052, 0.0493}};
  Form16 best{Form16::kTile128, 1e30};
  for(const Shape& s : shapes) {
    const double workgroups = (double)((M + s.rows - 1) / s.rows) * ((N + s.cols - 1) / s.cols);
    if(workgroups * kTile16Threads >= 4294967296.0) continue;   // (a launch has fewer threads than that)
    double per_cu = workgroups > 256.0 ? workgroups / 256.0 : 1.0;
    if(s.form == Form16::kTile128) per_cu = std::ceil(per_cu);
    const int rows = M < s.rows ? M : s.rows;   // (rows past the end repeat the last one, which is in the cache)
    const double ns = s.launch_ns + per_cu * (s.workgroup_ns + K * (s.a_byte_ns * rows * a_bytes + s.b_byte_ns * s.cols * 2));
    if(ns < best.ns) best = Form16{s.form, ns};
  }
  return best;
}

// Whether float32 activations are quantized by a launch of their own first: where the multiplication then saves more
// than the launch costs, 2 us and 0.75 ns per thousand values (the pass over them, and the multiplication's wait for values
// that were just written).  Only the 128 x 128 tiles take rows in often enough: the other forms are never more than 1 % behind two
// launches with one.
inline bool quantize_first16(int64_t M, int64_t K, int64_t N) {
  const Form16 one = plan16((int)M, (int)K, (int)N, 4);
  return one.form == Form16::kTile128 && one.ns - plan16((int)M, (int)K, (int)N, 2).ns > 2000.0 + 0.00075 * (double)M * (double)K;
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
    case Form16::kTile64: return launch_tile16<AT, 64, 64, 2, 4, DUMP>(g, st);
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
  MH_LAUNCH(quantize16_a_kernel, dim3((unsigned)blocks), dim3(256), 0, reinterpret_cast<hipStream_t>(stream), A, n8, Aq, (int)blocks);
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
  MH_LAUNCH(quantize16_b_transpose_kernel, grid, dim3(256), 0, reinterpret_cast<hipStream_t>(stream), W, (int)K, (int)N, Bq);
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
