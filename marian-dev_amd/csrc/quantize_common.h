// Device helpers of the quantizers: the int8 rounding and packing, wave and workgroup maxima, the
// quantMult, and the layout of the workspace.  Shared by every translation unit that quantizes.
#pragma once

#include "int8_common.h"
#include "shared_quotient.h"

namespace marian_hip {

constexpr int kQuantThreads = 256;
// Workspace layout, 12 KB: 31 lines of abs-max partials of the two-pass forms, a line with a generation word, four copies of the words that
// workgroups exchange within a launch, 256 of 8 bytes each.  No two of them overlap: partials are written by one launch
// and read by the next, and a launch that exchanges words may come in between.
constexpr int kMaxPartials = 31 * 32;
constexpr int kOnePassMaxGroups = 256;              // workgroups of the one-pass forms (one per CU)
constexpr int kOnePassCopies = 4;
constexpr size_t kOnePassGenOffset = kMaxPartials * sizeof(float);
constexpr size_t kOnePassWordsOffset = 4096;
constexpr size_t kWorkspaceBytes = kOnePassWordsOffset + kOnePassCopies * kOnePassMaxGroups * 8;
static_assert(kOnePassGenOffset + 128 == kOnePassWordsOffset && kWorkspaceBytes == 12288, "workspace layout");
constexpr int kSingleBlockThreads = 1024;
constexpr int kSingleBlockMaxElems = 32 * 1024;     // one workgroup does abs-max and quantize (beyond: 8.6 us against 6.4 us for two launches)

// Four clamped products -> four int8 in one word.  Adding 1.5 * 2^23 rounds to nearest-even and
// leaves the integer in the low byte of the sum; the SDWA form of the add writes that low byte
// straight into byte 0..3 of the destination, so no byte shuffles are needed afterwards.
__device__ __forceinline__ uint32_t round_pack4(float c0, float c1, float c2, float c3) {
  const float magic = 12582912.0f;
  uint32_t q;
  asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_0 dst_unused:UNUSED_PAD src0_sel:DWORD src1_sel:DWORD"
      : "=v"(q) : "v"(c0), "v"(magic));
  asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_1 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
      : "+v"(q) : "v"(c1), "v"(magic));
  asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_2 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
      : "+v"(q) : "v"(c2), "v"(magic));
  asm("v_add_f32_sdwa %0, %1, %2 dst_sel:BYTE_3 dst_unused:UNUSED_PRESERVE src0_sel:DWORD src1_sel:DWORD"
      : "+v"(q) : "v"(c3), "v"(magic));
  return q;
}

// q = clamp(rne(fl32(x * qm)), -127, 127); products that are NaN or outside int32 give -127 (x86 cvtps2dq integer-indefinite followed
// by saturating packs and max(-127)).  Clamping first commutes with the rounding (the bounds are integers), and med3 returns -127
// for NaN.  With a finite quantMult every product lies within [-127.0001, 127.0001]: finite values are at most the abs-max in
// magnitude, and an infinite value makes the quantMult 0 and its product NaN.  An abs-max of zero, or one below 127 / FLT_MAX, gives an
// infinite quantMult, and then products that are infinite or NaN: all -127, so NaN stands in for such a multiplier (a second path
// for it was half of the quantizing code of a launch, which fetches what it passes over).
__device__ __forceinline__ float quantizer(float qm) { return qm < __builtin_inff() ? qm : __builtin_nanf(""); }
// qm: a quantizer's
__device__ __forceinline__ uint32_t quantize_pack4(v4f x, float qm) {
  return round_pack4(__builtin_amdgcn_fmed3f(x.x * qm, -127.0f, 127.0f),
                     __builtin_amdgcn_fmed3f(x.y * qm, -127.0f, 127.0f),
                     __builtin_amdgcn_fmed3f(x.z * qm, -127.0f, 127.0f),
                     __builtin_amdgcn_fmed3f(x.w * qm, -127.0f, 127.0f));
}

__device__ __forceinline__ float abs4max(v4f x, float m) {
  m = fmaxf(m, fabsf(x.x));
  m = fmaxf(m, fabsf(x.y));
  m = fmaxf(m, fabsf(x.z));
  m = fmaxf(m, fabsf(x.w));
  return m;
}

// Max over each row of 16 lanes, left in all 16 of them: four DPP steps (the two lane swaps within
// a quad, the mirror within half a row and within the row).  All lanes of the wave must be active.
// The magnitudes that are reduced here are zero or positive and never NaN (fmaxf passes over NaN operands), so their bits order as
// unsigned numbers do, and a step is one instruction: a float maximum has its operands made quiet first, four more
// (ten steps stand between the arrival of a row and its quantization; a block of 64 x 512 x 2048 and back 10.43 -> 10.27 us).
template <int CTRL, int ROWS = 0xF>
__device__ __forceinline__ unsigned max_step(unsigned m) {
  const unsigned t = (unsigned)__builtin_amdgcn_update_dpp(0, (int)m, CTRL, ROWS, 0xF, false);
  return t > m ? t : m;
}
__device__ __forceinline__ unsigned row16_max_bits(unsigned m) {
  return max_step<0x140>(max_step<0x141>(max_step<0x4E>(max_step<0xB1>(m))));   // quad_perm [1,0,3,2], [2,3,0,1], row_half_mirror, row_mirror
}
__device__ __forceinline__ float row16_max(float m) { return __uint_as_float(row16_max_bits(__float_as_uint(m))); }
// Max over the wave, in all lanes: within the rows, then across them with the two row-broadcast
// DPP steps (rows 1 and 3 take in the last lane of the row before them, then rows 2 and 3 the last
// lane of row 1), which leaves the result in lane 63, read from there as a scalar.  No step goes
// through the LDS crossbar (a lane exchange there costs ten times a DPP step, and these reductions
// sit between the arrival of the activations and their quantization in every fused call).  All
// lanes of the wave must be active.
__device__ __forceinline__ float wave_max(float m) {
  const unsigned r = max_step<0x143, 0xC>(max_step<0x142, 0xA>(row16_max_bits(__float_as_uint(m))));   // row_bcast:15, row_bcast:31
  return __uint_as_float((unsigned)__builtin_amdgcn_readlane((int)r, 63));
}

// Max over the workgroup of WAVES waves (at most 16); every thread returns the result.
// red: >= WAVES floats of LDS.
// (The sizes of a launch are template or kernel arguments throughout: a kernel that asks the runtime for them has
// 256 bytes of hidden arguments, and its launch costs the host 0.35 us more.)
template <int WAVES>
__device__ __forceinline__ float block_max(float m, float* red) {
  m = wave_max(m);
  const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
  __syncthreads();
  if(lane == 0) red[wave] = m;
  __syncthreads();
  // every row of 16 lanes reads all the wave maxima, so the rows need no exchange afterwards
  const float r = (lane % 16 < WAVES) ? red[lane % 16] : 0.0f;
  return row16_max(r);
}

// The abs-max partials a launch starts from, n of them, 1 .. kAbsmaxSlots: up to four a load (a load takes the CU's address unit
// sixteen clocks whatever its width, and four of them a wave were a third of what a call of few rows asks for).
template <int THREADS>
struct PartialMaxima {
  static_assert(kAbsmaxSlots % (4 * THREADS) == 0, "whole vectors a thread");
  static constexpr int kVecs = kAbsmaxSlots / (4 * THREADS);
  v4f v[kVecs];
  __device__ __forceinline__ void load(const float* partials, int n) {
    if(__builtin_expect(n % 4 == 0, 1)) {
#pragma unroll
      for(int i = 0; i < kVecs; ++i) v[i] = *reinterpret_cast<const v4f_any*>(partials + 4 * min((int)threadIdx.x + i * THREADS, n / 4 - 1));
    } else {
#pragma unroll
      for(int i = 0; i < kVecs; ++i)
#pragma unroll
        for(int e = 0; e < 4; ++e) v[i][e] = partials[min(4 * ((int)threadIdx.x + i * THREADS) + e, n - 1)];
    }
  }
  __device__ __forceinline__ float max() const {   // (of this thread's, at least 0)
    float m = 0.0f;
#pragma unroll
    for(int i = 0; i < kVecs; ++i) m = fmaxf(fmaxf(fmaxf(m, v[i].x), fmaxf(v[i].y, v[i].z)), v[i].w);
    return m;
  }
};

// quantMult = 127.0f / maxabs as one correctly rounded fp32 division (via double).
__device__ __forceinline__ float quant_mult_from_maxabs(float maxabs) {
  return (float)(127.0 / (double)maxabs);
}

}  // namespace marian_hip
