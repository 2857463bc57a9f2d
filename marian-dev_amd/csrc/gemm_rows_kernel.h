// Small-M int8 GEMM that quantizes its float32 activations on the way, every wave for itself: an abs-max launch (or the
// producer of the activations) has left values whose maximum is max|A|.
//
// A workgroup makes ROWS x 32 outputs; its eight waves split K into pairs of sub-steps (64 values of k), wave w takes
// pairs w, w + 8, ..  A wave loads the float32 rows of its pairs itself - sixteen lanes a row, whole 128-byte lines -,
// quantizes them into LDS of its own in matrix-operand order, multiplies with weights that go from memory straight into
// operand registers, and keeps D pairs on their way.  No value is quantized twice in a workgroup and nothing but the
// abs-max and the partial sums at the end changes hands between the waves, so there is no barrier in the loop: one wave's
// loads are in flight while another quantizes.  (The form before staged a chunk of K for all waves: loads, barrier,
// quantization, barrier, products, in turn.  Reading alone takes 6.4 us of a 128 x 4096 x 1024 call in 16 x 32 tiles; the staged form
// took 11.2, this one 8.5; 64 x 1024 x 1024 4.5 and 3.9, 65 x 512 x 1536 4.3 and 3.7, 40 x 3072 x 768 7.7 and 5.7.)
// ROWS: 32, or 16 or 8 where few tiles would leave most CUs idle (half or a quarter of the float32 bytes and of the
// quantizing per workgroup, twice or four times the workgroups).
#pragma once

#include <type_traits>

#include "gemm_stream32_kernel.h"
#include "onepass_exchange.h"

namespace marian_hip {

constexpr int kRowsThreads = kRowsWaves * kWave;
// LDS of a wave: the four 16-value chunks of a pair, 16 bytes a row; the padding spreads the dwords of four rows over the banks
template <int ROWS>
constexpr int rows_chunk_bytes() { return ROWS * 16 + 64; }
template <int ROWS>
constexpr int rows_lds_bytes() {   // the staging, or the partial sums
  return kRowsWaves * (ROWS * 128 > 4 * rows_chunk_bytes<ROWS>() ? ROWS * 128 : 4 * rows_chunk_bytes<ROWS>());
}

// pairs of a wave that are on their way at a time, as registers allow
constexpr int rows_depth(int rows) { return rows == 32 ? 2 : 4; }

// Where the abs-max of the activations comes from.  AbsMaxSlots: n_partials values at `partials`, whose maximum it is.
// AbsMaxExchange: nobody has taken it.  Every workgroup takes that of its share of the activations (kRowsShare values at most, read
// ahead of its operands) and they exchange it while their first operands are on their way, instead of a launch in front: calls on a stream
// 64 x 1024 x 1024 7.4 -> 5.3 us, 256 x 512 x 512 6.7 -> 5.3, 256 x 1024 x 1000 7.4 -> 6.5, and 2.2 us less of the host's time each.
struct AbsMaxSlots {};
struct AbsMaxExchange {
  unsigned long long* words;
  unsigned nonce;
  int polls;
};
constexpr int kRowsShareVecs = 4;   // of four values, of a thread
constexpr int kRowsShare = kRowsThreads * kRowsShareVecs * 4;

// Arguments behind those that come in registers.
template <typename GROUPS, typename ABSMAX>
struct RowsRest {
  GemmArgs args;
  int8_t* aq_out;
  GROUPS groups;
  ABSMAX absmax;
};

// STEPS: pairs that the first waves take, ceil(K / 512); the others take one fewer.  tile_block: h | w << 16; flags: 1 with a shortlist,
// plus 2 (shift + 1).  (The fields of args that are arguments of their own as well are those.)
template <int ROWS, int STEPS, typename GROUPS = NoGroups, typename ABSMAX = AbsMaxSlots>
__global__ __launch_bounds__(kRowsThreads) void gemm_rows_kernel(const float* A, const int8_t* Bq, const float* partials, unsigned long long M_K,
                                                                 unsigned long long N_n_out, unsigned long long n_partials_flags,
                                                                 unsigned tile_block, RowsRest<GROUPS, ABSMAX> rest) {
  const int M = int_pair(M_K).first, K = int_pair(M_K).second, N = int_pair(N_n_out).first, n_out = int_pair(N_n_out).second;
  const int n_partials = int_pair(n_partials_flags).first, flags = int_pair(n_partials_flags).second;
  GemmArgs args = rest.args;
  int8_t* const aq_out = rest.aq_out;
  const GROUPS& groups = rest.groups;
  const ABSMAX& absmax = rest.absmax;
  args.Bq = Bq; args.M = M; args.K = K; args.N = N; args.n_out = n_out;   // (what is needed first comes in registers, see the Makefile)
  constexpr bool GROUPED = std::is_same<GROUPS, GroupTable>::value, EXCHANGE = std::is_same<ABSMAX, AbsMaxExchange>::value;
  constexpr int CHUNK = rows_chunk_bytes<ROWS>(), LOADS = ROWS / 4;   // of four rows a load
  extern __shared__ __attribute__((aligned(16))) int8_t lds[];
  __shared__ float red[kRowsWaves + 1];
  __shared__ __attribute__((aligned(16))) float bias_lds[32];
  const int tid = threadIdx.x, lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int li = lane % 32, lg = lane / 32;
  const RowsTile tile = rows_tile(RowsTiles{(flags >> 1) - 1, (int)(tile_block & 0xFFFFu), (int)(tile_block >> 16)}, blockIdx.x, blockIdx.y, blockIdx.z);
  const bool first_column = tile.bx == 0;
  int bx = tile.bx;
  if constexpr(GROUPED) bx = groups.select(args, bx);
  const int m_base = tile.by * ROWS;

  // The order of the loads: see gemm_stream32_kernel (ids first, then what is needed first, all unconditional).
  const int n0 = bx * 32;
  int wsrc = stream32_lane_column(n0, li, args.n_out);
  if(flags & 1) wsrc = (int)args.idx[wsrc];   // through a shortlist
  asm volatile("" : "+v"(wsrc));
  const float bqm = tail_quant_mult(args.Bq, (size_t)K * (size_t)args.N);
  [[maybe_unused]] PartialMaxima<kRowsThreads> pm;
  v4f share[kRowsShareVecs];
  const int block = tile.by * args.blocks_x + tile.bx, blocks = args.blocks_x * args.blocks_y;
  if constexpr(EXCHANGE) {
    const int n4 = M * K / 4, each = (n4 + blocks - 1) / blocks;   // (past the share: the tensor's last values, again)
#pragma unroll
    for(int i = 0; i < kRowsShareVecs; ++i) share[i] = reinterpret_cast<const v4f*>(A)[rows_share_vec(block, each, i, tid, kRowsThreads, n4)];
  } else {
    pm.load(partials, n_partials);
  }

  // lane: value group v (four values) of row 4 j + lane / 16 of load j
  const int v = lane % 16;
  unsigned a_off[LOADS];   // bytes from A (M * K <= 2^20, 2^28 where a measurement id asks for the form)
#pragma unroll
  for(int j = 0; j < LOADS; ++j) a_off[j] = rows_a_offset(m_base, j, lane, v, M, K);
  const unsigned w_off = stream32_lane_offset(wsrc, lg);   // bytes from a sub-step's first column
  const unsigned w_step = 32u * (unsigned)args.N;
  // (as buffers: a scalar base, a scalar offset along K and a 32-bit lane offset, no vector arithmetic between the loads)
  const auto a_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(A), 0, (int)(4u * (unsigned)M * (unsigned)K), kRawBuffer);
  const auto w_buf = __builtin_amdgcn_make_buffer_rsrc(const_cast<int8_t*>(args.Bq), 0, (int)((unsigned)K * (unsigned)args.N), kRawBuffer);
  const float* bias_src = args.bias ? args.bias : reinterpret_cast<const float*>(args.Bq);   // (without a bias: dropped in the epilogue)
  int8_t* const mine = lds + wave * 4 * CHUNK;
  int8_t* const put = mine + (v / 4) * CHUNK + (lane / 16) * 16 + (v % 4) * 4;
  const int8_t* const get = mine + lg * CHUNK + (li % ROWS) * 16;   // (rows past ROWS: others again, their outputs are not stored)
  float bias_v = 0.0f, unquant = 0.0f;   // (bias_v: of the column that this lane loads)
  v16i_s acc;
  // The whole of a wave's share of K, for T steps: straight-line code, because a load behind a branch would be waited for at
  // once.  WRITE_AQ: the quantized activations leave as well (rows past M: the last one again, to the same place).
  constexpr bool EARLY = STEPS > 2;   // of the abs-max that is in slots
  auto exchange_of = [&]() __attribute__((always_inline)) {
    if constexpr(EXCHANGE) return OnepassExchange(block, absmax.nonce, 0u, absmax.words, blocks);
    else return 0;
  };
  auto run = [&](auto steps_tag, auto write_tag) __attribute__((always_inline)) {
    constexpr int T = decltype(steps_tag)::value, D = T < rows_depth(ROWS) ? T : rows_depth(ROWS);
    constexpr bool WRITE_AQ = decltype(write_tag)::value;
    v4f a[D > 0 ? D : 1][LOADS];
    v4i w[D > 0 ? D : 1][2];
    auto load = [&](int t, int d) __attribute__((always_inline)) {
      const unsigned pair = (unsigned)rows_pair(wave, t);
#pragma unroll
      for(int j = 0; j < LOADS; ++j) a[d][j] = __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(a_buf, a_off[j], pair * kRowsPairBytes, 0));
#pragma unroll
      for(int s = 0; s < 2; ++s) w[d][s] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(w_buf, w_off, (2u * pair + s) * w_step, 0));
      __builtin_amdgcn_sched_barrier(0);
    };
    __builtin_amdgcn_sched_barrier(0);
    // The abs-max comes between the first pair's loads and the others': a wave goes on only when its loads have been accepted, and those of the later
    // four waves stand behind all of the earlier ones', 3000 clocks of a launch of 14 000 before anyone knew it or sent its share of it.  All loads
    // first: 64 x 512 x 2048 and back 10.19 us, now 9.78, 256 x 1024 x 1000 of a shortlist with its four best words 11.03 and 10.13, a step of 65 x 512
    // 300.8 and 298.9; none first: 9.90 and 10.21.  (Two pairs and fewer are all on their way together.)
    float amax = 0.0f;
    [[maybe_unused]] const auto exchange = exchange_of();
    if(D > 0) load(0, 0);
    if constexpr(EXCHANGE) {
#pragma unroll
      for(int i = 0; i < kRowsShareVecs; ++i) amax = abs4max(share[i], amax);
      amax = block_max<kRowsWaves>(amax, red);
      if(blocks > 1) exchange.publish(amax);
    } else if constexpr(EARLY) {
      amax = block_max<kRowsWaves>(pm.max(), red);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for(int d = 1; d < D; ++d) load(d, d);
    bias_v = bias_src[wsrc];
    __builtin_amdgcn_sched_barrier(0);
    if constexpr(EXCHANGE) {
      if(blocks > 1)
        amax = exchange.collect(amax, 0u, nullptr, absmax.polls, &red[kRowsWaves], [&] { return onepass_scan<kRowsThreads>(A, (size_t)M * K / 4, red); });
    } else if constexpr(!EARLY) {
      amax = block_max<kRowsWaves>(pm.max(), red);
    }
    const float aqm = __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(quant_mult_from_maxabs(amax))));
    unquant = unquant_mult(aqm, bqm, args.scale);
    const float by = quantizer(aqm);
    if(WRITE_AQ && tile.by == 0 && tid == 0) *reinterpret_cast<float*>(aq_out + (size_t)M * K) = aqm;
#pragma unroll
    for(int e = 0; e < 16; ++e) acc[e] = 0;
#pragma unroll
    for(int t = 0; t < T; ++t) {
      const int d = t % (D > 0 ? D : 1);
      uint32_t q[LOADS];
#pragma unroll
      for(int j = 0; j < LOADS; ++j) q[j] = quantize_pack4(a[d][j], by);
#pragma unroll
      for(int j = 0; j < LOADS; ++j) *reinterpret_cast<uint32_t*>(put + j * 64) = q[j];
      if(WRITE_AQ) {
#pragma unroll
        for(int j = 0; j < LOADS; ++j)
          *reinterpret_cast<uint32_t*>(aq_out + (a_off[j] / 4 + (unsigned)(rows_pair(wave, t) * 64))) = q[j];
      }
      // (a wave's LDS operations keep their order)
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for(int s = 0; s < 2; ++s) {
        const v4i x = *reinterpret_cast<const v4i*>(get + 2 * s * CHUNK);
        acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(w[d][s], x, acc, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      if(t + D < T) load(t + D, d);
    }
  };
  // The waves of a workgroup run different instances of this code, and meet at its barriers all the same: the hardware counts
  // the waves that have come to a barrier, whichever instruction they came by, and every instance has the same barriers in the same order.
  const bool more = rows_has_all_steps(K, STEPS, wave);
  if(aq_out && first_column) {
    if(more) run(std::integral_constant<int, STEPS>(), std::true_type());
    else run(std::integral_constant<int, STEPS - 1>(), std::true_type());
  } else {
    if(more) run(std::integral_constant<int, STEPS>(), std::false_type());
    else run(std::integral_constant<int, STEPS - 1>(), std::false_type());
  }

  // ---- partial sums: every wave drops its ROWS x 32 NT tile into LDS (row-major, the 16-byte pieces of a row permuted by
  //      the row number) and finishes an eighth of the rows, as in gemm_stream32_kernel ----
  constexpr int kTileBytes = ROWS * 128;
  if(tid < 32) bias_lds[tid] = bias_v;
  __syncthreads();   // (the tiles lie over the staging of other waves)
  if(li < ROWS) {
#pragma unroll
    for(int q = 0; q < 4; ++q)
      *reinterpret_cast<v4i*>(lds + wave * kTileBytes + li * 128 + ((2 * q + lg) ^ (li & 7)) * 16) =
          v4i{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
  }
  __syncthreads();
  float omax = 0.0f;
  const int n = n0 + 4 * (lane % 8), mrow = wave * (ROWS / kRowsWaves) + lane / 8, m = m_base + mrow;
  if(lane < ROWS * 8 / kRowsWaves && m < M && n < args.n_out) {
    const int8_t* src = lds + mrow * 128 + (((lane % 8) ^ (mrow & 7)) * 16);
    v4i sum = *reinterpret_cast<const v4i*>(src);
#pragma unroll
    for(int k = 1; k < kRowsWaves; ++k) sum += *reinterpret_cast<const v4i*>(src + k * kTileBytes);
    const v4f bias4 = reinterpret_cast<const v4f*>(bias_lds)[lane % 8];
    float y[4];
#pragma unroll
    for(int e = 0; e < 4; ++e) {   // y = float(acc) * unquant (+ bias); relu: y > 0 ? y : 0; multiply and add round separately
      y[e] = (float)sum[e] * unquant;
      if(args.bias) y[e] = y[e] + bias4[e];
      if(args.relu) y[e] = y[e] > 0.0f ? y[e] : 0.0f;
      omax = fmaxf(omax, fabsf(y[e]));
    }
    v4f* dst = reinterpret_cast<v4f*>(reinterpret_cast<float*>(args.out) + (size_t)m * (size_t)args.n_out + (size_t)n);
    const v4f yv = v4f{y[0], y[1], y[2], y[3]};
    if(args.stream_out) asm volatile("global_store_dwordx4 %0, %1, off nt" : : "v"(dst), "v"(yv) : "memory");
    else *dst = yv;
  }
  if(args.absmax_out) {   // a slot per wave; workgroup 0 zeroes the slots nobody owns
    const int used = blocks * kRowsWaves;
    omax = wave_max(omax);
    if(lane == 0) args.absmax_out[block * kRowsWaves + wave] = omax;
    if(block == 0)
      for(int sl = used + tid; sl < kAbsmaxSlots; sl += kRowsThreads) args.absmax_out[sl] = 0.0f;
  }
}

}  // namespace marian_hip
