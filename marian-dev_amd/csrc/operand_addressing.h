// Where the GEMM kernels read their operands: every byte offset a lane computes for a weight or
// activation load, as functions that compile for the host as well.  The kernels call them, and a
// CPU program (tests/addressing_check.cpp) walks all lanes, waves, tiles and K steps of edge shapes
// through the same functions and checks that every 16-byte load stays inside its operand.
#pragma once

#include <stddef.h>
#include <stdint.h>

#if !defined(__HIPCC__)
#define __host__
#define __device__
#define __forceinline__ inline
#endif

namespace marian_hip {

__host__ __device__ __forceinline__ int addr_min(int a, int b) { return a < b ? a : b; }

// Prepared weights ("K-blocked"): the K*N int8 values of W^T are stored by K sub-step of 32 values;
// within a sub-step the N columns follow each other, 32 bytes (the sub-step's 32 K values) each:
//   byte of (column n, k) = (k / 32) * 32 * N + n * 32 + k % 32
// The operand of one matrix instruction for 32 (or 16) consecutive columns is then 1 KB (512 bytes)
// of consecutive memory, which a wave fetches with one fully coalesced load; advancing along K adds
// 32 * N bytes for every column alike.  (With the plain [N x K] rows every lane of such a load reads
// a different 128-byte line: the address unit then takes four times as long per load, measured as
// 2 k of 16 k clocks of the dominant decode call.  A gathered column - shortlist - still finds the
// two 16-byte halves of a sub-step side by side.)
__host__ __device__ __forceinline__ unsigned b_column_offset(int n) { return (unsigned)n * 32u; }
// 16-byte chunk k16 (K values 16 * k16 .. + 15) of column n
__host__ __device__ __forceinline__ size_t b_chunk_offset(int n, int k16, int N) {
  return (size_t)(k16 >> 1) * 32u * (size_t)N + b_column_offset(n) + (unsigned)(k16 & 1) * 16u;
}

// ---- small-M kernels on 32x32x32 instructions (gemm_stream32_kernel, proj_attention_kernel) ----
// Lane (li, lg) of the wave that owns output columns n0 .. n0 + 31 reads half lg of column
// min(n0 + li, n_out - 1) (through the shortlist ids when there are any), sub-step after sub-step.
__host__ __device__ __forceinline__ int stream32_lane_column(int n0, int li, int n_out) {
  return addr_min(n0 + li, n_out - 1);
}
__host__ __device__ __forceinline__ unsigned stream32_lane_offset(int src_column, int lg) {
  return b_column_offset(src_column) + (unsigned)lg * 16u;
}
// A chunk is CS sub-steps; wave kw of the K split takes sub-steps kw * PW .. + PW - 1 of it.  When
// they all exist the loads use one pointer and constant offsets, otherwise every sub-step is
// clamped to the last one (and its weights are replaced by zeros afterwards).
__host__ __device__ __forceinline__ bool stream32_chunk_is_whole(int chunk, int CS, int kw, int PW, int S) {
  return chunk * CS + (kw + 1) * PW <= S;
}
__host__ __device__ __forceinline__ int stream32_clamped_substep(int s, int S) { return addr_min(s, S - 1); }

// ---- small-M kernel on 16x16x64 instructions (gemm_stream_kernel) ----
// Lane (li, lg) reads 16-byte chunk lg of a K step of 64 of column n (column 0 stands in for columns
// past the output; K steps past the end are not loaded at all).
__host__ __device__ __forceinline__ size_t stream16_lane_offset(int src_column, int lg, int N) {
  return b_chunk_offset(src_column, lg, N);
}

// ---- large-M kernels (gemm_mfma32_kernel, gemm_pair_kernel): global -> LDS staging ----
// Activations: load j of wave `wave` (of `waves`) fills rows (j * waves + wave) * 8 .. + 7 of a stage;
// a lane takes the 16-byte chunk that the XOR swizzle of its row puts at its place.  Rows past the
// matrix re-read the last one.  Offset within a K block of 128 bytes.
__host__ __device__ __forceinline__ int stage_a_row(int j, int waves, int wave, int lane) {
  return (j * waves + wave) * 8 + lane / 8;
}
__host__ __device__ __forceinline__ int stage_a_chunk(int row, int lane) { return (lane % 8) ^ ((row >> 1) & 7); }
__host__ __device__ __forceinline__ int stage_a_offset(int j, int waves, int wave, int lane, int m0, int M, int K) {
  const int row = stage_a_row(j, waves, wave, lane);
  return addr_min(m0 + row, M - 1) * K + stage_a_chunk(row, lane) * 16;
}
// A last block of 64 instead of 128 columns has no chunks 4 .. 7: such lanes go 64 bytes back.
// (The chunk of a lane is the same for all its loads when the number of waves is even.)
__host__ __device__ __forceinline__ int stage_a_tail_adjust(int wave, int lane) {
  return stage_a_chunk(stage_a_row(0, 0, wave, lane), lane) >= 4 ? 64 : 0;
}
// Weights: load g of a stage brings sub-step g / tiles_n of the 32 columns of tile g % tiles_n; lane q
// fetches half q >> 5 of column q & 31 of the tile (clamped to the last output column).
__host__ __device__ __forceinline__ int stage_b_column(int g, int tiles_n, int lane, int n0, int n_out) {
  return addr_min(n0 + (g % tiles_n) * 32 + (lane & 31), n_out - 1);
}
__host__ __device__ __forceinline__ size_t stage_b_offset(int g, int tiles_n, int lane, int src_column, int N) {
  return b_chunk_offset(src_column, 2 * (g / tiles_n) + (lane >> 5), N);
}
// A last block of 64 columns has no sub-steps 2, 3: such loads go two sub-steps (64 * N bytes) back.
__host__ __device__ __forceinline__ bool stage_b_goes_back(int g, int tiles_n) { return g / tiles_n >= 2; }

// ---- projections + attention in one launch (proj_attention_kernel): which input rows a workgroup takes ----
// Caches that are complete and shared - `sentences` entries per head, row m attends to sentence
// m % sentences, M = hypotheses * sentences - let a workgroup take `per_wg` hypotheses of
// 1 << shift neighbouring sentences (per_wg << shift <= 8) instead of eight consecutive rows, so
// that the waves reading the same keys and values sit on one CU; the hypotheses of a sentence are
// taken in `chunks` of per_wg.  Row r of a workgroup: hypothesis chunk * per_wg + (r >> shift) of
// sentence first + (r & ((1 << shift) - 1)); rows whose hypothesis does not exist are idle.
// shift < 0: eight consecutive rows.
struct ProjRowPlan {
  int shift;       // log2 of the sentences per workgroup, or -1
  int sentences;
  int hyps;        // hypotheses per sentence
  int per_wg;      // hypotheses of a sentence a workgroup takes; shift -1: consecutive rows it takes
  int stage;       // the sentences' keys and values are staged in LDS (shift 0 or 1, len <= stage_len)
  long long blocks_y;   // workgroups per head
};
__host__ __device__ __forceinline__ ProjRowPlan proj_row_plan(long long n_proj, long long M, long long heads, long long batchKV,
                                                              long long len, int stage_len, size_t lds_without,
                                                              size_t lds_max) {
  ProjRowPlan plan = {-1, 0, 0, 8, 0, (M + 7) / 8};
  if(n_proj != 1 || heads <= 0 || batchKV % heads != 0) return plan;
  const long long nb = batchKV / heads;
  if(nb <= 0 || nb >= M || M % nb != 0 || nb > 2147483647LL) return plan;
  const long long hyps = M / nb;
  if(hyps > 2147483647LL) return plan;
  // the fewest workgroups (each reads the head's weights), then the fewest chunks (each reads the
  // sentences' keys and values); two hypotheses a sentence keep four sentences per workgroup
  int best_shift = -1, best_per = 0;
  long long best_blocks = 0, best_chunks = 0;
  for(int shift = 2; shift >= 0; --shift) {
    if(nb % (1 << shift) != 0) continue;
    const int room = 8 >> shift;                        // hypotheses a workgroup has rows for
    const long long chunks = (hyps + room - 1) / room;
    const int per = (int)((hyps + chunks - 1) / chunks);
    if(per < 2 || (per << shift) < 4) continue;         // (at least half of a workgroup's rows in use)
    if(shift == 2 && hyps != 2) continue;               // (four sentences are not staged: only where nothing else fits)
    const long long blocks = chunks * (nb >> shift);
    if(best_shift < 0 || blocks < best_blocks || (blocks == best_blocks && chunks < best_chunks)) {
      best_shift = shift; best_per = per; best_blocks = blocks; best_chunks = chunks;
    }
  }
  if(best_shift < 0) return plan;
  plan.shift = best_shift;
  plan.sentences = (int)nb;
  plan.hyps = (int)hyps;
  plan.per_wg = best_per;
  plan.blocks_y = best_blocks;
  const size_t kv_bytes = (size_t)(2 << best_shift) * (size_t)len * 256;
  plan.stage = best_shift <= 1 && len <= stage_len && lds_without + kv_bytes <= lds_max;
  return plan;
}
// Input row r (0 .. 7) of the workgroup of sentence group `group` and hypothesis chunk `chunk` (shift < 0: of rows number
// `group`); rows that do not exist: a value of at least M (= hyps * sentences).  The launch has a dimension for either, so
// that no workgroup divides.
__host__ __device__ __forceinline__ int proj_row_of(int shift, int sentences, int hyps, int per_wg, int group, int chunk, int r) {
  if(shift < 0) return group * per_wg + r;
  const int j = r >> shift, hyp = chunk * per_wg + j;
  if(j >= per_wg || hyp >= hyps) return 0x7fffffff;
  return hyp * sentences + (group << shift) + (r & ((1 << shift) - 1));
}
// The other way round: as which row the workgroup takes input row `row` (below M), or -1.
__host__ __device__ __forceinline__ int proj_place_of(int shift, int sentences, int hyps, int per_wg, int group, int chunk, int row) {
  if(shift < 0) {
    const int r = row - group * per_wg;
    return r >= 0 && r < per_wg ? r : -1;
  }
  const int hyp = (int)((unsigned)row / (unsigned)sentences), j = hyp - chunk * per_wg, s = row - hyp * sentences - (group << shift);
  return s >= 0 && s < 1 << shift && j >= 0 && j < per_wg && hyp < hyps ? (j << shift) + s : -1;
}
// sentence groups of a launch (shift >= 0), and the first sentence of one
__host__ __device__ __forceinline__ int proj_groups(int shift, int sentences) { return sentences >> shift; }
__host__ __device__ __forceinline__ int proj_first_sentence(int shift, int group) { return group << shift; }

// ---- gemm_rows_kernel: tiles of rows x 32 columns, every wave its own share of K ----
constexpr int kRowsWaves = 8;
// Which tile a workgroup of gx x gy takes.  Workgroups are dealt out to the eight XCDs in turn; a split of r = 1 << shift (r divides gy,
// 8 / r divides gx) is launched as 8 x h x w workgroups, h = gy / r, w = gx r / 8, and gives each XCD a block of h x w tiles, so
// that its L2 fetches fewer operands.  shift < 0: launched as gx x gy.
struct RowsTiles {
  int shift, h, w;
};
struct RowsTile {
  int bx, by;
};
__host__ __device__ __forceinline__ RowsTile rows_tile(RowsTiles t, int x, int y, int z) {
  if(t.shift < 0) return RowsTile{x, y};
  return RowsTile{(x >> t.shift) * t.w + z, (x & ((1 << t.shift) - 1)) * t.h + y};
}
// The split of gx x gy tiles with which the XCDs' L2 caches fetch the fewest bytes (as they come where the tiles don't divide into eight blocks).
__host__ __device__ __forceinline__ RowsTiles rows_tiles(int gx, int gy, long long row_bytes, long long column_bytes) {
  RowsTiles best{-1, 0, 0};
  long long least = 0;
  for(int shift = 0; shift <= 3; ++shift) {
    const int r = 1 << shift;
    if(gy % r != 0 || gx % (8 / r) != 0) continue;
    const RowsTiles t{shift, gy / r, gx / (8 / r)};
    const long long bytes = t.h * row_bytes + t.w * column_bytes;
    if(best.shift < 0 || bytes < least) { best = t; least = bytes; }
  }
  return best;
}
// K is taken in pairs of sub-steps (64 values of k): pair number t of a wave, and whether the wave has `steps` of them, ceil(K / 512), or one fewer
__host__ __device__ __forceinline__ int rows_pair(int wave, int t) { return wave + t * kRowsWaves; }
__host__ __device__ __forceinline__ bool rows_has_all_steps(int K, int steps, int wave) { return wave < K / 64 - (steps - 1) * kRowsWaves; }
// Load j of a pair brings rows 4 j .. 4 j + 3 of the tile, sixteen lanes a row: byte offset of the four float32 values of a lane at
// pair 0, v = lane % 16 (M * K <= 2^28); a pair is kRowsPairBytes of a row
constexpr unsigned kRowsPairBytes = 256;
__host__ __device__ __forceinline__ unsigned rows_a_offset(int m_base, int j, int lane, int v, int M, int K) {
  return (unsigned)(addr_min(m_base + 4 * j + lane / 16, M - 1) * K + 4 * v) * 4u;
}
// Vector i of a thread's share of the activations, of workgroup `block` with `each` vectors (past the share or the tensor: the last ones again)
__host__ __device__ __forceinline__ int rows_share_vec(int block, int each, int i, int tid, int threads, int n4) {
  return addr_min(block * each + addr_min(tid + i * threads, each - 1), n4 - 1);
}

// ---- 16-bit kernels (rows of K values, K % 32 == 0, taken in steps of 64) ----
// The four lanes of a quad take a row's step: piece q eight values from piece16_offset(q) and eight from 32 behind (where K % 64 != 0 the last
// step has only the former: it reads them twice, and the kernels drop the second).  Index of a row's first value (rows past the end: the last one);
// a step is kStep16 values.
constexpr int kStep16 = 64;
__host__ __device__ __forceinline__ size_t row16_offset(int row, int rows, int K) { return (size_t)addr_min(row, rows - 1) * K; }
__host__ __device__ __forceinline__ int piece16_offset(int piece) { return piece * 8; }
// The tile of workgroup `block` of tiles_n x tiles_m: workgroups are dealt out to the eight XCDs in turn, and those of one XCD
// take neighbouring tiles - bands of eight columns - so that its L2 holds what they share.
__host__ __device__ __forceinline__ void xcd_order16(int tiles_n, int tiles_m, int block, int& tn, int& tm) {
  const int total = tiles_n * tiles_m, x = block % 8, rest = total % 8;
  const int t = x * (total / 8) + addr_min(x, rest) + block / 8;
  const int band = 8, b = t / (band * tiles_m), r = t % (band * tiles_m), width = addr_min(tiles_n - b * band, band);
  tn = b * band + r % width;
  tm = r / width;
}

}  // namespace marian_hip
