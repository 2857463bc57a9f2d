// Which attentions of several query rows a head take attention_heads_kernel, and how (host code, no HIP).
#pragma once

#include <stdint.h>

namespace marian_hip {

struct AttentionHeadsPlan {
  int tiles, waves;      // blocks of sixteen keys, waves of a workgroup (sixteen query rows each)
  int64_t workgroups;    // of a head; 0: attention_rows_kernel
};

// groups: workgroups of a head in attention_rows_kernel.  Measured on 256 CUs, this form's time over that one's:
// - Where that deal leaves some CUs two workgroups, and not where each of them has one block of rows (80 heads of 64 x 64 1.20) unless a head has
//   two blocks at the most.
// - Where a quarter of the waves or more would have no rows it is slower: one block of rows to three or four waves 1.03 - 1.86 (288 heads of 16 x 64 1.36,
//   of 16 x 128 1.62), two 0.97 - 1.41 (1024 of 30 x 100 1.34), four to twice three 0.97 - 1.36 (512 of 64 x 80 1.21), five and six to twice four
//   1.02 - 1.18; with fewer 0.68 - 1.1, most 0.75 - 0.95 (144 heads of 64 x 64 0.89, of 80 x 80 0.87, 640 of 64 x 64 0.91, 512 of 128 x 128
//   0.92; the most, 1.04 - 1.1, for seven and eight blocks of rows and 81 .. 96 keys with 192 .. 256 heads).
// - Of two waves (up to 32 keys) it is the faster one all the same: 0.68 - 1.01.
// - Three blocks to four waves: 0.80 - 0.93 where a head has two workgroups in the other form, too, 0.98 - 1.10 where it has one.
inline AttentionHeadsPlan attention_heads_plan(int64_t heads, int64_t groups, int64_t row_blocks, int64_t len) {
  const AttentionHeadsPlan none{0, 0, 0};
  if(heads * groups <= 256 || len > 128 || (groups == row_blocks && row_blocks > 2)) return none;
  const int tiles = len <= 32 ? 2 : len <= 48 ? 3 : len <= 64 ? 4 : len <= 80 ? 5 : len <= 96 ? 6 : 8;   // (97 .. 112 keys: eight as well)
  const int waves = tiles == 2 ? 2 : tiles % 4 == 0 ? 4 : 3;
  const int64_t workgroups = (row_blocks + waves - 1) / waves, slots = workgroups * waves, idle = slots - row_blocks;
  if(waves > 2 && 4 * idle >= slots && !(4 * idle == slots && workgroups == 1 && groups > 1)) return none;
  return AttentionHeadsPlan{tiles, waves, workgroups};
}

}  // namespace marian_hip
