// Which kernel and tile shape a launch takes, from its sizes: host arithmetic alone, with no
// device or HIP header, so that it can be looked at without either.
#pragma once

#include <cstdint>

namespace iehip {

// The matrix-core prefill's forms: a workgroup per (pair of 16-row blocks, KV head) with one or
// two teams of waves, or per (one or two row blocks, query head) with 8 or 4 waves.
enum class PrefillKernel { kPairsTwoTeams, kPairsOneTeam, kRows1x8, kRows2x8, kRows2x4 };

// 16-bit caches; `split`: hi + lo operands.
// A workgroup per (pair of blocks, KV head) shares every K/V tile among the group's heads,
// which pays where more than four do and those workgroups fill enough of the compute units: two
// thirds (32 / 48) where hi + lo products weigh more against the tiles' way in, 29 / 48 with
// single operands; in prompts under 1,120 rows, whose row blocks are few enough to end unevenly,
// 29 and 24. Below, and up to two thirds for smaller groups, workgroups per (row block, query
// head). Measured (us, f16 / bf16; rows on cached positions), pairs of blocks against row
// blocks: 4,000 on 0: 54 / 82 against 68 / 95; 2,000 on 0: 31 / 46 against 28 / 34; 2,000 on
// 2,000: 67 / 107 against 54 / 73; 600 on 0: 18 / 23 against 11 / 12; 130 on 4,000: 81 / 135
// against 17 / 19; 2,720 on 0: 36.7 / 62 against 37.7 / 52; 64/8 heads, 512 on 0: 17.8 / 23
// against 17.3 / 20, 640 on 0: 18.6 / 23.7 against 23.8 / 27.1.
// Of the row-block shapes: one block and 8 waves while that gives at most a workgroup per unit
// (64 on 2,000, f16: 11.1, two blocks 13); two blocks, 32-key tiles and 8 waves up to 2.5 (512
// on 8,000, f16: 37, 4 waves 53), or up to the 2 that a unit holds at once where the few that
// come after those hold the launch up (hi + lo operands: 1,280 on 0 22.0, 4 waves 17.2; on
// 4,000 78 and 76; short prompts of small groups: 32/8 heads, f16, 576 on 0 16.6, 4 waves
// 14.0); 64-key tiles and 4 waves above (2,000 on 2,000, bf16: 73, 8 waves 77).
// Two teams of waves split a pair's key tiles while the pairs leave units without a workgroup
// or with one: twice the waves, half the chain of tiles of each.
inline PrefillKernel choose_prefill(int T, int n_heads, int n_kv_heads, bool split, int64_t cus) {
  const int group = n_heads / n_kv_heads;
  const int64_t blocks = (int64_t(T) + 15) / 16;
  const int64_t grid = (blocks + 1) / 2 * n_kv_heads;
  const bool longer = blocks >= 70;
  const int64_t share = group <= 4 || (split && longer) ? 32 : split || longer ? 29 : 24;
  if (48 * grid > share * cus)
    return grid <= cus ? PrefillKernel::kPairsTwoTeams : PrefillKernel::kPairsOneTeam;
  if (blocks * n_heads <= cus) return PrefillKernel::kRows1x8;
  const int64_t pairs = (int64_t(T) + 31) / 32 * n_heads;
  return 2 * pairs <= (split || (group <= 4 && !longer) ? 4 : 5) * cus ? PrefillKernel::kRows2x8
                                                                       : PrefillKernel::kRows2x4;
}

// f32 caches: row blocks always. Two blocks of 16 rows per workgroup halve the splitting of K
// and V; 8 waves halve a workgroup's chain of key tiles, 4 leave more of them resident. Measured
// (us; rows on cached positions): 2 blocks x 4 waves from 1.75 workgroups per compute unit on
// (1,333 on 1,000: 73, with 8 waves 82, one block 82); 8 waves below (512 on 8,000: 113, with 4
// 142); one block where two leave half the units idle (130 on 4,000: 44, two 57).
inline PrefillKernel choose_prefill_f32(int T, int n_heads, int64_t cus) {
  const int64_t pairs = (int64_t(T) + 31) / 32 * n_heads;
  if (4 * pairs >= 7 * cus) return PrefillKernel::kRows2x4;
  return 2 * pairs > cus ? PrefillKernel::kRows2x8 : PrefillKernel::kRows1x8;
}

}  // namespace iehip
