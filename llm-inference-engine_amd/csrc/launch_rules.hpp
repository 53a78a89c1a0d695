// Which kernel and tile shape a launch takes, from its sizes: host arithmetic alone, with no
// device or HIP header, so that it can be looked at without either.
#pragma once

#include <cstdint>
#include <iterator>

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
// against 17 / 19; 2,720 on 0: 37.0 / 55.7 against 37.7 / 47.4; 64/8 heads, 512 on 0: 17.4 / 21.7
// against 17.2 / 19.2, 640 on 0: 18.7 / 23.8 against 23.9 / 27.3.
// Of the row-block shapes: one block and 8 waves while that gives at most a workgroup per unit
// (64 on 2,000, f16: 11.1, two blocks 13); two blocks, 32-key tiles and 8 waves up to 2.5 (512
// on 8,000, f16: 37, 4 waves 53), or up to the 2 that a unit holds at once where the few that
// come after those hold the launch up (hi + lo operands, 1,280 on 0: 22.0, 4 waves 17.2; on
// 4,000 79.5 and 77.7; short prompts of small groups: 32/8 heads, f16, 576 on 0 16.6, 4 waves
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

// The projections' LDS tiles (matmul_tiled_kernel). A shape is chosen by the time its launch should take:
// rounds over the compute units times a workgroup's time, which is a fixed part plus a part
// per K block of a slot. The parts (ns) were fitted on an MI355X to o_proj (896 x 896) and
// down (896 x 4,864) with at most one workgroup per compute unit, launch overhead taken
// off; the choice was then within 8% of the fastest shape for q/k/v, o_proj, gate/up and
// down at 21 batch sizes from 1 to 4,000 tokens. What the shapes gain over one 16- or
// 32-row tile per workgroup at every size (us, bf16): gate/up 16.3 -> 12.1 at 64 tokens,
// 104 -> 44 at 600, 630 -> 252 at 4,000; down 11.1 -> 8.7, 47 -> 27, 246 -> 123.
struct Tile {
  int nr, ct, w;           // row tiles (of all weight matrices) and token tiles, waves
  int fixed_ns, block_ns;  // a workgroup's time: fixed + block * (K blocks of a slot)
};
constexpr Tile kPlainTiles[] = {{1, 1, 8, 600, 280},  {2, 1, 8, 750, 390},  {2, 2, 8, 700, 620},
                                {3, 2, 4, 1300, 900}, {4, 2, 4, 1600, 940}, {6, 2, 4, 2000, 1210},
                                {8, 2, 4, 2500, 1470}};
constexpr Tile kGateTiles[] = {{2, 1, 8, 750, 390}, {4, 1, 8, 700, 680}, {4, 2, 8, 1000, 850},
                               {6, 2, 4, 2000, 1210}, {8, 2, 4, 2500, 1470}};
inline int choose_tile(bool gate, int rows, int cols, int T, int cus) {
  const Tile* tiles = gate ? kGateTiles : kPlainTiles;
  const int count = gate ? int(std::size(kGateTiles)) : int(std::size(kPlainTiles));
  const int64_t blocks = (cols / 32 + 7) / 8;
  int best = 0;
  int64_t best_ns = INT64_MAX;
  for (int i = 0; i < count; ++i) {
    const Tile& t = tiles[i];
    const int64_t rt = 16 * (gate ? t.nr / 2 : t.nr), tt = 16 * t.ct;
    const int64_t groups = ((rows + rt - 1) / rt) * ((T + tt - 1) / tt);
    const int64_t ns = ((groups + cus - 1) / cus) * (t.fixed_ns + t.block_ns * blocks);
    if (ns < best_ns) {
      best_ns = ns;
      best = i;
    }
  }
  return best;
}

// K below a 32-wide block for each of the 8 slots: 32 rows x 32 tokens in LDS from 2 16 x 16 tiles
// per compute unit on, direct loads below, where a launch's fixed time is all there is (us,
// one staged 16 x 16 tile / direct / 32 x 32: 256 x 192 at 600 tokens 3.67 / 4.20 / 3.56, 896 x
// 192 at 4,000 35 / 26 / 17, 4,864 x 96 at 600 25 / 15 / 12; 896 x 192 with the norm at 64
// 3.9 / 3.9 / 4.8, 896 x 32 with the norm at 600 11.5 / 6.1 / 7.1).
inline bool short_k_staged(int64_t tiles, int cols, bool norm, int cus) {
  return tiles >= 2 * int64_t(cus) && (!norm || cols >= 96);
}

// Whether a tile's byte offsets from its first row and token fit the 32 bits that its loads
// take them in (128 bf16 rows: up to 16.7 M columns).
inline bool tile_offsets_fit(int tile_rows, int tile_tokens, int64_t cols, int weight_bytes) {
  return tile_rows * cols * weight_bytes <= int64_t(UINT32_MAX) &&
         tile_tokens * cols * 4 <= int64_t(UINT32_MAX);
}

// Wide matrices (16 row tiles per compute unit: LM heads): tiles of 64 rows x 16 tokens or
// 128 x 32, or their weights streamed past up to 16 or 64 tokens whose split activations stay
// in registers (K up to 1,024). The stream counts 8 K blocks per slot whatever there are, so it
// pays where K comes near that: from 768 columns at 33 to 64 tokens, 896 at up to 16; at 17 to
// 32, 128 x 32 tiles take as long and spill nothing. The 151,936-row LM head with 896 columns,
// us, direct loads before / tiles / streamed: bf16, 1 token 59 / 52 / 49, 16 tokens 74 / 64 / 57,
// 32 tokens 90 / 65 / 63, 64 tokens 138 / 92 / 76; INT8, 1 token 58 / 36 / 34, 16 tokens 65 /
// 43 / 39, 64 tokens 177 / 73 / 64. (HBM's share, at the 5.1 TB/s of a large copy: bf16 53 to 61,
// INT8 27 to 34.) With 512 columns, tiles / streamed: bf16, 16 tokens 26.5 / 31.9, 64 tokens
// 45.6 / 53.2; with 128: 12.5 / 26.8 and 24.9 / 47.8 (direct loads 15.8 and 42.6).
enum class WideKernel { kGateTiles, kTiles16, kTiles32, kStream16, kStream64 };
inline WideKernel choose_wide(bool gate, int cols, int T) {
  if (gate) return WideKernel::kGateTiles;
  if (T <= 16) return cols >= 896 && cols <= 1024 ? WideKernel::kStream16 : WideKernel::kTiles16;
  return T > 32 && T <= 64 && cols >= 768 && cols <= 1024 ? WideKernel::kStream64
                                                          : WideKernel::kTiles32;
}

// Waves per chunk of an f32 cache's decode, from the chunk's size alone, so that a row's result
// does not depend on the launch. attention_chunk_tokens chooses 192 where workgroups abound and
// 32, 64 and 128 for small grids (us; rows x positions): 192: 64 x 128-4,096 one wave 28.8, four
// 32.0; 32, two pages: 16 x 512-2,048 11.5, four 15.7; 64: 16 x 512-2,048 four 12.2, two 12.9, one
// 12.7; 128: 48 x 256-2,048 four 18.4, one 19.6. Between those, two waves waste least where the grid
// is large and lose little where it is not (48: 1,024 x 16-512 one 61, two 64, four 85, 1 x 600 9.8,
// 9.4 and 8.9; 96: 256 x 1,024-4,096 139, 138 and 148). More than 192 is a long chain for one
// wave (256: 16 x 512-2,048 26.6, four 15.7).
inline int decode_f32_waves(int chunk_tokens) {
  if (chunk_tokens <= 32 || (chunk_tokens > 128 && chunk_tokens <= 192)) return 1;
  return chunk_tokens != 64 && chunk_tokens <= 96 ? 2 : 4;
}

}  // namespace iehip
