// Chunked-prefill attention into pages on the matrix cores (gfx950), for KV
// caches of every type with head_dim 64: 16-bit caches in their own type
// (prefill_mfma_kernel), f32 caches in three bf16 parts
// (prefill_mfma_f32_kernel, further down).
//
// Reference semantics: each row's causal GQA attention over positions
// 0..row_pos[t] of its sequence (src/ops.cpp:70-108); the reference's GPU
// prompt kernels are src/cuda/kernels.cu:527-776. Rows are consecutive
// positions of ONE sequence (row_pos[t] = row_pos[0] + t), already appended.
//
// Here QK^T and PV are dense tiles: a block of 16 query rows against 64-key
// tiles, per query head,
//     S^T[16 keys x 16 rows]   = K_tile[16 x 64] . Q^T[64 x 16]          (2 k-steps)
//     O^T[64 dims x 16 rows]  += V_tile^T[64 x 32 keys] . P^T[32 x 16 rows]
// on v_mfma_f32_16x16x32_{f16,bf16} in the cache's own 16-bit type. As in the
// decode kernel, lane (g, r) of every tile belongs to query row r, so the
// online-softmax statistics of a row never leave its lanes except for the
// reductions over the 4 lane groups.
//
// Precision: K and V enter exactly. With an f16 cache, q (pre-scaled by
// log2(e)/8) and P (weights <= 2^kLazyMax) enter as single f16 values rounded
// to nearest -- the operand rounding of the reference's tensor-core kernel
// (src/cuda/kernels.cu:673-674,741), here with the row sums taken from the same
// rounded P on the matrix cores, so the output is a weighted mean with weights
// off by <= 2^-11 relative (errors ~6e-4 at 4,000 keys against the 2e-3
// absolute bound). bf16 keeps 8 mantissa bits, too few for that bound:
// with a bf16 cache q and P are split into hi + lo halves and each product is
// done twice (float32-level scores and weights, errors ~1e-6).
//
// Layout of the work:
//   One workgroup per (pair of 16-row blocks, KV head); one wave per query head
//   of the KV head (the 7 heads of a Qwen2.5 group share every K/V tile through
//   LDS). Two heads per wave (each K/V operand feeding both) was measured
//   slower: half the waves leave the dependency and barrier stalls exposed.
//   The pair is block b and block n-1-b: the causal triangle gives block b b+1
//   key tiles of work, so every pair carries about the same total and the
//   ceil(n/2) x n_kv_heads workgroups finish together (the heavier block goes
//   first). When that grid leaves compute units with at most one workgroup,
//   two teams of waves split each block's key tiles (even and odd) and merge
//   their (m, l, O) through LDS at the end.
//   K/V tiles of 64 keys (4 pages, 16 KB) go through an LDS ring by DMA
//   (global_load_lds_dwordx4, 16 x 1 KB per tile spread over 4 waves of a team):
//   4 tiles with one team, 3 steps of 2 tiles with two. The page ids of up to
//   512 tiles are staged in LDS at a block's start (scalar loads of the table
//   inside the loop would share lgkmcnt with the K reads and put the table's
//   round trip on every step). K rows are stored with their 16-byte pieces
//   swizzled (piece ^ (row/2 % 8)) so the A-operand reads (16 rows, one piece each) hit
//   distinct banks; V rows with piece ^ 2*(row/2 % 4) so the transposed reads
//   (ds_read_b64_tr_b16: 8 rows x 32 bytes per half-wave) do.
//   Keys past the block's last position and pages outside the pool are masked
//   (-inf scores, and their V rows zeroed in LDS before use, so stale or
//   non-finite memory cannot reach the output through 0 * x).
#include <algorithm>
#include <type_traits>

#include "common.hpp"
#include "launch_rules.hpp"
#include "mfma.hpp"
#include "prefill.hpp"

namespace iehip {
namespace {

constexpr int kRows = 16;                  // query rows per block (one MFMA column tile)
constexpr int kKeys = 64;                  // keys per LDS tile
constexpr int kTileBytes = kKeys * 128;    // 64 keys x 64 dims x 2 B
constexpr int kBufBytes = 2 * kTileBytes;  // K tile + V tile
constexpr int kMaxGroup = 8;
constexpr int kHeadsPerWave = 1;           // query heads per wave (2 measured slower: fewer waves)
static_assert(kHeadsPerWave == 1, "the team exchange hands over one head per wave");
constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLazyMax = 8.0f;           // log2 headroom of the lazily raised softmax max
constexpr float kSumMax = 16384.0f;        // largest tile row sum taken without a new max
constexpr int kSegTiles = 512;             // key tiles (32,768 keys) with page ids in LDS at once
constexpr int kRopeStride = 68;            // floats per staged RoPE row (64 + 4 of padding)

// kWaves = group / kHeadsPerWave waves per team (rounded up), wave w of a team
// taking query heads kHeadsPerWave * w .. of the KV head. kTeams teams of
// kWaves waves split each block's key tiles (team t takes tiles kTeams s + t)
// and merge their (m, l, O) through LDS at the end of the block.
template <int KV, int kWaves, int kTeams, bool kSplitF16>
__global__ void __launch_bounds__(64 * kWaves * kTeams)
prefill_mfma_kernel(float* __restrict__ out, const float* __restrict__ q,
                    const uint16_t* __restrict__ k_pool, const uint16_t* __restrict__ v_pool,
                    int T, const int32_t* __restrict__ row_pos, const int32_t* __restrict__ row_seq,
                    const int32_t* __restrict__ tables, int max_pages, int num_pages, int n_heads,
                    int n_kv_heads, int n_blocks, const float* __restrict__ rope,
                    int rope_positions) {
  using M = Mfma<KV>;
  using op = typename M::op;
  using E = typename M::elem;
  // hi + lo operands: always for bf16; for f16 under IE_HIP_PREFILL_SPLIT.
  constexpr bool kSplit = kSplitF16 || !std::is_same_v<E, _Float16>;
  constexpr int kRingSteps = kTeams == 1 ? 4 : 3;  // steps of kTeams tiles in LDS
  static_assert(kSegTiles % kTeams == 0, "a step's tiles never straddle two segments");
  constexpr int kRingBytes = kRingSteps * kTeams * kBufBytes;
  op ones;  // all-ones A operand: row sums of P^T on the matrix cores
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = static_cast<E>(1.0f);
  // A tile's 16 loads of 1 KB, spread evenly over kDmaWaves waves of its team.
  constexpr int kDmaWaves = kWaves >= 4 ? 4 : kWaves >= 2 ? 2 : 1;
  constexpr int kPerWave = 16 / kDmaWaves;
  extern __shared__ __align__(16) unsigned char smem[];
  const int group = n_heads / n_kv_heads;
  const int kvh = blockIdx.y;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave_id = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int team = wave_id / kWaves, wave = wave_id - team * kWaves;
  const int g = lane >> 4, r = lane & 15;
  const int h0 = kvh * group + kHeadsPerWave * wave;       // this wave's first head
  const int nh = min(kHeadsPerWave, group - kHeadsPerWave * wave);  // 1 or 2 (uniform)
  const int kv_dim = n_kv_heads * 64;
  const int pos0 = __builtin_amdgcn_readfirstlane(row_pos[0]);
  const int seq = __builtin_amdgcn_readfirstlane(row_seq[0]);
  const int32_t* tab = tables + size_t(seq) * max_pages;

  // The page ids of a segment of key tiles, staged in LDS after the ring by all
  // threads at the segment's start: ids[4 (tile - seg0) + j] is page j of the
  // tile, or -1 for a page past the table row or outside the pool (loaded as
  // page 0 and masked). A step then reads its tiles' ids from LDS instead of
  // the table: no memory round trip inside the tile loop.
  int* const ids = reinterpret_cast<int*>(smem + kRingBytes);
  // Per step of the segment, staged after the ids: bits 4 tm .. 4 tm + 3 = the
  // in-pool bits of team tm's tile, bit 8 = some tile of the step needs V rows
  // zeroed (past max_pos or a page outside the pool). One LDS read per step.
  int* const step_flags = ids + 4 * (kSegTiles + kTeams);
  // With a RoPE table: the cos/sin rows of the block's 16 positions, staged once
  // per block after the step flags and read by every wave; rows kRopeStride
  // floats apart (64 + 4), so that the 16 rows one lane group reads at the same
  // offset fall into different banks.
  float* const rope_rows = reinterpret_cast<float*>(step_flags + kSegTiles);
  int seg0 = 0;  // first tile of the segment in progress
  auto tile_ids = [&](const int tile) {
    return *reinterpret_cast<const int4*>(ids + 4 * (tile - seg0));
  };
  // Buffer of the tile a team takes at step s.
  auto buffer = [&](const int ring_step, const int tm) { return ring_step * kTeams + tm; };

  // DMA of a tile into buffer `buf`: 8 K loads and 8 V loads of 1 KB (8 key rows
  // of 128 bytes each), the same kPerWave for every tile, so a wave can wait for
  // "all but the newest steps" by count. Load u (rows 8u .. 8u+7) lands lane l at
  // base + 16 l: key row 8u + l/8, LDS slot l % 8, holding the global piece the
  // row's swizzle maps to that slot (K: piece ^ (row/2 % 8); V: piece ^ 2*(row/2 % 4)).
  // Per-lane byte offsets (row & 15 = 8 (u & 1) + l / 8) depend only on u & 1.
  const int row_bytes = kv_dim * 2;
  const int lrow = lane >> 3, lslot = lane & 7;
  int koff[2], voff[2];
#pragma unroll
  for (int odd = 0; odd < 2; ++odd) {
    const int row15 = 8 * odd + lrow;
    koff[odd] = row15 * row_bytes + 16 * (lslot ^ (4 * odd + (lrow >> 1)));
    voff[odd] = row15 * row_bytes + 16 * (lslot ^ (2 * (lrow >> 1)));
  }
  const unsigned smem_lds = lds_address(smem);
  const char* kbase_g = reinterpret_cast<const char*>(k_pool) + kvh * 128;
  const char* vbase_g = reinterpret_cast<const char*>(v_pool) + kvh * 128;
  const size_t page_bytes = size_t(IE_HIP_PAGE_SIZE) * row_bytes;
  auto issue = [&](const int buf, const int tile) {
    if (wave >= kDmaWaves) return;
    const int4 v = tile_ids(tile);
    const int id[4] = {max(__builtin_amdgcn_readfirstlane(v.x), 0),
                       max(__builtin_amdgcn_readfirstlane(v.y), 0),
                       max(__builtin_amdgcn_readfirstlane(v.z), 0),
                       max(__builtin_amdgcn_readfirstlane(v.w), 0)};
    // Quarter qt of the loads: qt = 0, 1 the K rows 0-31, 32-63; qt = 2, 3 the V rows.
#pragma unroll
    for (int k = 0; k < 4 / kDmaWaves; ++k) {
      const int qt = wave + k * kDmaWaves;
      const bool is_v = qt >= 2;
      const int half = qt & 1;  // rows 32 half .. 32 half + 31: pages 2 half, 2 half + 1
      const int ida = half ? id[2] : id[0], idb = half ? id[3] : id[1];
      const char* base = is_v ? vbase_g : kbase_g;
      const char* pa = base + size_t(ida) * page_bytes;
      const char* pb = base + size_t(idb) * page_bytes;
      const unsigned dst = smem_lds + buf * kBufBytes + (is_v ? kTileBytes : 0) + half * 4096;
#pragma unroll
      for (int j = 0; j < 4; ++j) {  // u = 4 half + j: page u / 2 of the tile
        const int off = is_v ? voff[j & 1] : koff[j & 1];
        dma16(((j >> 1) ? pb : pa) + off, dst + j * 1024);
      }
    }
  };
  // Wait until this wave's loads of all but the newest `newer` steps have landed.
  auto wait_steps = [&](const int newer) {
    if (newer >= 2) wait_vmcnt<2 * kPerWave>();
    else if (newer == 1) wait_vmcnt<kPerWave>();
    else wait_vmcnt<0>();
  };

  for (int pass = 0; pass < 2; ++pass) {
    const int hi_block = n_blocks - 1 - int(blockIdx.x);
    const int rb = pass == 0 ? hi_block : int(blockIdx.x);
    if (pass == 1 && rb == hi_block) break;  // the middle block of an odd count
    const int t0 = rb * kRows;
    const int t_last = min(t0 + kRows, T) - 1;
    const int max_pos = pos0 + t_last;  // last position any row of the block sees
    const int min_pos = pos0 + t0;      // first row's position
    const int n_tiles = max_pos / kKeys + 1;

    // Queries of row t0 + r for the wave's heads, times log2(e)/8 (split hi + lo
    // for bf16): the B operands of S^T (dims 32 ks + 8g .. +8). Their loads (and
    // the RoPE table rows') are issued here and turned into operands (make_q) only
    // after the block's first page-id staging is under way, so that the query's
    // round trip and the table's overlap instead of following each other.
    const int t = t0 + r;
    const bool row_ok = t < T;
    const int rp = pos0 + t;  // this lane's row position
    float4 qa[kHeadsPerWave][2][2];
#pragma unroll
    for (int hh = 0; hh < kHeadsPerWave; ++hh)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        qa[hh][ks][0] = qa[hh][ks][1] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (row_ok && hh < nh) {
          const float4* src = reinterpret_cast<const float4*>(
              q + (size_t(t) * n_heads + h0 + hh) * 64 + 32 * ks + 8 * g);
          qa[hh][ks][0] = src[0];
          qa[hh][ks][1] = src[1];
        }
      }
    // With a RoPE table (ie_hip_rope_cache_attention_prefill) q arrives unrotated,
    // and the rotation ie_hip_rope_and_cache would have applied in place happens
    // in make_q: lane (g, r) holds dims 8g + j and 32 + 8g + j, the rotation
    // pairs, and takes cos/sin of its row's position from the table; the same
    // fmaf in the same order, so the same float32 values. Rows whose position
    // lies outside the table are used unrotated, as there. The table is read for
    // every lane (row 0's entries where the row is not rotated), the rotation
    // applied by selection.
    const bool rot = rope && row_ok && rp >= 0 && rp < rope_positions;
    op qhi[kHeadsPerWave][2], qlo[kHeadsPerWave][2];
    auto make_q = [&]() {
      float4 tcs[4] = {};  // cos of dims 8g .. 8g+7, then sin (rows staged in LDS)
      if (rope) {
        const float* trow = rope_rows + r * kRopeStride + 8 * g;
        tcs[0] = *reinterpret_cast<const float4*>(trow);
        tcs[1] = *reinterpret_cast<const float4*>(trow + 4);
        tcs[2] = *reinterpret_cast<const float4*>(trow + 32);
        tcs[3] = *reinterpret_cast<const float4*>(trow + 36);
      }
#pragma unroll
      for (int hh = 0; hh < kHeadsPerWave; ++hh) {
        float x[2][8] = {{qa[hh][0][0].x, qa[hh][0][0].y, qa[hh][0][0].z, qa[hh][0][0].w,
                          qa[hh][0][1].x, qa[hh][0][1].y, qa[hh][0][1].z, qa[hh][0][1].w},
                         {qa[hh][1][0].x, qa[hh][1][0].y, qa[hh][1][0].z, qa[hh][1][0].w,
                          qa[hh][1][1].x, qa[hh][1][1].y, qa[hh][1][1].z, qa[hh][1][1].w}};
        if (rope) {
          const float cs[8] = {tcs[0].x, tcs[0].y, tcs[0].z, tcs[0].w,
                               tcs[1].x, tcs[1].y, tcs[1].z, tcs[1].w};
          const float sn[8] = {tcs[2].x, tcs[2].y, tcs[2].z, tcs[2].w,
                               tcs[3].x, tcs[3].y, tcs[3].z, tcs[3].w};
          const bool on = rot && hh < nh;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const float x0 = x[0][j], x1 = x[1][j];
            const float r0 = __builtin_fmaf(x0, cs[j], -(x1 * sn[j]));  // x0*c - x1*s
            const float r1 = __builtin_fmaf(x1, cs[j], x0 * sn[j]);     // x1*c + x0*s
            x[0][j] = on ? r0 : x0;
            x[1][j] = on ? r1 : x1;
          }
        }
        const float qs = 0.125f * kLog2e;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            E hv, lv = static_cast<E>(0.0f);
            if constexpr (kSplit) {
              split16(x[ks][j] * qs, hv, lv);
            } else {
              // The float32 product, then its f16 rounding: kept opaque so that no
              // instantiation folds the two into one mixed-precision fma (a single
              // rounding of the exact product), whether q was rotated here or not.
              float xq = x[ks][j] * qs;
              asm("" : "+v"(xq));
              hv = static_cast<E>(xq);
            }
            qhi[hh][ks][j] = hv;
            qlo[hh][ks][j] = lv;
          }
        }
      }
    };

    // nref: every entry -(the reference max, 0 while m = -inf), the value the S
    // accumulators start from; kept across steps and changed only when m is raised.
    float m[kHeadsPerWave];
    float lsum[kHeadsPerWave];  // the row's sum of weights
    f32x4 nref[kHeadsPerWave];
    f32x4 o[kHeadsPerWave][4];
#pragma unroll
    for (int hh = 0; hh < kHeadsPerWave; ++hh) {
      m[hh] = -INFINITY;
      lsum[hh] = 0.0f;
      nref[hh] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) o[hh][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
    }

    // The block's key tiles in segments of kSegTiles, each with its page ids
    // staged in LDS. Within a segment, a ring of kRingSteps steps of kTeams tile
    // buffers: steps 0 .. kRingSteps-2 are issued up front; at step s, step
    // s + kRingSteps - 1 goes into the buffers step s - 1 used. A step past the
    // last tile still loads (page 0 or in-pool pages, never read), keeping every
    // step's load count the same for the counted waits. Segments hold an even
    // number of tiles, so a step never straddles two.
    // Staging of the segment starting at seg0: its page ids and step flags into
    // LDS, and the ring's first steps issued.
    int n_steps = 0;
    auto stage = [&]() {
      n_steps = (min(kSegTiles, n_tiles - seg0) + kTeams - 1) / kTeams;
      // The ring is idle here and every wave is past its last read of the previous
      // segment's ids (the last step, or the team exchange, ended in a barrier).
      for (int i = tid; i < 4 * kTeams * n_steps; i += 64 * kWaves * kTeams) {
        const int pi = 4 * seg0 + i;
        const int id = pi < max_pages ? tab[pi] : -1;
        ids[i] = id >= 0 && id < num_pages ? id : -1;
      }
      // The block's RoPE rows (first segment only; rows outside the table or past
      // the block's rows are not used and stay as they are).
      if (rope && seg0 == 0) {
        for (int i = tid; i < kRows * 16; i += 64 * kWaves * kTeams) {
          const int ri = i >> 4, p = pos0 + t0 + ri;
          if (t0 + ri < T && p >= 0 && p < rope_positions)
            reinterpret_cast<float4*>(rope_rows + ri * kRopeStride)[i & 15] =
                reinterpret_cast<const float4*>(rope + size_t(p) * 64)[i & 15];
        }
      }
      __syncthreads();
      for (int i = tid; i < n_steps; i += 64 * kWaves * kTeams) {
        int f = 0;
#pragma unroll
        for (int tm = 0; tm < kTeams; ++tm) {
          const int tile = seg0 + kTeams * i + tm;
          const int4 v = tile_ids(tile);
          const int ok = int(v.x >= 0) | (int(v.y >= 0) << 1) | (int(v.z >= 0) << 2) |
                         (int(v.w >= 0) << 3);
          f |= ok << (4 * tm);
          if (tile < n_tiles && (tile * kKeys + kKeys - 1 > max_pos || ok != 15)) f |= 1 << 8;
        }
        step_flags[i] = f;
      }  // read after the barrier below
      for (int pre = 0; pre < kRingSteps - 1 && pre < n_steps; ++pre)
        issue(buffer(pre, team), seg0 + kTeams * pre + team);
    };
    seg0 = 0;
    stage();
    make_q();  // the query's loads landed with the staging's
    for (;;) {
      wait_steps(min(kRingSteps - 2, n_steps - 1));  // step 0 has landed
      __syncthreads();

      int rs = 0;               // ring slot of step s
      int is = kRingSteps - 1;  // ring slot of step s + kRingSteps - 1
      for (int st = 0; st < n_steps; ++st) {
        const int fl = __builtin_amdgcn_readfirstlane(step_flags[st]);  // read with the ids below
        const int ahead = st + kRingSteps - 1;
        if (ahead < n_steps)  // its buffers held step s - 1: free since the last barrier
          issue(buffer(is, team), seg0 + kTeams * ahead + team);
        is = is + 1 == kRingSteps ? 0 : is + 1;
        const int kb = seg0 + kTeams * st + team;  // this team's tile
        const int buf = buffer(rs, team);
        rs = rs + 1 == kRingSteps ? 0 : rs + 1;
        const int kbase = kb * kKeys;
        const unsigned char* kt = smem + buf * kBufBytes;
        unsigned char* vt = smem + buf * kBufBytes + kTileBytes;
        // Keys past max_pos (the last tile) or in pages outside the pool: zero
        // their V rows before the team reads the tile. The decision covers every
        // tile of the step, so every wave takes the same branch and barrier.
        const bool zero_step = (fl >> 8) & 1;
        const int okb = (fl >> (4 * team)) & 15;
        if (zero_step) {
          if (kb < n_tiles) {
            for (int i = tid - 64 * kWaves * team; i < kKeys * 8; i += 64 * kWaves) {
              const int key = i >> 3;
              if (kbase + key > max_pos || !((okb >> (key >> 4)) & 1))
                *reinterpret_cast<uint4*>(vt + key * 128 + (i & 7) * 16) = make_uint4(0, 0, 0, 0);
            }
          }
          __syncthreads();
        }

        if (kb < n_tiles) {  // uniform per team (the odd last step of team 1 skips)
          // S^T for the tile's 4 key groups of 16: A = K rows 16 kt4 + r, dims 32 ks + 8g.
          op ka[4][2];
#pragma unroll
          for (int kt4 = 0; kt4 < 4; ++kt4) {
            const int row = 16 * kt4 + r;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
              ka[kt4][ks] = *reinterpret_cast<const op*>(kt + row * 128 +
                                                         16 * ((4 * ks + g) ^ ((row >> 1) & 7)));
          }
          // The accumulators start at -mref (the row's reference max, 0 before any
          // visible key), so the products come out as s - mref directly.
          f32x4 s[kHeadsPerWave][4];
#pragma unroll
          for (int kt4 = 0; kt4 < 4; ++kt4)
#pragma unroll
            for (int hh = 0; hh < kHeadsPerWave; ++hh) {
              f32x4 acc = nref[hh];
#pragma unroll
              for (int ks = 0; ks < 2; ++ks) {
                acc = M::mma(ka[kt4][ks], qhi[hh][ks], acc);
                if constexpr (kSplit) acc = M::mma(ka[kt4][ks], qlo[hh][ks], acc);
              }
              s[hh][kt4] = acc;
            }
          // Causal mask (and masked pages) where the tile is not entirely visible.
          if (kbase + kKeys - 1 > min_pos || okb != 15) {
#pragma unroll
            for (int kt4 = 0; kt4 < 4; ++kt4)
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                const int kp = kbase + 16 * kt4 + 4 * g + e;
                const bool vis = kp <= rp && ((okb >> kt4) & 1);
#pragma unroll
                for (int hh = 0; hh < kHeadsPerWave; ++hh)
                  s[hh][kt4][e] = vis ? s[hh][kt4][e] : -INFINITY;
              }
          }
          // Online softmax per head on s - mref; P^T operands per 32-key group kg:
          // slots 0-3 = keys 32kg + 4g + e (group 2kg), slots 4-7 = keys 32kg + 16 +
          // 4g + e. The reference max mref is raised lazily: weights are 2^(s - mref)
          // with mref the row's max when it was last raised, and O and l are rescaled
          // only when the reference has to move.
          //   Until every row of the wave has a reference (its first visible tile),
          //   each tile's max is taken and the reference raised when a row's max
          //   passes mref + kLazyMax (weights then <= 2^kLazyMax).
          //   After that (single-rounded f16 operands; split hi + lo operands take
          //   the max on every tile) a tile's weights are formed against the standing reference
          //   without a max, and the tile's row sums (from the matrix cores, from the
          //   same rounded operands as O) tell whether it may: while every row's sum
          //   is <= kSumMax, so is every weight -- in range for f16, whose largest
          //   value is 65504, and at a magnitude where rounding is relative, as it
          //   is at any normal magnitude. A larger sum (or an f16 weight rounded to
          //   inf) sends the tile through the max and the raise above, and its
          //   weights are formed again. The row sums l come from the matrix cores.
          op phi[kHeadsPerWave][2], plo[kHeadsPerWave][2];
#pragma unroll
          for (int hh = 0; hh < kHeadsPerWave; ++hh) {
            auto raise = [&]() {
              settle(s[hh]);
              const f32x4(&sh)[4] = s[hh];
              float mx = max_nn(max3_nn(max3_nn(sh[0][0], sh[0][1], sh[0][2]),
                                        max3_nn(sh[0][3], sh[1][0], sh[1][1]),
                                        max3_nn(sh[1][2], sh[1][3], sh[2][0])),
                                max3_nn(max3_nn(sh[2][1], sh[2][2], sh[2][3]),
                                        max3_nn(sh[3][0], sh[3][1], sh[3][2]), sh[3][3]));
              mx = group_max4(mx);  // the tile's row max, relative to mref
              // m = -inf (nothing visible yet) always counts as growth when mx is finite.
              const bool grow = mx > (m[hh] == -INFINITY ? -INFINITY : kLazyMax);
              if (__builtin_amdgcn_ballot_w64(grow) != 0) {
                const float mref = -nref[hh][0];
                const float m_new = fmaxf(m[hh], mref + mx);
                // m = -inf (nothing seen yet): the old terms are all zero
                const float corr = m_new == -INFINITY ? 1.0f : exp2_weight(m[hh] - m_new);
                lsum[hh] *= corr;
#pragma unroll
                for (int mt = 0; mt < 4; ++mt) o[hh][mt] *= corr;
                m[hh] = m_new;
                // Re-reference this tile's scores to the new max.
                const float ref = m_new == -INFINITY ? 0.0f : m_new;
                const float shift = ref - mref;
#pragma unroll
                for (int kt4 = 0; kt4 < 4; ++kt4) s[hh][kt4] -= shift;
                nref[hh] = f32x4{-ref, -ref, -ref, -ref};
              }
            };
            auto weights = [&]() {
#pragma unroll
              for (int kg = 0; kg < 2; ++kg)
#pragma unroll
                for (int e = 0; e < 4; e += 2) {
                  const float pa0 = exp2_weight(s[hh][2 * kg][e]);
                  const float pa1 = exp2_weight(s[hh][2 * kg][e + 1]);
                  const float pb0 = exp2_weight(s[hh][2 * kg + 1][e]);
                  const float pb1 = exp2_weight(s[hh][2 * kg + 1][e + 1]);
                  E h0, h1, l0, l1;
                  if constexpr (kSplit) {
                    split16x2(pa0, pa1, h0, h1, l0, l1);
                    plo[hh][kg][e] = l0;
                    plo[hh][kg][e + 1] = l1;
                  } else {
                    round16x2(pa0, pa1, h0, h1);
                  }
                  phi[hh][kg][e] = h0;
                  phi[hh][kg][e + 1] = h1;
                  if constexpr (kSplit) {
                    split16x2(pb0, pb1, h0, h1, l0, l1);
                    plo[hh][kg][4 + e] = l0;
                    plo[hh][kg][5 + e] = l1;
                  } else {
                    round16x2(pb0, pb1, h0, h1);
                  }
                  phi[hh][kg][4 + e] = h0;
                  phi[hh][kg][5 + e] = h1;
                }
            };
            // The tile's row sums: an all-ones A operand against P^T puts sum_k P[r][k]
            // of the tile's keys in every entry of lane r's accumulator.
            auto row_sum = [&]() {
              f32x4 tl = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int kg = 0; kg < 2; ++kg) {
                tl = M::mma(ones, phi[hh][kg], tl);
                if constexpr (kSplit) tl = M::mma(ones, plo[hh][kg], tl);
              }
              return tl[0];
            };
            if constexpr (kSplit) {
              // hi + lo operands: twice the weight registers, no room for a second
              // formation; every tile takes the max.
              raise();
              weights();
              lsum[hh] += row_sum();
            } else {
              const bool fresh = __builtin_amdgcn_ballot_w64(m[hh] == -INFINITY) != 0;
              if (fresh) raise();
              weights();
              float tl = row_sum();
              if (!fresh && __builtin_amdgcn_ballot_w64(!(tl <= kSumMax)) != 0) {
                raise();
                weights();
                tl = row_sum();
              }
              lsum[hh] += tl;
            }
          }
          // O^T += V^T P^T. Lane L reads tile row 32kg + 4g + L/4 (and +16), dims
          // 16 mt + 4 (L%4) .. +3: after the transpose lane r holds dim 16 mt + r of
          // keys 32kg + 4g + e and 32kg + 16 + 4g + e -- P^T's slots.
          const int rbyte = (r & 1) * 8;
#pragma unroll
          for (int kg = 0; kg < 2; ++kg) {
            const int vrow = 32 * kg + 4 * g + (r >> 2);
            const int sw = 2 * ((vrow >> 1) & 3);  // same for vrow + 16
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
              const int slot = (2 * mt + ((r >> 1) & 1)) ^ sw;
              const s16x4 lo4 = lds_read_tr16(vt + vrow * 128 + slot * 16 + rbyte);
              const s16x4 hi4 = lds_read_tr16(vt + (vrow + 16) * 128 + slot * 16 + rbyte);
              const op a = join_tr<op>(lo4, hi4);
#pragma unroll
              for (int hh = 0; hh < kHeadsPerWave; ++hh) {
                o[hh][mt] = M::mma(a, phi[hh][kg], o[hh][mt]);
                if constexpr (kSplit) o[hh][mt] = M::mma(a, plo[hh][kg], o[hh][mt]);
              }
            }
          }
        }
        // This wave's loads of step s + 1 have landed (later steps may still be in
        // flight); after the barrier every wave's have, and every wave is done
        // with step s's buffers.
        wait_steps(max(0, min(kRingSteps - 2, n_steps - st - 2)));
        __syncthreads();
      }
      seg0 += kSegTiles;
      if (seg0 >= n_tiles) break;
      stage();
    }

    // Teams 1.. hand their (m, l, O) to team 0 through LDS (the ring is idle:
    // every load has landed and every tile was consumed before the last barrier).
    // Lane L of a head's waves holds the same rows and dims in every team.
    float* xo = reinterpret_cast<float*>(smem);                       // [kWaves][4][64] f32x4
    float* xml = reinterpret_cast<float*>(smem + kWaves * 4096);      // [kWaves][64] float2
    if constexpr (kTeams > 1) {
#pragma unroll
      for (int tm = 1; tm < kTeams; ++tm) {
        if (team == tm) {
#pragma unroll
          for (int mt = 0; mt < 4; ++mt)
            *reinterpret_cast<f32x4*>(xo + ((wave * 4 + mt) * 64 + lane) * 4) = o[0][mt];
          *reinterpret_cast<float2*>(xml + (wave * 64 + lane) * 2) = make_float2(m[0], lsum[0]);
        }
        __syncthreads();
        if (team == 0) {
          const float2 ml = *reinterpret_cast<const float2*>(xml + (wave * 64 + lane) * 2);
          const float m_new = fmaxf(m[0], ml.x);
          const float c0 = m[0] == -INFINITY ? 0.0f : exp2_weight(m[0] - m_new);
          const float c1 = ml.x == -INFINITY ? 0.0f : exp2_weight(ml.x - m_new);
          lsum[0] = lsum[0] * c0 + ml.y * c1;
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) {
            const f32x4 o1 = *reinterpret_cast<const f32x4*>(xo + ((wave * 4 + mt) * 64 + lane) * 4);
            o[0][mt] = o[0][mt] * c0 + o1 * c1;
          }
          m[0] = m_new;
        }
        __syncthreads();  // the exchange area is free again (next team or next pass)
      }
    }

    if (team == 0 && row_ok) {
#pragma unroll
      for (int hh = 0; hh < kHeadsPerWave; ++hh) {
        if (hh >= nh) break;
        const float il = 1.0f / lsum[hh];
        float* dst = out + (size_t(t) * n_heads + h0 + hh) * 64 + 4 * g;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) *reinterpret_cast<f32x4*>(dst + 16 * mt) = o[hh][mt] * il;
      }
    }
  }
}

// LDS of the kernel: the ring of steps (which also holds the team exchange
// area), then the page ids of one segment of key tiles.
template <int kTeams>
constexpr int prefill_lds_bytes() {
  return (kTeams == 1 ? 4 : 3) * kTeams * kBufBytes + 16 * (kSegTiles + kTeams) +
         4 * kSegTiles + kRows * kRopeStride * 4;
}

template <int KV, int W, int kTeams, bool kSplitF16>
int launch_prefill_split(const dim3 grid, float* out, const float* q, const uint16_t* kp,
                         const uint16_t* vp, int T, const int32_t* row_pos,
                         const int32_t* row_seq, const ie_kv_layout& kv, int n_heads,
                         int n_kv_heads, int n_blocks, const PrefillRope& rope,
                         hipStream_t stream) {
  constexpr int lds = prefill_lds_bytes<kTeams>();
  static_assert(lds - 16 * (kSegTiles + kTeams) - 4 * kSegTiles - kRows * kRopeStride * 4 >=
                    W * 4096 + W * 512,
                "team exchange area must fit in the ring");
  if (lds > 65536) {  // above the default dynamic-LDS cap, within gfx950's 160 KB
    static const hipError_t attr = hipFuncSetAttribute(
        reinterpret_cast<const void*>(prefill_mfma_kernel<KV, W, kTeams, kSplitF16>),
        hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    if (int rc = check_hip(attr, "hipFuncSetAttribute(attention_prefill_mfma)")) return rc;
  }
  hipLaunchKernelGGL((prefill_mfma_kernel<KV, W, kTeams, kSplitF16>), grid,
                     dim3(64 * W * kTeams), lds, stream, out, q, kp, vp, T, row_pos, row_seq,
                     kv.tables, kv.max_pages, kv.num_pages, n_heads, n_kv_heads, n_blocks,
                     rope.table, rope.positions);
  return check_launch("attention_prefill_mfma");
}

// f16 caches take q and P as single f16 values unless the process asked for the
// split operands (ie_hip_set_prefill_rounding); bf16 caches always split.
template <int KV, int W, int kTeams>
int launch_prefill_variant(const dim3 grid, float* out, const float* q, const uint16_t* kp,
                           const uint16_t* vp, int T, const int32_t* row_pos,
                           const int32_t* row_seq, const ie_kv_layout& kv, int n_heads,
                           int n_kv_heads, int n_blocks, const PrefillRope& rope,
                           hipStream_t stream) {
  if (KV == IE_KV_F16 && prefill_rounding() == IE_HIP_PREFILL_SPLIT)
    return launch_prefill_split<KV, W, kTeams, true>(grid, out, q, kp, vp, T, row_pos, row_seq,
                                                     kv, n_heads, n_kv_heads, n_blocks, rope,
                                                     stream);
  return launch_prefill_split<KV, W, kTeams, false>(grid, out, q, kp, vp, T, row_pos, row_seq,
                                                    kv, n_heads, n_kv_heads, n_blocks, rope,
                                                    stream);
}

// The work of workgroup blockIdx.x in the kernels with a workgroup per row block and query
// head. Workgroups go to the 8 XCDs in turn; where the KV heads divide 8, an XCD takes one KV
// head's work only, so its L2 holds that head's K and V.
__device__ __forceinline__ void unit_of_block(int n_kv_heads, int& kvh, int& unit) {
  const int b = blockIdx.x;
  if (8 % n_kv_heads == 0) {
    kvh = (b & 7) % n_kv_heads;
    unit = (b >> 3) * (8 / n_kv_heads) + (b & 7) / n_kv_heads;
  } else {
    kvh = b % n_kv_heads;
    unit = b / n_kv_heads;
  }
}

// Workgroups for n_units row blocks; -1 where the launch's size would not fit 32 bits.
inline int64_t unit_grid(int64_t n_units, int n_heads, int n_kv_heads, int threads) {
  const int64_t per_head = n_units * (n_heads / n_kv_heads);
  const int spread = 8 % n_kv_heads == 0 ? 8 / n_kv_heads : 1;
  const int64_t grid = 8 % n_kv_heads == 0 ? 8 * ((per_head + spread - 1) / spread)
                                           : per_head * n_kv_heads;
  return grid * threads > int64_t(UINT32_MAX) ? -1 : grid;
}

// The waves' (o, m, l) through LDS (their stages are idle: no DMA is left in flight) and the
// output: wave w < 4 finishes row r's dims 16g + 4w .. +3. l is the row's whole sum, in every
// lane; o[b][mt][t] is dim 16g + 4t + mt. after(b, w, x, dst) follows dims
// 16g + 4w .. of block b's result x into `out`.
// n_tiles == 1: only wave 0 took keys, and writes its own result (32/8 heads, 2 rows: 5.7 us
// through the merge, 4.7, by pairs 5.3). The f32 kernel has no registers to spare for that and
// gives kTeams.
template <int NB, int kTeams, typename After>
__device__ __forceinline__ void merge_teams(unsigned char* smem, float* out, const f32x4 (&o)[NB][4],
                                            const float (&m)[NB], const float (&l)[NB], int t0,
                                            int T, int n_heads, int head, int lane, int wave,
                                            int n_tiles, After after) {
  const int g = lane >> 4, r = lane & 15;
  if (n_tiles == 1) {  // wave 0 has it all
    if (wave > 0) return;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      const int t = t0 + 16 * b + r;
      f32x4* const dst = reinterpret_cast<f32x4*>(out + (size_t(t) * n_heads + head) * 64 + 16 * g);
      const float il = 1.0f / l[b];
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const f32x4 x = f32x4{o[b][0][w], o[b][1][w], o[b][2][w], o[b][3][w]} * il;
        if (t < T) dst[w] = x;
        after(b, w, x, dst + w);
      }
    }
    return;
  }
  __syncthreads();
  f32x4* const xo = reinterpret_cast<f32x4*>(smem);                          // [wave][b][t][lane]
  float2* const xml = reinterpret_cast<float2*>(smem + kTeams * NB * 4096);  // [wave][b][lane]
#pragma unroll
  for (int b = 0; b < NB; ++b) {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      xo[((wave * NB + b) * 4 + t) * 64 + lane] = f32x4{o[b][0][t], o[b][1][t], o[b][2][t], o[b][3][t]};
    xml[(wave * NB + b) * 64 + lane] = make_float2(m[b], l[b]);
  }
  __syncthreads();
  if (wave >= 4) return;
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    float2 ml[kTeams];
    float top = -INFINITY;
#pragma unroll
    for (int w = 0; w < kTeams; ++w) {
      ml[w] = xml[(w * NB + b) * 64 + lane];
      top = fmaxf(top, ml[w].x);
    }
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    float total = 0.0f;
#pragma unroll
    for (int w = 0; w < kTeams; ++w) {
      const float c = ml[w].x == -INFINITY ? 0.0f : exp2_weight(ml[w].x - top);
      total += ml[w].y * c;
      sum += xo[((w * NB + b) * 4 + wave) * 64 + lane] * c;
    }
    const int t = t0 + 16 * b + r;
    f32x4* const dst =
        reinterpret_cast<f32x4*>(out + (size_t(t) * n_heads + head) * 64 + 16 * g + 4 * wave);
    const f32x4 x = sum * (1.0f / total);
    if (t < T) *dst = x;
    after(b, wave, x, dst);
  }
}

// A block's 16 rows over all their keys with whole float32 operands, on the f32 matrix
// instruction: for what a row-block kernel's own operands got wrong, by one wave for dims
// 16g + 4 part + e of row r. qv: row r's query times log2(e)/8, [8 ks + j] dim 32 ks + 8g + j.
// Keys up to `pos` are row r's, up to `last` the block's (V rows past it are taken as zeros).
template <typename E, typename Page>
__device__ __forceinline__ f32x4 rows_in_f32(const float (&qv)[16], const char* k_base,
                                             const char* v_base, size_t page_bytes,
                                             unsigned row_bytes, Page page, int pos, int last,
                                             int lane, int part) {
  const int g = lane >> 4, r = lane & 15;
  float top = -INFINITY, total = 0.0f;  // running max, this lane's part of the sum
  f32x4 x = {0.f, 0.f, 0.f, 0.f};
#pragma nounroll
  for (int u = 0; 16 * u <= last; ++u) {
    const int id = page(u);
    if (id < 0) continue;
    const size_t at = size_t(id) * page_bytes;
    const E* krow = reinterpret_cast<const E*>(k_base + at + r * row_bytes) + 8 * g;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 16; ++i)  // step i: dim 32 (i/8) + 8g + i%8 of key r
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(static_cast<float>(krow[32 * (i >> 3) + (i & 7)]), qv[i],
                                               s, 0, 0, 0);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (16 * u + 4 * g + e > pos) s[e] = -INFINITY;
    const float was = top;
    top = fmaxf(top, group_max4(fmaxf(fmaxf(s[0], s[1]), fmaxf(s[2], s[3]))));
    if (top != -INFINITY) {
      const float corr = exp2_weight(was - top);
      total *= corr;
      x *= corr;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {  // step e: key 4g + e, row r of the tile dim 16 (r/4) + 4 part + r%4
      const float w = top == -INFINITY ? 0.0f : exp2_weight(s[e] - top);
      total += w;
      const E* vrow = reinterpret_cast<const E*>(v_base + at + (4 * g + e) * row_bytes);
      const float v = 16 * u + 4 * g + e <= last
                          ? static_cast<float>(vrow[16 * (r >> 2) + 4 * part + (r & 3)]) : 0.0f;
      x = __builtin_amdgcn_mfma_f32_16x16x4f32(v, w, x, 0, 0, 0);
    }
  }
  return x * (1.0f / group_sum4(total));
}

// ---------------------------------------------------------------------------
// 16-bit caches again, one workgroup per (NB blocks of 16 rows, query head) instead of per
// (pair of blocks, KV head): its waves take tiles of 16 KT keys in turn, each with its own K
// stage, softmax state and output, merged through LDS at the end, as in the f32 kernel below.
// No wave waits for another inside the key loop, and T / 16 / NB x heads workgroups fill the
// chip where pairs of blocks x KV heads leave most of it idle. Every wave brings its own K and
// V (prefill_mfma_kernel's 7 waves share theirs), so long prompts are bound by what a
// compute unit can take in (4,000 rows: 68 us here, 54 there) and stay there; see
// choose_prefill for the line.
//   S^T and the softmax as in prefill_mfma_kernel (same operands, rounding and row sums).
//   O^T[64 dims x 16 rows] += V^T . P^T: row i of tile mt is dim 4i + mt, so lane (g, r)'s
//     A operand is dim 4r + mt of keys 4g + e of a page pair, and its 8-byte loads of V
//     (16 lanes a whole 128-byte row) hold all four tiles' values: V comes straight from
//     memory into registers, sent for before the scores, and is packed by 4 byte permutes a
//     tile. Lane (g, r) ends up with row r's dims 16g + 4t + mt (o[mt][t]).
template <int KV, int NB, int KT, int kTeams, bool kSplit>
__global__ void __launch_bounds__(64 * kTeams)
prefill_rows_kernel(float* __restrict__ out, const float* __restrict__ q,
                    const uint16_t* __restrict__ k_pool, const uint16_t* __restrict__ v_pool, int T,
                    const int32_t* __restrict__ row_pos, const int32_t* __restrict__ row_seq,
                    const int32_t* __restrict__ tables, int max_pages, int num_pages, int n_heads,
                    int n_kv_heads, int n_units, const float* __restrict__ rope,
                    int rope_positions) {
  using M = Mfma<KV>;
  using op = typename M::op;
  using E = typename M::elem;
  static_assert(kSplit || std::is_same_v<E, _Float16>, "bf16 operands are split");
  constexpr int kTileKeys = 16 * KT, kStage = kTileKeys * 128;
  static_assert(KT % 2 == 0, "products over V take pages in pairs");
  constexpr int kMerge = kTeams * NB * (4 * 1024 + 512);
  __shared__ __align__(16) unsigned char smem[kTeams * kStage > kMerge ? kTeams * kStage : kMerge];
  op ones;
#pragma unroll
  for (int i = 0; i < 8; ++i) ones[i] = static_cast<E>(1.0f);
  const int group = n_heads / n_kv_heads;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  int kvh, unit;
  unit_of_block(n_kv_heads, kvh, unit);
  if (unit >= n_units * group) return;
  const int block = n_units - 1 - unit / group;  // longest contexts first
  const int head = kvh * group + unit % group;
  const int pos0 = __builtin_amdgcn_readfirstlane(row_pos[0]);
  const int seq = __builtin_amdgcn_readfirstlane(row_seq[0]);
  const int32_t* tab = tables + size_t(seq) * max_pages;
  const int t0 = block * 16 * NB;
  const int max_pos = pos0 + min(t0 + 16 * NB, T) - 1;
  const int min_pos = pos0 + t0;
  const int n_tiles = max_pos / kTileKeys + 1;

  // Page ids of a tile, -1 past the table row or outside the pool.
  auto page = [&](int at) {
    const int id = at < max_pages ? tab[at] : -1;
    return __builtin_amdgcn_readfirstlane(id >= 0 && id < num_pages ? id : -1);
  };
  // DMA of a tile's K rows, two loads a page: load h moves rows 8h .. 8h+7, lane l row
  // 8h + l/8, LDS slot l % 8, holding piece slot ^ (row/2 % 8).
  const unsigned row_bytes = unsigned(n_kv_heads) * 128;
  const size_t page_bytes = size_t(IE_HIP_PAGE_SIZE) * row_bytes;
  const char* const kbase_g = reinterpret_cast<const char*>(k_pool) + kvh * 128;
  const char* const vbase_g = reinterpret_cast<const char*>(v_pool) + kvh * 128;
  unsigned char* const stage = smem + wave * kStage;
  const unsigned stage_lds = lds_address(stage);
  unsigned koff[2], voff[4];
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int row = 8 * h + (lane >> 3);
    koff[h] = row * row_bytes + 16 * ((lane & 7) ^ ((row >> 1) & 7));
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) voff[e] = (4 * g + e) * row_bytes + 8 * r;
  auto issue_k = [&](const int (&id)[KT]) {
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) {
      const char* base = kbase_g + size_t(max(id[kt], 0)) * page_bytes;
      dma16_at(base, koff[0], stage_lds + kt * 2048);
      dma16_at(base, koff[1], stage_lds + kt * 2048 + 1024);
    }
  };
  int id[KT];
#pragma unroll
  for (int kt = 0; kt < KT; ++kt) id[kt] = wave < n_tiles ? page(KT * wave + kt) : -1;
  if (wave < n_tiles) issue_k(id);

  // Row r's query of each block, times log2(e)/8: the B operands of S^T (dims 32 ks + 8g ..
  // +7), rotated here when a RoPE table is given (the arithmetic of ie_hip_rope_and_cache;
  // rows outside the table as they are).
  auto query = [&](int b, float (&x)[2][8]) {
    const int t = t0 + 16 * b + r;
    const bool row_ok = t < T;
    const float4* src = reinterpret_cast<const float4*>(
        q + (size_t(row_ok ? t : t0) * n_heads + head) * 64 + 8 * g);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const float4 a = src[8 * ks], c = src[8 * ks + 1];
      const float v[8] = {a.x, a.y, a.z, a.w, c.x, c.y, c.z, c.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) x[ks][j] = row_ok ? v[j] : 0.0f;
    }
    const int rp = pos0 + t;
    if (rope) {
      const bool rot = row_ok && rp >= 0 && rp < rope_positions;
      const float4* trow = reinterpret_cast<const float4*>(rope + size_t(rot ? rp : 0) * 64 + 8 * g);
      const float4 c0 = trow[0], c1 = trow[1], s0 = trow[8], s1 = trow[9];
      const float cs[8] = {c0.x, c0.y, c0.z, c0.w, c1.x, c1.y, c1.z, c1.w};
      const float sn[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float x0 = x[0][j], x1 = x[1][j];
        const float r0 = __builtin_fmaf(x0, cs[j], -(x1 * sn[j]));  // x0*c - x1*s
        const float r1 = __builtin_fmaf(x1, cs[j], x0 * sn[j]);     // x1*c + x0*s
        x[0][j] = rot ? r0 : x0;
        x[1][j] = rot ? r1 : x1;
      }
    }
  };
  op qhi[NB][2], qlo[NB][2];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    float x[2][8];
    query(b, x);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        E hv, lv = static_cast<E>(0.0f);
        if constexpr (kSplit) {
          split16(x[ks][j] * (0.125f * kLog2e), hv, lv);
        } else {
          float xq = x[ks][j] * (0.125f * kLog2e);  // the float32 product, then its f16 rounding
          asm("" : "+v"(xq));
          hv = static_cast<E>(xq);
        }
        qhi[b][ks][j] = hv;
        qlo[b][ks][j] = lv;
      }
  }

  float m[NB], lsum[NB], nref[NB];  // nref: -(the reference max, 0 while m = -inf)
  f32x4 o[NB][4];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    m[b] = -INFINITY;
    lsum[b] = nref[b] = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) o[b][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  for (int tile = wave; tile < n_tiles; tile += kTeams) {
    const int kbase = tile * kTileKeys;
    const bool more = tile + kTeams < n_tiles;
    int next[KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) next[kt] = more ? page(KT * (tile + kTeams) + kt) : -1;
    wait_vmcnt<0>();  // the tile's K rows have landed
    op ka[KT][2];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
        ka[kt][ks] = *reinterpret_cast<const op*>(stage + (16 * kt + r) * 128 +
                                                  16 * ((4 * ks + g) ^ ((r >> 1) & 7)));
    if (more) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage's reads are done
      issue_k(next);
    }
    uint2 v[KT][4];  // key 16 kt + 4g + e, dims 4r .. 4r+3
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[kt][e] = *reinterpret_cast<const uint2*>(
            vbase_g + size_t(max(id[kt], 0)) * page_bytes + voff[e]);

    f32x4 s[NB][KT];
#pragma unroll
    for (int kt = 0; kt < KT; ++kt)
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        f32x4 acc = {nref[b], nref[b], nref[b], nref[b]};
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
          acc = M::mma(ka[kt][ks], qhi[b][ks], acc);
          if constexpr (kSplit) acc = M::mma(ka[kt][ks], qlo[b][ks], acc);
        }
        s[b][kt] = acc;
      }
#pragma unroll
    for (int b = 0; b < NB; ++b) settle(s[b]);
    int all = 0;
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) all |= id[kt];
    if (kbase + kTileKeys - 1 > min_pos || all < 0) {
#pragma unroll
      for (int kt = 0; kt < KT; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int kp = kbase + 16 * kt + 4 * g + e;
#pragma unroll
          for (int b = 0; b < NB; ++b)
            s[b][kt][e] = id[kt] >= 0 && kp <= pos0 + t0 + 16 * b + r ? s[b][kt][e] : -INFINITY;
          if (id[kt] < 0 || kp > max_pos) v[kt][e] = make_uint2(0, 0);
        }
    }
    // The softmax of prefill_mfma_kernel: lazily raised reference, row sums on the matrix
    // cores from the rounded weights, the max taken only until every row has a reference
    // (single-rounded f16) or on every tile (hi + lo).
    op phi[NB][KT / 2], plo[NB][KT / 2];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      auto raise = [&]() {
        float mx = max_nn(max_nn(s[b][0][0], s[b][0][1]), max_nn(s[b][0][2], s[b][0][3]));
#pragma unroll
        for (int kt = 1; kt < KT; ++kt)
          mx = max3_nn(mx, max_nn(s[b][kt][0], s[b][kt][1]), max_nn(s[b][kt][2], s[b][kt][3]));
        mx = group_max4(mx);
        const bool grow = mx > (m[b] == -INFINITY ? -INFINITY : kLazyMax);
        if (__builtin_amdgcn_ballot_w64(grow) != 0) {
          const float mref = -nref[b];
          const float m_new = fmaxf(m[b], mref + mx);
          const float corr = m_new == -INFINITY ? 1.0f : exp2_weight(m[b] - m_new);
          lsum[b] *= corr;
#pragma unroll
          for (int mt = 0; mt < 4; ++mt) o[b][mt] *= corr;
          m[b] = m_new;
          const float ref = m_new == -INFINITY ? 0.0f : m_new;
          const float shift = ref - mref;
#pragma unroll
          for (int kt = 0; kt < KT; ++kt) s[b][kt] -= shift;
          nref[b] = -ref;
        }
      };
      auto weights = [&]() {
#pragma unroll
        for (int kg = 0; kg < KT / 2; ++kg)
#pragma unroll
          for (int e = 0; e < 8; e += 2) {
            const f32x4& sv = s[b][2 * kg + (e >> 2)];
            const float p0 = exp2_weight(sv[e & 3]), p1 = exp2_weight(sv[(e & 3) + 1]);
            E h0, h1, l0, l1;
            if constexpr (kSplit) {
              split16x2(p0, p1, h0, h1, l0, l1);
              plo[b][kg][e] = l0;
              plo[b][kg][e + 1] = l1;
            } else {
              round16x2(p0, p1, h0, h1);
            }
            phi[b][kg][e] = h0;
            phi[b][kg][e + 1] = h1;
          }
      };
      auto row_sum = [&]() {
        f32x4 tl[1] = {{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int kg = 0; kg < KT / 2; ++kg) {
          tl[0] = M::mma(ones, phi[b][kg], tl[0]);
          if constexpr (kSplit) tl[0] = M::mma(ones, plo[b][kg], tl[0]);
        }
        // All four parts stay taken until the matrix core has written them: the next
        // block's maxima would otherwise be put in the three that are not read.
        settle(tl);
        return tl[0][0];
      };
      if constexpr (kSplit) {
        raise();
        weights();
        lsum[b] += row_sum();
      } else {
        const bool fresh = __builtin_amdgcn_ballot_w64(m[b] == -INFINITY) != 0;
        if (fresh) raise();
        weights();
        float tl = row_sum();
        if (!fresh && __builtin_amdgcn_ballot_w64(!(tl <= kSumMax)) != 0) {
          raise();
          weights();
          tl = row_sum();
        }
        lsum[b] += tl;
      }
    }
#pragma unroll
    for (int kg = 0; kg < KT / 2; ++kg)
#pragma unroll
      for (int mt = 0; mt < 4; ++mt) {
        typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
        u32x4 a;
#pragma unroll
        for (int j = 0; j < 4; ++j) {  // keys 2j, 2j + 1 of the lane's 8
          const uint2 k0 = v[2 * kg + (j >> 1)][2 * (j & 1)], k1 = v[2 * kg + (j >> 1)][2 * (j & 1) + 1];
          a[j] = __builtin_amdgcn_perm(mt >> 1 ? k1.y : k1.x, mt >> 1 ? k0.y : k0.x,
                                       mt & 1 ? 0x07060302u : 0x05040100u);
        }
        const op av = __builtin_bit_cast(op, a);
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          o[b][mt] = M::mma(av, phi[b][kg], o[b][mt]);
          if constexpr (kSplit) o[b][mt] = M::mma(av, plo[b][kg], o[b][mt]);
        }
      }
#pragma unroll
    for (int kt = 0; kt < KT; ++kt) id[kt] = next[kt];
  }
  // Blocks before the last: their products take in V rows of the later blocks' positions, with
  // weight 0, which passes infinities and NaN on. A wave that has written such an output of a
  // block takes its rows again without them.
  auto redo = [&](int b, int part, f32x4 y, f32x4* dst) {
    if (b == NB - 1) return;
    const int row = t0 + 16 * b + r;
    const bool odd = !(fabsf(y[0]) + fabsf(y[1]) + (fabsf(y[2]) + fabsf(y[3])) < INFINITY);
    if (__builtin_amdgcn_ballot_w64(odd && row < T) == 0) return;
    float x[2][8], qv[16];
    query(b, x);
#pragma unroll
    for (int i = 0; i < 16; ++i) qv[i] = x[i >> 3][i & 7] * (0.125f * kLog2e);
    y = rows_in_f32<E>(qv, kbase_g, vbase_g, page_bytes, row_bytes, page, pos0 + row,
                       min(pos0 + t0 + 16 * b + 15, max_pos), lane, part);
    if (odd && row < T) *dst = y;
  };
  merge_teams<NB, kTeams>(smem, out, o, m, lsum, t0, T, n_heads, head, lane, wave, n_tiles, redo);
}

// ---------------------------------------------------------------------------
// float32 KV caches. Queries, keys, weights and values enter the 16-bit matrix cores in
// three bf16 parts each, x = hi + mid + lo exactly (split3; for what has no such split see
// `redo` at the end), and every product is the six largest of the nine partial ones: what is
// left out is at most about 2^-24 of the product (parts of up to 2^-8 and 2^-17 of a value), a
// float32 rounding of it. The whole is as exact as float32 products: against float64 4.4e-7 at
// 1,333 rows on 1,000 cached, where v_mfma_f32_16x16x4_f32 on the whole values gave 8.0e-7.
// The f32 instruction takes 256 cycles for the 16x16x32 product that six bf16 ones do in 96,
// and the bf16 ones leave the VALU free for the splits and the softmax.
//
// One workgroup per (NB blocks of 16 rows, query head); its waves take 32-key tiles in turn,
// each with its own K stage, softmax state and output, merged through LDS at the end: no
// barrier and no sharing until then, and T / 16 / NB x heads workgroups, the longest
// contexts first, where a workgroup per pair of blocks and KV head left two thirds of the
// compute units idle at 1,333 rows. What bounds it now: a tile's K and V take 352 VALU
// instructions to split, shared by NB blocks and done again by every query head; VALU issue
// takes 50% of the cycles at 1,333 rows on 1,000, the matrix cores 28%, in turn for the most
// part. Times (us, was 7 waves on shared f32 tiles): 1,333 rows on 1,000 cached 237 -> 72,
// 4,000 rows 281 -> 193, 130 rows on 4,000 cached 548 -> 44.
//   S^T[16 keys x 16 rows] per key group of 16: step ks takes dims 16g + 8ks .. +7, so lane
//     (g, r) reads key r's dims 16g .. 16g+15 (64 bytes, 4 LDS reads).
//   O^T[64 dims x 16 rows] += V^T . P^T: one step of 32 keys; lane (g, r)'s B operand is its
//     own 8 weights, keys 16 kt + 4g + e; row i of tile mt is dim 4i + mt, so its A operand
//     is one component of the 16-byte pieces r of those keys' V rows: 16 lanes read a whole
//     256-byte row, so V comes straight from memory into registers, sent for before the
//     scores and used after the softmax. Lane (g, r) ends up with row r's dims
//     16g + 4t + mt (o[mt][t]).
// K tiles (8 KB) come through LDS by DMA, one stage per wave: read whole into registers,
// then the next tile is sent for. K loads take a scalar page base and a 32-bit lane offset, V
// loads a 64-bit lane address made from the two (both from 64-bit lane pointers: 1,000 rows
// 30.6 -> 29.5 us, 4,000 rows 198 -> 193). Four waves a SIMD with one block need its registers
// at 128, as asked for; three with two blocks spill (1,000 rows 30.6, 4,000 rows 189: not
// kept); three or four blocks hold so many registers that too few waves are left (4,000 rows
// 242 and 236 us). K rows are stored with their 16-byte pieces swizzled (piece ^ (key & 15)),
// so the 16 lanes of a group reading the same dims of 16 keys hit distinct banks.
constexpr int kKeysF32 = 32;                      // keys per wave tile (2 pages)
constexpr int kStageF32 = kKeysF32 * 64 * 4;      // 8 KB of K
// The six products of two operands in three parts (0 the largest), the smallest first.
__device__ constexpr int kPartA[6] = {2, 0, 1, 1, 0, 0};
__device__ constexpr int kPartB[6] = {0, 2, 1, 0, 1, 0};

template <int NB, int kTeams>
__global__ void __launch_bounds__(64 * kTeams)
__attribute__((amdgpu_waves_per_eu(NB == 1 ? 4 : 2)))
prefill_mfma_f32_kernel(float* __restrict__ out, const float* __restrict__ q,
                        const float* __restrict__ k_pool, const float* __restrict__ v_pool, int T,
                        const int32_t* __restrict__ row_pos, const int32_t* __restrict__ row_seq,
                        const int32_t* __restrict__ tables, int max_pages, int num_pages,
                        int n_heads, int n_kv_heads, int n_units) {
  // The K stages; at the end each wave's (o, m, l).
  constexpr int kMergeF32 = kTeams * NB * (4 * 1024 + 512);
  __shared__ __align__(16) unsigned char smem[kTeams * kStageF32 > kMergeF32
                                                  ? kTeams * kStageF32 : kMergeF32];
  const int group = n_heads / n_kv_heads;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  int kvh, unit;
  unit_of_block(n_kv_heads, kvh, unit);
  if (unit >= n_units * group) return;
  const int block = n_units - 1 - unit / group;  // longest contexts first
  const int head = kvh * group + unit % group;
  const int pos0 = __builtin_amdgcn_readfirstlane(row_pos[0]);
  const int seq = __builtin_amdgcn_readfirstlane(row_seq[0]);
  const int32_t* tab = tables + size_t(seq) * max_pages;
  const int t0 = block * 16 * NB;
  const int max_pos = pos0 + min(t0 + 16 * NB, T) - 1;  // last position any row sees
  const int min_pos = pos0 + t0;
  const int n_tiles = max_pos / kKeysF32 + 1;

  // Row r's query of each block, times log2(e)/8, in three parts: B of the scores' step ks is
  // dims 16g + 8ks .. +7.
  bf16x8 qp[NB][2][3];
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    const int t = t0 + 16 * b + r;
    const float4* src =
        reinterpret_cast<const float4*>(q + (size_t(t < T ? t : t0) * n_heads + head) * 64 + 16 * g);
    const float qs = t < T ? 0.125f * kLog2e : 0.0f;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const float4 x = src[2 * ks], y = src[2 * ks + 1];
      split3(make_float4(x.x * qs, x.y * qs, x.z * qs, x.w * qs),
             make_float4(y.x * qs, y.y * qs, y.z * qs, y.w * qs), qp[b][ks][0], qp[b][ks][1],
             qp[b][ks][2]);
    }
  }

  // Page ids of a tile, -1 past the table row or outside the pool.
  auto page = [&](int at) {
    const int id = at < max_pages ? tab[at] : -1;
    return __builtin_amdgcn_readfirstlane(id >= 0 && id < num_pages ? id : -1);
  };
  // DMA of a tile's K rows: load u moves keys 4u .. 4u+3, lane l key 4u + l/16, LDS slot
  // l % 16, holding piece slot ^ (key & 15).
  const unsigned row_bytes = unsigned(n_kv_heads) * 256;
  const size_t page_bytes = size_t(IE_HIP_PAGE_SIZE) * row_bytes;
  const char* const kbase_g = reinterpret_cast<const char*>(k_pool) + kvh * 256;
  const char* const vbase_g = reinterpret_cast<const char*>(v_pool) + kvh * 256;
  unsigned char* const stage = smem + wave * kStageF32;
  const unsigned stage_lds = lds_address(stage);
  unsigned koff[4], voff[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int key = 4 * u + g;
    koff[u] = key * row_bytes + 16 * (r ^ key);
    voff[u] = (4 * g + u) * row_bytes + 16 * r;
  }
  auto issue_k = [&](int ida, int idb) {
#pragma unroll
    for (int u = 0; u < 8; ++u)
      dma16_at(kbase_g + size_t(max(u < 4 ? ida : idb, 0)) * page_bytes, koff[u & 3],
               stage_lds + u * 1024);
  };

  float m[NB], l[NB];  // running max (base 2), this lane's part of the sum
  f32x4 o[NB][4];      // o[b][mt][t]: row r of block b, dim 16g + 4t + mt
#pragma unroll
  for (int b = 0; b < NB; ++b) {
    m[b] = -INFINITY;
    l[b] = 0.0f;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) o[b][mt] = f32x4{0.f, 0.f, 0.f, 0.f};
  }

  int id0 = -1, id1 = -1;  // the tile's pages
  if (wave < n_tiles) {
    id0 = page(2 * wave);
    id1 = page(2 * wave + 1);
    issue_k(id0, id1);
  }
  for (int tile = wave; tile < n_tiles; tile += kTeams) {
    const int kbase = tile * kKeysF32;
    const bool more = tile + kTeams < n_tiles;
    int next0 = -1, next1 = -1;
    if (more) {
      next0 = page(2 * (tile + kTeams));
      next1 = page(2 * (tile + kTeams) + 1);
    }
    wait_vmcnt<0>();  // the tile's K rows have landed
    float4 ka[2][4];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        ka[kt][i] = *reinterpret_cast<const float4*>(stage + (16 * kt + r) * 256 +
                                                     16 * ((4 * g + i) ^ r));
    if (more) {
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage's reads are done
      issue_k(next0, next1);
    }
    // V rows of the tile: step (kt, e) is key 16 kt + 4g + e, dims 4r .. 4r+3.
    float4 v[2][4];
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[kt][e] = *reinterpret_cast<const float4*>(
            vbase_g + size_t(max(kt ? id1 : id0, 0)) * page_bytes + voff[e]);

    float mref[NB];
    f32x4 s[NB][2];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      mref[b] = m[b] == -INFINITY ? 0.0f : m[b];
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) s[b][kt] = f32x4{-mref[b], -mref[b], -mref[b], -mref[b]};
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        bf16x8 kp[3];
        split3(ka[kt][2 * ks], ka[kt][2 * ks + 1], kp[0], kp[1], kp[2]);
#pragma unroll
        for (int p = 0; p < 6; ++p)
#pragma unroll
          for (int b = 0; b < NB; ++b)
            s[b][kt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kp[kPartA[p]], qp[b][ks][kPartB[p]],
                                                               s[b][kt], 0, 0, 0);
      }
#pragma unroll
    for (int b = 0; b < NB; ++b) settle(s[b]);
    // Keys a row may not see, or in pages outside the pool: no weight, and V rows that
    // nothing may see zeroed (stale or non-finite memory must not reach O through 0 * x).
    if (kbase + kKeysF32 - 1 > min_pos || (id0 | id1) < 0) {
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const bool ok = (kt ? id1 : id0) >= 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int kp = kbase + 16 * kt + 4 * g + e;
#pragma unroll
          for (int b = 0; b < NB; ++b)
            s[b][kt][e] = ok && kp <= pos0 + t0 + 16 * b + r ? s[b][kt][e] : -INFINITY;
          if (!ok || kp > max_pos) v[kt][e] = make_float4(0.f, 0.f, 0.f, 0.f);
        }
      }
    }
    // Online softmax on s - mref, the reference max raised lazily (as in the
    // 16-bit kernel: O and l rescaled only when a row's max grows past
    // m + kLazyMax somewhere in the wave).
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      float mx = max_nn(max3_nn(s[b][0][0], s[b][0][1], s[b][0][2]),
                        max3_nn(max_nn(s[b][0][3], s[b][1][0]), s[b][1][1],
                                max_nn(s[b][1][2], s[b][1][3])));
      mx = group_max4(mx);
      const bool grow = m[b] == -INFINITY ? mx != -INFINITY : mx > kLazyMax;
      if (__builtin_amdgcn_ballot_w64(grow) != 0) {
        const float m_new = fmaxf(m[b], mref[b] + mx);
        const float corr = m_new == -INFINITY ? 1.0f : exp2_weight(m[b] - m_new);  // m = -inf: 0
        l[b] *= corr;
#pragma unroll
        for (int mt = 0; mt < 4; ++mt) o[b][mt] *= corr;
        m[b] = m_new;
        const float shift = (m_new == -INFINITY ? 0.0f : m_new) - mref[b];
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) s[b][kt] -= shift;
      }
      float sum = 0.0f;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          s[b][kt][e] = exp2_weight(s[b][kt][e]);
          sum += s[b][kt][e];
        }
      l[b] += sum;
    }
    bf16x8 wp[NB][3];  // the weights in three parts: B, keys 16 kt + 4g + e
#pragma unroll
    for (int b = 0; b < NB; ++b)
      split3(make_float4(s[b][0][0], s[b][0][1], s[b][0][2], s[b][0][3]),
             make_float4(s[b][1][0], s[b][1][1], s[b][1][2], s[b][1][3]), wp[b][0], wp[b][1],
             wp[b][2]);
#pragma unroll
    for (int mt = 0; mt < 4; ++mt) {
      auto dim = [&](const float4 x) { return mt == 0 ? x.x : mt == 1 ? x.y : mt == 2 ? x.z : x.w; };
      bf16x8 vp[3];
      split3(make_float4(dim(v[0][0]), dim(v[0][1]), dim(v[0][2]), dim(v[0][3])),
             make_float4(dim(v[1][0]), dim(v[1][1]), dim(v[1][2]), dim(v[1][3])), vp[0], vp[1], vp[2]);
#pragma unroll
      for (int p = 0; p < 6; ++p)
#pragma unroll
        for (int b = 0; b < NB; ++b)
          o[b][mt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vp[kPartA[p]], wp[b][kPartB[p]],
                                                             o[b][mt], 0, 0, 0);
    }
    id0 = next0;
    id1 = next1;
  }

#pragma unroll
  for (int b = 0; b < NB; ++b) l[b] = group_sum4(l[b]);

  // What three bf16 parts cannot hold: infinities, NaN and what rounds to infinity in bf16 (from
  // 3.3962e38 on) make every output that they reach NaN, their last part being one, and
  // outputs all of whose values are below 2^-110 lack the values' low parts. A wave that
  // has written such an output (not finite, or below 2^-100) takes block b's rows over all their
  // keys again with the whole float32 values, on the f32 instruction, for its own 16 dims.
  // (Looked for after the write: no size is slower by more than 2%; every wave looking at its
  // own sums before the merge took 1.4 us more a launch.)
  auto redo = [&](int b, int part, f32x4 x, f32x4* dst) {
    const int row = t0 + 16 * b + r;
    bool odd = false;
#pragma unroll
    for (int e = 0; e < 4; ++e)
      odd |= !(x[e] == 0.0f || (fabsf(x[e]) >= 0x1p-100f && fabsf(x[e]) < INFINITY));
    if (__builtin_amdgcn_ballot_w64(odd && row < T) == 0) return;
    const float* src = q + (size_t(row < T ? row : t0) * n_heads + head) * 64 + 8 * g;
    float qv[16];
#pragma unroll
    for (int i = 0; i < 16; ++i)
      qv[i] = row < T ? src[32 * (i >> 3) + (i & 7)] * (0.125f * kLog2e) : 0.0f;
    x = rows_in_f32<float>(qv, kbase_g, vbase_g, page_bytes, row_bytes, page, pos0 + row,
                           min(pos0 + t0 + 16 * b + 15, max_pos), lane, part);
    if (row < T) *dst = x;
  };
  merge_teams<NB, kTeams>(smem, out, o, m, l, t0, T, n_heads, head, lane, wave, kTeams, redo);
}

template <int NB, int kTeams>
int launch_prefill_f32(float* out, const float* q, const float* kp, const float* vp, int T,
                       const int32_t* row_pos, const int32_t* row_seq, const ie_kv_layout& kv,
                       int n_heads, int n_kv_heads, hipStream_t stream) {
  const int n_units = (T - 1) / (16 * NB) + 1;
  const int64_t grid = unit_grid(n_units, n_heads, n_kv_heads, 64 * kTeams);
  if (grid < 0) return fail(IE_HIP_EINVAL, "attention_prefill: too many rows");
  hipLaunchKernelGGL((prefill_mfma_f32_kernel<NB, kTeams>), dim3(unsigned(grid)),
                     dim3(64 * kTeams), 0, stream, out, q, kp, vp, T, row_pos, row_seq, kv.tables,
                     kv.max_pages, kv.num_pages, n_heads, n_kv_heads, n_units);
  return check_launch("attention_prefill_mfma_f32");
}

template <int KV, int NB, int KT, int kTeams>
int launch_prefill_rows(float* out, const float* q, const uint16_t* kp, const uint16_t* vp, int T,
                        const int32_t* row_pos, const int32_t* row_seq, const ie_kv_layout& kv,
                        int n_heads, int n_kv_heads, const PrefillRope& rope, hipStream_t stream) {
  const int n_units = (T - 1) / (16 * NB) + 1;
  const int64_t grid = unit_grid(n_units, n_heads, n_kv_heads, 64 * kTeams);
  if (grid < 0) return fail(IE_HIP_EINVAL, "attention_prefill: too many rows");
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(unsigned(grid)), dim3(64 * kTeams), 0, stream, out, q, kp, vp, T,
                       row_pos, row_seq, kv.tables, kv.max_pages, kv.num_pages, n_heads, n_kv_heads,
                       n_units, rope.table, rope.positions);
  };
  if (KV == IE_KV_BF16 || prefill_rounding() == IE_HIP_PREFILL_SPLIT)
    go(prefill_rows_kernel<KV, NB, KT, kTeams, true>);
  else if constexpr (KV == IE_KV_F16)
    go(prefill_rows_kernel<KV, NB, KT, kTeams, false>);
  return check_launch("attention_prefill_rows");
}

template <int KV>
int launch_prefill_mfma(float* out, const float* q, const uint16_t* kp, const uint16_t* vp, int T,
                        const int32_t* row_pos, const int32_t* row_seq, const ie_kv_layout& kv,
                        int n_heads, int n_kv_heads, const PrefillRope& rope, hipStream_t stream) {
  const int group = n_heads / n_kv_heads;
  const int waves = (group + kHeadsPerWave - 1) / kHeadsPerWave;
  const int n_blocks = (T + kRows - 1) / kRows;
  const dim3 grid((n_blocks + 1) / 2, n_kv_heads);
  const bool split = KV == IE_KV_BF16 || prefill_rounding() == IE_HIP_PREFILL_SPLIT;
  const PrefillKernel kernel = choose_prefill(T, n_heads, n_kv_heads, split, device_compute_units());
  if (kernel == PrefillKernel::kRows1x8)
    return launch_prefill_rows<KV, 1, 4, 8>(out, q, kp, vp, T, row_pos, row_seq, kv, n_heads,
                                            n_kv_heads, rope, stream);
  if (kernel == PrefillKernel::kRows2x8)
    return launch_prefill_rows<KV, 2, 2, 8>(out, q, kp, vp, T, row_pos, row_seq, kv, n_heads,
                                            n_kv_heads, rope, stream);
  if (kernel == PrefillKernel::kRows2x4)
    return launch_prefill_rows<KV, 2, 4, 4>(out, q, kp, vp, T, row_pos, row_seq, kv, n_heads,
                                            n_kv_heads, rope, stream);
  const bool teams2 = kernel == PrefillKernel::kPairsTwoTeams;
#define IE_PF_CASE(W)                                                                             \
  case W:                                                                                         \
    return teams2 ? launch_prefill_variant<KV, W, 2>(grid, out, q, kp, vp, T, row_pos, row_seq,   \
                                                      kv, n_heads, n_kv_heads, n_blocks, rope,    \
                                                      stream)                                     \
                  : launch_prefill_variant<KV, W, 1>(grid, out, q, kp, vp, T, row_pos, row_seq,   \
                                                      kv, n_heads, n_kv_heads, n_blocks, rope,    \
                                                      stream);
  switch (waves) {
    IE_PF_CASE(1)
    IE_PF_CASE(2)
    IE_PF_CASE(3)
    IE_PF_CASE(4)
    IE_PF_CASE(5)
    IE_PF_CASE(6)
    IE_PF_CASE(7)
    IE_PF_CASE(8)
    default:
      return fail(IE_HIP_EINVAL, "attention_prefill: at most 8 query heads per KV head");
  }
#undef IE_PF_CASE
}

}  // namespace

bool prefill_mfma_supported(int kv_dtype, int n_heads, int n_kv_heads, int head_dim) {
  return (kv_dtype == IE_KV_F16 || kv_dtype == IE_KV_BF16 || kv_dtype == IE_KV_F32) &&
         head_dim == 64 && n_kv_heads > 0 && n_heads % n_kv_heads == 0 &&
         n_heads / n_kv_heads <= kMaxGroup;
}

int prefill_mfma_launch(float* out, const float* q, const void* k_pool, const void* v_pool, int T,
                        const int32_t* row_pos, const int32_t* row_seq, const ie_kv_layout& kv,
                        int n_heads, int n_kv_heads, const PrefillRope& rope,
                        hipStream_t stream) {
  if (rope.table && (reinterpret_cast<uintptr_t>(rope.table) & 15))
    return fail(IE_HIP_EINVAL, "attention_prefill: the RoPE table must be 16-byte aligned");
  if ((reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(out) |
       reinterpret_cast<uintptr_t>(k_pool) | reinterpret_cast<uintptr_t>(v_pool)) & 15)
    return fail(IE_HIP_EINVAL, "attention_prefill: q, out and the pools must be 16-byte aligned");
  if (kv.kv_dtype == IE_KV_F32) {
    // The f32 kernel takes q already rotated (its lanes hold 16 consecutive dims,
    // not the rotation pairs; reading the partner dims and the table per lane
    // cost more than the append's q traffic saves).
    if (rope.table)
      return fail(IE_HIP_EINVAL, "attention_prefill: f32 caches take q rotated by rope_and_cache");
    const float* kf = static_cast<const float*>(k_pool);
    const float* vf = static_cast<const float*>(v_pool);
    switch (choose_prefill_f32(T, n_heads, device_compute_units())) {
      case PrefillKernel::kRows2x4:
        return launch_prefill_f32<2, 4>(out, q, kf, vf, T, row_pos, row_seq, kv, n_heads, n_kv_heads,
                                        stream);
      case PrefillKernel::kRows2x8:
        return launch_prefill_f32<2, 8>(out, q, kf, vf, T, row_pos, row_seq, kv, n_heads, n_kv_heads,
                                        stream);
      default:
        return launch_prefill_f32<1, 8>(out, q, kf, vf, T, row_pos, row_seq, kv, n_heads, n_kv_heads,
                                        stream);
    }
  }
  const uint16_t* kp = static_cast<const uint16_t*>(k_pool);
  const uint16_t* vp = static_cast<const uint16_t*>(v_pool);
  if (kv.kv_dtype == IE_KV_F16)
    return launch_prefill_mfma<IE_KV_F16>(out, q, kp, vp, T, row_pos, row_seq, kv, n_heads,
                                          n_kv_heads, rope, stream);
  return launch_prefill_mfma<IE_KV_BF16>(out, q, kp, vp, T, row_pos, row_seq, kv, n_heads,
                                         n_kv_heads, rope, stream);
}

}  // namespace iehip
