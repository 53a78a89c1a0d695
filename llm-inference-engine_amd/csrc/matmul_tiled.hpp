// The projections' matrix-core kernel (gfx950): y (+)= (x . W^T) * s + b over LDS tiles, with
// the rmsnorm before it and the SiLU product after it folded in.
#pragma once

#include "common.hpp"
#include "mfma.hpp"

namespace iehip {

// Outputs: rows [0, split0) go to y ([T, split0]), rows [split0, split1) to y1
// ([T, split1 - split0]) and the rest to y2 ([T, rows - split1]); a plain
// matmul has split0 = split1 = rows.
struct RowSplit {
  float* y1;
  float* y2;
  int split0, split1;
};

// NORM: the rmsnorm before the matmul, folded into it (the decode step's
// xn = rmsnorm(x); y = xn . W^T pairs). y = (x * w_norm) . W^T * inv_rms(x):
// the activations are scaled by the norm weight as they are split, each lane
// sums the squares of the raw x it loads, those sums are added in the same fixed
// tree as the tiles, and the epilogue takes the row's 1 / sqrt(mean(x^2) + eps).
// The orders depend on the matrix shape alone.
struct RowNorm {
  const float* weight;  // [cols]
  float eps;
};

// 8 INT8 weights as bf16 (exact for |q| <= 127).
__device__ __forceinline__ bf16x8 widen_i8(const uint2 raw) {
  bf16x8 a;
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    const uint32_t word = j < 4 ? raw.x : raw.y;
    const int8_t q = static_cast<int8_t>((word >> (8 * (j & 3))) & 0xFF);
    a[j] = static_cast<bf16>(static_cast<float>(q));
  }
  return a;
}

__device__ __forceinline__ float silu(float v) { return v / (1.0f + expf(-v)); }

// Waits until at most min(newer, MAX) steps of PER loads each are still in flight.
template <int MAX, int PER>
__device__ __forceinline__ void wait_steps(int newer) {
  if constexpr (MAX == 0) {
    wait_vmcnt<0>();
  } else {
    if (newer >= MAX)
      wait_vmcnt<MAX * PER>();
    else
      wait_steps<MAX - 1, PER>(newer);
  }
}

// A workgroup's tile: RT row tiles of 16 per weight matrix by CT token tiles of 16. Its W
// waves share the K blocks, each with S stages of its own in LDS.
template <bool GATE, int RT, int CT, int W, int S, bool I8>
struct TiledShape {
  static constexpr int kRows = 16 * RT, kTokens = 16 * CT;
  static constexpr int kNA = GATE ? 2 : 1;                       // weight matrices
  static constexpr int kWTile = I8 ? 512 : 1024;                 // 16 rows x 32 columns
  static constexpr int kABytes = kNA * RT * kWTile;
  static constexpr int kStage = kABytes + CT * 2048;             // + 16 tokens x 32 floats each
  static constexpr int kTiles = kNA * RT * CT;
  static constexpr int kSums = W * (kTiles * 1024 + CT * 256);   // the waves' partial tiles
  static constexpr int kLds = W * S * kStage > kSums ? W * S * kStage : kSums;
};

// The tile of workgroup b. Workgroups go to the 8 XCDs in turn, so XCD b % 8 takes a
// contiguous run of tiles, ordered by groups of 8 row tiles, tokens, rows: what runs at
// once on an XCD shares its weight and activation tiles in that XCD's L2 (q/k/v at 4,000
// tokens: 50.5 us with the tiles in plain order, 48.2 so). With two weight matrices and few token
// tiles: rows, then tokens, so that the runs do not part a row tile's tokens and with them its
// weights (gate/up 640 x 20,480 at 32 tokens: 39.2 us by groups, 36.1 so, 34.3 where an XCD had
// whole columns of row tiles; one matrix gains nothing by it).
template <bool GATE>
__device__ __forceinline__ void tile_of_block(int b, int row_tiles, int tok_tiles, int& row,
                                              int& tok) {
  constexpr int kXcds = 8, kGroup = 8, kFewTokens = 4;
  const int n = row_tiles * tok_tiles, q = n / kXcds, rem = n % kXcds, xcd = b % kXcds;
  const int t = xcd * q + min(xcd, rem) + b / kXcds;
  if (GATE && tok_tiles <= kFewTokens) {
    row = t / tok_tiles;
    tok = t - row * tok_tiles;
    return;
  }
  const int group = t / (kGroup * tok_tiles), in = t - group * kGroup * tok_tiles;
  const int width = min(kGroup, row_tiles - group * kGroup);
  tok = in / width;
  row = group * kGroup + in - tok * width;
}

// One lane's 4 rows of a finished tile: token `tok`, rows row .. row + 3.
// vec: the row counts of every output are multiples of 4 and all pointers 16-byte
// aligned, so they are one 16-byte access.
template <bool GATE, bool I8, bool NORM>
__device__ __forceinline__ void put_rows(const f32x4 (&v)[GATE ? 2 : 1], float inv, int tok, int row,
                                         float* y, const float* scale, const float* scale2,
                                         const float* bias, int T, int rows, int accumulate,
                                         const RowSplit& out, int vec) {
  constexpr int NA = GATE ? 2 : 1;
  if (tok >= T || row >= rows) return;
  auto place = [&](int at) {
    if (at < out.split0) return y + size_t(tok) * out.split0 + at;
    if (at < out.split1) return out.y1 + size_t(tok) * (out.split1 - out.split0) + (at - out.split0);
    return out.y2 + size_t(tok) * (rows - out.split1) + (at - out.split1);
  };
  if (vec) {
    f32x4 o = v[0];
    if constexpr (I8) o *= *reinterpret_cast<const f32x4*>(scale + row);
    if constexpr (NORM) o *= inv;
    f32x4* dst = reinterpret_cast<f32x4*>(place(row));
    if constexpr (GATE) {
      f32x4 up = v[NA - 1];
      if constexpr (I8) up *= *reinterpret_cast<const f32x4*>(scale2 + row);
      if constexpr (NORM) up *= inv;
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = silu(o[e]) * up[e];
    } else {
      if (bias) o += *reinterpret_cast<const f32x4*>(bias + row);
      if (accumulate) o += *dst;
    }
    *dst = o;
    return;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (row + e >= rows) break;
    float o = v[0][e] * (I8 ? scale[row + e] : 1.0f);
    if constexpr (NORM) o *= inv;
    float* dst = place(row + e);
    if constexpr (GATE) {
      float up = v[NA - 1][e] * (I8 ? scale2[row + e] : 1.0f);
      if constexpr (NORM) up *= inv;
      o = silu(o) * up;
    } else {
      if (bias) o += bias[row + e];
      if (accumulate) o += *dst;
    }
    *dst = o;
  }
}

// GATE: out = silu(x . Wg^T * sg) * (x . Wu^T * su) (gate_up_silu); otherwise
// y (+)= x . W^T * s + bias.
//
// The order of every output's sum depends on the matrix alone: its 32-wide K blocks go to
// SLOTS slots in turn (block k to slot k % SLOTS), a slot's blocks are added in order by the
// matrix cores (hi, mid, lo of each block), and the slots' sums in a fixed tree (s and
// s + SLOTS/2, then s and s + SLOTS/4, ..). So a token's result is the same bit for bit
// whatever tile, wave count and batch it is computed in. W = SLOTS waves take a slot each;
// W = SLOTS / 2 waves take two, one after the other, each with accumulators of its own.
//
// Each wave brings its K block's weight and activation tiles into LDS stages of its own by
// DMA (global_load_lds_dwordx4, whole 64- and 128-byte row pieces, swizzled so that the
// operand reads spread over the banks), reads them all into registers, sends the stage's
// next loads, and only then splits and multiplies: the loads have the whole block's
// arithmetic to land, with one stage, and no wave waits for another before the end (stages
// shared by several waves, with a barrier per block, were slower at every size but one).
//
// What bounds it: at many tokens the VALU and matrix cores in turn (the x3 split of the
// activations, 5.5 instructions a value, done again by every row tile: hence tiles of up to
// 128 rows; norm + gate/up at 4,000 tokens: VALU issue 54%, matrix cores 36% of the cycles, and
// with INT8 weights, widened again by every token tile, 60 and 30%). At few
// tokens a launch's fixed time and the 16-token tile's split.
//
// SHORT: K has fewer blocks than slots; a slot without one adds zeros.
template <bool GATE, int RT, int CT, int W, int SLOTS, int S, bool I8, bool NORM, bool SHORT>
__global__ void __launch_bounds__(64 * W)
matmul_tiled_kernel(float* __restrict__ y, const float* __restrict__ x, const void* __restrict__ w,
                    const float* __restrict__ scale, const void* __restrict__ w2,
                    const float* __restrict__ scale2, const float* __restrict__ bias, int T,
                    int rows, int cols, int accumulate, RowSplit out, RowNorm norm, int vec,
                    int row_tiles, int tok_tiles) {
  using Shape = TiledShape<GATE, RT, CT, W, S, I8>;
  constexpr int NA = Shape::kNA, NR = NA * RT;
  constexpr int N = SLOTS / W;                 // slots of a wave
  constexpr int kLA = I8 ? (NR + 1) / 2 : NR;  // 1 KB weight loads of a block
  constexpr int kPerStep = kLA + 2 * CT;
  static_assert(N == 1 || N == 2, "a wave takes one slot or two");
  extern __shared__ __align__(16) unsigned char dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  int row_tile, tok_tile;
  tile_of_block<GATE>(blockIdx.x, row_tiles, tok_tiles, row_tile, tok_tile);
  const int row0 = row_tile * 16 * RT, tok0 = tok_tile * 16 * CT;
  // [0, cols * 4): the norm weight (NORM); then each wave's stages.
  unsigned char* const tiles = dyn + (NORM ? cols * 4 : 0);
  unsigned char* const stages = tiles + wave * S * Shape::kStage;
  const unsigned stages_lds = lds_address(stages);

  // DMA sources: a lane's byte offsets from the tile's first row and token. Weight tiles:
  // bf16, load u is row tile u, lane l row l/4, 16-byte piece (l%4) ^ (row/2 % 4); int8,
  // load u is row tiles 2u and 2u + 1, lane l row l/2 of the 32, piece (l%2) ^ (row/4 % 2).
  // Activations: load p is tokens 8p .. 8p+7, lane l token l/8, piece (l%8) ^ (l/8). LDS
  // slot = lane. (The host takes this kernel where a tile's offsets fit 32 bits: tile_offsets_fit.)
  constexpr int kWBytes = I8 ? 1 : 2;
  const int wr = I8 ? lane >> 1 : lane >> 2;
  const int wp = I8 ? (lane & 1) ^ ((wr >> 2) & 1) : (lane & 3) ^ ((wr >> 1) & 3);
  unsigned woff[kLA];
  bool second[kLA];  // INT8, two matrices: this lane's row tile belongs to w2
#pragma unroll
  for (int u = 0; u < kLA; ++u) {
    const int tile = I8 ? min(2 * u + (wr >> 4), NR - 1) : u;
    woff[u] = unsigned(min(16 * (tile % RT) + (wr & 15), rows - 1 - row0)) * unsigned(cols * kWBytes) +
              16 * wp;
    second[u] = tile >= RT;
  }
  const int xq = (lane & 7) ^ ((lane >> 3) & 7);
  unsigned xoff[2 * CT];
#pragma unroll
  for (int p = 0; p < 2 * CT; ++p)
    xoff[p] = unsigned(min(8 * p + (lane >> 3), T - 1 - tok0)) * unsigned(cols * 4) + 16 * xq;
  const char* const wbase = static_cast<const char*>(w) + size_t(row0) * cols * kWBytes;
  const char* const w2base = GATE ? static_cast<const char*>(w2) + size_t(row0) * cols * kWBytes : wbase;
  const char* const xbase = reinterpret_cast<const char*>(x + size_t(tok0) * cols);

  const int nblocks = cols >> 5;  // at least SLOTS, unless SHORT (the launcher)
  auto blocks_of = [&](int slot) { return (nblocks - slot + SLOTS - 1) / SLOTS; };
  const int first = blocks_of(wave);  // blocks of this wave's first slot
  const int nsteps = N == 1 ? first : first + blocks_of(wave + W);
  // Step s of the wave: block s of its first slot, then the second slot's.
  auto column_of = [&](int s) {
    return N == 1 || s < first ? 32 * (wave + SLOTS * s) : 32 * (wave + W + SLOTS * (s - first));
  };
  auto issue = [&](int step, int stage) {
    const int kb = column_of(step);
    const unsigned base = stages_lds + stage * Shape::kStage;
#pragma unroll
    for (int u = 0; u < kLA; ++u) {
      // One matrix per load, except where a pair of INT8 row tiles straddles the two.
      constexpr bool kPairs = I8 && GATE && RT % 2 == 1;
      if constexpr (I8 && NR % 2 == 1) {
        if (2 * u + (lane >> 5) < NR) dma16_at(wbase + kb * kWBytes, woff[u], base + u * 1024);
      } else if (kPairs && 2 * u + 1 == RT) {
        dma16((second[u] ? w2base : wbase) + kb * kWBytes + woff[u], base + u * 1024);
      } else {
        const bool two = GATE && (I8 ? 2 * u : u) >= RT;
        dma16_at((two ? w2base : wbase) + kb * kWBytes, woff[u], base + u * 1024);
      }
    }
#pragma unroll
    for (int p = 0; p < 2 * CT; ++p)
      dma16_at(xbase + kb * 4, xoff[p], base + Shape::kABytes + p * 1024);
  };
#pragma unroll
  for (int s = 0; s < S; ++s)
    if (s < nsteps) issue(s, s);
  // The norm weight, also by DMA (so that every wait here is on this wave's own count of
  // DMAs), after the first blocks': its round trip overlaps theirs.
  if constexpr (NORM) {
    const int n4 = cols / 4;  // 16-byte pieces; lane l of a DMA lands at base + 16 l
    const unsigned norm_lds = lds_address(dyn);
    for (int i0 = 64 * wave; i0 < n4; i0 += 64 * W)
      if (i0 + lane < n4) dma16(norm.weight + 4 * (i0 + lane), norm_lds + 16 * i0);
    wait_vmcnt<0>();
    __syncthreads();
  }

  // Operand offsets in a stage (the inverse of the swizzles above).
  const int aoff = I8 ? 16 * (2 * r + ((g >> 1) ^ ((r >> 2) & 1))) + 8 * (g & 1)
                      : 16 * (4 * r + (g ^ ((r >> 1) & 3)));
  const int boff0 = Shape::kABytes + 16 * (8 * r + ((2 * g) ^ (r & 7)));
  const int boff1 = Shape::kABytes + 16 * (8 * r + ((2 * g + 1) ^ (r & 7)));

  f32x4 sums[N][NR][CT];  // per slot
  float squares[N][CT];   // NORM: this lane's sum of x^2 of its token (row r of token tile j)
  int step = 0, stage = 0;
#pragma unroll
  for (int n = 0; n < N; ++n) {
    f32x4(&acc)[NR][CT] = sums[n];
    float(&ss)[CT] = squares[n];
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      ss[j] = 0.0f;
#pragma unroll
      for (int i = 0; i < NR; ++i) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    const int end = n == 0 ? first : nsteps;
    if (SHORT && step == end) continue;
    do {
      wait_steps<S - 1, kPerStep>(nsteps - 1 - step);  // this step's tiles have landed
      const unsigned char* st = stages + stage * Shape::kStage;
      float4 xr[CT][2];
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        xr[j][0] = *reinterpret_cast<const float4*>(st + j * 2048 + boff0);
        xr[j][1] = *reinterpret_cast<const float4*>(st + j * 2048 + boff1);
      }
      bf16x8 a[I8 ? 1 : NR];
      uint2 a8[I8 ? NR : 1];
#pragma unroll
      for (int i = 0; i < NR; ++i) {
        if constexpr (I8)
          a8[i] = *reinterpret_cast<const uint2*>(st + i * 512 + aoff);
        else
          a[i] = *reinterpret_cast<const bf16x8*>(st + i * 1024 + aoff);
      }
      if (step + S < nsteps) {
        __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage's reads are done
        issue(step + S, stage);
      }
      bf16x8 xb[3][CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        float4 x0 = xr[j][0], x1 = xr[j][1];
        if constexpr (NORM) {
          const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) ss[j] = __builtin_fmaf(v[e], v[e], ss[j]);
          const float* wn = reinterpret_cast<const float*>(dyn) + column_of(step) + 8 * g;
          const float4 wn0 = *reinterpret_cast<const float4*>(wn);
          const float4 wn1 = *reinterpret_cast<const float4*>(wn + 4);
          x0 = make_float4(x0.x * wn0.x, x0.y * wn0.y, x0.z * wn0.z, x0.w * wn0.w);
          x1 = make_float4(x1.x * wn1.x, x1.y * wn1.y, x1.z * wn1.z, x1.w * wn1.w);
        }
        split3(x0, x1, xb[0][j], xb[1][j], xb[2][j]);
      }
      constexpr int kI = NR % 2 == 0 ? 2 : 1;  // row tiles interleaved in the products
#pragma unroll
      for (int i = 0; i < NR; i += kI) {
        bf16x8 af[kI];
#pragma unroll
        for (int k = 0; k < kI; ++k) {
          if constexpr (I8)
            af[k] = widen_i8(a8[i + k]);
          else
            af[k] = a[i + k];
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int k = 0; k < kI; ++k)
#pragma unroll
            for (int j = 0; j < CT; ++j)
              acc[i + k][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(af[k], xb[p][j],
                                                                      acc[i + k][j], 0, 0, 0);
      }
      stage = stage + 1 == S ? 0 : stage + 1;
    } while (++step < end);
    // The token's sum over the 4 lane groups of its K slices (lanes r, r + 16, ..).
    if constexpr (NORM) {
#pragma unroll
      for (int j = 0; j < CT; ++j) ss[j] = group_sum4(ss[j]);
    }
  }
  if constexpr (N == 2) {
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      squares[0][j] += squares[1][j];
#pragma unroll
      for (int i = 0; i < NR; ++i) sums[0][i][j] += sums[1][i][j];
    }
  }

  // The waves' partial tiles through LDS (the stages are idle: every load was waited for
  // and read), added in the fixed tree by whichever wave finishes the tile.
  __syncthreads();
  f32x4* const red = reinterpret_cast<f32x4*>(tiles);                              // [W][tile][lane]
  float* const red_ss = reinterpret_cast<float*>(tiles + W * Shape::kTiles * 1024);  // [W][CT][lane]
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    if constexpr (NORM) red_ss[(wave * CT + j) * 64 + lane] = squares[0][j];
#pragma unroll
    for (int i = 0; i < NR; ++i)
      red[(wave * Shape::kTiles + i * CT + j) * 64 + lane] = sums[0][i][j];
  }
  __syncthreads();
  auto total = [&](auto part) {
    static_assert(W == 4 || W == 8, "the tree below");
    if constexpr (W == 4)
      return (part(0) + part(2)) + (part(1) + part(3));
    else
      return ((part(0) + part(4)) + (part(2) + part(6))) + ((part(1) + part(5)) + (part(3) + part(7)));
  };
  for (int u = wave; u < RT * CT; u += W) {
    const int i = u / CT, j = u % CT;
    f32x4 v[NA];
#pragma unroll
    for (int n = 0; n < NA; ++n)
      v[n] = total([&](int k) {
        return red[(k * Shape::kTiles + (n * RT + i) * CT + j) * 64 + lane];
      });
    float inv = 1.0f;  // NORM: the token's 1 / rms
    if constexpr (NORM) {
      const float sum = total([&](int k) { return red_ss[(k * CT + j) * 64 + lane]; });
      inv = 1.0f / sqrtf(sum / float(cols) + norm.eps);
    }
    put_rows<GATE, I8, NORM>(v, inv, tok0 + 16 * j + r, row0 + 16 * i + 4 * g, y, scale, scale2,
                             bias, T, rows, accumulate, out, vec);
  }
}

// The same product for a wide matrix and few tokens (the LM head of a decode step), where the
// time is the weights' way from HBM: a persistent workgroup keeps its tokens' split
// activations in registers and streams row tiles past them, so that nothing but weights is
// loaded and nothing split again per tile. 4 slots x TG waves; wave (slot, tg) holds the
// slot's at most KB K blocks of CT token tiles (12 registers a block and tile) and runs through
// tiles of RT x 16 rows, its weights arriving in a ring of D blocks. The slots' sums meet
// in LDS, in two buffers in turn: one barrier a tile. The order of every sum is
// matmul_tiled_kernel's.
template <int RT, int CT, int TG, bool I8>
struct StreamShape {
  static constexpr int kSlots = 4, kKB = 8, kD = 4;
  static constexpr int kWaves = kSlots * TG;
  static constexpr int kStage = RT * (I8 ? 512 : 1024);
  static constexpr int kTiles = RT * CT;
  static constexpr int kRing = kWaves * kD * kStage;
  static constexpr int kLds = kRing + 2 * kWaves * kTiles * 1024;
};

template <int RT, int CT, int TG, bool I8>
__global__ void __launch_bounds__(256 * TG)
matmul_stream_kernel(float* __restrict__ y, const float* __restrict__ x, const void* __restrict__ w,
                     const float* __restrict__ scale, const float* __restrict__ bias, int T,
                     int rows, int cols, int accumulate, RowSplit out, int vec, int row_tiles) {
  using Shape = StreamShape<RT, CT, TG, I8>;
  constexpr int kSlots = Shape::kSlots, KB = Shape::kKB, D = Shape::kD;
  constexpr int kPer = I8 ? RT / 2 : RT;  // 1 KB loads of a block
  static_assert(!I8 || RT % 2 == 0, "INT8 loads take row tiles in pairs");
  extern __shared__ __align__(16) unsigned char dyn[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int slot = wave / TG, tg = wave % TG;
  const int g = lane >> 4, r = lane & 15;
  unsigned char* const ring = dyn + wave * D * Shape::kStage;
  const unsigned ring_lds = lds_address(ring);
  const int nb = ((cols >> 5) - slot + kSlots - 1) / kSlots;  // this slot's blocks, 1 .. KB

  // Weights: as in matmul_tiled_kernel. A tile's steps are always KB; those past the
  // slot's blocks load 16 bytes, so that every step counts the same loads.
  constexpr int kWBytes = I8 ? 1 : 2;
  const int wr = I8 ? lane >> 1 : lane >> 2;
  const int wp = I8 ? (lane & 1) ^ ((wr >> 2) & 1) : (lane & 3) ^ ((wr >> 1) & 3);
  auto issue = [&](int tile, int b) {
    const int kb = 32 * (slot + kSlots * min(b, nb - 1));
    const int row0 = tile * 16 * RT;
    const char* base = static_cast<const char*>(w) + (size_t(row0) * cols + kb) * kWBytes;
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
      const unsigned off = unsigned(min((I8 ? 32 : 16) * u + wr, rows - 1 - row0)) *
                               unsigned(cols * kWBytes) + 16 * wp;
      if (b < nb || lane == 0) dma16_at(base, off, ring_lds + (b % D) * Shape::kStage + u * 1024);
    }
  };
  int tile = blockIdx.x;
#pragma unroll
  for (int b = 0; b < D; ++b) issue(tile, b);

  bf16x8 xb[KB][CT][3];
#pragma unroll
  for (int b = 0; b < KB; ++b) {
    const int kb = 32 * (slot + kSlots * min(b, nb - 1)) + 8 * g;
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const float4* src = reinterpret_cast<const float4*>(
          x + size_t(min((tg * CT + j) * 16 + r, T - 1)) * cols + kb);
      split3(src[0], src[1], xb[b][j][0], xb[b][j][1], xb[b][j][2]);
    }
  }
  const int aoff = I8 ? 16 * (2 * r + ((g >> 1) ^ ((r >> 2) & 1))) + 8 * (g & 1)
                      : 16 * (4 * r + (g ^ ((r >> 1) & 3)));
  f32x4* const red = reinterpret_cast<f32x4*>(dyn + Shape::kRing);  // [2][wave][tile][lane]
  for (int turn = 0; tile < row_tiles; turn ^= 1) {
    const int next = tile + int(gridDim.x);
    f32x4 acc[RT][CT];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      wait_vmcnt<(D - 1) * kPer>();  // this step's tile has landed
      const unsigned char* st = ring + (b % D) * Shape::kStage;
      bf16x8 a[RT];
      uint2 a8[RT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        if constexpr (I8)
          a8[i] = *reinterpret_cast<const uint2*>(st + i * 512 + aoff);
        else
          a[i] = *reinterpret_cast<const bf16x8*>(st + i * 1024 + aoff);
      }
      __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the stage's reads are done
      // The step D ahead; past the last tile, that tile again (read by no one).
      if (b + D < KB)
        issue(tile, b + D);
      else
        issue(next < row_tiles ? next : tile, b + D - KB);
      if (b < nb) {
        if constexpr (I8) {
#pragma unroll
          for (int i = 0; i < RT; ++i) a[i] = widen_i8(a8[i]);
        }
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
          for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j)
              acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[i], xb[b][j][p], acc[i][j], 0, 0, 0);
      }
    }
    f32x4* const part = red + turn * Shape::kWaves * Shape::kTiles * 64;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < CT; ++j) part[(wave * Shape::kTiles + i * CT + j) * 64 + lane] = acc[i][j];
    __syncthreads();
    for (int u = wave; u < TG * Shape::kTiles; u += Shape::kWaves) {
      const int t = u / Shape::kTiles, ij = u % Shape::kTiles;
      auto of = [&](int sl) { return part[((sl * TG + t) * Shape::kTiles + ij) * 64 + lane]; };
      const f32x4 v[1] = {(of(0) + of(2)) + (of(1) + of(3))};
      put_rows<false, I8, false>(v, 1.0f, (t * CT + ij % CT) * 16 + r,
                                 tile * 16 * RT + 16 * (ij / CT) + 4 * g, y, scale, nullptr, bias, T,
                                 rows, accumulate, out, vec);
    }
    tile = next;
  }
  wait_vmcnt<0>();  // no load may land in LDS that is another workgroup's by then
}

}  // namespace iehip
