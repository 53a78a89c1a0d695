// The dense ops of the decode step around the paged-KV path (gfx950): the
// embedding lookup, rmsnorm, the projections (q/k/v, o_proj, down) and the
// fused gate/up + SiLU. Reference: src/cuda/kernels.cuh:40-66 and
// src/cuda/kernels.cu:191-241,1236-1285; CPU semantics src/ops.cpp:23-32,68,
// src/matrix.cpp:131-146,247-289, src/model.cpp:53-90.
//
// Weights are BF16 bits or INT8 with one f32 scale per row (the reference's
// DeviceMatrix). Activations are f32.
//
// matmul_mfma_kernel: y[t][o] (+)= (sum_k W[o][k] x[t][k]) * s[o] + bias[o] on
// v_mfma_f32_16x16x32_bf16, in 16-row x 16-token output tiles:
//   D[16 rows x 16 tokens] = W[16 x K] . x^T[K x 16]
// The weights enter the MFMA exactly (BF16 as stored; INT8 values widened to
// bf16, exact for |q| <= 127). Each activation is split into three bf16
// parts, x = hi + mid + lo exactly (each remainder is exact in f32 and holds
// at most 16, then 8, significant bits), and each block is multiplied three
// times, so every product is the f32-exact w * x. Only the summation order
// differs from the CPU's: the results agree to float32 rounding of the sum.
// matmul_tiled_kernel (matmul_tiled.hpp) is that product with its operands staged in LDS,
// in one of several tile shapes (see choose_tile), for K in whole 32-wide blocks and
// weights aligned for the DMA; matmul_mfma_kernel here loads its operands directly, for
// every other shape (launch_rules.hpp says which). Both add every output in the same order,
// fixed by the matrix alone.
// Lane (g, r) of a tile: A = W[row r][k + 8g .. +8], B = x[token r][k + 8g ..
// +8]; the result lane holds rows 4g .. 4g+3 of token r.
#include <algorithm>

#include "common.hpp"
#include "launch_rules.hpp"
#include "matmul_tiled.hpp"
#include "mfma.hpp"

namespace iehip {
namespace {

constexpr int kMmWaves = 8;  // waves of a workgroup, splitting K

template <bool I8>
__device__ __forceinline__ bf16x8 load_weights(const void* w, size_t idx) {
  bf16x8 a;
  if constexpr (!I8) {
    a = *reinterpret_cast<const bf16x8*>(static_cast<const uint16_t*>(w) + idx);
  } else {
    a = widen_i8(*reinterpret_cast<const uint2*>(static_cast<const int8_t*>(w) + idx));
  }
  return a;
}

__device__ __forceinline__ f32x4 mma3(bf16x8 a, bf16x8 bh, bf16x8 bm, bf16x8 bl, f32x4 c) {
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bh, c, 0, 0, 0);
  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bm, c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, bl, c, 0, 0, 0);
}

// GATE: out = silu(x . Wg^T * sg) * (x . Wu^T * su) (gate_up_silu); otherwise
// y (+)= x . W^T * s + bias. A workgroup owns RT x TT tiles of 16 rows x 16
// tokens: each weight fragment is loaded once per K block and used for all TT
// token tiles (so the weights are read once per launch when T <= 16 TT), each
// activation fragment split once and used for all RT row tiles. cols % 8 == 0;
// the K tail past cols is zero. Lane (g, r)'s direct loads of its operands touch 16
// rows per quarter-wave, and the L1's access rate bounds the kernel: shapes that the
// LDS tiles take run there (down 896 x 4,864 at 64 tokens: 15.3 us here, 8.7 us there).
template <bool GATE, int RT, int TT, int W, bool I8, bool NORM = false>
__global__ void __launch_bounds__(64 * W)
matmul_mfma_kernel(float* __restrict__ y, const float* __restrict__ x, const void* __restrict__ w,
                   const float* __restrict__ scale, const void* __restrict__ w2,
                   const float* __restrict__ scale2, const float* __restrict__ bias,
                   int T, int rows, int cols, int accumulate, RowSplit out, RowNorm norm) {
  constexpr int NA = GATE ? 2 : 1, NT = NA * RT * TT;
  static_assert(NT <= 16, "at most 16 accumulator tiles (64 KB of LDS for the reduction)");
  __shared__ f32x4 red[W / 2][NT][64];
  __shared__ float red_ss[NORM ? W / 2 : 1][TT][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, r = lane & 15;
  const int row0 = blockIdx.x * 16 * RT, tok0 = blockIdx.y * 16 * TT;
  size_t wrow[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) wrow[i] = size_t(min(row0 + 16 * i + r, rows - 1)) * cols;
  const float* xrow[TT];
#pragma unroll
  for (int j = 0; j < TT; ++j) xrow[j] = x + size_t(min(tok0 + 16 * j + r, T - 1)) * cols;
  f32x4 acc[NA][RT][TT];
#pragma unroll
  for (int n = 0; n < NA; ++n)
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
      for (int j = 0; j < TT; ++j) acc[n][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  float ss[TT];  // NORM: this lane's sum of x^2 of its token (row r of token tile j)
#pragma unroll
  for (int j = 0; j < TT; ++j) ss[j] = 0.0f;
  for (int kb = 32 * wave; kb < cols; kb += 32 * W) {
    const int k = kb + 8 * g;
    const bool kin = k < cols;
    float4 wn0 = make_float4(1.f, 1.f, 1.f, 1.f), wn1 = wn0;
    if constexpr (NORM) {
      if (kin) {
        wn0 = *reinterpret_cast<const float4*>(norm.weight + k);
        wn1 = *reinterpret_cast<const float4*>(norm.weight + k + 4);
      }
    }
    bf16x8 a[NA][RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      a[0][i] = kin ? load_weights<I8>(w, wrow[i] + k) : bf16x8{};
      if constexpr (GATE) a[NA - 1][i] = kin ? load_weights<I8>(w2, wrow[i] + k) : bf16x8{};
    }
#pragma unroll
    for (int j = 0; j < TT; ++j) {
      bf16x8 bh = {}, bm = {}, bl = {};
      if (kin) {
        const float4* xp = reinterpret_cast<const float4*>(xrow[j] + k);
        float4 x0 = xp[0], x1 = xp[1];
        if constexpr (NORM) {
          const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) ss[j] = __builtin_fmaf(v[e], v[e], ss[j]);
          x0 = make_float4(x0.x * wn0.x, x0.y * wn0.y, x0.z * wn0.z, x0.w * wn0.w);
          x1 = make_float4(x1.x * wn1.x, x1.y * wn1.y, x1.z * wn1.z, x1.w * wn1.w);
        }
        split3(x0, x1, bh, bm, bl);
      }
#pragma unroll
      for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < RT; ++i) acc[n][i][j] = mma3(a[n][i], bh, bm, bl, acc[n][i][j]);
    }
  }
  // NORM: the token's sum over the 4 lane groups of its K slices (lanes r,
  // r + 16, r + 32, r + 48), then with the tiles through the waves' tree.
  if constexpr (NORM) {
#pragma unroll
    for (int j = 0; j < TT; ++j) ss[j] = group_sum4(ss[j]);
  }
  // The waves' partial tiles summed through LDS in a fixed tree (waves 4-7
  // into 0-3, 2-3 into 0-1, 1 into 0), so results do not depend on timing.
#pragma unroll
  for (int half = W / 2; half >= 1; half /= 2) {
    if (wave >= half && wave < 2 * half) {
#pragma unroll
      for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < TT; ++j) red[wave - half][(n * RT + i) * TT + j][lane] = acc[n][i][j];
      if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < TT; ++j) red_ss[wave - half][j][lane] = ss[j];
      }
    }
    __syncthreads();
    if (wave < half) {
#pragma unroll
      for (int n = 0; n < NA; ++n)
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
          for (int j = 0; j < TT; ++j) acc[n][i][j] += red[wave][(n * RT + i) * TT + j][lane];
      if constexpr (NORM) {
#pragma unroll
        for (int j = 0; j < TT; ++j) ss[j] += red_ss[wave][j][lane];
      }
    }
    __syncthreads();
  }
  if (wave > 0) return;
#pragma unroll
  for (int j = 0; j < TT; ++j) {
    const int tok = tok0 + 16 * j + r;
    if (tok >= T) break;
    // NORM: the token's 1 / rms (1 otherwise)
    const float inv = NORM ? 1.0f / sqrtf(ss[j] / float(cols) + norm.eps) : 1.0f;
#pragma unroll
    for (int i = 0; i < RT; ++i) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = row0 + 16 * i + 4 * g + e;
        if (row >= rows) break;
        float v = acc[0][i][j][e] * (I8 ? scale[row] : 1.0f);
        if constexpr (NORM) v *= inv;
        float* dst;
        if (row < out.split0)
          dst = y + size_t(tok) * out.split0 + row;
        else if (row < out.split1)
          dst = out.y1 + size_t(tok) * (out.split1 - out.split0) + (row - out.split0);
        else
          dst = out.y2 + size_t(tok) * (rows - out.split1) + (row - out.split1);
        if constexpr (GATE) {
          float u = acc[NA - 1][i][j][e] * (I8 ? scale2[row] : 1.0f);
          if constexpr (NORM) u *= inv;
          v = silu(v) * u;
        } else {
          if (bias) v += bias[row];
          if (accumulate) v += *dst;
        }
        *dst = v;
      }
    }
  }
}

// y[t] = x[t] * (1 / sqrt(mean(x[t]^2) + eps)) * weight; one workgroup per row.
// Each element is read and written by the same thread, so y may equal x.
__global__ void __launch_bounds__(256)
rmsnorm_kernel(float* y, const float* x, const float* __restrict__ weight, int dim, float eps) {
  __shared__ float part[4];
  const float* xt = x + size_t(blockIdx.x) * dim;
  float* yt = y + size_t(blockIdx.x) * dim;
  // Rows up to 8 elements a thread (2,048 floats) stay in registers between
  // the sum and the scaling, so the row is read once.
  constexpr int kHeld = 8;
  const bool held = dim <= kHeld * int(blockDim.x);
  float xv[kHeld];
  float ss = 0.0f;
  if (held) {
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const int i = int(threadIdx.x) + j * int(blockDim.x);
      xv[j] = i < dim ? xt[i] : 0.0f;
      ss += xv[j] * xv[j];
    }
  } else {
    for (int i = threadIdx.x; i < dim; i += blockDim.x) ss += xt[i] * xt[i];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) ss += __shfl_xor(ss, off, 64);
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = ss;
  __syncthreads();
  const float total = (part[0] + part[1]) + (part[2] + part[3]);
  const float inv_rms = 1.0f / sqrtf(total / float(dim) + eps);
  if (held) {
#pragma unroll
    for (int j = 0; j < kHeld; ++j) {
      const int i = int(threadIdx.x) + j * int(blockDim.x);
      if (i < dim) yt[i] = xv[j] * inv_rms * weight[i];
    }
  } else {
    for (int i = threadIdx.x; i < dim; i += blockDim.x) yt[i] = xt[i] * inv_rms * weight[i];
  }
}

// x[t] = E[ids[t]] widened to f32 (times the row's scale for INT8).
__global__ void __launch_bounds__(256)
embedding_kernel(float* __restrict__ x, const int32_t* __restrict__ ids, const void* __restrict__ e,
                 const float* __restrict__ scale, int int8, int dim) {
  const int id = ids[blockIdx.x];
  float* xt = x + size_t(blockIdx.x) * dim;
  if (int8) {
    const int8_t* row = static_cast<const int8_t*>(e) + size_t(id) * dim;
    const float s = scale[id];
    for (int i = threadIdx.x; i < dim; i += blockDim.x) xt[i] = s * static_cast<float>(row[i]);
  } else {
    const uint16_t* row = static_cast<const uint16_t*>(e) + size_t(id) * dim;
    for (int i = threadIdx.x; i < dim; i += blockDim.x)
      xt[i] = __uint_as_float(static_cast<uint32_t>(row[i]) << 16);
  }
}

int check_matrix(const ie_matrix& m, const char* who) {
  if (!m.data || m.rows <= 0 || m.cols <= 0)
    return fail(IE_HIP_EINVAL, std::string(who) + ": empty weight matrix");
  if (m.int8 && !m.scale) return fail(IE_HIP_EINVAL, std::string(who) + ": INT8 needs row scales");
  return IE_HIP_OK;
}

constexpr int kTiledMaxLds = 160 * 1024;  // a gfx950 compute unit's LDS

// One launch of a tile shape; false (nothing launched) where its LDS, its grid or its offsets do
// not fit.
struct TiledLaunch {
  float* y;
  const float* x;
  const ie_matrix* w;
  const ie_matrix* w2;
  const float* bias;
  int T, accumulate;
  RowSplit split;
  RowNorm norm;
  int vec;
  hipStream_t stream;

  template <bool GATE, int NR, int CT, int W, int SLOTS, int S, bool I8, bool NORM, bool SHORT>
  bool go(int* rc) const {
    constexpr int RT = NR / (GATE ? 2 : 1);
    using Shape = TiledShape<GATE, RT, CT, W, S, I8>;
    const int64_t lds = int64_t(Shape::kLds) + (NORM ? int64_t(w->cols) * 4 : 0);
    const int64_t row_tiles = (int64_t(w->rows) + Shape::kRows - 1) / Shape::kRows;
    const int64_t tok_tiles = (int64_t(T) + Shape::kTokens - 1) / Shape::kTokens;
    if (lds > kTiledMaxLds || row_tiles * tok_tiles * 64 * W > int64_t(UINT32_MAX) ||
        !tile_offsets_fit(Shape::kRows, Shape::kTokens, w->cols, I8 ? 1 : 2))
      return false;
    const auto kernel = matmul_tiled_kernel<GATE, RT, CT, W, SLOTS, S, I8, NORM, SHORT>;
    if (lds > 64 * 1024) {  // above the default dynamic-LDS cap
      static const hipError_t attr =
          hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, kTiledMaxLds);
      if ((*rc = check_hip(attr, "hipFuncSetAttribute(matmul)"))) return true;
    }
    hipLaunchKernelGGL(kernel, dim3(unsigned(row_tiles * tok_tiles)), dim3(64 * W), unsigned(lds),
                       stream, y, x, w->data, w->scale, w2 ? w2->data : nullptr,
                       w2 ? w2->scale : nullptr, bias, T, w->rows, w->cols, accumulate, split, norm,
                       vec, int(row_tiles), int(tok_tiles));
    *rc = IE_HIP_OK;
    return true;
  }
  template <bool GATE, int NR, int CT, int W, int SLOTS, int S, bool SHORT = false>
  bool with_types(int* rc) const {
    if constexpr (SLOTS == 8) {  // the folded rmsnorm: matrices below 16 row tiles per unit
      if (norm.weight)
        return w->int8 ? go<GATE, NR, CT, W, SLOTS, S, true, true, SHORT>(rc)
                       : go<GATE, NR, CT, W, SLOTS, S, false, true, SHORT>(rc);
    }
    return w->int8 ? go<GATE, NR, CT, W, SLOTS, S, true, false, SHORT>(rc)
                   : go<GATE, NR, CT, W, SLOTS, S, false, false, SHORT>(rc);
  }
  bool run_short(bool gate, int* rc) const {
    return gate ? with_types<true, 4, 2, 8, 8, 1, true>(rc) : with_types<false, 2, 2, 8, 8, 1, true>(rc);
  }
  template <bool GATE>
  bool run(int shape, int* rc) const {
    if constexpr (GATE) {
      switch (shape) {
        case 0: return with_types<true, 2, 1, 8, 8, 2>(rc);
        case 1: return with_types<true, 4, 1, 8, 8, 1>(rc);
        case 2: return with_types<true, 4, 2, 8, 8, 1>(rc);
        case 3: return with_types<true, 6, 2, 4, 8, 1>(rc);
        default: return with_types<true, 8, 2, 4, 8, 1>(rc);
      }
    } else {
      switch (shape) {
        case 0: return with_types<false, 1, 1, 8, 8, 2>(rc);
        case 1: return with_types<false, 2, 1, 8, 8, 1>(rc);
        case 2: return with_types<false, 2, 2, 8, 8, 1>(rc);
        case 3: return with_types<false, 3, 2, 4, 8, 1>(rc);
        case 4: return with_types<false, 4, 2, 4, 8, 1>(rc);
        case 5: return with_types<false, 6, 2, 4, 8, 1>(rc);
        default: return with_types<false, 8, 2, 4, 8, 1>(rc);
      }
    }
  }
  template <int RT, int CT, int TG, bool I8>
  bool stream_go(int per_cu, int* rc) const {
    using Shape = StreamShape<RT, CT, TG, I8>;
    static_assert(Shape::kLds <= kTiledMaxLds, "a compute unit's LDS");
    const auto kernel = matmul_stream_kernel<RT, CT, TG, I8>;
    if (Shape::kLds > 64 * 1024) {
      static const hipError_t attr =
          hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, Shape::kLds);
      if ((*rc = check_hip(attr, "hipFuncSetAttribute(matmul)"))) return true;
    }
    const int row_tiles = (w->rows - 1) / (16 * RT) + 1;
    const int grid = std::min(row_tiles, per_cu * device_compute_units());
    hipLaunchKernelGGL(kernel, dim3(unsigned(grid)), dim3(64 * Shape::kWaves), unsigned(Shape::kLds),
                       stream, y, x, w->data, w->scale, bias, T, w->rows, w->cols, accumulate, split,
                       vec, row_tiles);
    *rc = IE_HIP_OK;
    return true;
  }
  // Wide matrices (4 slots, one wave each).
  bool run_wide(bool gate, int* rc) const {
    switch (choose_wide(gate, w->cols, T)) {
      case WideKernel::kGateTiles: return with_types<true, 8, 2, 4, 4, 1>(rc);
      case WideKernel::kTiles16: return with_types<false, 4, 1, 4, 4, 2>(rc);
      case WideKernel::kTiles32: return with_types<false, 8, 2, 4, 4, 1>(rc);
      case WideKernel::kStream16:
        return w->int8 ? stream_go<4, 1, 1, true>(2, rc) : stream_go<2, 1, 1, false>(1, rc);
      default: return w->int8 ? stream_go<2, 2, 2, true>(1, rc) : stream_go<2, 2, 2, false>(1, rc);
    }
  }
};

int launch_matmul(bool gate, float* y, const float* x, const ie_matrix& w, const ie_matrix* w2,
                  const float* bias, int T, int accumulate, hipStream_t stream, const char* who,
                  RowSplit split = RowSplit{nullptr, nullptr, 0, 0},
                  RowNorm norm = RowNorm{nullptr, 0.0f}) {
  if (split.split0 == 0 && split.split1 == 0) split.split0 = split.split1 = w.rows;
  if (int rc = check_matrix(w, who)) return rc;
  if (w2) {
    if (int rc = check_matrix(*w2, who)) return rc;
    if (w2->rows != w.rows || w2->cols != w.cols || w2->int8 != w.int8)
      return fail(IE_HIP_EINVAL, std::string(who) + ": gate and up shapes differ");
  }
  if (T < 0) return fail(IE_HIP_EINVAL, std::string(who) + ": T < 0");
  if (T == 0) return IE_HIP_OK;
  if (!y || !x) return fail(IE_HIP_EINVAL, std::string(who) + ": null pointer");
  if (w.cols % 8)
    return fail(IE_HIP_EINVAL, std::string(who) + ": cols must be a multiple of 8");
  const uintptr_t align = reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w.data) |
                          (w2 ? reinterpret_cast<uintptr_t>(w2->data) : 0);
  if (align & (w.int8 ? 7 : 15))
    return fail(IE_HIP_EINVAL, std::string(who) + ": x and the weights must be 16-byte aligned");
  // K is split over slots whose count fixes every output's summation order. It depends on
  // the matrix alone, never on T: a token's result is then the same bit for bit whatever
  // batch it is computed in (the reference's "batch of N == N single tokens" contract,
  // src/cuda/cuda_runner.cu:798-829): 4 for wide matrices (row tiles alone reach 16 per
  // compute unit: the 151,936-row LM head), where fewer, longer waves fill the chip, else 8.
  const int cus = device_compute_units();
  const bool wide = (w.rows + 15) / 16 >= 16 * cus;
  const int waves = wide ? 4 : kMmWaves;
  if (norm.weight && wide)
    return fail(IE_HIP_EINVAL, std::string(who) + ": too many rows for the folded rmsnorm");
  const int tok_tiles = (T + 15) / 16;  // kernels exist for 1, 2 and 4 token tiles
  const int TT = !wide ? 1 : tok_tiles > 2 ? 4 : tok_tiles;
  if ((T + 16 * TT - 1) / (16 * TT) > 65535)
    return fail(IE_HIP_EINVAL, std::string(who) + ": too many tokens");
  // LDS tiles: K in whole 32-wide blocks, at least one per slot or a launch of many tiles, and
  // 16-byte aligned weights for the DMA (x always is).
  const uintptr_t weights = reinterpret_cast<uintptr_t>(w.data) |
                            reinterpret_cast<uintptr_t>(w2 ? w2->data : nullptr);
  const int64_t tiles = int64_t((w.rows + 15) / 16) * tok_tiles;
  const bool short_k = w.cols < 32 * waves;
  const bool staged = !short_k || (!wide && short_k_staged(tiles, w.cols, norm.weight != nullptr, cus));
  if (w.cols % 32 == 0 && staged && ((reinterpret_cast<uintptr_t>(x) | weights) & 15) == 0) {
    const uintptr_t out = reinterpret_cast<uintptr_t>(y) | reinterpret_cast<uintptr_t>(split.y1) |
                          reinterpret_cast<uintptr_t>(split.y2) | reinterpret_cast<uintptr_t>(bias) |
                          reinterpret_cast<uintptr_t>(w.scale) |
                          reinterpret_cast<uintptr_t>(w2 ? w2->scale : nullptr);
    const int vec = (out & 15) == 0 && ((w.rows | split.split0 | split.split1) & 3) == 0;
    const TiledLaunch launch{y, x, &w, w2, bias, T, accumulate, split, norm, vec, stream};
    int rc = IE_HIP_OK;
    bool launched;
    if (wide) {
      launched = launch.run_wide(gate, &rc);
    } else if (short_k) {
      launched = launch.run_short(gate, &rc);
    } else {
      const int shape = choose_tile(gate, w.rows, w.cols, T, cus);
      launched = gate ? launch.run<true>(shape, &rc) : launch.run<false>(shape, &rc);
      // A folded rmsnorm's weights can leave too little LDS for the shape: the smallest one.
      if (!launched && shape != 0)
        launched = gate ? launch.run<true>(0, &rc) : launch.run<false>(0, &rc);
    }
    if (launched) return rc != IE_HIP_OK ? rc : check_launch(who);
  }
  // Direct loads. Tiles per workgroup from the count of 16 x 16 output tiles: two row tiles
  // from 4 per compute unit on, 4 x 4 (or the token tiles there are) for wide matrices.
  int RT = wide ? 4 : tiles >= 4 * int64_t(cus) ? 2 : 1;
  if (gate) RT = std::min(RT, 2);
  const dim3 grid((w.rows + 16 * RT - 1) / (16 * RT), (T + 16 * TT - 1) / (16 * TT));
  const dim3 block(64 * waves);
  const void* w2d = gate ? w2->data : nullptr;
  const float* s2 = gate ? w2->scale : nullptr;
  if (norm.weight) {
#define IE_MM_NORM(G, R)                                                                          \
  do {                                                                                            \
    if (w.int8)                                                                                   \
      hipLaunchKernelGGL((matmul_mfma_kernel<G, R, 1, kMmWaves, true, true>), grid, block, 0,     \
                         stream, y, x, w.data, w.scale, w2d, s2, bias, T, w.rows, w.cols,         \
                         accumulate, split, norm);                                                \
    else                                                                                          \
      hipLaunchKernelGGL((matmul_mfma_kernel<G, R, 1, kMmWaves, false, true>), grid, block, 0,    \
                         stream, y, x, w.data, w.scale, w2d, s2, bias, T, w.rows, w.cols,         \
                         accumulate, split, norm);                                                \
  } while (0)
    if (gate) {
      if (RT == 2)
        IE_MM_NORM(true, 2);
      else
        IE_MM_NORM(true, 1);
    } else {
      if (RT == 2)
        IE_MM_NORM(false, 2);
      else
        IE_MM_NORM(false, 1);
    }
#undef IE_MM_NORM
    return check_launch(who);
  }
#define IE_MM_LAUNCH_W(G, R, C, W)                                                               \
  do {                                                                                           \
    if (w.int8)                                                                                  \
      hipLaunchKernelGGL((matmul_mfma_kernel<G, R, C, W, true>), grid, block, 0, stream, y, x,   \
                         w.data, w.scale, w2d, s2, bias, T, w.rows, w.cols, accumulate, split,   \
                         norm);                                                                  \
    else                                                                                         \
      hipLaunchKernelGGL((matmul_mfma_kernel<G, R, C, W, false>), grid, block, 0, stream, y, x,  \
                         w.data, w.scale, w2d, s2, bias, T, w.rows, w.cols, accumulate, split,   \
                         norm);                                                                  \
  } while (0)
#define IE_MM_LAUNCH(G, R, C)            \
  do {                                   \
    if (wide)                            \
      IE_MM_LAUNCH_W(G, R, C, 4);        \
    else                                 \
      IE_MM_LAUNCH_W(G, R, C, kMmWaves); \
  } while (0)
#define IE_MM_TT(G, R)            \
  if (TT == 4)                    \
    IE_MM_LAUNCH(G, R, 4);        \
  else if (TT == 2)               \
    IE_MM_LAUNCH(G, R, 2);        \
  else                            \
    IE_MM_LAUNCH(G, R, 1);
  if (gate) {
    if (RT == 2) {
      IE_MM_TT(true, 2)
    } else {
      IE_MM_TT(true, 1)
    }
  } else if (RT == 4) {
    IE_MM_TT(false, 4)
  } else if (RT == 2) {
    IE_MM_TT(false, 2)
  } else {
    IE_MM_TT(false, 1)
  }
#undef IE_MM_TT
#undef IE_MM_LAUNCH
#undef IE_MM_LAUNCH_W
  return check_launch(who);
}

}  // namespace
}  // namespace iehip

using namespace iehip;

extern "C" int ie_hip_embedding(float* x, const int32_t* ids, ie_matrix e, int T,
                                hipStream_t stream) {
  clear_error();
  if (int rc = check_matrix(e, "embedding")) return rc;
  if (T < 0) return fail(IE_HIP_EINVAL, "embedding: T < 0");
  if (T == 0) return IE_HIP_OK;
  if (!x || !ids) return fail(IE_HIP_EINVAL, "embedding: null pointer");
  hipLaunchKernelGGL(embedding_kernel, dim3(T), dim3(256), 0, stream, x, ids, e.data, e.scale,
                     e.int8, e.cols);
  return check_launch("embedding");
}

extern "C" int ie_hip_rmsnorm(float* y, const float* x, const float* weight, int T, int dim,
                              float eps, hipStream_t stream) {
  clear_error();
  if (T < 0 || dim <= 0) return fail(IE_HIP_EINVAL, "rmsnorm: bad sizes");
  if (T == 0) return IE_HIP_OK;
  if (!y || !x || !weight) return fail(IE_HIP_EINVAL, "rmsnorm: null pointer");
  hipLaunchKernelGGL(rmsnorm_kernel, dim3(T), dim3(256), 0, stream, y, x, weight, dim, eps);
  return check_launch("rmsnorm");
}

extern "C" int ie_hip_matmul(float* y, const float* x, ie_matrix w, const float* bias, int T,
                             int accumulate, hipStream_t stream) {
  clear_error();
  return launch_matmul(false, y, x, w, nullptr, bias, T, accumulate, stream, "matmul");
}

extern "C" int ie_hip_qkv_proj(float* q, float* k, float* v, const float* x, ie_matrix w_qkv,
                               const float* b_qkv, int T, int q_dim, int kv_dim,
                               hipStream_t stream) {
  clear_error();
  if (q_dim <= 0 || kv_dim <= 0 || w_qkv.rows != q_dim + 2 * kv_dim)
    return fail(IE_HIP_EINVAL, "qkv_proj: weight rows must be q_dim + 2 kv_dim");
  if (T > 0 && (!q || !k || !v)) return fail(IE_HIP_EINVAL, "qkv_proj: null pointer");
  return launch_matmul(false, q, x, w_qkv, nullptr, b_qkv, T, 0, stream, "qkv_proj",
                       RowSplit{k, v, q_dim, q_dim + kv_dim});
}

extern "C" int ie_hip_gate_up_silu(float* out, const float* x, ie_matrix w_gate, ie_matrix w_up,
                                   int T, hipStream_t stream) {
  clear_error();
  return launch_matmul(true, out, x, w_gate, &w_up, nullptr, T, 0, stream, "gate_up_silu");
}

extern "C" int ie_hip_rmsnorm_qkv_proj(float* q, float* k, float* v, const float* x,
                                       const float* norm_weight, float eps, ie_matrix w_qkv,
                                       const float* b_qkv, int T, int q_dim, int kv_dim,
                                       hipStream_t stream) {
  clear_error();
  if (q_dim <= 0 || kv_dim <= 0 || w_qkv.rows != q_dim + 2 * kv_dim)
    return fail(IE_HIP_EINVAL, "rmsnorm_qkv_proj: weight rows must be q_dim + 2 kv_dim");
  if (T > 0 && (!q || !k || !v || !norm_weight))
    return fail(IE_HIP_EINVAL, "rmsnorm_qkv_proj: null pointer");
  if (reinterpret_cast<uintptr_t>(norm_weight) & 15)
    return fail(IE_HIP_EINVAL, "rmsnorm_qkv_proj: the norm weight must be 16-byte aligned");
  return launch_matmul(false, q, x, w_qkv, nullptr, b_qkv, T, 0, stream, "rmsnorm_qkv_proj",
                       RowSplit{k, v, q_dim, q_dim + kv_dim}, RowNorm{norm_weight, eps});
}

extern "C" int ie_hip_rmsnorm_gate_up_silu(float* out, const float* x, const float* norm_weight,
                                           float eps, ie_matrix w_gate, ie_matrix w_up, int T,
                                           hipStream_t stream) {
  clear_error();
  if (T > 0 && !norm_weight) return fail(IE_HIP_EINVAL, "rmsnorm_gate_up_silu: null pointer");
  if (reinterpret_cast<uintptr_t>(norm_weight) & 15)
    return fail(IE_HIP_EINVAL, "rmsnorm_gate_up_silu: the norm weight must be 16-byte aligned");
  return launch_matmul(true, out, x, w_gate, &w_up, nullptr, T, 0, stream, "rmsnorm_gate_up_silu",
                       RowSplit{nullptr, nullptr, 0, 0}, RowNorm{norm_weight, eps});
}
