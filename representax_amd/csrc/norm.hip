// The normalisations between the quantized linears of a transformer layer, in
// bf16 with f32 statistics and frozen weights: LayerNorm and RMSNorm over a
// row, with the residual addition before them fused, and the per-head RMSNorm
// of queries and keys with the rotary rotation after it
// (src/representax/models/components.py:110-150,
// src/representax/models/qwen3_vl/text.py:30-61). Forward and the gradient of
// the input; values are rounded to bf16 where the unfused steps round them (the
// residual sum, the normalised value, the rotated value), everything between
// is f32.
//
// These are passes over memory: a row lives in the registers of 8 to 64
// lanes, each tensor is read and written once in 16-byte vectors, and the
// backward recomputes the statistics from the row it reads anyway instead of
// loading saved ones. Residual LayerNorm over 32768 x 768: 37 us forward (200
// MB, 5.4 TB/s) and 32 us backward (151 MB), where torch's addition and norm
// took 72 and 102 us. An RMSNorm without a residual also writes its row to a
// copy for the backward when there will be one (its caller may change the row in
// place): 14 MB more at 3500 x 2048, and 0 to 13 us of the 1.8 ms layer that it
// stands in (three runs of both, whose noise is 10 us). The RMSNorms and the rotation, with their residual
// additions, were 70 launches of torch expressions in a Qwen3-wide layer of 7
// sequences of 500 tokens, forward and backward: 1000 of its 2870 us.
#include <hip/hip_runtime.h>

#include "common.h"
#include "kernels.h"

namespace rpx {

namespace {

constexpr int kThreads = 256;

// Sum over the L lanes of a row, the same value in each (fixed order).
template <int L>
__device__ __forceinline__ float row_sum(float v) {
#pragma unroll
  for (int off = L / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ void unpack8(u32x4_t w, float* v) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = bf16lo_to_f32(w[i]);
    v[2 * i + 1] = bf16hi_to_f32(w[i]);
  }
}

__device__ __forceinline__ u32x4_t pack8(const float* v) {
  return u32x4_t{pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]), pack_bf16x2(v[4], v[5]),
                 pack_bf16x2(v[6], v[7])};
}

__device__ __forceinline__ void load8(const uint16_t* p, float* v) {
  unpack8(*reinterpret_cast<const u32x4_t*>(p), v);
}

// Eight weights as f32. ROUND: the f32 master rounded to bf16 first (the
// LayerNorm's weight and bias take the value's dtype).
template <bool ROUND>
__device__ __forceinline__ void load_weight8(const void* w, int dtype, int e, float* v) {
  if (dtype == kBF16) {
    load8(static_cast<const uint16_t*>(w) + e, v);
    return;
  }
  const f32x4_t* p = reinterpret_cast<const f32x4_t*>(static_cast<const float*>(w) + e);
  const f32x4_t a = p[0], b = p[1];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[i] = ROUND ? round_bf16(a[i]) : a[i];
    v[4 + i] = ROUND ? round_bf16(b[i]) : b[i];
  }
}

// Mean (LayerNorm only) and 1 / sqrt(var + eps) or 1 / sqrt(mean square +
// eps) of the row in v; entries past the row's end are zero and not counted.
template <int KIND, int L, int C>
__device__ __forceinline__ void row_stats(const float (&v)[C][8], int lane, int size, float eps,
                                          float* mean, float* rstd) {
  float s = 0.0f;
  *mean = 0.0f;
  if constexpr (KIND == kNormLayer) {
#pragma unroll
    for (int c = 0; c < C; ++c)
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[c][i];
    *mean = row_sum<L>(s) / static_cast<float>(size);
    s = 0.0f;
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    if ((c * L + lane) * 8 >= size) continue;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float d = v[c][i] - *mean;
      s = __builtin_fmaf(d, d, s);
    }
  }
  *rstd = rsqrtf(row_sum<L>(s) / static_cast<float>(size) + eps);
}

// y = norm(t), t = x or bf16(x + r), also written where there is a `sum` for
// it: L lanes a row, C chunks of 8 elements a lane.
template <int KIND, bool ADD, int L, int C>
__global__ void __launch_bounds__(kThreads)
    k_norm_fwd(const uint16_t* __restrict__ x, const uint16_t* __restrict__ r,
               const void* __restrict__ w, const void* __restrict__ b, int w_dtype, int64_t rows,
               int size, float eps, uint16_t* __restrict__ sum, uint16_t* __restrict__ y) {
  const int lane = threadIdx.x & (L - 1);
  const int64_t row = block_of_grid() * (kThreads / L) + threadIdx.x / L;
  if (row >= rows) return;
  const int64_t base = row * size;
  float v[C][8];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = (c * L + lane) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[c][i] = 0.0f;
    if (e >= size) continue;
    u32x4_t t = *reinterpret_cast<const u32x4_t*>(x + base + e);
    unpack8(t, v[c]);
    if constexpr (ADD) {
      float a[8];
      load8(r + base + e, a);
#pragma unroll
      for (int i = 0; i < 8; ++i) a[i] += v[c][i];
      t = pack8(a);
      unpack8(t, v[c]);
    }
    if (ADD || sum != nullptr) *reinterpret_cast<u32x4_t*>(sum + base + e) = t;
  }
  // the weights' loads are in flight while the statistics are summed
  float g[C][8], h[KIND == kNormLayer ? C : 1][8];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = (c * L + lane) * 8;
    if (e >= size) continue;
    load_weight8<KIND == kNormLayer>(w, w_dtype, e, g[c]);
    if constexpr (KIND == kNormLayer) load_weight8<true>(b, w_dtype, e, h[c]);
  }
  float mean, rstd;
  row_stats<KIND, L, C>(v, lane, size, eps, &mean, &rstd);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = (c * L + lane) * 8;
    if (e >= size) continue;
    if constexpr (KIND == kNormLayer) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        v[c][i] = __builtin_fmaf((v[c][i] - mean) * rstd, g[c][i], h[c][i]);
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) v[c][i] = v[c][i] * rstd * g[c][i];
    }
    *reinterpret_cast<u32x4_t*>(y + base + e) = pack8(v[c]);
  }
}

// v = the normalised row (in place of the row), g = the gradient of w * v:
// the input's gradient, left in g.
template <int KIND, int L, int C>
__device__ __forceinline__ void row_gradient(float (&v)[C][8], float (&g)[C][8], int size,
                                             float rstd) {
  float sg = 0.0f, sgv = 0.0f;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (KIND == kNormLayer) sg += g[c][i];
      sgv = __builtin_fmaf(g[c][i], v[c][i], sgv);
    }
  const float n = static_cast<float>(size);
  const float mg = KIND == kNormLayer ? row_sum<L>(sg) / n : 0.0f;
  const float mgv = row_sum<L>(sgv) / n;
#pragma unroll
  for (int c = 0; c < C; ++c)
#pragma unroll
    for (int i = 0; i < 8; ++i) g[c][i] = rstd * (g[c][i] - mg - v[c][i] * mgv);
}

// dx of y = norm(t) (+ the gradient that reaches t by its other use).
template <int KIND, bool ADD, int L, int C>
__global__ void __launch_bounds__(kThreads)
    k_norm_bwd(const uint16_t* __restrict__ dy, const uint16_t* __restrict__ dt,
               const uint16_t* __restrict__ t, const void* __restrict__ w, int w_dtype,
               int64_t rows, int size, float eps, uint16_t* __restrict__ dx) {
  const int lane = threadIdx.x & (L - 1);
  const int64_t row = block_of_grid() * (kThreads / L) + threadIdx.x / L;
  if (row >= rows) return;
  const int64_t base = row * size;
  float v[C][8], g[C][8];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = (c * L + lane) * 8;
#pragma unroll
    for (int i = 0; i < 8; ++i) v[c][i] = g[c][i] = 0.0f;
    if (e >= size) continue;
    load8(t + base + e, v[c]);
    load8(dy + base + e, g[c]);
  }
  float mean, rstd;
  row_stats<KIND, L, C>(v, lane, size, eps, &mean, &rstd);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = (c * L + lane) * 8;
    if (e >= size) continue;
    float wv[8];
    load_weight8<KIND == kNormLayer>(w, w_dtype, e, wv);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      v[c][i] = (v[c][i] - mean) * rstd;
      g[c][i] *= wv[i];
    }
  }
  row_gradient<KIND, L, C>(v, g, size, rstd);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int e = (c * L + lane) * 8;
    if (e >= size) continue;
    if constexpr (ADD) {
      float a[8];
      load8(dt + base + e, a);
#pragma unroll
      for (int i = 0; i < 8; ++i) g[c][i] += a[i];
    }
    *reinterpret_cast<u32x4_t*>(dx + base + e) = pack8(g[c]);
  }
}

// Heads of D = 8 * L elements, one per L lanes: lane l holds the elements
// 8 l .. 8 l + 7, so the rotation's other half is lane l ^ (L / 2). The parts
// (queries, keys and the values that only repeat) share a launch: blocks
// [first[p], first[p + 1]) are part p's, and first[kHeadParts] is their end. x [tokens, heads, D] dense; y [tokens,
// heads * repeat, D] dense, head h written `repeat` times.
__device__ __forceinline__ int head_part(const HeadNormArgs& a, int64_t block) {
  int p = 0;
  while (block >= a.first[p + 1]) ++p;
  return p;
}

template <int L>
__global__ void __launch_bounds__(kThreads) k_head_norm_fwd(HeadNormArgs a) {
  constexpr int kD = 8 * L;
  const int64_t block = block_of_grid();
  if (block >= a.first[kHeadParts]) return;
  const int p = head_part(a, block);
  const HeadPart& part = a.part[p];
  const int lane = threadIdx.x & (L - 1);
  const int64_t row = (block - a.first[p]) * (kThreads / L) + threadIdx.x / L;
  if (row >= a.tokens * part.heads) return;
  const int64_t token = row / part.heads;
  const int e = 8 * lane;
  u32x4_t out = *reinterpret_cast<const u32x4_t*>(part.x + row * kD + e);
  if (part.weight != nullptr) {
    float v[1][8], wv[8], cs[8], sn[8];
    unpack8(out, v[0]);
    load_weight8<false>(part.weight, part.weight_dtype, e, wv);
    const int64_t at = (token % a.sequence) * kD + e;
    load_weight8<false>(a.cosines + at, kF32, 0, cs);
    load_weight8<false>(a.sines + at, kF32, 0, sn);
    float mean, rstd;
    row_stats<kNormRms, L, 1>(v, lane, kD, part.eps, &mean, &rstd);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float n = round_bf16(v[0][i] * rstd * wv[i]);
      const float other = __shfl_xor(n, L / 2, 64);
      v[0][i] = n * cs[i] + (lane < L / 2 ? -other : other) * sn[i];
    }
    out = pack8(v[0]);
  }
  for (int j = 0; j < part.repeat; ++j)
    *reinterpret_cast<u32x4_t*>(part.out + (row * part.repeat + j) * kD + e) = out;
}

// dx; g's element (b, s, h, d) at b * stride_b + s * stride_s + h * stride_h + d.
template <int L>
__global__ void __launch_bounds__(kThreads) k_head_norm_bwd(HeadNormArgs a) {
  constexpr int kD = 8 * L;
  const int64_t block = block_of_grid();
  if (block >= a.first[kHeadParts]) return;
  const int p = head_part(a, block);
  const HeadPart& part = a.part[p];
  const int lane = threadIdx.x & (L - 1);
  const int64_t row = (block - a.first[p]) * (kThreads / L) + threadIdx.x / L;
  if (row >= a.tokens * part.heads) return;
  const int64_t token = row / part.heads;
  const int64_t s = token % a.sequence;
  const int64_t head = row % part.heads;
  const int e = 8 * lane;
  float dv[1][8];
#pragma unroll
  for (int i = 0; i < 8; ++i) dv[0][i] = 0.0f;
  const uint16_t* gr = part.g + (token / a.sequence) * part.stride_b + s * part.stride_s +
                       head * part.repeat * part.stride_h + e;
  for (int j = 0; j < part.repeat; ++j) {
    float t[8];
    load8(gr + j * part.stride_h, t);
#pragma unroll
    for (int i = 0; i < 8; ++i) dv[0][i] += t[i];
  }
  if (part.weight != nullptr) {
    float v[1][8], wv[8], cs[8], sn[8];
    load8(part.x + row * kD + e, v[0]);
    load_weight8<false>(part.weight, part.weight_dtype, e, wv);
    load_weight8<false>(a.cosines + s * kD + e, kF32, 0, cs);
    load_weight8<false>(a.sines + s * kD + e, kF32, 0, sn);
    float mean, rstd;
    row_stats<kNormRms, L, 1>(v, lane, kD, part.eps, &mean, &rstd);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // the rotation's transpose: the other half's gradient times its sine
      const float other = __shfl_xor(dv[0][i] * sn[i], L / 2, 64);
      const float dn = dv[0][i] * cs[i] + (lane < L / 2 ? other : -other);
      dv[0][i] = dn * wv[i];
      v[0][i] *= rstd;
    }
    row_gradient<kNormRms, L, 1>(v, dv, kD, rstd);
  }
  *reinterpret_cast<u32x4_t*>(part.out + row * kD + e) = pack8(dv[0]);
}

// Lanes a row and chunks a lane: the fewest that hold the row, so that short
// rows share a wave and no lane keeps more than 64 elements.
template <int KIND, bool ADD, int L, int C>
void norm_fwd(const NormArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((k_norm_fwd<KIND, ADD, L, C>),
                     grid_of(ceil_div(a.rows, kThreads / L)), dim3(kThreads), 0, stream, a.x, a.residual, a.weight, a.bias, a.weight_dtype, a.rows, a.size,
                     a.eps, a.sum, a.y);
}

template <int KIND, bool ADD, int L, int C>
void norm_bwd(const NormArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((k_norm_bwd<KIND, ADD, L, C>),
                     grid_of(ceil_div(a.rows, kThreads / L)), dim3(kThreads), 0, stream, a.x, a.residual, a.sum, a.weight, a.weight_dtype, a.rows, a.size,
                     a.eps, a.y);
}

template <int KIND, bool ADD>
void norm_sized(const NormArgs& a, bool backward, hipStream_t stream) {
#define RPX_NORM(L, C) \
  return backward ? norm_bwd<KIND, ADD, L, C>(a, stream) : norm_fwd<KIND, ADD, L, C>(a, stream)
  if (a.size <= 128) RPX_NORM(16, 1);
  if (a.size <= 768) RPX_NORM(32, 3);
  if (a.size <= 2048) RPX_NORM(64, 4);
  RPX_NORM(64, 8);
#undef RPX_NORM
}

}  // namespace

hipError_t launch_norm(const NormArgs& a, int kind, bool backward, hipStream_t stream) {
  if (a.rows <= 0) return hipSuccess;
  const bool add = a.residual != nullptr;
  if (kind == kNormLayer)
    add ? norm_sized<kNormLayer, true>(a, backward, stream)
        : norm_sized<kNormLayer, false>(a, backward, stream);
  else
    add ? norm_sized<kNormRms, true>(a, backward, stream)
        : norm_sized<kNormRms, false>(a, backward, stream);
  return hipGetLastError();
}

hipError_t launch_head_norm(HeadNormArgs a, int parts, bool backward, hipStream_t stream) {
  const int lanes = a.head_dim / 8;
  a.first[0] = 0;
  for (int p = 0; p < kHeadParts; ++p)
    a.first[p + 1] =
        a.first[p] + (p < parts ? ceil_div(a.tokens * a.part[p].heads, kThreads / lanes) : 0);
  if (a.first[parts] == 0) return hipSuccess;
  const auto kernel = a.head_dim == 128 ? (backward ? k_head_norm_bwd<16> : k_head_norm_fwd<16>)
                                        : (backward ? k_head_norm_bwd<8> : k_head_norm_fwd<8>);
  hipLaunchKernelGGL(kernel, grid_of(a.first[parts]), dim3(kThreads), 0, stream, a);
  return hipGetLastError();
}

}  // namespace rpx
