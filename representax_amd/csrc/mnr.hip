// In-batch multiple-negatives ranking loss, fused: the fp32 casts and row
// normalisation of both embedding sets, the scaled cosine logits, each
// query's log-sum-exp, the mean over queries, and the gradient of all of it
// (src/representax/tasks/retrieval/mnr.py:48-52 `_normalize`, :132-158
// `_direction_row_terms` with query i's positive = document i and unit
// weights, :338-341 the forward loss). Five launches (four forward, one
// backward) replace the ~30 small elementwise, reduction and matmul kernels of
// the unfused objective.
//
// Every sum runs in a fixed order (per-thread strided partials, then a
// shuffle tree, then the waves in order; MFMA chains, then the waves in
// order), so results do not depend on scheduling.
#include <hip/hip_runtime.h>

#include <cmath>

#include "common.h"
#include "kernels.h"

namespace rpx {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / 64;
constexpr int64_t kMnrMaxDim = 4096;

__device__ __forceinline__ float load_elem(const void* p, int dtype, int64_t i) {
  return dtype == kBF16 ? bf16_to_f32(static_cast<const uint16_t*>(p)[i])
                        : static_cast<const float*>(p)[i];
}

__device__ __forceinline__ void store_elem(void* p, int dtype, int64_t i, float v) {
  if (dtype == kBF16)
    static_cast<uint16_t*>(p)[i] = f32_to_bf16(v);
  else
    static_cast<float*>(p)[i] = v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
  return v;
}

// Block-wide sum, the same value in every thread: wave trees, then the
// waves' partials in wave order.
__device__ __forceinline__ float block_sum(float v, float* sh) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[wave] = v;
  __syncthreads();
  float s = sh[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) s += sh[w];
  return s;
}

__device__ __forceinline__ float block_max(float v, float* sh) {
  v = wave_max(v);
  const int wave = threadIdx.x >> 6;
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[wave] = v;
  __syncthreads();
  float m = sh[0];
#pragma unroll
  for (int w = 1; w < kWaves; ++w) m = fmaxf(m, sh[w]);
  return m;
}

// Block r: row r of the queries (r < nq) or row r - nq of the documents,
// cast to f32 and divided by max(||row||, 1e-12) (mnr.py:48-52); the
// unclamped norm is kept for the backward.
__global__ void __launch_bounds__(kThreads)
    k_mnr_normalize(const void* __restrict__ q, const void* __restrict__ d, int dtype, int64_t nq,
                    int64_t dim, float* __restrict__ unit, float* __restrict__ norms) {
  __shared__ float sh[kWaves];
  const int64_t r = blockIdx.x;
  const void* src = r < nq ? q : d;
  const int64_t row = r < nq ? r : r - nq;
  float ss = 0.0f;
  for (int64_t e = threadIdx.x; e < dim; e += kThreads) {
    const float v = load_elem(src, dtype, row * dim + e);
    ss = __builtin_fmaf(v, v, ss);
  }
  const float norm = sqrtf(block_sum(ss, sh));
  const float denom = fmaxf(norm, 1e-12f);
  for (int64_t e = threadIdx.x; e < dim; e += kThreads)
    unit[r * dim + e] = load_elem(src, dtype, row * dim + e) / denom;
  if (threadIdx.x == 0) norms[r] = norm;
}

// The two products of the loss and of its gradient run on the f32 MFMAs
// (v_mfma_f32_16x16x4: operands stay f32, products and sums are f32 FMAs).
// One 64-lane step covers 16 of the summed dimension: lane l = (r, g) with
// r = l % 16, g = l / 16 holds row r's four consecutive values 4g .. 4g + 3,
// and MFMA t sums position 4g + t of every group, the same permutation on
// both operands.
using f32x4 = float __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 mfma16(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Four consecutive values of a row at `e`, zeros from `end` on. VEC: `end`
// is a multiple of 4 and the rows are 16-byte aligned.
template <bool VEC>
__device__ __forceinline__ f32x4 load4(const float* row, int64_t e, int64_t end) {
  f32x4 v = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (VEC) {
    if (e < end) v = *reinterpret_cast<const f32x4*>(row + e);
  } else {
#pragma unroll
    for (int t = 0; t < 4; ++t)
      if (e + t < end) v[t] = row[e + t];
  }
  return v;
}

constexpr int kDotWaves = 8;
constexpr int kDotBatch = 6;  // steps of a wave in flight: all of them at width 768

// dots[i][j] = <q_i, d_j>: one 16 x 16 tile per workgroup, the embedding
// width dealt to eight waves in steps of 16 and their partial tiles summed in
// wave order. What bounds it is latency, not work (0.1 GFLOP at 256 x 256 x
// 768), hence the small tile (256 workgroups there) and the split sum. One
// query per workgroup with a shuffle tree per document, which this replaces,
// took 216 us of a 256-pair step; this one 5.4 us and the log-sum-exps 4.3.
template <bool VEC>
__global__ void __launch_bounds__(64 * kDotWaves)
    k_mnr_dots(const float* __restrict__ unit, int64_t nq, int64_t nd, int64_t dim,
               float* __restrict__ dots) {
  __shared__ float part[kDotWaves][256];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int64_t i0 = static_cast<int64_t>(blockIdx.y) * 16;
  const int64_t j0 = static_cast<int64_t>(blockIdx.x) * 16;
  // rows past the end read the last row; their products are not stored
  const float* qi = unit + (i0 + r < nq ? i0 + r : nq - 1) * dim;
  const float* dj = unit + (nq + (j0 + r < nd ? j0 + r : nd - 1)) * dim;
  f32x4 acc[2] = {};
  const int64_t steps = (dim + 15) / 16;
  for (int64_t c0 = wave; c0 < steps; c0 += kDotBatch * kDotWaves) {
    f32x4 a[kDotBatch], b[kDotBatch];
#pragma unroll
    for (int n = 0; n < kDotBatch; ++n) {
      const int64_t e = (c0 + n * kDotWaves) * 16 + 4 * g;
      a[n] = load4<VEC>(qi, e, dim);
      b[n] = load4<VEC>(dj, e, dim);
    }
#pragma unroll
    for (int n = 0; n < kDotBatch; ++n) {
      if (c0 + n * kDotWaves >= steps) break;
#pragma unroll
      for (int t = 0; t < 4; ++t) acc[t & 1] = mfma16(a[n][t], b[n][t], acc[t & 1]);
    }
  }
  // lane (r, g) holds column r of rows 4g .. 4g + 3
#pragma unroll
  for (int t = 0; t < 4; ++t) part[wave][(4 * g + t) * 16 + r] = acc[0][t] + acc[1][t];
  __syncthreads();
  if (threadIdx.x >= 256) return;
  float s = part[0][threadIdx.x];
#pragma unroll
  for (int w = 1; w < kDotWaves; ++w) s += part[w][threadIdx.x];
  const int64_t i = i0 + (threadIdx.x >> 4);
  const int64_t j = j0 + (threadIdx.x & 15);
  if (i < nq && j < nd) dots[i * nd + j] = s;
}

// l = scale * dot, rounded: one value of a logit wherever it is used. (Fused
// into the subtraction after it, the product would differ from the rounded one
// inside the log-sum-exp by more than a small loss is worth.)
__device__ __forceinline__ float logit(float dot, float scale) {
#pragma clang fp contract(off)
  return dot * scale;
}

// Block i (query i): logits l_j = scale * dots_ij and their log-sum-exp
// m + log(sum_j exp(l_j - m)). The row is read twice (from L2) rather than
// kept in LDS.
__global__ void __launch_bounds__(kThreads)
    k_mnr_rows(const float* __restrict__ dots, int64_t nd, float scale, float* __restrict__ lse) {
  __shared__ float sh[kWaves];
  const int64_t i = blockIdx.x;
  const float* row = dots + i * nd;
  float m = -INFINITY;
  for (int64_t j = threadIdx.x; j < nd; j += kThreads) m = fmaxf(m, logit(row[j], scale));
  m = block_max(m, sh);
  float s = 0.0f;
  for (int64_t j = threadIdx.x; j < nd; j += kThreads) s += expf(logit(row[j], scale) - m);
  s = block_sum(s, sh);
  if (threadIdx.x == 0) lse[i] = m + logf(s);
}

// loss = mean over queries of lse_i - l_ii (mnr.py:338-341, every query
// active).
__global__ void __launch_bounds__(kThreads)
    k_mnr_mean(const float* __restrict__ dots, const float* __restrict__ lse, int64_t nq,
               int64_t nd, float scale, float* __restrict__ loss) {
  __shared__ float sh[kWaves];
  float s = 0.0f;
  for (int64_t i = threadIdx.x; i < nq; i += kThreads) s += lse[i] - logit(dots[i * nd + i], scale);
  s = block_sum(s, sh);
  if (threadIdx.x == 0) loss[0] = s / static_cast<float>(nq);
}

// Gradient. With p_ij = exp(l_ij - lse_i) and c_ij = g * scale *
// (p_ij - [i == j]) / nq:
//   query i:    du = sum_j c_ij d_j,   <u, du> = sum_j c_ij dots_ij;
//   document j: du = sum_i c_ij q_i,   <u, du> = sum_i c_ij dots_ij;
// then through the normalisation u = v / max(||v||, 1e-12):
//   dv = (du - u <u, du>) / ||v|| when ||v|| > 1e-12, else du / 1e-12.
// A workgroup owns 16 rows (of the queries, or of the documents) and 64
// columns; its four waves split the summed rows in steps of 16 and are summed
// in wave order. Taking <u, du> from the saved dot products is what lets the
// columns go to different workgroups (384 at 256 pairs of 768; the whole-row
// form kept 512 with one output chain per thread and took 264 us; this one
// 10.7 us).
constexpr int kGradWaves = 4;
constexpr int kGradCols = 64;
constexpr int kGradBatch = 2;  // steps of a wave in flight

template <bool VEC>
__global__ void __launch_bounds__(64 * kGradWaves)
    k_mnr_grad(const float* __restrict__ unit, const float* __restrict__ norms,
               const float* __restrict__ dots, const float* __restrict__ lse, int64_t nq,
               int64_t nd, int64_t dim, float scale, const float* __restrict__ grad_loss,
               void* __restrict__ dq, void* __restrict__ dd, int dtype) {
  __shared__ float part[kGradWaves][16][kGradCols];
  __shared__ float proj_part[kGradWaves][16];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int r = lane & 15;
  const int g = lane >> 4;
  const int64_t q_tiles = (nq + 15) / 16;
  const bool is_q = blockIdx.y < q_tiles;
  const int64_t row0 = (is_q ? blockIdx.y : blockIdx.y - q_tiles) * 16;
  const int64_t rows = is_q ? nq : nd;
  const int64_t others = is_q ? nd : nq;
  const float* other = is_q ? unit + nq * dim : unit;
  const int64_t e0 = static_cast<int64_t>(blockIdx.x) * kGradCols;
  const float c0 = grad_loss[0] * scale / static_cast<float>(nq);
  const int64_t row = row0 + r;
  f32x4 acc[4] = {};
  float proj = 0.0f;
  const int64_t steps = (others + 15) / 16;
  for (int64_t s0 = wave; s0 < steps; s0 += kGradBatch * kGradWaves) {
    f32x4 b[kGradBatch][4];
    float dot[kGradBatch][4], l[kGradBatch][4];
#pragma unroll
    for (int n = 0; n < kGradBatch; ++n) {
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int64_t o = (s0 + n * kGradWaves) * 16 + 4 * g + t;
        b[n][t] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        dot[n][t] = l[n][t] = 0.0f;
        if (o >= others) continue;
        b[n][t] = load4<VEC>(other + o * dim, e0 + 4 * r, dim);
        if (row >= rows) continue;
        const int64_t i = is_q ? row : o;
        dot[n][t] = dots[i * nd + (is_q ? o : row)];
        l[n][t] = lse[i];
      }
    }
#pragma unroll
    for (int n = 0; n < kGradBatch; ++n) {
      if (s0 + n * kGradWaves >= steps) break;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const int64_t o = (s0 + n * kGradWaves) * 16 + 4 * g + t;
        float c = 0.0f;
        if (o < others && row < rows) {
          c = c0 * (expf(logit(dot[n][t], scale) - l[n][t]) - (o == row ? 1.0f : 0.0f));
          proj = __builtin_fmaf(c, dot[n][t], proj);
        }
        // column tile u holds the columns e0 + 4 * r + u
#pragma unroll
        for (int u = 0; u < 4; ++u) acc[u] = mfma16(c, b[n][t][u], acc[u]);
      }
    }
  }
#pragma unroll
  for (int t = 0; t < 4; ++t)
#pragma unroll
    for (int u = 0; u < 4; ++u) part[wave][4 * g + t][4 * r + u] = acc[u][t];
  proj += __shfl_xor(proj, 16, 64);
  proj += __shfl_xor(proj, 32, 64);
  if (g == 0) proj_part[wave][r] = proj;
  __syncthreads();

  const int tr = threadIdx.x >> 4;
  const int64_t orow = row0 + tr;
  if (orow >= rows) return;
  float pr = proj_part[0][tr];
#pragma unroll
  for (int w = 1; w < kGradWaves; ++w) pr += proj_part[w][tr];
  const int64_t urow = is_q ? orow : nq + orow;
  const float norm = norms[urow];
  const bool clamped = !(norm > 1e-12f);
  void* out = is_q ? dq : dd;
#pragma unroll
  for (int t = 0; t < 4; ++t) {
    const int col = (threadIdx.x & 15) + 16 * t;
    const int64_t e = e0 + col;
    if (e >= dim) continue;
    float du = part[0][tr][col];
#pragma unroll
    for (int w = 1; w < kGradWaves; ++w) du += part[w][tr][col];
    const float v = clamped ? du / 1e-12f : (du - unit[urow * dim + e] * pr) / norm;
    store_elem(out, dtype, orow * dim + e, v);
  }
}

}  // namespace

int64_t mnr_saved_floats(int64_t nq, int64_t nd, int64_t dim) {
  // unit rows (queries, then documents), norms, dot products, log-sum-exps
  return (nq + nd) * dim + (nq + nd) + nq * nd + nq;
}

bool mnr_shape_ok(int64_t nq, int64_t nd, int64_t dim) {
  return nq >= 1 && nd >= nq && nd <= kMnrMaxDocuments && dim >= 1 && dim <= kMnrMaxDim;
}

// 16-byte loads of the unit rows: every row starts at a multiple of 16 bytes.
static bool mnr_vector_rows(const float* unit, int64_t dim) {
  return dim % 4 == 0 && reinterpret_cast<uintptr_t>(unit) % 16 == 0;
}

hipError_t launch_mnr_forward(const void* q, const void* d, int dtype, int64_t nq, int64_t nd,
                              int64_t dim, float scale, float* loss, float* saved,
                              hipStream_t stream) {
  float* unit = saved;
  float* norms = unit + (nq + nd) * dim;
  float* dots = norms + (nq + nd);
  float* lse = dots + nq * nd;
  hipLaunchKernelGGL(k_mnr_normalize, dim3(static_cast<unsigned>(nq + nd)), dim3(kThreads), 0,
                     stream, q, d, dtype, nq, dim, unit, norms);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const auto k_dots = mnr_vector_rows(unit, dim) ? k_mnr_dots<true> : k_mnr_dots<false>;
  hipLaunchKernelGGL(k_dots,
                     dim3(static_cast<unsigned>((nd + 15) / 16),
                          static_cast<unsigned>((nq + 15) / 16)),
                     dim3(64 * kDotWaves), 0, stream, unit, nq, nd, dim, dots);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mnr_rows, dim3(static_cast<unsigned>(nq)), dim3(kThreads), 0, stream, dots,
                     nd, scale, lse);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_mnr_mean, dim3(1), dim3(kThreads), 0, stream, dots, lse, nq, nd, scale,
                     loss);
  return hipGetLastError();
}

hipError_t launch_mnr_backward(const float* grad_loss, const float* saved, int64_t nq, int64_t nd,
                               int64_t dim, float scale, void* dq, void* dd, int dtype,
                               hipStream_t stream) {
  const float* unit = saved;
  const float* norms = unit + (nq + nd) * dim;
  const float* dots = norms + (nq + nd);
  const float* lse = dots + nq * nd;
  const auto k_grad = mnr_vector_rows(unit, dim) ? k_mnr_grad<true> : k_mnr_grad<false>;
  hipLaunchKernelGGL(k_grad,
                     dim3(static_cast<unsigned>((dim + kGradCols - 1) / kGradCols),
                          static_cast<unsigned>((nq + 15) / 16 + (nd + 15) / 16)),
                     dim3(64 * kGradWaves), 0, stream, unit, norms, dots, lse, nq, nd, dim, scale,
                     grad_loss, dq, dd, dtype);
  return hipGetLastError();
}

}  // namespace rpx
