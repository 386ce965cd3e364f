// float32 matrix products of any shape and stride for gfx950: out[M, N] f32 =
// sum_k A(m, k) B(n, k), with A and B float32, bf16 or (B) a packed INT4
// weight, each read along either of its dimensions. These carry the INT4 +
// LoRA linear in float32 compute, its promoted form (bf16 activations against
// float32 masters) and bf16 shapes the MFMA path does not take.
//
// Every product and sum is float32 (v_mfma_f32_*: no operand is rounded or
// split), so the results differ from a scalar fma chain only in the order of
// their sums. Two kernels:
//   k_gemm_f32       64 x 64 outputs per workgroup of four 32 x 32 waves, K
//                    in blocks of 32 through LDS as [k][row] (one conflict-
//                    free dword per lane and MFMA operand), the next block's
//                    global loads in registers under the MFMAs;
//   k_gemm_f32_thin  outputs with a side of at most 64 (the adapter products:
//                    rank-wide or rank-high), 16 x 16 outputs per workgroup
//                    of 16 waves that split K and sum in LDS in wave order.
// They replace one output per thread over 16 x 16 LDS tiles. Bound: at these
// sizes the loads' latency behind few workgroups (the f32 matrix rate, 157
// TFLOP/s nominal, would allow 30 us per large product). Measured at 1000 x
// 3072 <- 768, float32, group 64, rank 16 (kernel traces, us): the eight
// products of forward and backward 1107 -> 245, of them x W_b^T 74 and g W_b
// 99; the whole linear, forward and backward, 1080 -> 258.
#include <atomic>

#include "common.h"
#include "kernels.h"
#include "tuning.h"

namespace rpx {

namespace {

// One operand: element (row, k) at row * s_row + k * s_k, or the packed
// weight's W[row, k] (kInt4) or W[k, row] (kInt4T).
enum OperandKind : int {
  kAlongK = 0,    // s_k == 1: four consecutive k per load
  kAlongRow = 1,  // s_row == 1: four consecutive rows per load
  kStrided = 2,
  kInt4 = 3,
  kInt4T = 4,
};
struct F32Operand {
  const void* p = nullptr;
  int dtype = kF32;
  int64_t s_row = 0, s_k = 0;
  int kind = kStrided;
  bool vec = false;     // four-element loads (or two packed bytes) are aligned
  int group_shift = 0;  // packed: log2 of a group's columns (kNoShift: divide)
  Int4Operand w;
};
constexpr int kNoShift = -1;
constexpr int kOneGroup = 62;  // a shift that maps every column to group 0

__device__ __forceinline__ float load_elem(const void* p, int dtype, int64_t idx) {
  if (dtype == kBF16) return bf16_to_f32(static_cast<const uint16_t*>(p)[idx]);
  return static_cast<const float*>(p)[idx];
}

__device__ __forceinline__ float int4_value(uint32_t nib, float s) {
  return round_bf16(static_cast<float>(static_cast<int>((nib & 15u) ^ 8u) - 8) * s);
}

__device__ __forceinline__ float int4_elem(const Int4Operand& w, int64_t row, int64_t col) {
  const uint32_t byte = w.packed[row * w.packed_cols + col / 2];
  const int64_t g = w.n_groups == 1 ? 0 : col / w.group;
  return int4_value((col & 1) ? (byte >> 4) : byte, bf16_to_f32(w.scales[row * w.n_groups + g]));
}

__device__ __forceinline__ float elem(const F32Operand& o, int64_t row, int64_t k) {
  if (o.kind == kInt4) return int4_elem(o.w, row, k);
  if (o.kind == kInt4T) return int4_elem(o.w, k, row);
  return load_elem(o.p, o.dtype, row * o.s_row + k * o.s_k);
}

// Four consecutive elements at p, which is aligned for them.
__device__ __forceinline__ f32x4_t four_at(const uint8_t* p, int dtype) {
  if (dtype == kBF16) {
    const u32x2_t w = *reinterpret_cast<const u32x2_t*>(p);
    return f32x4_t{bf16lo_to_f32(w[0]), bf16hi_to_f32(w[0]), bf16lo_to_f32(w[1]),
                   bf16hi_to_f32(w[1])};
  }
  return *reinterpret_cast<const f32x4_t*>(p);
}

// Four elements along the operand's contiguous dimension, one at a time, from
// (row, k): k .. k + 3 (kAlongK, kStrided, kInt4) or row .. row + 3 (kAlongRow,
// kInt4T); zero outside rows x K.
__device__ __forceinline__ f32x4_t load4_any(const F32Operand& o, int64_t row, int64_t k,
                                             int64_t rows, int64_t K) {
  const bool by_row = o.kind == kAlongRow || o.kind == kInt4T;
  f32x4_t v{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int64_t r = by_row ? row + e : row;
    const int64_t c = by_row ? k : k + e;
    if (r < rows && c < K) v[e] = elem(o, r, c);
  }
  return v;
}

constexpr int kTile = 64;
constexpr int kBlockK = 32;
// LDS row of one k: 64 rows plus two words, so that the four k rows a
// row-major load writes land on different banks
constexpr int kPitch = kTile + 2;

// This thread's two loads of the 64-row x 32-k blocks of one operand, from
// block to block `step` k further on. KIND: the operand's kind, or kStrided
// for one that takes the element path everywhere. Blocks with all their k take
// vector loads through two running pointers; rows past the last re-read it
// (or its last four), which only feeds outputs that are not stored. With edge
// blocks on the element path their workgroups set the launch's time: 1000 x
// 3072 <- 768 took 104 us instead of 74.
template <int KIND>
struct BlockLoads {
  const F32Operand& o;
  int64_t row0, rows, K;
  int tid;
  const uint8_t* p[2];
  const uint16_t* sc[2];
  int64_t p_step = 0, sc_step = 0;

  __device__ __forceinline__ bool by_row() const {
    return KIND == kStrided ? o.kind == kAlongRow || o.kind == kInt4T
                            : KIND == kAlongRow || KIND == kInt4T;
  }
  __device__ __forceinline__ int64_t row_of(int i) const {
    return row0 + (by_row() ? 4 * (tid & 15) : (tid >> 3) + 32 * i);
  }
  __device__ __forceinline__ int k_of(int i) const {
    return by_row() ? (tid >> 4) + 16 * i : 4 * (tid & 7);
  }
  __device__ __forceinline__ BlockLoads(const F32Operand& op, int64_t r0, int64_t k0, int64_t step,
                                        int64_t nrows, int64_t depth, int t)
      : o(op), row0(r0), rows(nrows), K(depth), tid(t) {
    const int64_t es = o.dtype == kBF16 ? 2 : 4;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      int64_t row = row_of(i);
      const int64_t last = by_row() ? rows - 4 : rows - 1;
      if (row > last) row = last;
      const int64_t k = k0 + k_of(i);
      sc[i] = nullptr;
      if constexpr (KIND == kInt4) {
        p[i] = o.w.packed + row * o.w.packed_cols + k / 2;
        sc[i] = o.w.scales + row * o.w.n_groups;
      } else if constexpr (KIND == kInt4T) {
        p[i] = o.w.packed + k * o.w.packed_cols + row / 2;
        sc[i] = o.w.scales + k * o.w.n_groups + (row >> o.group_shift);
      } else {
        p[i] = static_cast<const uint8_t*>(o.p) + (row * o.s_row + k * o.s_k) * es;
      }
    }
    if constexpr (KIND == kInt4) {
      p_step = step / 2;
    } else if constexpr (KIND == kInt4T) {
      p_step = step * o.w.packed_cols;
      sc_step = step * o.w.n_groups;
    } else {
      p_step = step * o.s_k * es;
    }
  }
  // the block at k0, which the pointers are at; moves them on
  __device__ __forceinline__ void next(int64_t k0, f32x4_t* v) {
    const bool vec = KIND != kStrided && k0 + kBlockK <= K && (!by_row() || (rows & 3) == 0);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if (vec) {
        if constexpr (KIND == kInt4 || KIND == kInt4T) {
          const uint32_t two = *reinterpret_cast<const uint16_t*>(p[i]);
          const int64_t g = KIND == kInt4 ? (k0 + k_of(i)) >> o.group_shift : 0;
          const float s = bf16_to_f32(sc[i][g]);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[i][e] = int4_value(two >> (4 * e), s);
        } else {
          v[i] = four_at(p[i], o.dtype);
        }
      } else if (k0 < K) {
        v[i] = load4_any(o, row_of(i), k0 + k_of(i), rows, K);
      } else {
        v[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
      p[i] += p_step;
      sc[i] += sc_step;
    }
  }
};
template <int KIND>
__device__ __forceinline__ void store_block(const F32Operand& o, float* lds, int tid,
                                            const f32x4_t* v) {
  const bool by_row = KIND == kStrided ? o.kind == kAlongRow || o.kind == kInt4T
                                       : KIND == kAlongRow || KIND == kInt4T;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    if (by_row) {
      float* d = lds + ((tid >> 4) + 16 * i) * kPitch + 4 * (tid & 15);
      *reinterpret_cast<f32x2_t*>(d) = f32x2_t{v[i][0], v[i][1]};
      *reinterpret_cast<f32x2_t*>(d + 2) = f32x2_t{v[i][2], v[i][3]};
    } else {
      float* d = lds + 4 * (tid & 7) * kPitch + (tid >> 3) + 32 * i;
#pragma unroll
      for (int e = 0; e < 4; ++e) d[e * kPitch] = v[i][e];
    }
  }
}

// G groups of four waves take the K blocks in turn (block group + G i) and are
// summed in group order at the end: outputs too few to fill the chip with one
// group each get their waves from K.
template <int AK, int BK, int G>
__global__ void __launch_bounds__(256 * G)
    k_gemm_f32(F32Operand A, F32Operand B, int64_t M, int64_t N, int64_t K, int64_t tiles_n,
               float* __restrict__ out) {
  constexpr int kBuf = kBlockK * kPitch;  // floats of one operand's block
  extern __shared__ __align__(16) float lds[];
  const int tid = threadIdx.x & 255;
  const int group = threadIdx.x >> 8;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  float* const sa = lds + group * 4 * kBuf;  // two buffers each
  float* const sb = sa + 2 * kBuf;
  const int64_t tile = block_of_grid();
  if (tile >= ceil_div(M, kTile) * tiles_n) return;
  const int64_t m0 = tile / tiles_n * kTile;
  const int64_t n0 = tile % tiles_n * kTile;
  const int wm = 32 * (wave & 1);
  const int wn = 32 * (wave >> 1);
  f32x16_t acc;
#pragma unroll
  for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
  // the global loads of the next two blocks are in flight in registers
  constexpr int64_t kStep = int64_t{kBlockK} * G;
  int64_t k0 = int64_t{kBlockK} * group;
  f32x4_t va[2][2], vb[2][2];
  BlockLoads<AK> la(A, m0, k0, kStep, M, K, tid);
  BlockLoads<BK> lb(B, n0, k0, kStep, N, K, tid);
#pragma unroll
  for (int d = 0; d < 2; ++d) {
    la.next(k0 + d * kStep, va[d]);
    lb.next(k0 + d * kStep, vb[d]);
  }
  const int64_t rounds = (K + kStep - 1) / kStep;  // the same for every group
  int buf = 0;
  for (int64_t i = 0; i < rounds; ++i, k0 += kStep) {
    store_block<AK>(A, sa + buf * kBuf, tid, va[0]);
    store_block<BK>(B, sb + buf * kBuf, tid, vb[0]);
    // the two buffers alternate, so this barrier also keeps a block's stores
    // behind every wave's reads of the block before the last
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      va[0][j] = va[1][j];
      vb[0][j] = vb[1][j];
    }
    la.next(k0 + 2 * kStep, va[1]);
    lb.next(k0 + 2 * kStep, vb[1]);
    const int64_t left = K - k0;
    const int steps = left >= kBlockK ? kBlockK / 2 : (left > 0 ? static_cast<int>((left + 1) / 2) : 0);
    // lane: row lane % 32 of its operand, k = 2 step + lane / 32; B first, so
    // a lane's outputs are columns 8 (v / 4) + 4 (lane / 32) + v % 4 of row
    // lane % 32
    const float* pa = sa + buf * kBuf + (lane >> 5) * kPitch + wm + (lane & 31);
    const float* pb = sb + buf * kBuf + (lane >> 5) * kPitch + wn + (lane & 31);
    if (steps == kBlockK / 2) {
#pragma unroll
      for (int s = 0; s < kBlockK / 2; ++s)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(pb[2 * s * kPitch], pa[2 * s * kPitch], acc, 0,
                                                   0, 0);
    } else {
      for (int s = 0; s < steps; ++s)
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(pb[2 * s * kPitch], pa[2 * s * kPitch], acc, 0,
                                                   0, 0);
    }
    buf ^= 1;
  }
  if constexpr (G > 1) {
    __syncthreads();  // every wave is done with the blocks
    if (group > 0) {
#pragma unroll
      for (int v = 0; v < 16; ++v) sa[v * 256 + tid] = acc[v];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int g = 1; g < G; ++g)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[v] += lds[g * 4 * kBuf + v * 256 + tid];
  }
  const int64_t m = m0 + wm + (lane & 31);
  if (m >= M) return;
  const bool vec = (N & 3) == 0 && (reinterpret_cast<uintptr_t>(out) & 15) == 0;
#pragma unroll
  for (int vg = 0; vg < 4; ++vg) {
    const int64_t n = n0 + wn + 8 * vg + 4 * (lane >> 5);
    float* d = out + m * N + n;
    if (vec && n + 3 < N) {
      *reinterpret_cast<f32x4_t*>(d) =
          f32x4_t{acc[4 * vg], acc[4 * vg + 1], acc[4 * vg + 2], acc[4 * vg + 3]};
    } else {
      for (int e = 0; e < 4; ++e)
        if (n + e < N) d[e] = acc[4 * vg + e];
    }
  }
}

template <int AK, int BK, int G>
hipError_t run_f32_groups(const F32Operand& a, const F32Operand& b, int64_t m, int64_t n, int64_t k,
                          float* out, hipStream_t stream) {
  constexpr int kLds = G * 4 * kBlockK * kPitch * 4;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  auto kern = k_gemm_f32<AK, BK, G>;
  static std::atomic<unsigned> lds_set{0};
  const hipError_t e = ensure_lds_limit(reinterpret_cast<const void*>(kern), kLds, lds_set);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, grid_of(ceil_div(m, kTile) * ceil_div(n, kTile)), dim3(256 * G), kLds, stream, a, b, m, n, k, ceil_div(n, kTile), out);
  return hipGetLastError();
}

// Four groups where the 64 x 64 outputs give fewer than two workgroups per CU
// and K has blocks for them, else one (1000 x 768 <- 3072, 192 workgroups: 99
// us with four groups, although they spill 17 registers, 122 with two, about
// 200 with one).
template <int AK, int BK>
hipError_t run_f32(const F32Operand& a, const F32Operand& b, int64_t m, int64_t n, int64_t k,
                   float* out, hipStream_t stream) {
  if (ceil_div(m, kTile) * ceil_div(n, kTile) < 512 && k >= 8 * kBlockK)
    return run_f32_groups<AK, BK, 4>(a, b, m, n, k, out, stream);
  return run_f32_groups<AK, BK, 1>(a, b, m, n, k, out, stream);
}

constexpr int kThinWaves = 16;
constexpr int kThinK = 16;  // k per wave and step

// Lane fragment of a 16-row x 16-k step: element e is (row0 + lane % 16, k0 +
// 4 (lane / 16) + e), the same k for both operands.
template <int KIND>
__device__ __forceinline__ f32x4_t thin_frag(const F32Operand& o, int64_t row0, int64_t k0,
                                             int64_t rows, int64_t K, int lane) {
  const int64_t row = row0 + (lane & 15);
  const int64_t k = k0 + 4 * (lane >> 4);
  f32x4_t v{0.0f, 0.0f, 0.0f, 0.0f};
  if (row >= rows) return v;
  const bool four = k + 3 < K;
  if constexpr (KIND == kAlongK) {
    if (four && o.vec)
      return four_at(static_cast<const uint8_t*>(o.p) +
                         (row * o.s_row + k) * (o.dtype == kBF16 ? 2 : 4),
                     o.dtype);
  }
  if constexpr (KIND == kAlongRow) {
    if (four) {
      const int64_t at = row + k * o.s_k;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = load_elem(o.p, o.dtype, at + e * o.s_k);
      return v;
    }
  }
#pragma unroll
  for (int e = 0; e < 4; ++e)
    if (k + e < K) v[e] = elem(o, row, k + e);
  return v;
}

template <int AK, int BK>
__global__ void __launch_bounds__(64 * kThinWaves)
    k_gemm_f32_thin(F32Operand A, F32Operand B, int64_t M, int64_t N, int64_t K, int64_t tiles_n,
                    float* __restrict__ out) {
  __shared__ f32x4_t red[kThinWaves - 1][64];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int64_t tile = block_of_grid();
  if (tile >= ceil_div(M, 16) * tiles_n) return;
  const int64_t m0 = tile / tiles_n * 16;
  const int64_t n0 = tile % tiles_n * 16;
  f32x4_t acc{0.0f, 0.0f, 0.0f, 0.0f};
  constexpr int U = 4;  // steps in flight
  for (int64_t k0 = wave * kThinK; k0 < K; k0 += U * kThinWaves * kThinK) {
    f32x4_t fa[U], fb[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      fa[u] = thin_frag<AK>(A, m0, k0 + u * kThinWaves * kThinK, M, K, lane);
      fb[u] = thin_frag<BK>(B, n0, k0 + u * kThinWaves * kThinK, N, K, lane);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc = __builtin_amdgcn_mfma_f32_16x16x4f32(fb[u][e], fa[u][e], acc, 0, 0, 0);
  }
  if (wave > 0) red[wave - 1][lane] = acc;
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int w = 0; w < kThinWaves - 1; ++w) acc += red[w][lane];
  // columns 4 (lane / 16) + v of row lane % 16
  const int64_t m = m0 + (lane & 15);
  const int64_t n = n0 + 4 * (lane >> 4);
  if (m >= M) return;
#pragma unroll
  for (int v = 0; v < 4; ++v)
    if (n + v < N) out[m * N + n + v] = acc[v];
}

F32Operand dense_operand(const void* p, int dtype, int64_t s_row, int64_t s_k) {
  F32Operand o;
  o.p = p;
  o.dtype = dtype;
  o.s_row = s_row;
  o.s_k = s_k;
  const uintptr_t bytes = dtype == kBF16 ? 8 : 16;  // of four elements
  const bool base = (reinterpret_cast<uintptr_t>(p) & (bytes - 1)) == 0;
  if (s_k == 1) {
    o.kind = kAlongK;
    o.vec = base && s_row % 4 == 0;
  } else if (s_row == 1) {
    o.kind = kAlongRow;
    o.vec = base && s_k % 4 == 0;
  }
  return o;
}

}  // namespace

hipError_t launch_generic_gemm(const void* a, int a_dtype, int64_t a_sm, int64_t a_sk,
                               const void* b, int b_dtype, int64_t b_sn, int64_t b_sk,
                               const Int4Operand* b_int4, bool int4_transposed, int64_t m,
                               int64_t n, int64_t k, float* out, hipStream_t stream) {
  if (m == 0 || n == 0) return hipSuccess;
  const F32Operand oa = dense_operand(a, a_dtype, a_sm, a_sk);
  F32Operand ob;
  if (b_int4 != nullptr) {
    ob.kind = int4_transposed ? kInt4T : kInt4;
    ob.w = *b_int4;
    // two packed bytes (four columns) of one row and one scale group
    ob.group_shift = kNoShift;
    if (b_int4->n_groups == 1) {
      ob.group_shift = kOneGroup;
    } else {
      for (int sh = 2; sh < 32; ++sh)
        if (b_int4->group == (int64_t{1} << sh)) ob.group_shift = sh;
    }
    ob.vec = b_int4->packed_cols % 2 == 0 && ob.group_shift != kNoShift &&
             (reinterpret_cast<uintptr_t>(b_int4->packed) & 1) == 0;
  } else {
    ob = dense_operand(b, b_dtype, b_sn, b_sk);
  }
  const bool thin = m <= kTile || n <= kTile;
  const int64_t side = thin ? 16 : kTile;
  const int64_t tiles_n = ceil_div(n, side);
  const int64_t tiles = ceil_div(m, side) * tiles_n;
  if (tiles >= (int64_t{1} << 31)) return hipErrorInvalidValue;
  // the kinds the linear's products have; any other (or an operand without
  // aligned vectors, in the 64 x 64 kernel) takes the element path. A short
  // reduction (an adapter's up-projection, K = rank) gives the thin kernel's
  // waves nothing to split.
  if (thin && k > 2 * kThinK) {
    auto run = [&](auto kern) {
      hipLaunchKernelGGL(kern, grid_of(tiles), dim3(64 * kThinWaves), 0, stream, oa, ob, m, n, k, tiles_n, out);
    };
    if (oa.kind == kAlongK && ob.kind == kAlongK)
      run(k_gemm_f32_thin<kAlongK, kAlongK>);
    else if (oa.kind == kAlongK && ob.kind == kAlongRow)
      run(k_gemm_f32_thin<kAlongK, kAlongRow>);
    else if (oa.kind == kAlongRow && ob.kind == kAlongRow)
      run(k_gemm_f32_thin<kAlongRow, kAlongRow>);
    else
      run(k_gemm_f32_thin<kStrided, kStrided>);
  } else {
    const bool vec = oa.vec && ob.vec && oa.kind == kAlongK;
    if (vec && ob.kind == kInt4) return run_f32<kAlongK, kInt4>(oa, ob, m, n, k, out, stream);
    if (vec && ob.kind == kInt4T) return run_f32<kAlongK, kInt4T>(oa, ob, m, n, k, out, stream);
    if (vec && ob.kind == kAlongK) return run_f32<kAlongK, kAlongK>(oa, ob, m, n, k, out, stream);
    if (vec && ob.kind == kAlongRow) return run_f32<kAlongK, kAlongRow>(oa, ob, m, n, k, out, stream);
    return run_f32<kStrided, kStrided>(oa, ob, m, n, k, out, stream);
  }
  return hipGetLastError();
}

}  // namespace rpx
