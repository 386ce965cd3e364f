// bf16 MFMA "NT" GEMM on 256-row tiles for gfx950, for the large products of
// the INT4 + LoRA linear: the forward over a bf16 copy of W_b (dequantized
// into the call's workspace by a 3-8 us launch) and the input gradient over
// W_b^T, with the LoRA, bias and activation epilogues of k_gemm_nt.
//
// What bounds it: power, then the LDS reads and L2 loads. A workgroup of eight
// waves computes 256 x 256 (waves of 128 x 64) or 256 x 192 (waves of 64 x 96)
// outputs, so a 64-deep K slice moves 64 or 56 KB from L2 for 2048 or 1536
// MFMA clocks: about half the L2 traffic per MFMA of a 256 x 128 tile, which
// is what those tiles wait for. Without its LDS reads and its loads the main
// loop runs at 2.03 PFLOP/s (the chip clocks down to 1.8 GHz under it), with
// either at 1.55, with both at 1.25-1.35 (1.65 GHz, the MFMAs busy 72% of the
// cycles). Two stages of 128-byte rows measured 5-10% faster than three or
// four stages of 64-byte rows (half lines: every L2 line is asked for twice).
//
// The grid is persistent, at most one workgroup per CU: the direct-to-LDS
// loads run one slice ahead across tile boundaries, so a tile's first slices
// land under the previous tile's last MFMAs and epilogue. Each wave stages
// its outputs 32 rows at a time in its own few KB of LDS behind the two
// stages, so the epilogue needs no workgroup barrier and leaves the pipeline
// stages alone. The epilogue's arithmetic is not hidden (one workgroup per
// CU), so its registers are: no kernel below spills more than 3 (with 40-140
// spilled the gated forward took 553 us instead of 423).
//
// Measured against k_gemm_nt's tiles, kernel traces, us (the forward's
// dequantization, 4-10 us, not included):
//   16384 x 6144 <- 2048, rank 32     forward 441 -> 337, gated 483 -> 422
//   16384 x 2048 <- 6144              forward 441 -> 337, dx 412 -> 337
//   16384 x 6144 <- 2048, gated dx    641 -> 453
//   32768 x 3072 <- 768, rank 16      GELU forward 285 -> 238, GELU dx 316 -> 254
//   32768 x 768 <- 3072               forward 174 -> 134, dx 166 -> 134
// The MFMA sequence of an output (which k go into which MFMA, and the order)
// is k_gemm_nt's, so the outputs are the same bit for bit.
#include <atomic>
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "act.h"
#include "lds_pipeline.h"
#include "tuning.h"

namespace rpx {

namespace {

constexpr int kBK = 64;      // k elements per slice
constexpr int kStages = 2;   // pipeline stages
constexpr int kSteps = 4;    // 16-deep MFMA steps per slice

__device__ __forceinline__ bf16x8_t as_bf16x8(u32x4_t v) {
  return __builtin_bit_cast(bf16x8_t, v);
}

__device__ __forceinline__ void round2(float& a, float& b) {
  const uint32_t p = pack_bf16x2(a, b);
  a = bf16lo_to_f32(p);
  b = bf16hi_to_f32(p);
}

// One direct-to-LDS load of 16 bytes per lane: lane l writes dst + 16 l.
__device__ __forceinline__ void dma16(const uint8_t* src, uint8_t* dst) {
  __builtin_amdgcn_global_load_lds(
      src, reinterpret_cast<lds_void_t*>(reinterpret_cast<uintptr_t>(dst)), 16, 0, 0);
}

// Physical 16-byte chunk of logical chunk c in row r of a wave's staging rows
// (CPR chunks per row): 8 chunks use the low row bits; 12 chunks permute
// within groups of four.
template <int CPR>
__device__ __forceinline__ int stage_chunk(int r, int c) {
  return CPR == 8 ? (c ^ (r & 7)) : (c ^ ((r >> 2) & 3));
}

// JB: 16-rank blocks of the LoRA term, rank = 16 JB.
template <int BN, int WM, int WN, int JB, int ACT>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
    k_gemm_wide(const uint8_t* __restrict__ A, int64_t lda_bytes, const uint8_t* __restrict__ B,
                int64_t ldb_bytes, int M, int N, int K, uint16_t* __restrict__ out, int64_t ldc,
                LowRankEpilogue epi, int tiles_m, int tiles_n, int band) {
  constexpr int BM = 256;
  constexpr int NW = WM * WN;
  static_assert(NW == 8, "eight waves");
  constexpr int TM = BM / WM;
  constexpr int TN = BN / WN;
  constexpr int FM = TM / 32;
  constexpr int FN = TN / 32;
  constexpr int ROW = 2 * kBK;  // bytes of an LDS row
  constexpr int STAGE = (BM + BN) * ROW;
  constexpr int A_SEGS = BM / 8;
  constexpr int LPW = (BM + BN) / 8 / NW;  // loads per wave and slice
  static_assert((BM + BN) % (8 * NW) == 0, "DMA segments must split evenly over the waves");
  constexpr int CPR = TN / 8;  // 16-byte chunks per staged row
  static_assert(CPR == 8 || CPR == 12, "staging swizzle");
  constexpr int ITS = 32 * CPR / 64;
  constexpr int NMF = FM * FN;
  extern __shared__ __align__(16) uint8_t smem[];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM;
  const int wn = wave / WM;
  const int half = lane >> 5;
  const int frow = lane & 31;
  const int nk = K / kBK;
  const int tiles = tiles_m * tiles_n;
  const int grid = static_cast<int>(gridDim.x);
  const int first = xcd_block(static_cast<int>(blockIdx.x), grid);  // grid <= tiles

  // Load cursor (tile lt, slice ls), kStages slices ahead of the MFMAs and
  // running on into the workgroup's next tile. Segment wave + i NW is 8 rows
  // of A or of B; rows past the edge re-read the last row. Past the last
  // tile the loads repeat its last slice into a stage nothing reads again.
  uint32_t off[LPW];
  auto tile_offsets = [&](int t) {
    int tm, tn;
    band_tile(t, tiles_m, tiles_n, band, tm, tn);
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
      const int j = wave + i * NW;
      const int trow = (j < A_SEGS ? 8 * j : 8 * (j - A_SEGS)) + (lane >> 3);
      const int chunk = ((lane & 7) ^ swz(trow)) << 4;
      if (j < A_SEGS) {
        int r = tm * BM + trow;
        r = r < M ? r : M - 1;
        off[i] = static_cast<uint32_t>(r) * static_cast<uint32_t>(lda_bytes) + chunk;
      } else {
        int r = tn * BN + trow;
        r = r < N ? r : N - 1;
        off[i] = static_cast<uint32_t>(r) * static_cast<uint32_t>(ldb_bytes) + chunk;
      }
    }
  };
  int lt = first, ls = 0;
  tile_offsets(lt);
  auto advance = [&]() {
    if (++ls < nk) return;
    if (lt + grid < tiles) {
      lt += grid;
      ls = 0;
      tile_offsets(lt);
    } else {
      ls = nk - 1;
    }
  };
  auto load_seg = [&](int stage, int i) {
    const int j = wave + i * NW;
    const uint8_t* base = (j < A_SEGS ? A : B) + static_cast<int64_t>(ls) * ROW;
    dma16(base + off[i], smem + stage * STAGE + j * 1024);
  };

  // Fragment addresses within a stage: step kk takes k = 32 half + 8 kk +
  // [0, 8) of each row, as k_gemm_nt does.
  uint32_t a_off[kSteps], b_off[kSteps];
#pragma unroll
  for (int kk = 0; kk < kSteps; ++kk) {
    const int ar = wm * TM + frow;
    const int br = wn * TN + frow;
    a_off[kk] = ar * ROW + (((4 * half + kk) ^ swz(ar)) << 4);
    b_off[kk] = BM * ROW + br * ROW + (((4 * half + kk) ^ swz(br)) << 4);
  }
  f32x16_t acc[FN][FM];
  bf16x8_t af[2][FM], bf[2][FN];
  auto read_a = [&](uint32_t base, int kk, int buf) {
#pragma unroll
    for (int f = 0; f < FM; ++f)
      af[buf][f] = *reinterpret_cast<const bf16x8_t*>(smem + base + a_off[kk] + f * 32 * ROW);
  };
  auto read_b = [&](uint32_t base, int kk, int buf) {
#pragma unroll
    for (int f = 0; f < FN; ++f)
      bf[buf][f] = *reinterpret_cast<const bf16x8_t*>(smem + base + b_off[kk] + f * 32 * ROW);
  };
  auto mma = [&](int i, int buf) {
    acc[i / FM][i % FM] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bf[buf][i / FM], af[buf][i % FM],
                                                                  acc[i / FM][i % FM], 0, 0, 0);
  };

  for (int s = 0; s < kStages; ++s) {
#pragma unroll
    for (int i = 0; i < LPW; ++i) load_seg(s, i);
    advance();
  }
  wait_sync<(kStages - 1) * LPW>();
  read_a(0, 0, 0);
  read_b(0, 0, 0);
  int stage = 0;
  uint8_t* const st = smem + kStages * STAGE + wave * (32 * TN * 2);  // this wave's staging rows

  const uint32_t sbits = __builtin_bit_cast(uint32_t, epi.scale);
  // bf16(t) * scale is already a bf16 value when scale = 2^k, k >= 0
  const bool scale_exact = (sbits & 0x807FFFFFu) == 0 && sbits >= 0x3F800000u && sbits < 0x7F800000u;
  // (the backward epilogues carry no bias)
  const bool has_bias = (ACT == kActNone || ACT == kActGeluFwd || ACT == kActSiluMulFwd) && epi.bias != nullptr;
  const bool bias_vec = (reinterpret_cast<uintptr_t>(epi.bias) & 7) == 0;
  constexpr int kJB = JB > 0 ? JB : 1;

  for (int t = first; t < tiles; t += grid) {
#pragma unroll
    for (int fn = 0; fn < FN; ++fn)
#pragma unroll
      for (int fm = 0; fm < FM; ++fm)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[fn][fm][v] = 0.0f;

    int tm, tn;
    band_tile(t, tiles_m, tiles_n, band, tm, tn);
    const int mw = tm * BM + wm * TM;
    const int nw = tn * BN + wn * TN;
    constexpr bool AUX = ACT != kActNone && ACT != kActGeluFwd;
    constexpr bool TWO = ACT == kActSiluMulBwd;
    constexpr bool FWD = ACT == kActGeluFwd || ACT == kActSiluMulFwd;
    // The epilogue's operands: the LoRA fragments of the wave's columns and
    // of one 32-row block at a time, and that block's activation operands.
    // The first block's are issued under the last slice's MFMAs, ahead of
    // that slice's refill in the load queue, in the registers of the step-0
    // fragments that slice does not read ahead. All offsets within a 32-row
    // block are 32-bit per lane on a uniform base.
    //
    // el is the lane id made opaque here, once per tile: everything the
    // epilogue derives from it is computed after the main loop, where
    // registers are free, instead of being hoisted out of the tile loop and
    // carried (or spilled) through it.
    int el = lane;
    bf16x8_t cf[2][kJB], rf[kJB][FN];
    u32x4_t av[AUX ? ITS : 1], a2v[TWO ? ITS : 1];
    const int64_t tile_at = 2 * (mw * ldc + nw);  // bytes of the wave's first output
    const uint32_t ld2 = static_cast<uint32_t>(2 * ldc);
    auto piece_ok = [&](int fm, int it) {
      const int idx = it * 64 + el;
      return mw + fm * 32 + idx / CPR < M && nw + 8 * (idx % CPR) < N;
    };
    auto piece_off = [&](int it) {
      const int idx = it * 64 + el;
      return static_cast<uint32_t>(idx / CPR) * ld2 + 16 * (idx % CPR);
    };
    // the wave's whole sub-tile inside the matrix (uniform): no bounds checks
    const bool inside = mw + TM <= M && nw + TN <= N;
    auto load_piece = [&](int64_t at, int it) {
      if constexpr (AUX)
        av[it] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint8_t*>(epi.aux) + at +
                                                   piece_off(it));
      if constexpr (TWO)
        a2v[it] = *reinterpret_cast<const u32x4_t*>(reinterpret_cast<const uint8_t*>(epi.aux2) + at +
                                                    piece_off(it));
    };
    auto load_aux = [&](int fm) {
      const int64_t at = tile_at + static_cast<int64_t>(fm * 32) * ld2;
      if (inside) {
#pragma unroll
        for (int it = 0; it < ITS; ++it) load_piece(at, it);
      } else {
#pragma unroll
        for (int it = 0; it < ITS; ++it) {
          av[it] = u32x4_t{0u, 0u, 0u, 0u};
          if constexpr (TWO) a2v[it] = u32x4_t{0u, 0u, 0u, 0u};
          if (piece_ok(fm, it)) load_piece(at, it);
        }
      }
    };
    auto load_cols = [&](int fm) {
      int r = mw + fm * 32 + (el & 31);
      r = r < M ? r : M - 1;
      const uint32_t at = static_cast<uint32_t>(r) * static_cast<uint32_t>(2 * epi.cols_sm) + (el >> 5) * 16;
#pragma unroll
      for (int jb = 0; jb < kJB; ++jb)
        cf[fm & 1][jb] = *reinterpret_cast<const bf16x8_t*>(
            reinterpret_cast<const uint8_t*>(epi.cols) + at + jb * 32);
    };
    constexpr bool kBiasEarly = BN == 192;  // 256 columns leave no registers for it
    u32x2_t bias2[FN][4];  // bf16 pairs of columns 32 fn + 8 vg + 4 half + [0, 4)
    auto load_bias = [&]() {
#pragma unroll
      for (int fn = 0; fn < FN; ++fn)
#pragma unroll
        for (int vg = 0; vg < 4; ++vg) {
          int nb = nw + fn * 32 + 8 * vg + 4 * (el >> 5);
          nb = nb < N ? nb : 0;  // N % 8 == 0: all four inside, or none
          if (bias_vec)
            bias2[fn][vg] = *reinterpret_cast<const u32x2_t*>(epi.bias + nb);
          else
            bias2[fn][vg] = u32x2_t{epi.bias[nb] | (static_cast<uint32_t>(epi.bias[nb + 1]) << 16),
                                    epi.bias[nb + 2] | (static_cast<uint32_t>(epi.bias[nb + 3]) << 16)};
        }
    };
    auto load_epilogue = [&]() {
      asm volatile("" : "+v"(el));
      if (kBiasEarly && has_bias) load_bias();
      if constexpr (JB > 0) {
#pragma unroll
        for (int fn = 0; fn < FN; ++fn) {
          int n = nw + fn * 32 + (el & 31);
          n = n < N ? n : N - 1;
          const uint32_t at =
              static_cast<uint32_t>(n) * static_cast<uint32_t>(2 * epi.rows_sn) + (el >> 5) * 16;
#pragma unroll
          for (int jb = 0; jb < kJB; ++jb)
            rf[jb][fn] = *reinterpret_cast<const bf16x8_t*>(
                reinterpret_cast<const uint8_t*>(epi.rows) + at + jb * 32);
        }
        load_cols(0);
      }
      if constexpr (AUX) load_aux(0);
    };

    // One slice: steps 0-2 issue their MFMAs with the next step's fragment
    // reads behind the first two; the barrier before step 3 says that every
    // wave has read this stage and that the next slice has landed; step 3
    // refills the stage and reads the next slice's step-0 fragments (the
    // tile's last slice: loads the epilogue's operands instead).
    auto slice = [&](auto last_c) {
      constexpr bool LAST = decltype(last_c)::value;
      const uint32_t cur = stage * STAGE;
      const uint32_t nxt = (stage ^ 1) * STAGE;
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int kk = 0; kk < kSteps - 1; ++kk) {
#pragma unroll
        for (int i = 0; i < NMF; ++i) {
          mma(i, kk & 1);
          __builtin_amdgcn_sched_barrier(0);
          if (i == 0) read_a(cur, kk + 1, (kk + 1) & 1);
          if (i == 1) read_b(cur, kk + 1, (kk + 1) & 1);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      wait_sync<(kStages - 2) * LPW>();
#pragma unroll
      for (int i = 0; i < NMF; ++i) {
        mma(i, 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (LAST) {
          if (i == 0) load_epilogue();
        } else {
          if (i == 0) read_a(nxt, 0, 0);
          if (i == 1) read_b(nxt, 0, 0);
        }
#pragma unroll
        for (int d = i * LPW / NMF; d < (i + 1) * LPW / NMF; ++d) load_seg(stage, d);
        __builtin_amdgcn_sched_barrier(0);
      }
      advance();
      stage ^= 1;
    };
    for (int s = 0; s + 1 < nk; ++s) slice(std::false_type{});
    slice(std::true_type{});

    // Epilogue: y = bf16(bf16(acc) + bf16(bf16(t) * scale)) (+ bias, rounded
    // again) with t = C R^T, then the activation on whole 16-byte row pieces
    // read back from the wave's staging rows. N and the output's row stride
    // are multiples of 8, so a piece is wholly inside or outside.
    if (!kBiasEarly && has_bias) load_bias();
    // sched_barrier fences keep the unrolled blocks from being interleaved,
    // which would spill.
#pragma unroll
    for (int fm = 0; fm < FM; ++fm) {
      if constexpr (JB > 0) {
        if (fm + 1 < FM) load_cols(fm + 1);
      }
#pragma unroll
      for (int fn = 0; fn < FN; ++fn) {
        __builtin_amdgcn_sched_barrier(0);
        f32x16_t lr;
#pragma unroll
        for (int v = 0; v < 16; ++v) lr[v] = 0.0f;
        if constexpr (JB > 0) {
#pragma unroll
          for (int jb = 0; jb < kJB; ++jb)
            lr = __builtin_amdgcn_mfma_f32_32x32x16_bf16(rf[jb][fn], cf[fm & 1][jb], lr, 0, 0, 0);
        }
        // one copy of the block per uniform case, so that no element pays for
        // the other cases' selects
        auto block = [&](auto exact_c, auto bias_c) {
          // no fma of the scaling and the sum: an overflowing product is inf
#pragma clang fp contract(off)
          constexpr bool EXACT = decltype(exact_c)::value;
          constexpr bool BIAS = decltype(bias_c)::value;
#pragma unroll
          for (int vg = 0; vg < 4; ++vg) {
            uint32_t w2[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
              const int v = 4 * vg + 2 * p;
              float a0 = acc[fn][fm][v];
              float a1 = acc[fn][fm][v + 1];
              if constexpr (JB > 0) {
                round2(a0, a1);
                float t0 = lr[v];
                float t1 = lr[v + 1];
                round2(t0, t1);
                t0 *= epi.scale;
                t1 *= epi.scale;
                if constexpr (!EXACT) round2(t0, t1);
                a0 += t0;
                a1 += t1;
              }
              if constexpr (BIAS) {
                round2(a0, a1);
                a0 += bf16lo_to_f32(bias2[fn][vg][p]);
                a1 += bf16hi_to_f32(bias2[fn][vg][p]);
              }
              w2[p] = pack_bf16x2(a0, a1);
            }
            *reinterpret_cast<u32x2_t*>(st + (el & 31) * (TN * 2) +
                                        (stage_chunk<CPR>((el & 31), fn * 4 + vg) << 4) +
                                        (el >> 5) * 8) = u32x2_t{w2[0], w2[1]};
          }
        };
        if (scale_exact) {
          if (has_bias)
            block(std::true_type{}, std::true_type{});
          else
            block(std::true_type{}, std::false_type{});
        } else {
          if (has_bias)
            block(std::false_type{}, std::true_type{});
          else
            block(std::false_type{}, std::false_type{});
        }
      }
      // the wave's LDS operations run in order: the staged rows are complete
      // before they are read, and read before the next 32 rows replace them
      const int64_t at = tile_at + static_cast<int64_t>(fm * 32) * ld2;
#pragma unroll
      for (int it = 0; it < ITS; ++it) {
        __builtin_amdgcn_sched_barrier(0);
        const int idx = it * 64 + el;
        const int r = idx / CPR;
        const int c = idx % CPR;
        const u32x4_t v = *reinterpret_cast<const u32x4_t*>(st + r * (TN * 2) +
                                                            (stage_chunk<CPR>(r, c) << 4));
        u32x4_t o = v, o2{0u, 0u, 0u, 0u};
        if constexpr (ACT != kActNone) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            float x0 = 0.0f, x1 = 0.0f, y0 = 0.0f, y1 = 0.0f, s0 = 0.0f, s1 = 0.0f;
            if constexpr (AUX) {
              x0 = bf16lo_to_f32(av[it][q]);
              x1 = bf16hi_to_f32(av[it][q]);
            }
            if constexpr (TWO) {
              y0 = bf16lo_to_f32(a2v[it][q]);
              y1 = bf16hi_to_f32(a2v[it][q]);
            }
            const float r0 = act_apply<ACT>(bf16lo_to_f32(v[q]), x0, y0, &s0);
            const float r1 = act_apply<ACT>(bf16hi_to_f32(v[q]), x1, y1, &s1);
            o[q] = pack_bf16x2(r0, r1);
            if constexpr (TWO) o2[q] = pack_bf16x2(s0, s1);
          }
        }
        if (inside || piece_ok(fm, it)) {
          const uint32_t po = piece_off(it);
          *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint8_t*>(out) + at + po) = o;
          if constexpr (FWD)
            *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint8_t*>(epi.pre_out) + at + po) = v;
          if constexpr (TWO)
            *reinterpret_cast<u32x4_t*>(reinterpret_cast<uint8_t*>(epi.out2) + at + po) = o2;
        }
      }
      if constexpr (AUX) {
        __builtin_amdgcn_sched_barrier(0);
        if (fm + 1 < FM) load_aux(fm + 1);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // the next tile's slice 0 landed before the last slice's barrier
    read_a(stage * STAGE, 0, 0);
    read_b(stage * STAGE, 0, 0);
  }
  // no LDS DMA may still be in flight when the workgroup ends
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Row-blocks per band of the tile order: an XCD runs 32 tiles at once, and
// with b-row bands those span about b A row-blocks and 32 / b B
// column-blocks; b minimizes their rows together (the band knob forces one).
int wide_band(int tiles_m, int tiles_n, int bn) {
  const int forced = tune(kTuneBand);
  if (forced > 0) return forced < tiles_m ? forced : tiles_m;
  int best = 1;
  int64_t best_cost = -1;
  const int64_t t = 32;
  for (int b = 1; b <= tiles_m && b <= 32; ++b) {
    const int64_t band_tiles = static_cast<int64_t>(b) * tiles_n;
    int64_t rows, cols;
    if (t <= band_tiles) {
      rows = b;
      cols = ceil_div(t, b);
    } else {
      rows = ceil_div(t, tiles_n);
      cols = tiles_n;
    }
    const int64_t cost = rows * 256 + cols * bn;
    if (best_cost < 0 || cost < best_cost) {
      best_cost = cost;
      best = b;
    }
  }
  return best;
}

template <int BN, int WM, int WN, int JB, int ACT>
hipError_t run_wide(const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, int64_t m,
                    int64_t n, int64_t k, uint16_t* out, int64_t ldc, const LowRankEpilogue& epi,
                    hipStream_t stream) {
  constexpr int kLds = kStages * (256 + BN) * 2 * kBK + 8 * 32 * (BN / WN) * 2;
  static_assert(kLds <= 160 * 1024, "LDS budget");
  auto kern = k_gemm_wide<BN, WM, WN, JB, ACT>;
  static std::atomic<unsigned> lds_set{0};
  hipError_t e = ensure_lds_limit(reinterpret_cast<const void*>(kern), kLds, lds_set);
  if (e != hipSuccess) return e;
  const int tiles_m = static_cast<int>(ceil_div(m, 256));
  const int tiles_n = static_cast<int>(ceil_div(n, BN));
  const int tiles = tiles_m * tiles_n;
  hipLaunchKernelGGL(kern, dim3(static_cast<unsigned>(tiles < 256 ? tiles : 256)), dim3(512), kLds,
                     stream, reinterpret_cast<const uint8_t*>(a), 2 * lda,
                     reinterpret_cast<const uint8_t*>(b), 2 * ldb, static_cast<int>(m),
                     static_cast<int>(n), static_cast<int>(k), out, ldc, epi, tiles_m, tiles_n,
                     wide_band(tiles_m, tiles_n, BN));
  return hipGetLastError();
}

template <int BN, int WM, int WN, int JB>
hipError_t run_wide_act(const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, int64_t m,
                        int64_t n, int64_t k, uint16_t* out, int64_t ldc,
                        const LowRankEpilogue& epi, hipStream_t stream) {
#define RPX_WIDE(ACT) run_wide<BN, WM, WN, JB, ACT>(a, lda, b, ldb, m, n, k, out, ldc, epi, stream)
  switch (epi.act) {
    case kActNone: return RPX_WIDE(kActNone);
    case kActGeluFwd: return RPX_WIDE(kActGeluFwd);
    case kActSiluMulFwd: return RPX_WIDE(kActSiluMulFwd);
    case kActGeluBwd: return RPX_WIDE(kActGeluBwd);
    case kActSiluMulBwd: return RPX_WIDE(kActSiluMulBwd);
    case kActAddBwd: return RPX_WIDE(kActAddBwd);
    default: return hipErrorInvalidValue;
  }
#undef RPX_WIDE
}

template <int BN, int WM, int WN>
hipError_t run_wide_jb(const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, int64_t m,
                       int64_t n, int64_t k, uint16_t* out, int64_t ldc,
                       const LowRankEpilogue& epi, hipStream_t stream) {
  if (epi.rank == 0 && epi.act == kActNone)
    return run_wide<BN, WM, WN, 0, kActNone>(a, lda, b, ldb, m, n, k, out, ldc, epi, stream);
  if (epi.rank == 16)
    return run_wide_act<BN, WM, WN, 1>(a, lda, b, ldb, m, n, k, out, ldc, epi, stream);
  return run_wide_act<BN, WM, WN, 2>(a, lda, b, ldb, m, n, k, out, ldc, epi, stream);
}

}  // namespace

// Estimated microseconds of both forms, fitted to graph-timed sweeps of the
// six BERT-base and Qwen3-wide projections at 700 to 32768 rows (each tile
// forced): the wide tiles take one round per 256 tiles, each its slices and a
// fixed epilogue, on a launch; k_gemm_nt's
// tiles run at about 0.93 PFLOP/s less what short reductions lose. A wide
// tile must look 5% faster (10% under an activation, whose arithmetic a lone
// workgroup per CU does not overlap): near the line both measured within 4%
// of each other, for instance (us, old / 256 / 192 columns)
//   forward 4096 x 6144 <- 2048   127 / 136 / 118   taken
//   forward 2600 x 2048 <- 2048    49 /  61 /  55   not taken
//   dx      6144 x 2048 <- 6144   262 / 222 / 301   taken (192 of 256 tiles)
//   dx     12000 x 2048 <- 6144   431 / 450 / 474   not taken (376 of 512 tiles)
int wide_plan(int64_t m, int64_t n, int64_t k, int knob, int act, bool dequant) {
  if (knob == kTileWide_256x256 || knob == kTileWide_256x192) return knob;
  if (knob != kTileAuto) return 0;
  const double s = static_cast<double>(k) / kBK;
  const int64_t tm = ceil_div(m, 256);
  // the forward's dequantization and what a further launch costs a caller
  // that is not running in a graph
  const double first = dequant ? 16.0 : 4.0;
  const double t256 = first + ceil_div(tm * ceil_div(n, 256), 256) * (1.65 * s + 6.0);
  const double t192 = first + ceil_div(tm * ceil_div(n, 192), 256) * (1.30 * s + 5.0);
  const double other =
      10.0 + 2.0 * static_cast<double>(m) * n * k / 0.93e9 * (1.0 + 200.0 / static_cast<double>(k));
  const double margin = act == kActNone || act == kActAddBwd ? 0.95 : 0.90;
  const double t = t256 <= t192 ? t256 : t192;
  if (t >= margin * other) return 0;
  return t256 <= t192 ? kTileWide_256x256 : kTileWide_256x192;
}

bool wide_gemm_ok(const uint16_t* a, int64_t lda, const uint16_t* b, int64_t ldb, int64_t m,
                  int64_t n, int64_t k, const uint16_t* out, int64_t ldc,
                  const LowRankEpilogue& epi) {
  const uintptr_t ptrs =
      reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) |
      reinterpret_cast<uintptr_t>(out) | reinterpret_cast<uintptr_t>(epi.aux) |
      reinterpret_cast<uintptr_t>(epi.aux2) | reinterpret_cast<uintptr_t>(epi.pre_out) |
      reinterpret_cast<uintptr_t>(epi.out2) | reinterpret_cast<uintptr_t>(epi.rows) |
      reinterpret_cast<uintptr_t>(epi.cols);
  // 32-bit row offsets of the operands; 16-byte pieces everywhere; a LoRA
  // term of rank 16 or 32 with unit stride: two 16-rank blocks are what the
  // epilogue has registers for (48 and 64 would spill), and its loads read whole
  // blocks, so other ranks, also below 16, stay with k_gemm_nt, which pads them
  const int64_t lim = int64_t{1} << 32;
  return m > 0 && n > 0 && k > 0 && k % kBK == 0 && lda % 8 == 0 && ldb % 8 == 0 && n % 8 == 0 &&
         ldc % 8 == 0 && (ptrs & 15) == 0 && m * lda * 2 < lim && n * ldb * 2 < lim &&
         m < (int64_t{1} << 31) - 256 && n < (int64_t{1} << 31) - 256 &&
         ceil_div(m, 256) * ceil_div(n, 192) < (int64_t{1} << 30) &&
         (epi.rank == 16 || epi.rank == 32 || (epi.rank == 0 && epi.act == kActNone)) &&
         (epi.rank == 0 || (epi.rows_sj == 1 && epi.cols_sj == 1 && epi.rows_sn % 8 == 0 &&
                            epi.cols_sm % 8 == 0 && m * epi.cols_sm * 2 < lim &&
                            n * epi.rows_sn * 2 < lim)) &&
         ldc * 64 < lim;
}

hipError_t launch_gemm_wide(int tile, const uint16_t* a, int64_t lda, const uint16_t* b,
                            int64_t ldb, int64_t m, int64_t n, int64_t k, uint16_t* out,
                            int64_t ldc, const LowRankEpilogue& epi, hipStream_t stream) {
  if (!wide_gemm_ok(a, lda, b, ldb, m, n, k, out, ldc, epi)) return hipErrorInvalidValue;
  if (tile == kTileWide_256x256)
    return run_wide_jb<256, 2, 4>(a, lda, b, ldb, m, n, k, out, ldc, epi, stream);
  if (tile == kTileWide_256x192)
    return run_wide_jb<192, 4, 2>(a, lda, b, ldb, m, n, k, out, ldc, epi, stream);
  return hipErrorInvalidValue;
}

}  // namespace rpx
