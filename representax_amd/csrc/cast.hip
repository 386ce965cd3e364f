// bf16 compute views of float32 masters, several tensors a launch. One
// adapter's A and B are a few tens of thousands of elements, so a cast is a
// launch and nothing else (4.4 us each in kernel traces, whatever it moves):
// a feed-forward block of three linears casts its six masters in one launch.
#include <hip/hip_runtime.h>

#include "common.h"
#include "kernels.h"

namespace rpx {

namespace {

constexpr int kThreads = 256;
constexpr int kPerBlock = kThreads * 8;

// Block b belongs to the tensor t with first[t] <= b < first[t + 1] (the last,
// first[kCastMany], is the blocks' end); a thread converts 8 consecutive
// elements.
__global__ void __launch_bounds__(kThreads) k_cast_many(CastMany args) {
  const int64_t block = block_of_grid();
  if (block >= args.first[kCastMany]) return;
  int t = 0;
  while (block >= args.first[t + 1]) ++t;
  const int64_t i = (block - args.first[t]) * kPerBlock + static_cast<int64_t>(threadIdx.x) * 8;
  const int64_t n = args.count[t];
  const float* src = args.src[t];
  uint16_t* dst = args.dst[t];
  if (i + 8 <= n) {
    const f32x4_t a = *reinterpret_cast<const f32x4_t*>(src + i);
    const f32x4_t b = *reinterpret_cast<const f32x4_t*>(src + i + 4);
    *reinterpret_cast<u32x4_t*>(dst + i) =
        u32x4_t{pack_bf16x2(a[0], a[1]), pack_bf16x2(a[2], a[3]), pack_bf16x2(b[0], b[1]),
                pack_bf16x2(b[2], b[3])};
    return;
  }
  for (int64_t e = i; e < n; ++e) dst[e] = f32_to_bf16(src[e]);
}

}  // namespace

hipError_t launch_cast_many(CastMany args, int tensors, hipStream_t stream) {
  args.first[0] = 0;
  for (int t = 0; t < kCastMany; ++t)
    args.first[t + 1] = args.first[t] + (t < tensors ? ceil_div(args.count[t], kPerBlock) : 0);
  if (args.first[tensors] == 0) return hipSuccess;
  hipLaunchKernelGGL(k_cast_many, grid_of(args.first[tensors]), dim3(kThreads), 0, stream, args);
  return hipGetLastError();
}

}  // namespace rpx
