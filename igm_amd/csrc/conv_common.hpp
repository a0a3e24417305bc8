// Types and helpers shared by the emulator's kernels (conv.hip, conv3x3.hip, conv_in.hip, wgrad3x3.hip).
#pragma once

#include "common.hpp"
#include "../../include/igm_amd.h"

#include <cstdlib>

namespace igm {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int kC = 32;   // hidden channels
constexpr int kCin = 5;  // input fields

__device__ __forceinline__ float leaky(float x) { return x > 0.f ? x : 0.01f * x; }
__device__ __forceinline__ float bf2f(bf16 h) { return (float)h; }
__device__ __forceinline__ bf16 f2bf(float f) { return (bf16)f; }
__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

__device__ __forceinline__ void extent_of(const int32_t* ext, int b, int H, int W, int& ny, int& nx) {
  ny = ext ? min(ext[2 * b], H) : H;
  nx = ext ? min(ext[2 * b + 1], W) : W;
}

// A lane's 16 B of a 3x3 layer's weights [tap][out][in]: rows in the order that
// leaves lane n + 16 g of a product with channels 8 g + 4 cb .. + 3 of pixel n.
__device__ __forceinline__ const u32x4* conv_weight_frag(const bf16* wt, int n, int g, int tap, int cb) {
  return reinterpret_cast<const u32x4*>(wt + ((tap * kC + 8 * (n >> 2) + 4 * cb + (n & 3)) * kC + 8 * g));
}

// cache policy of a kernel's stores: cached, non-temporal, written through
constexpr int kStoreCached = 0, kStoreStream = 2, kStoreThrough = 16;

// How a layer's output of so many bytes is stored.  The caches write it back
// at the kernel's end otherwise: written through, 500 x 500 takes 8.6 us
// instead of 10.5 and 1000 x 1000 (64 MB) 22.7 instead of 24.0.  Buffers that
// do not stay in the 256 MB last-level cache together gain nothing from it:
// 1500 x 1500 (144 MB, forward) took 59 to 61 us either way, and the data
// gradient, which also reads the activation, 75.7 us with non-temporal
// stores, 88 without (8 x 512 x 512, 134 MB: 63.9 and 71.9).  The forward
// pass of such a batch keeps them cached (41 us, 50 non-temporal).
inline int conv_store_mode(int64_t bytes, bool dgrad) {
  if (bytes <= (80 << 20)) return kStoreThrough;
  return dgrad && bytes >= (120 << 20) ? kStoreStream : kStoreCached;
}

// Per-block partial sums of a 3x3 layer's weight gradient (wgrad3x3.hip).
int wgrad3x3_launch(const void* act, const void* dz, const int32_t* ext, int B, int H, int W, int nblocks,
                    float* partials, int accumulate, hipStream_t st);

}  // namespace igm
