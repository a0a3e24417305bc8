// Types and helpers shared by the emulator's kernels (conv.hip, conv3x3.hip).
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

// Per-block partial sums of a 3x3 layer's weight gradient (wgrad3x3.hip).
int wgrad3x3_launch(const void* act, const void* dz, const int32_t* ext, int B, int H, int W, int nblocks,
                    float* partials, int accumulate, hipStream_t st);

}  // namespace igm
