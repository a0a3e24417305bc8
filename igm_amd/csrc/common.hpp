// Shared helpers for the gfx950 kernels: error reporting for the C-ABI and
// cross-lane exchange inside a 64-wide wavefront.
#pragma once

#include <hip/hip_runtime.h>
#include <cstdint>
#include <cstdio>
#include <string>

namespace igm {

// Last error message of the calling host thread (read by igm_last_error()).
void set_error(const std::string& msg);
const char* last_error();

#define IGM_CHECK_ARG(cond, msg)                         \
  do {                                                   \
    if (!(cond)) {                                       \
      ::igm::set_error(std::string(__func__) + ": " + (msg)); \
      return -1;                                         \
    }                                                    \
  } while (0)

#define IGM_CHECK_LAUNCH()                                                    \
  do {                                                                        \
    hipError_t e_ = hipGetLastError();                                        \
    if (e_ != hipSuccess) {                                                   \
      ::igm::set_error(std::string(__func__) + ": launch failed: " + hipGetErrorString(e_)); \
      return -2;                                                              \
    }                                                                         \
  } while (0)

constexpr int kWave = 64;

// Lane l receives the value held by lane l+1 (lane 63 receives 0).
// DPP wave_shl:1 -- one VALU move, no LDS traffic.
__device__ __forceinline__ float lane_from_right(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x130, 0xF, 0xF, true));
}
// Lane l receives the value held by lane l-1 (lane 0 receives 0).
// DPP wave_shr:1.
__device__ __forceinline__ float lane_from_left(float x) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), 0x138, 0xF, 0xF, true));
}
__device__ __forceinline__ double lane_from_right(double x) {
  int lo = __double2loint(x), hi = __double2hiint(x);
  lo = __builtin_amdgcn_update_dpp(0, lo, 0x130, 0xF, 0xF, true);
  hi = __builtin_amdgcn_update_dpp(0, hi, 0x130, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double lane_from_left(double x) {
  int lo = __double2loint(x), hi = __double2hiint(x);
  lo = __builtin_amdgcn_update_dpp(0, lo, 0x138, 0xF, 0xF, true);
  hi = __builtin_amdgcn_update_dpp(0, hi, 0x138, 0xF, 0xF, true);
  return __hiloint2double(hi, lo);
}

// Sum over the 64 lanes of a wavefront (every lane gets the total).
// Raw buffer resources with 32-bit byte offsets: an offset at or beyond the
// resource size reads 0 and drops a store, in hardware, so out-of-grid and
// masked lanes need no branch.  kOOB is above every resource size (the host
// checks that each buffer is below 2 GiB).
using rsrc_t = __amdgpu_buffer_rsrc_t;
constexpr uint32_t kOOB = 0x80000000u;
constexpr int kRsrcWord3 = 0x00020000;  // raw buffer, gfx9 data format

__device__ __forceinline__ rsrc_t make_rsrc(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, kRsrcWord3);
}

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// Every 16-B store goes through here: to byte offset off (kOOB: dropped), with
// nothing in the instruction's scalar offset.  The store reads its data
// registers after it has issued, and the compiler keeps the wait states until
// they are written again only behind stores without a scalar offset.  (The ISA
// documents exempt the other form, but a forward layer that used it, with two
// waves on a SIMD, stored the next values in its last lanes.)  An offset of all
// lanes is therefore added to off.
template <int AUX = 0>
__device__ __forceinline__ void store_b128(u32x4 v, rsrc_t r, uint32_t off) {
  __builtin_amdgcn_raw_buffer_store_b128(v, r, off, 0, AUX);
}

// MI355X dispatches the workgroups of a launch to its 8 XCDs round-robin
// (workgroup p runs on XCD p % 8), and each XCD has an L2 of its own.
// xcd_remap turns the dispatch index p of nb workgroups into a logical index
// such that every XCD gets one contiguous range of logical indices: tiles
// that are neighbours in the logical order then share an L2, and the cache
// lines on their common edges are fetched from HBM once.  A bijection on
// [0, nb) whatever the hardware order, so only speed depends on it.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_remap(int p, int nb) {
  const int q = nb / kXcds, r = nb % kXcds;
  const int x = p % kXcds, i = p / kXcds;
  return x * q + (x < r ? x : r) + i;
}

__device__ __forceinline__ double wave_sum(double x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, kWave);
  return x;
}
__device__ __forceinline__ float wave_sum(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_xor(x, off, kWave);
  return x;
}
__device__ __forceinline__ float wave_max(float x) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) x = fmaxf(x, __shfl_xor(x, off, kWave));
  return x;
}

// x^e for x > 0 via the hardware log2/exp2 (fp32) or libm (fp64).
__device__ __forceinline__ float pow_pos(float x, float e) {
  return __builtin_amdgcn_exp2f(e * __builtin_amdgcn_logf(x));
}
__device__ __forceinline__ double pow_pos(double x, double e) { return pow(x, e); }
// d * x^e for x, d > 0, with l2d = log2(d): one exp2 of e log2(x) + log2(d)
// in fp32 (the multiply by d folds into the exponent)
__device__ __forceinline__ float scaled_pow(float x, float e, float d, float l2d) {
  return __builtin_amdgcn_exp2f(__builtin_fmaf(e, __builtin_amdgcn_logf(x), l2d));
}
__device__ __forceinline__ double scaled_pow(double x, double e, double d, double l2d) {
  return d * pow(x, e);
}
// x^e for x >= 0 and e within 1e-12 of -1/3, which n = 3 and m = 3 give (the
// rounding of e included): the float32 power y of the mantissa m, which is good
// to 2^-22, and one third-order step of y (1 - r)^(-1/3), r = 1 - m y^3.  y^2 is
// exact, the rounding of m y is put back into r, and the step and x^(e + 1/3)
// are added with one rounding.  The largest error sampled over [1e-10, 1e3] is
// 0.50 ulp, 0.29 in the root mean square (pow: 0.7 and 0.30; two roundings and r
// as computed: 1.3 and 0.42); over 3,100 values of all exponents, subnormal ones
// too, x x^e as a pass computes it is within 1.61 x 2^-53.  About 30 instructions
// where pow takes 250.
__device__ __forceinline__ double pow_third(double x, double e) {
  const int ex = __builtin_amdgcn_frexp_exp(x), q = (int)floorf((float)ex * (1.0f / 3.0f) + 0.125f);
  const double m = __builtin_amdgcn_ldexp(__builtin_amdgcn_frexp_mant(x), ex - 3 * q);  // [1/2, 4)
  const float l = __builtin_amdgcn_logf((float)m);
  const double y = (double)__builtin_amdgcn_exp2f(l * (-1.0f / 3.0f));
  const double yy = y * y, my = m * y;
  const double r = __builtin_fma(-yy, __builtin_fma(m, y, -my), __builtin_fma(-yy, my, 1.0));
  // x^(e + 1/3), with the rounding of 1/3
  const double d = ((e + 1.0 / 3.0) + 0x1.5555555555555p-56) * 0.6931471805599453;
  const double c = __builtin_fma(r, __builtin_fma(r, 2.0 / 9.0, 1.0 / 3.0), d * (double)(l + (float)(3 * q)));
  const double w = __builtin_amdgcn_ldexp(__builtin_fma(y, c, y), -q);
  return __builtin_amdgcn_class(x, 0x260) ? y : w;  // of zero and infinity
}
__device__ __forceinline__ float rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ double rcp(double x) { return 1.0 / x; }
// hardware square root (v_sqrt_f32, ~1 ulp) -- not the correctly rounded expansion
__device__ __forceinline__ float sqrt_(float x) { return __builtin_amdgcn_sqrtf(x); }
__device__ __forceinline__ double sqrt_(double x) { return sqrt(x); }
// clamp of x to [lo, hi] in one v_med3_f32
__device__ __forceinline__ float clamp_(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }
__device__ __forceinline__ double clamp_(double x, double lo, double hi) { return fmin(fmax(x, lo), hi); }

}  // namespace igm
