// Layer 1 of the emulator on gfx950: 3x3 "same" convolution of the 5 float32
// input fields to 32 channels, bias, LeakyReLU(0.01), bf16 out
// (emulate/neural_network.py:9-66).  Raw inputs such as the surface elevation
// need float32 (bf16 spacing is 16 m at 2500-3000 m).
//
// Every channel is the chain of float32 FMAs bias, taps 0 .. 8, fields 0 .. 4
// of a tap.  A float32 matrix product adds its k = 2 products in order, each
// with one rounding, so 23 products in a row are that chain, at twice the rate
// of vector FMAs.  A wave owns a strip of 64 columns and walks down its rows;
// its ring of four rows in LDS is its own, so nothing waits for a barrier, and
// the next row's loads are in flight during a row's products.
//
// What bounds it: the products and the vector instructions, which share the
// units (the activation and its rounding are most of the latter): 46 x 64
// cycles and about 110 x 4 for 64 pixels, 24 us for 1000 x 1000, which takes 34
// us.  16x16x4 products, of four, took 36 us; vector FMAs with the weights from
// scalar loads 61 us.
#include "conv_common.hpp"

namespace igm {

constexpr int kInPx = 64;                 // columns of a wave's strip
constexpr int kInRow = 512;               // floats of a ring row in LDS
constexpr int kInField = 68;              // floats of a field's row in it
constexpr int kInZero = kCin * kInField;  // zeros behind the fields' rows
constexpr int kInSpare = kInRow - 64;      // written, never read
constexpr int kInSteps = (9 * kCin + 1) / 2;  // products of k = 2

typedef float f32x16 __attribute__((ext_vector_type(16)));

__global__ void __launch_bounds__(256, 2)
conv_in_kernel(const float* __restrict__ f0, const float* __restrict__ f1, const float* __restrict__ f2,
               const float* __restrict__ f3, const float* __restrict__ f4, int64_t fb, int64_t fr, int64_t fc,
               const int32_t* __restrict__ ext, int H, int W, int nstrips, int nchunk, int rows, int ntask,
               const float* __restrict__ w, const float* __restrict__ bias, bf16* __restrict__ out) {
  __shared__ __attribute__((aligned(16))) float lds[4][4 * kInRow];
  const int lane = threadIdx.x & 63, n = lane & 31, g = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int task = blockIdx.x * 4 + wave;
  if (task >= ntask) return;
  const int x0 = (task % nstrips) * kInPx;
  const int y0 = ((task / nstrips) % nchunk) * rows;
  const int b = task / (nstrips * nchunk);
  int ny, nx;
  extent_of(ext, b, H, W, ny, nx);
  const int yend = min(y0 + rows, H), y1 = x0 < nx ? max(min(yend, ny), y0) : y0;
  bf16* o = out + (((int64_t)b * H + y0) * W + x0) * kC;  // the chunk's first pixel
  const int64_t orow = (int64_t)W * kC;

  if (y1 > y0) {
    // Step q: k = 2 q + g is (tap, field) = (k / 5, k % 5).  A lane's results
    // are channels 8 g .. + 7 and 16 + 8 g .. + 7 of pixel n: row n of the
    // weights is the channel that has its place there.
    const int co = 16 * (n >> 4) + 8 * ((n >> 2) & 1) + 4 * ((n >> 3) & 1) + (n & 3);
    float wf[kInSteps];
#pragma unroll
    for (int q = 0; q < kInSteps; ++q) {
      const int k = 2 * q + g;
      const float v = w[min(k, 9 * kCin - 1) * kC + co];
      wf[q] = k < 9 * kCin ? v : 0.f;
    }
    f32x16 bl;
#pragma unroll
    for (int i = 0; i < 16; ++i) bl[i] = bias[16 * (i >> 3) + 8 * g + (i & 7)];

    float* ring = lds[wave];
#pragma unroll
    for (int r = 0; r < 4; ++r) ring[r * kInRow + kInZero + lane] = 0.f;
    // a row's pixels x0 - 1 .. x0 + 62, one per lane and field, and the two
    // after them, a field and pixel per lane; addresses are clamped into the
    // extent, values outside are zeroed on their way to LDS
    const float* fs[kCin] = {f0, f1, f2, f3, f4};
    const int xa = x0 - 1 + lane, hf = min(lane >> 1, kCin - 1), xh = x0 + 63 + (lane & 1);
    const bool oka = (xa >= 0) & (xa < nx), okh = xh < nx;
    const int64_t base = (int64_t)b * fb;
    const int64_t ca = base + (int64_t)min(max(xa, 0), nx - 1) * fc, ch = base + (int64_t)min(xh, nx - 1) * fc;
    const float* ph = hf == 0 ? f0 : hf == 1 ? f1 : hf == 2 ? f2 : hf == 3 ? f3 : f4;
    const int oh = lane < 2 * kCin ? hf * kInField + kInPx + (lane & 1) : kInSpare + lane;
    struct Row {
      float v[kCin + 1];
    };
    auto load1 = [&](int y, int f) {
      const int64_t r = (int64_t)min(max(y, 0), ny - 1) * fr;
      return f < kCin ? fs[f][r + ca] : ph[r + ch];
    };
    auto put1 = [&](int y, int f, float v) {
      float* s = ring + ((y - y0 + 1) & 3) * kInRow;
      const bool ok = (y >= 0) & (y < ny);
      if (f < kCin) s[f * kInField + lane] = (ok & oka) ? v : 0.f;
      else s[oh] = (ok & okh) ? v : 0.f;
    };
    Row next;
    {
      Row r[3];
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int f = 0; f <= kCin; ++f) r[j].v[f] = load1(y0 - 1 + j, f);
#pragma unroll
      for (int f = 0; f <= kCin; ++f) next.v[f] = load1(y0 + 2, f);
#pragma unroll
      for (int j = 0; j < 3; ++j)
#pragma unroll
        for (int f = 0; f <= kCin; ++f) put1(y0 - 1 + j, f, r[j].v[f]);
    }

    uint32_t os[2];  // of the lane's first 16 B in a row of the strip
#pragma unroll
    for (int p = 0; p < 2; ++p) os[p] = x0 + 32 * p + n < nx ? (uint32_t)((32 * p + n) * kC + 8 * g) * 2 : kOOB;
    // Where a step's inputs are in its row of the ring: the two lane halves
    // read neighbouring fields, or field 4 and field 0 of the next tap, where
    // k is a multiple of 5 less one: in the next row for step 7, and beyond
    // the last input (zeros) for step 22.
    const int near = n + g * kInField, far = n + (g ? 1 : 4 * kInField);
    const int over = n + (g ? kInRow : 4 * kInField + 2), last = n + (g ? kInZero : 4 * kInField + 2);
    float x[2][2];
    auto read = [&](int q, int y) {  // row y's inputs of step q
      const int r = 2 * q / 15, j = 2 * q % 15;
      const int slot = ((y - y0 + r) & 3) * kInRow;
      const float* s = ring + (q == 7    ? (over + slot) & (4 * kInRow - 1)
                               : q == 22 ? last + slot
                                         : (j % 5 == 4 ? far + slot : near + slot));
      const int c = q == 7 || q == 22 ? 0 : j / 5 + (j % 5 == 4 ? 0 : j % 5 * kInField);
#pragma unroll
      for (int p = 0; p < 2; ++p) x[q & 1][p] = s[c + 32 * p];
    };
    read(0, y0);
    for (int y = y0; y < y1; ++y) {
      f32x16 acc[2];
#pragma unroll
      for (int q = 0; q < kInSteps; ++q) {
        if (q + 1 < kInSteps) read(q + 1, y);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int p = 0; p < 2; ++p)
          acc[p] = __builtin_amdgcn_mfma_f32_32x32x2f32(wf[q], x[q & 1][p], q == 0 ? bl : acc[p], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      read(0, y + 1);
#pragma unroll
      for (int f = 0; f <= kCin; ++f) put1(y + 2, f, next.v[f]);
#pragma unroll
      for (int f = 0; f <= kCin; ++f) next.v[f] = load1(y + 3, f);
      const rsrc_t ro = make_rsrc(o, kInPx * kC * 2);
#pragma unroll
      for (int p = 0; p < 2; ++p)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          bf16x8 v;
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const float a = acc[p][8 * c + e];
            v[e] = f2bf(__builtin_elementwise_maximum(a, 0.01f * a));  // LeakyReLU
          }
          store_b128(__builtin_bit_cast(u32x4, v), ro, os[p] + 32 * c);
        }
      o += orow;
    }
  }
  // zeros outside the extent
  const uint4 z = {0, 0, 0, 0};
  o = out + (((int64_t)b * H + y0) * W + x0) * kC;
  for (int y = nx < min(x0 + kInPx, W) ? y0 : y1; y < yend; ++y)
#pragma unroll
    for (int p = 0; p < 4; ++p) {
      const int px = 16 * p + (lane >> 2), x = x0 + px;
      if (x < W && (y >= y1 || x >= nx)) *reinterpret_cast<uint4*>(o + (y - y0) * orow + px * kC + 8 * (lane & 3)) = z;
    }
}

}  // namespace igm

using namespace igm;

extern "C" int igm_conv_in_fwd(const float* f0, const float* f1, const float* f2, const float* f3, const float* f4,
                               int64_t fb, int64_t fr, int64_t fc, const int32_t* extents, int32_t B, int32_t H,
                               int32_t W, const float* w_hwio, const float* bias, void* out_bf16, void* stream) {
  IGM_CHECK_ARG(f0 && f1 && f2 && f3 && f4 && w_hwio && bias && out_bf16, "null pointer");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && H <= 65535 && B <= 65535, "bad sizes");
  const int nstrips = (W + kInPx - 1) / kInPx;
  // two waves per SIMD, with equal shares of the strips' rows (1000 x 1000: 34
  // us; 35 with one wave per SIMD, 36 with four)
  const int64_t rows = ((int64_t)B * nstrips * H + 2047) / 2048;
  const int nchunk = (int)((H + rows - 1) / rows);
  const int64_t ntask = (int64_t)B * nstrips * nchunk;
  hipLaunchKernelGGL(conv_in_kernel, dim3((unsigned)((ntask + 3) / 4)), dim3(256), 0, (hipStream_t)stream, f0, f1, f2,
                     f3, f4, fb, fr, fc, extents, H, W, nstrips, nchunk, (int)rows, (int)ntask, w_hwio, bias,
                     (bf16*)out_bf16);
  IGM_CHECK_LAUNCH();
  return 0;
}
