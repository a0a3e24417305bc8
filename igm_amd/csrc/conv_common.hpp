// Types and helpers shared by the emulator's kernels (conv.hip, conv3x3.hip, conv_in.hip, wgrad3x3.hip).
#pragma once

#include "common.hpp"
#include "../../include/igm_amd.h"

#include <cstdlib>

namespace igm {

typedef __bf16 bf16;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kC = 32;   // hidden channels
constexpr int kCin = 5;  // input fields

// floats of a block's partial sums of the weight gradient (kernel, then 32 of
// the bias): layer 1, a 3x3 layer, the output layer
constexpr int kWgIn = 9 * kCin * kC + kC, kWg9 = 9 * kC * kC + kC, kWg1 = kC * kC + kC;

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

// A layer's rows, split over the n waves of one launch by its kernel itself:
// the strips of kPx columns one after the other, their rows in groups of kRows,
// and every wave an equal range of that sequence, none a group longer than
// another's.  Of a batch of uneven entries only what is inside the extents
// counts, which the host does not know.  A range that runs on into the next
// strip costs another start of the march; without extents every strip is cut
// into `chunks` ranges of its own where that is no worse (strip_chunks).
struct StripRange {
  int b, x0;   // batch entry, first column
  int y0, y1;  // rows
  int ny, nx;  // the entry's extent
};
template <int kPx, int kRows>
struct StripShare {
  const int32_t* ext;
  int B, H, W;
  int u, hi;    // units (groups of rows) left to this wave
  int b, base;  // entry of unit u and that entry's first unit

  // sum over this and the lower lanes
  __device__ __forceinline__ static int scan(int v) {
    v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, false);  // row_shr 1, 2, 4, 8
    v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, false);
    v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // row_bcast 15, 31
    v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);
    return v;
  }
  __device__ __forceinline__ void units(int e, int& q, int& strips, int& ny, int& nx) const {
    extent_of(ext, e, H, W, ny, nx);
    q = (max(ny, 0) + kRows - 1) / kRows;
    strips = (max(nx, 0) + kPx - 1) / kPx;
  }
  __device__ __forceinline__ void range(int total, int w, int n) {
    const int k = total / n, r = total % n;
    u = w * k + min(w, r);
    hi = u + k + (w < r ? 1 : 0);
  }
  // wave w of n
  __device__ __forceinline__ StripShare(const int32_t* ext_, int B_, int H_, int W_, int chunks, int w, int n)
      : ext(ext_), B(B_), H(H_), W(W_), u(0), hi(0), b(0), base(0) {
    int q, strips, ny, nx;
    if (ext == nullptr) {
      units(0, q, strips, ny, nx);
      if (chunks > 0) {
        const int strip = w / chunks, k = w % chunks;
        if (strip >= B * strips) return;
        u = strip * q + k * (q / chunks) + min(k, q % chunks);
        hi = u + q / chunks + (k < q % chunks ? 1 : 0);
      } else {
        range(B * strips * q, w, n);
      }
      b = u / (strips * q);
      base = b * strips * q;
      return;
    }
    // 64 entries at a time, one per lane: their units and the sum up to them
    int v = 0, p = 0;
    auto entries = [&](int e0) {
      const int e = e0 + (threadIdx.x & 63);
      v = 0;
      if (e < B) {
        units(e, q, strips, ny, nx);
        v = q * strips;
      }
      p = scan(v);
      return __builtin_amdgcn_readlane(p, 63);
    };
    int total = 0;
    for (int e0 = 0; e0 < B; e0 += 64) total += entries(e0);
    range(total, w, n);
    if (u >= hi) return;
    int e0 = 0;
    if (B > 64) {
      for (int t; base + (t = entries(e0)) <= u; e0 += 64) base += t;
    }
    const int f = __builtin_ctzll(__ballot(base + p > u));
    b = e0 + f;
    base += __builtin_amdgcn_readlane(p, f) - __builtin_amdgcn_readlane(v, f);
  }
  // (a loop over the ranges leaves out empty ones, which there are none of:
  // without that test the compiler spills the accumulators around next)
  __device__ __forceinline__ bool more() const { return u < hi; }
  __device__ __forceinline__ StripRange next() {
    StripRange s;
    int q, strips;
    units(b, q, strips, s.ny, s.nx);
    while (u - base >= q * strips) {  // the next entry with rows
      base += q * strips;
      units(++b, q, strips, s.ny, s.nx);
    }
    const int i = (u - base) / q, g = (u - base) % q, k = min(q - g, hi - u);
    s.b = b;
    s.x0 = i * kPx;
    s.y0 = g * kRows;
    s.y1 = min((g + k) * kRows, s.ny);
    u += k;
    return s;
  }
};

// The ranges a strip of a batch without extents is cut into, for n waves, or
// 0 for one sequence of all strips: whichever leaves the longest wave the
// fewest rows, with `start` rows' time for each start of the march.
inline int strip_chunks(const int32_t* ext, int B, int H, int W, int px, int rows, int start, int n) {
  if (ext != nullptr) return 0;
  const int64_t strips = (int64_t)B * ((W + px - 1) / px), q = ((int64_t)H + rows - 1) / rows;
  const int64_t chunks = n / strips < q ? n / strips : q;
  if (chunks < 1) return 0;
  const int64_t apart = (q + chunks - 1) / chunks * rows + start, joined = (strips * q + n - 1) / n * rows + 2 * start;
  return apart <= joined ? (int)chunks : 0;
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
