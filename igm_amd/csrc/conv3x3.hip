// The emulator's 32 -> 32 3x3 layers on gfx950 (v_mfma_f32_16x16x32_bf16):
// forward (bias + LeakyReLU), data gradient, and two forward layers in one
// launch (emulate/neural_network.py:9-66).
//
// A wave owns a strip of 64 pixel columns and walks down its rows with the
// three input rows of a 3x3 window in registers, loading the next one while
// it multiplies.  A product takes 16 output channels (A: the weights, one
// 16-B fragment per lane and tap from LDS) and 16 pixels (B: lane n + 16 g
// holds channels 8 g .. 8 g + 7 of pixel slot n, the 16 B that NHWC rows hold
// them in, so activations go from memory to the products without LDS).  The
// weight rows are taken in the order that leaves a lane with 8 consecutive
// channels of its pixel: 16-B stores, and the layout of the next layer's
// operand.  Every output sums taps 0 .. 8 in order from zero and adds the
// bias last, in all of these kernels: they agree bit for bit.
//
// What bounds them: one layer, memory.  At 1000 x 1000 it moves 128 MB, where
// the products alone take 7.5 us: 18.2 us back and forth between two buffers,
// which the last-level cache holds, and 29.5 us (4.3 TB/s) in a pass that keeps
// its activations, sixteen buffers from and to HBM.  (From one buffer to
// another over and over, as the benchmark times it, 21 us; the earlier kernel,
// which staged tiles of rows in LDS between barriers, 33.)  Two layers in one
// launch move half the bytes and are bound by the matrix and the vector
// instructions of the one wave a SIMD holds, 72 products of 16 cycles and about
// 170 others of 4 per row and layer, which hardly overlap (43 % of a wave's time
// are products): at 1000 x 1000 31 us for both in a loop and 33.6 in a pass, at
// 100 x 100 7.1 either way (4.5 and 5.1 for one), most of it the launch and the
// first loads.
#include "conv_common.hpp"

#include <type_traits>

namespace igm {

constexpr int kStripPx = 64;            // pixels of a wave's row
constexpr int kPairPx = kStripPx - 2;   // columns a wave of the two-layer kernel owns

struct ConvGeom {
  int nstrips, nrowblk, rows, blocks;
};
// Strips of `own` columns, their rows in blocks of `rows`: the most blocks
// that leave one wave per SIMD, 1024 in all (256 x 319: 7.4 us a layer, 8.8
// with 2048; 1000 x 1000: 24.9 and 25.9), so that every wave of one field
// takes as long.  In a batch of uneven entries (ext) some waves only write
// padding; blocks of at most 32 rows keep the others short enough to fill in
// for them.  The two-layer kernel holds one wave per SIMD, so it keeps to one
// round instead.  (IGM_CONV_BLOCKS overrides the number of blocks of four
// waves the split aims at, for tuning sweeps.)
constexpr int kConvBlocks = 256;
constexpr int kConvRows = 32;
inline int64_t conv_target_waves() {
  static const int64_t n = [] {
    const char* e = getenv("IGM_CONV_BLOCKS");
    const long long r = e ? atoll(e) : kConvBlocks;
    return 4 * (int64_t)((r >= 64 && r <= (1 << 22)) ? r : kConvBlocks);
  }();
  return n;
}
inline ConvGeom conv_geom(int B, int H, int W, int own, bool ext) {
  ConvGeom c;
  c.nstrips = (W + own - 1) / own;
  const int64_t strips = (int64_t)B * c.nstrips;
  const int64_t blk = conv_target_waves() / strips < 1 ? 1 : conv_target_waves() / strips;
  const int64_t rows = (H + blk - 1) / blk;
  c.rows = (int)(ext && own == kStripPx && rows > kConvRows ? kConvRows : rows);
  c.nrowblk = (H + c.rows - 1) / c.rows;
  c.blocks = (int)((strips * c.nrowblk + 3) / 4);
  return c;
}

struct ConvArgs {
  const bf16* in;
  const bf16* wt[2];
  const float* bias[2];
  const bf16* aux;
  bf16* out;
  const bf16* head;       // output layer (HEAD): weights [32 out][32 in], bias,
  const float* headb;     // its result (B, H, W, cout)
  float* Y;
  int cout;
  const int32_t* ext;
  int B, H, W;
  ConvGeom g;
};

// This wave's part of the image.
struct ConvTile {
  int lane, n, g;  // pixel slot n of 16, channel group g of 4 (8 channels each)
  int x0, y0, y1;  // first column, rows
  int ny, nx;
  uint32_t bytes, rowbytes, img;
  bool live;
};
__device__ __forceinline__ ConvTile conv_tile(const ConvArgs& a, int own) {
  ConvTile t;
  t.lane = threadIdx.x & 63;
  t.n = t.lane & 15;
  t.g = t.lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wid = xcd_remap(blockIdx.x, gridDim.x) * 4 + wave;
  t.live = wid < a.B * a.g.nstrips * a.g.nrowblk;
  t.x0 = (wid % a.g.nstrips) * own;
  t.y0 = ((wid / a.g.nstrips) % a.g.nrowblk) * a.g.rows;
  const int b = wid / (a.g.nstrips * a.g.nrowblk);
  t.y1 = min(t.y0 + a.g.rows, a.H);
  t.ny = t.nx = 0;
  if (t.live) extent_of(a.ext, b, a.H, a.W, t.ny, t.nx);
  t.bytes = (uint32_t)((int64_t)a.B * a.H * a.W * kC * 2);
  t.rowbytes = (uint32_t)a.W * kC * 2;
  t.img = (uint32_t)b * a.H * t.rowbytes;
  return t;
}
// A block's weights on their way to LDS.  Their loads, and then the first rows',
// are under way together before a wave waits for the former: one latency at the
// start of a launch instead of two.  In a loop between two buffers, two layers at
// 100 x 100 8.3 -> 7.3 us, 256 x 319 10.8 -> 9.3, 1000 x 1000 35 -> 30; one layer
// 5.15 -> 4.7, 6.2 -> 5.65 and 19.6 -> 18.6.
template <int F, int N>  // F fragments, at least 4 N - 3
__device__ __forceinline__ void weights_load(u32x4 (&w)[N], const bf16* const (&wt)[2], const ConvTile& t) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int f = min(4 * i + (int)(threadIdx.x >> 6), F - 1);
    const int l = f >= 18 ? 1 : 0, k = f - 18 * l;
    w[i] = *conv_weight_frag(wt[l], t.n, t.g, k >> 1, k & 1);
  }
}
template <int N>
__device__ __forceinline__ void weights_put(u32x4 (*wl)[64], const u32x4 (&w)[N]) {
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < N; ++i) wl[4 * i + (threadIdx.x >> 6)][threadIdx.x & 63] = w[i];
}
// byte offset of pixel x of a row, this lane's channels; kOOB unless ok
__device__ __forceinline__ uint32_t px_off(const ConvTile& t, int x, bool ok) {
  return ok ? (uint32_t)(x * kC + 8 * t.g) * 2 : kOOB;
}

// One layer.  MODE 0: out = LeakyReLU(conv + bias).  MODE 1 (dgrad): out =
// conv * (aux > 0 ? 1 : 0.01), aux = activation of the layer below (its sign
// is the sign of its pre-activation); the network's backward pass runs
// bwd3x3_kernel instead, this mode serves igm_conv3x3_dgrad_bf16.  Slots n hold pairs of neighbouring
// pixels, 8 (n / 2) + 2 q + n % 2 for slot group q: an access of the wave
// covers whole 128-B lines (interleaved by 4 n + q instead, half lines, 1500
// x 1500 took 74 us a layer, now 60).  Tap column s of group q is then the
// row shifted by s - 1: nine fragments a row, whose overlap is read from L1.
//
// HEAD (forward): the 1x1 output layer with it, Y = head * out + headb.  A
// lane's 8 channels are the output layer's operand as they are, so a row's Y
// follows its activations (a.out NULL: those are not stored).  1000 x 1000, 20
// outputs: 38 us, 34 without the activations, where the two launches take 52.
template <int MODE, int ST, bool HEAD>
__global__ void __launch_bounds__(256, 2)
conv3x3_kernel(const ConvArgs a) {
  __shared__ u32x4 wl[20][64];  // 18 fragments (and two unused)
  const ConvTile t = conv_tile(a, kStripPx);
  u32x4 ws[5];
  weights_load<18>(ws, a.wt, t);
  const int xl = t.x0 + 8 * (t.n >> 1) + (t.n & 1);  // pixel of slot q: xl + 2 q
  const int yv = t.x0 < t.nx ? min(t.y1, t.ny) : t.y0;  // rows y0 .. yv - 1 are computed
  // fragment f: pixels xl + f - 1, f = 0 .. 8
  uint32_t voff[9];
#pragma unroll
  for (int f = 0; f < 9; ++f) voff[f] = px_off(t, xl + f - 1, (xl + f - 1 >= 0) & (xl + f - 1 < t.nx));
  auto load_row = [&](u32x4 (&r)[9], int y) {
    const bool ok = (y >= 0) & (y < t.ny) & (y <= yv);
    const rsrc_t rs = make_rsrc(a.in, ok ? t.bytes : 0u);
    const uint32_t so = ok ? t.img + (uint32_t)y * t.rowbytes : 0u;
#pragma unroll
    for (int f = 0; f < 9; ++f) r[f] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff[f], so, 0);
  };
  u32x4 r0[9], r1[9], r2[9];
  load_row(r0, t.y0 - 1);
  load_row(r1, t.y0);
  load_row(r2, t.y0 + 1);
  weights_put(wl, ws);
  __syncthreads();
  if (!t.live) return;
  uint32_t ooff[4];
  bool xin[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    ooff[q] = px_off(t, xl + 2 * q, xl + 2 * q < a.W);
    xin[q] = xl + 2 * q < t.nx;
  }
  const rsrc_t rout = make_rsrc(a.out, !HEAD || a.out ? t.bytes : 0u);
  // HEAD: Y of pixel slot q, output channels 16 c + 4 g .. + 3, in a row
  const uint32_t ybytes = HEAD ? (uint32_t)a.W * a.cout * 4 : 0u;
  const bool vec = HEAD && (a.cout % 4) == 0 && (reinterpret_cast<uintptr_t>(a.Y) & 15) == 0;
  const int b = HEAD ? (int)(t.img / ((uint32_t)a.H * t.rowbytes)) : 0;
  auto store_y = [&](int y, int q, int c, f32x4 v) {
    const rsrc_t ry = make_rsrc(a.Y + ((int64_t)b * a.H + y) * a.W * a.cout, ybytes);
    const int x = xl + 2 * q, co = 16 * c + 4 * t.g;
    const uint32_t o = ((x < a.W) & (co < a.cout)) ? (uint32_t)(x * a.cout + co) * 4 : kOOB;
    if (vec) {
      store_b128(__builtin_bit_cast(u32x4, v), ry, o);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v[e]), ry, co + e < a.cout ? o + 4 * e : kOOB, 0, 0);
    }
  };
  for (int y = max(yv, t.y0); y < t.y1; ++y) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      store_b128(u32x4{0, 0, 0, 0}, rout, ooff[q] + t.img + y * t.rowbytes);
      if constexpr (HEAD) {
#pragma unroll
        for (int c = 0; c < 2; ++c) store_y(y, q, c, f32x4{0.f, 0.f, 0.f, 0.f});
      }
    }
  }
  if (yv <= t.y0) return;

  float bias_r[8];
  if constexpr (MODE == 0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) bias_r[e] = a.bias[0][8 * t.g + e];
  }
  bf16x8 hw[2];
  f32x4 hb[2];
  if constexpr (HEAD) {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      hw[c] = as_bf16x8(*reinterpret_cast<const u32x4*>(a.head + (c * 16 + t.n) * kC + 8 * t.g));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int co = c * 16 + 4 * t.g + e;
        hb[c][e] = co < a.cout ? a.headb[co] : 0.f;
      }
    }
  }
  // row y from input rows y - 1 (ra), y (rb), y + 1 (rc); loads row y + 2 into ra
  auto step = [&](int y, u32x4 (&ra)[9], const u32x4 (&rb)[9], const u32x4 (&rc)[9]) {
    const uint32_t so = t.img + (uint32_t)y * t.rowbytes;
    u32x4 av[4];
    if constexpr (MODE == 1) {
      const rsrc_t raux = make_rsrc(a.aux, t.bytes);
#pragma unroll
      for (int q = 0; q < 4; ++q) av[q] = __builtin_amdgcn_raw_buffer_load_b128(raux, ooff[q], so, 0);
    }
    f32x4 acc[4][2];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      const u32x4 (&r)[9] = tap < 3 ? ra : (tap < 6 ? rb : rc);
      const bf16x8 w0 = as_bf16x8(wl[2 * tap][t.lane]), w1 = as_bf16x8(wl[2 * tap + 1][t.lane]);
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const bf16x8 v = as_bf16x8(r[2 * q + tap % 3]);
        const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
        acc[q][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, v, tap == 0 ? zero : acc[q][0], 0, 0, 0);
        acc[q][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, v, tap == 0 ? zero : acc[q][1], 0, 0, 0);
      }
      if (tap == 2) {
        load_row(ra, y + 2);
        asm volatile("" ::: "memory");  // keeps the loads here: they would sink into the next step
      }
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      bf16x8 h;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        float v = acc[q][e >> 2][e & 3];
        if constexpr (MODE == 0) {
          v += bias_r[e];
          v = fmaxf(v, 0.01f * v);
        } else {
          const uint32_t w = av[q][e >> 1];
          v *= __uint_as_float((e & 1) ? (w & 0xFFFF0000u) : (w << 16)) > 0.f ? 1.f : 0.01f;
        }
        h[e] = f2bf(v);
      }
      u32x4 o = __builtin_bit_cast(u32x4, h);
#pragma unroll
      for (int i = 0; i < 4; ++i) o[i] = xin[q] ? o[i] : 0u;
      if (!HEAD || a.out) store_b128<ST>(o, rout, ooff[q] + so);
      if constexpr (HEAD) {
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
          f32x4 v = __builtin_amdgcn_mfma_f32_16x16x32_bf16(hw[c], as_bf16x8(o), zero, 0, 0, 0);
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = xin[q] ? v[e] + hb[c][e] : 0.f;
          store_y(y, q, c, v);
        }
      }
    }
  };

  for (int y = t.y0;; y += 3) {
    step(y, r0, r1, r2);
    if (y + 1 >= yv) break;
    step(y + 1, r1, r2, r0);
    if (y + 2 >= yv) break;
    step(y + 2, r2, r0, r1);
    if (y + 3 >= yv) break;
  }
}

// lane n of each 16 receives lane n - 1's (lane n + 1's) value; 0 at the end
__device__ __forceinline__ u32x4 px_left(u32x4 v) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_update_dpp(0, (int)v[i], 0x111, 0xF, 0xF, true);
  return r;
}
__device__ __forceinline__ u32x4 px_right(u32x4 v) {
  u32x4 r;
#pragma unroll
  for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_update_dpp(0, (int)v[i], 0x101, 0xF, 0xF, true);
  return r;
}

// Two forward layers: the first one's rows stay in registers, three at a time
// like the input's, and its outputs are the second layer's operand as they
// are.  Slot n of group q is pixel 4 n + q: tap columns are other groups'
// fragments, and the neighbours of a row's ends come from the next lane (DPP).
// The second layer is complete on 62 of the 64 columns, and a wave computes
// two more rows of the first layer than it owns.  Outside the extent the
// first layer is zero, the second one's padding.
//
// The row that a layer has finished gets its bias, LeakyReLU and rounding while
// the other layer multiplies: its second layer's rows during the first layer's
// next one, the first layer's row during the second layer's first six taps,
// which don't read it, three vector instructions after each product.  Left to
// the scheduler, a layer's chains ran one after the other with waits between:
// an emulator pass at 1000 x 1000 385 us, now 363; 1500 x 1500 88 us a launch,
// now 83.
template <int ST>
__global__ void __launch_bounds__(256, 1)
conv3x3_pair_kernel(const ConvArgs a) {
  __shared__ u32x4 wl[2][18][64];
  __shared__ __attribute__((aligned(16))) float bl[2][kC];
  const ConvTile t = conv_tile(a, kPairPx);
  u32x4 ws[9];
  weights_load<36>(ws, a.wt, t);
  const float bs = (threadIdx.x < kC ? a.bias[0] : a.bias[1])[threadIdx.x & (kC - 1)];
  const int xl = t.x0 - 1 + 4 * t.n;  // pixel of slot q: xl + q
  const int yv = t.x0 < t.nx ? min(t.y1, t.ny) : t.y0;  // rows y0 .. yv - 1 are computed
  uint32_t voff[6];  // fragment f: pixels xl + f - 1
#pragma unroll
  for (int f = 0; f < 6; ++f) voff[f] = px_off(t, xl + f - 1, (xl + f - 1 >= 0) & (xl + f - 1 < t.nx));
  auto load_row = [&](u32x4 (&r)[6], int y) {
    const bool ok = (y >= 0) & (y < t.ny) & (y <= yv + 1);
    const rsrc_t rs = make_rsrc(a.in, ok ? t.bytes : 0u);
    const uint32_t so = ok ? t.img + (uint32_t)y * t.rowbytes : 0u;
#pragma unroll
    for (int f = 0; f < 6; ++f) r[f] = __builtin_amdgcn_raw_buffer_load_b128(rs, voff[f], so, 0);
  };
  u32x4 r[3][6];  // input rows
#pragma unroll
  for (int i = 0; i < 3; ++i) load_row(r[i], t.y0 - 2 + i);
  weights_put(&wl[0][0], ws);
  if (threadIdx.x < 2 * kC) bl[threadIdx.x / kC][threadIdx.x & (kC - 1)] = bs;
  __syncthreads();
  if (!t.live) return;
  uint32_t ooff[4];
  bool xin[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int p = 4 * t.n + q;
    ooff[q] = px_off(t, xl + q, (p >= 1) & (p <= kPairPx) & (xl + q < a.W));
    xin[q] = (xl + q >= 0) & (xl + q < t.nx);
  }
  const rsrc_t rout = make_rsrc(a.out, t.bytes);
  for (int y = max(yv, t.y0); y < t.y1; ++y) {
#pragma unroll
    for (int q = 0; q < 4; ++q)
      store_b128(u32x4{0, 0, 0, 0}, rout, ooff[q] + t.img + y * t.rowbytes);
  }
  if (yv <= t.y0) return;

  f32x4 bl_r[2][2];
  bf16x8 wr[2][18];
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int f = 0; f < 18; ++f) wr[l][f] = as_bf16x8(wl[l][f][t.lane]);
#pragma unroll
  for (int l = 0; l < 2; ++l)
#pragma unroll
    for (int c = 0; c < 2; ++c) bl_r[l][c] = *reinterpret_cast<const f32x4*>(&bl[l][8 * t.g + 4 * c]);
  u32x4 m[3][6];  // the first layer's rows

  // The products of one tap of layer l.
  auto mult = [&](int l, int tap, f32x4 (&acc)[4][2], const u32x4 (&ra)[6], const u32x4 (&rb)[6], const u32x4 (&rc)[6]) __attribute__((always_inline)) {
    const u32x4 (&rr)[6] = tap < 3 ? ra : (tap < 6 ? rb : rc);
    const bf16x8 w0 = wr[l][2 * tap], w1 = wr[l][2 * tap + 1];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const bf16x8 v = as_bf16x8(rr[q + tap % 3]);
      const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
      acc[q][0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w0, v, tap == 0 ? zero : acc[q][0], 0, 0, 0);
      acc[q][1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w1, v, tap == 0 ? zero : acc[q][1], 0, 0, 0);
    }
  };
  // Part u of 8 of a row's epilogue: half of slot group u / 2's channels.
  auto finish = [&](int l, int u, const f32x4 (&acc)[4][2], bool rv, u32x4 (&o)[4]) __attribute__((always_inline)) {
    const int q = u >> 1, c = u & 1;
    typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));
    bf16x4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float v = acc[q][c][e] + bl_r[l][c][e];
      v = fmaxf(v, 0.01f * v);
      h[e] = f2bf(v);
    }
    const uint2 w = __builtin_bit_cast(uint2, h);
    const bool ok = xin[q] & rv;
    o[q][2 * c] = ok ? w.x : 0u;
    o[q][2 * c + 1] = ok ? w.y : 0u;
  };
  // a row of the first layer, with its neighbours' end pixels
  auto put = [&](u32x4 (&d)[6], const u32x4 (&o)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < 4; ++q) d[q + 1] = o[q];
    d[0] = px_left(o[3]);
    d[5] = px_right(o[0]);
  };
  // One tap's products with `valu` vector instructions between each two.
  auto interleave = [](auto valu) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, valu.value, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  f32x4 acc0[4][2], acc1[4][2];
  // Row c of the first layer, from r[I], r[I + 1], r[I + 2], and between its
  // products the epilogue of the second layer's row c - 2, or (HEAD) of the
  // first layer's row c - 1, into m[I - 1].
  auto first = [&](int I, int c, auto head) __attribute__((always_inline)) {
    u32x4 o[4];
    const uint32_t so = t.img + (uint32_t)(c - 2) * t.rowbytes;
    const bool rv = (c - 1 >= 0) & (c - 1 < t.ny);
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      mult(0, tap, acc0, r[I], r[(I + 1) % 3], r[(I + 2) % 3]);
      if (tap < 8) finish(head.value ? 0 : 1, tap, acc1, head.value ? rv : true, o);
      if (tap == 3) load_row(r[I], c + 2);
      if (!head.value && tap >= 2 && tap % 2 == 0) store_b128<ST>(o[tap / 2 - 1], rout, ooff[tap / 2 - 1] + so);
      if (head.value && tap == 8) put(m[(I + 2) % 3], o);
      interleave(std::integral_constant<int, 3>{});
    }
  };
  // row y of the second layer: its products, and the epilogue of the first
  // layer's row y + 1, into m[I], which the last three taps read
  auto second = [&](int I, int y) __attribute__((always_inline)) {
    const bool rv = y + 1 < t.ny;
    u32x4 o[4];
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      mult(1, tap, acc1, m[(I + 1) % 3], m[(I + 2) % 3], m[I]);
      if (tap < 2) finish(0, 2 * tap, acc0, rv, o), finish(0, 2 * tap + 1, acc0, rv, o);
      else if (tap < 6) finish(0, tap + 2, acc0, rv, o);
      if (tap == 5) put(m[I], o);
      if (tap < 2) interleave(std::integral_constant<int, 5>{});
      else interleave(std::integral_constant<int, 3>{});
    }
  };
  auto step = [&](int I, int y) __attribute__((always_inline)) {
    first(I, y + 1, std::false_type{});
    second(I, y);
  };
  // the first layer's rows y0 - 1, y0 and y0 + 1
#pragma unroll
  for (int tap = 0; tap < 9; ++tap) mult(0, tap, acc0, r[0], r[1], r[2]);
  load_row(r[0], t.y0 + 1);
  {
    u32x4 o[4];
    const bool rv = t.y0 > 0;
#pragma unroll
    for (int tap = 0; tap < 9; ++tap) {
      mult(0, tap, acc1, r[1], r[2], r[0]);
      if (tap < 8) finish(0, tap, acc0, rv, o);
      if (tap == 3) load_row(r[1], t.y0 + 2);
      if (tap == 8) put(m[0], o);
      interleave(std::integral_constant<int, 3>{});
    }
  }
  int y = t.y0;
  first(2, y + 1, std::true_type{});
  second(2, y);
  for (++y; y + 3 <= yv; y += 3) {
    step(0, y);
    step(1, y + 1);
    step(2, y + 2);
  }
  if (yv - y == 1) {
    step(0, y);
  } else if (yv - y == 2) {
    step(0, y);
    step(1, y + 1);
  }
  u32x4 o[4];
#pragma unroll
  for (int u = 0; u < 8; ++u) finish(1, u, acc1, true, o);
#pragma unroll
  for (int q = 0; q < 4; ++q) store_b128<ST>(o[q], rout, ooff[q] + t.img + (uint32_t)(yv - 1) * t.rowbytes);
}

}  // namespace igm

using namespace igm;

namespace {
ConvArgs conv_args(const void* in, const void* w, const float* bias, const void* aux, const int32_t* ext, int B,
                   int H, int W, void* out, int own) {
  ConvArgs a{};
  a.in = (const bf16*)in;
  a.wt[0] = (const bf16*)w;
  a.bias[0] = bias;
  a.aux = (const bf16*)aux;
  a.out = (bf16*)out;
  a.ext = ext;
  a.B = B;
  a.H = H;
  a.W = W;
  a.g = conv_geom(B, H, W, own, ext != nullptr);
  return a;
}
int64_t act_bytes(int B, int H, int W) { return (int64_t)B * H * W * kC * 2; }
}  // namespace

extern "C" {

int igm_conv3x3_fwd_bf16(const void* in, const void* wpacked, const float* bias,
                         const int32_t* extents, int32_t B, int32_t H, int32_t W, void* out,
                         void* stream) {
  IGM_CHECK_ARG(in && wpacked && bias && out, "null pointer");
  IGM_CHECK_ARG(in != out, "in and out must differ");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535, "bad sizes");
  IGM_CHECK_ARG(act_bytes(B, H, W) < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  const ConvArgs a = conv_args(in, wpacked, bias, nullptr, extents, B, H, W, out, kStripPx);
  const dim3 grid(a.g.blocks), block(256);
  hipStream_t st = (hipStream_t)stream;
  switch (conv_store_mode(act_bytes(B, H, W), false)) {
    case kStoreThrough: hipLaunchKernelGGL((conv3x3_kernel<0, kStoreThrough, false>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((conv3x3_kernel<0, kStoreCached, false>), grid, block, 0, st, a); break;
  }
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_conv3x3_head_fwd_bf16(const void* in, const void* wpacked, const float* bias,
                              const void* head_wpacked, const float* head_bias, const int32_t* extents,
                              int32_t B, int32_t H, int32_t W, int32_t cout, void* out, float* Y,
                              void* stream) {
  IGM_CHECK_ARG(in && wpacked && bias && head_wpacked && head_bias && Y, "null pointer");
  IGM_CHECK_ARG(in != out, "in and out must differ");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC, "cout must be in [1, 32]");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535, "bad sizes");
  IGM_CHECK_ARG(act_bytes(B, H, W) < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  ConvArgs a = conv_args(in, wpacked, bias, nullptr, extents, B, H, W, out, kStripPx);
  a.head = (const bf16*)head_wpacked;
  a.headb = head_bias;
  a.Y = Y;
  a.cout = cout;
  const dim3 grid(a.g.blocks), block(256);
  hipStream_t st = (hipStream_t)stream;
  switch (conv_store_mode(act_bytes(B, H, W), false)) {
    case kStoreThrough: hipLaunchKernelGGL((conv3x3_kernel<0, kStoreThrough, true>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((conv3x3_kernel<0, kStoreCached, true>), grid, block, 0, st, a); break;
  }
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_conv3x3_pair_fwd_bf16(const void* in, const void* w1, const float* b1, const void* w2,
                              const float* b2, const int32_t* extents, int32_t B, int32_t H,
                              int32_t W, void* out, void* stream) {
  IGM_CHECK_ARG(in && w1 && b1 && w2 && b2 && out, "null pointer");
  IGM_CHECK_ARG(in != out, "in and out must differ");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535, "bad sizes");
  IGM_CHECK_ARG(act_bytes(B, H, W) < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  ConvArgs a = conv_args(in, w1, b1, nullptr, extents, B, H, W, out, kPairPx);
  a.wt[1] = (const bf16*)w2;
  a.bias[1] = b2;
  const dim3 grid(a.g.blocks), block(256);
  hipStream_t st = (hipStream_t)stream;
  switch (conv_store_mode(act_bytes(B, H, W), false)) {
    case kStoreThrough: hipLaunchKernelGGL((conv3x3_pair_kernel<kStoreThrough>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((conv3x3_pair_kernel<kStoreCached>), grid, block, 0, st, a); break;
  }
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_conv3x3_dgrad_bf16(const void* dz, const void* wpacked_dgrad, const void* act_below,
                           const int32_t* extents, int32_t B, int32_t H, int32_t W, void* dz_below,
                           void* stream) {
  IGM_CHECK_ARG(dz && wpacked_dgrad && act_below && dz_below, "null pointer");
  IGM_CHECK_ARG(dz != dz_below, "in and out must differ");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535, "bad sizes");
  IGM_CHECK_ARG(act_bytes(B, H, W) < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  const ConvArgs a = conv_args(dz, wpacked_dgrad, nullptr, act_below, extents, B, H, W, dz_below, kStripPx);
  const dim3 grid(a.g.blocks), block(256);
  hipStream_t st = (hipStream_t)stream;
  switch (conv_store_mode(act_bytes(B, H, W), true)) {
    case kStoreThrough: hipLaunchKernelGGL((conv3x3_kernel<1, kStoreThrough, false>), grid, block, 0, st, a); break;
    case kStoreStream: hipLaunchKernelGGL((conv3x3_kernel<1, kStoreStream, false>), grid, block, 0, st, a); break;
    default: hipLaunchKernelGGL((conv3x3_kernel<1, kStoreCached, false>), grid, block, 0, st, a); break;
  }
  IGM_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
