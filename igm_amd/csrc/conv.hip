// Convolutional emulator of IGM's ice flow on gfx950: forward and backward
// kernels of the "cnn" network (emulate/neural_network.py:9-66):
//   16 x [Conv2D 3x3 "same" + bias -> LeakyReLU(0.01)] -> Conv2D 1x1 + bias.
//
// Data layout: activations are NHWC bf16 (B, H, W, 32); the network output Y
// is NHWC fp32 (B, H, W, 2Nz).  Per-batch (ny, nx) extents mask padded
// batches: every kernel writes zeros outside a batch entry's extent, which
// makes a padded batch behave exactly like per-entry "same" zero padding.
//
// Kernels:
//  (layer 1: conv_in.hip)
//  (the 32 -> 32 3x3 layers, forward and data gradient: conv3x3.hip)
//  head_mfma_kernel     1x1 32 -> 2Nz (<= 32) output layer, fp32 out.
//  wgrad1x1_kernel      weight gradient of the head: K = pixels; tiles are
//                       transposed into LDS as [channel][pixel]; per-block
//                       partial sums.  (3x3 layers and layer 1: wgrad3x3.hip)
//  wgrad_reduce_*       deterministic sums of the partials: every layer of a
//                       network in one launch, or one layer in two stages.
//  head_bwd_kernel      dY -> dA16 * LeakyReLU'(A16) (fp32 VALU) and a padded
//                       bf16 copy of dY for the head's wgrad.
//  Adam: per-tensor clip_by_norm + legacy Adam on the fp32 master weights,
//  then bf16 packing of the MFMA operands.
#include "conv_common.hpp"

namespace igm {

constexpr int kTileW = 64;    // pixels per tile row
constexpr int kChStride = 72; // LDS channel-row stride in bf16 (144 B) for wgrad

// Gradient of the network with respect to its 5 input fields, through
// layer 1: the transpose of its cross-correlation,
//   dX[b, y, x, ci] = sum_{r, s, co} W[r][s][ci][co] * dz1[b, y - r + 1, x - s + 1, co],
// zero padding, fp32 accumulation in a fixed order; dz1 (bf16 NHWC, 32
// channels) is the gradient at layer 1's pre-activation output.  Zeros
// outside an entry's extent.
__global__ void __launch_bounds__(256)
conv_in_dgrad_kernel(const bf16* __restrict__ dz1, const int32_t* __restrict__ ext, int H, int W,
                     const float* __restrict__ w, float* __restrict__ dX) {
  __shared__ float ws[9 * kCin * kC];
  for (int i = threadIdx.x; i < 9 * kCin * kC; i += blockDim.x) ws[i] = w[i];
  __syncthreads();
  const int x = blockIdx.x * blockDim.x + threadIdx.x;
  const int y = blockIdx.y;
  const int b = blockIdx.z;
  if (x >= W) return;
  int ny, nx;
  extent_of(ext, b, H, W, ny, nx);
  float* o = dX + (((int64_t)b * H + y) * W + x) * kCin;
  float acc[kCin];
#pragma unroll
  for (int ci = 0; ci < kCin; ++ci) acc[ci] = 0.f;
  if (y < ny && x < nx) {
#pragma unroll 1
    for (int r = 0; r < 3; ++r) {
      const int yy = y - r + 1;
#pragma unroll 1
      for (int s = 0; s < 3; ++s) {
        const int xx = x - s + 1;
        if (yy < 0 || yy >= ny || xx < 0 || xx >= nx) continue;
        const uint4* src = reinterpret_cast<const uint4*>(dz1 + (((int64_t)b * H + yy) * W + xx) * kC);
        const float* wr = ws + (r * 3 + s) * kCin * kC;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const uint4 u = src[q];
          const uint32_t wv[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            const int co = 8 * q + e;
            const uint32_t bits = (e & 1) ? (wv[e >> 1] & 0xFFFF0000u) : (wv[e >> 1] << 16);
            const float d = __uint_as_float(bits);
#pragma unroll
            for (int ci = 0; ci < kCin; ++ci) acc[ci] += d * wr[ci * kC + co];
          }
        }
      }
    }
  }
#pragma unroll
  for (int ci = 0; ci < kCin; ++ci) o[ci] = acc[ci];
}

// ------------------------------------------------------- 1x1 head (MFMA) --
// wt: [32 out (zero-padded beyond cout)][32 in] bf16; Y fp32 (B,H,W,cout).
__global__ void __launch_bounds__(256)
head_mfma_kernel(const bf16* __restrict__ in, const bf16* __restrict__ wt,
                 const float* __restrict__ bias, const int32_t* __restrict__ ext, int H, int W,
                 int cout, float* __restrict__ Y) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int64_t npx = (int64_t)H * W;
  const int64_t p0 = ((int64_t)blockIdx.x * 4 + wave) * 64;  // 64 pixels per wave
  const int b = blockIdx.y;
  if (p0 >= npx) return;
  int ny, nx;
  extent_of(ext, b, H, W, ny, nx);
  bf16x8 wf[2];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
    wf[cb] = *reinterpret_cast<const bf16x8*>(wt + ((cb * 16 + (lane & 15)) * kC + 8 * (lane >> 4)));
  const bf16* ib = in + (int64_t)b * npx * kC;
  float* Yb = Y + (int64_t)b * npx * cout;
  // this lane's output channels co = cb*16 + 4*(lane/16) + e: their biases,
  // and whether all 4 are real (cout % 4 == 0 makes a pixel's row of cout
  // floats 16-B aligned: one 16-B store per lane and channel block)
  float bl[2][4];
#pragma unroll
  for (int cb = 0; cb < 2; ++cb)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int co = cb * 16 + 4 * (lane >> 4) + e;
      bl[cb][e] = co < cout ? bias[co] : 0.f;
    }
  const bool vec = (cout % 4) == 0 && (reinterpret_cast<uintptr_t>(Y) & 15) == 0;
#pragma unroll
  for (int pb = 0; pb < 4; ++pb) {
    const int64_t p = p0 + pb * 16 + (lane & 15);
    f32x4 acc[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
    for (int kc = 0; kc < 1; ++kc) {
      bf16x8 bfr;
      if (p < npx) bfr = *reinterpret_cast<const bf16x8*>(ib + p * kC + 8 * (lane >> 4));
      else {
#pragma unroll
        for (int e = 0; e < 8; ++e) bfr[e] = f2bf(0.f);
      }
      acc[0] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[0], bfr, acc[0], 0, 0, 0);
      acc[1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[1], bfr, acc[1], 0, 0, 0);
    }
    if (p >= npx) continue;
    const int yy = (int)(p / W), xx = (int)(p % W);
    const bool valid = yy < ny && xx < nx;
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const int co = cb * 16 + 4 * (lane >> 4);
      float o[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o[e] = valid ? acc[cb][e] + bl[cb][e] : 0.f;
      if (vec) {
        if (co < cout) *reinterpret_cast<float4*>(Yb + p * cout + co) = make_float4(o[0], o[1], o[2], o[3]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (co + e < cout) Yb[p * cout + co + e] = o[e];
      }
    }
  }
}

// ------------------------------------------------------- head backward --
// dZ16 = (dY W17^T) * LeakyReLU'(A16) (bf16); dYb = bf16(dY) zero-padded to 32.
// w17: HWIO [32 in][cout] fp32.
__global__ void __launch_bounds__(256)
head_bwd_kernel(const float* __restrict__ dY, const bf16* __restrict__ a16,
                const float* __restrict__ w17, const int32_t* __restrict__ ext, int H, int W,
                int cout, bf16* __restrict__ dz16, bf16* __restrict__ dYb) {
  // ws[ci][co] = w17[ci][co], zero for co >= cout: the loops below run over
  // whole groups of 4 output channels with static register indices (the
  // padded terms add exact zeros)
  __shared__ __attribute__((aligned(16))) float ws[kC][kC];
  for (int i = threadIdx.x; i < kC * kC; i += blockDim.x) {
    const int ci = i / kC, co = i % kC;
    ws[ci][co] = co < cout ? w17[ci * cout + co] : 0.f;
  }
  __syncthreads();
  const int64_t npx = (int64_t)H * W;
  const int64_t p = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (p >= npx) return;
  int ny, nx;
  extent_of(ext, b, H, W, ny, nx);
  const int yy = (int)(p / W), xx = (int)(p % W);
  const bool valid = yy < ny && xx < nx;
  const int64_t q = (int64_t)b * npx + p;
  if (!valid) {  // outside the extent: zero gradients, no arithmetic
    const uint4 z = {0, 0, 0, 0};
#pragma unroll
    for (int c4 = 0; c4 < 4; ++c4) {
      reinterpret_cast<uint4*>(dz16 + q * kC)[c4] = z;
      reinterpret_cast<uint4*>(dYb + q * kC)[c4] = z;
    }
    return;
  }
  // dY's row of cout floats: 16-B loads when cout % 4 == 0 (the row is then
  // 16-B aligned in a 16-B aligned dY), 4-B loads otherwise
  float d[kC];
  if ((cout % 4) == 0 && (reinterpret_cast<uintptr_t>(dY) & 15) == 0) {
#pragma unroll
    for (int g = 0; g < kC / 4; ++g) {
      const float4 t = 4 * g < cout ? *reinterpret_cast<const float4*>(dY + q * cout + 4 * g)
                                    : make_float4(0.f, 0.f, 0.f, 0.f);
      d[4 * g] = t.x;
      d[4 * g + 1] = t.y;
      d[4 * g + 2] = t.z;
      d[4 * g + 3] = t.w;
    }
  } else {
#pragma unroll
    for (int c = 0; c < kC; ++c) d[c] = c < cout ? dY[q * cout + c] : 0.f;
  }
  // s[ci] = sum over co = 0 .. cout-1, in order, of d[co] * w[ci][co]
  float s[kC];
#pragma unroll
  for (int ci = 0; ci < kC; ++ci) s[ci] = 0.f;
#pragma unroll
  for (int g = 0; g < kC / 4; ++g) {
    if (4 * g < cout) {  // wave-uniform
#pragma unroll
      for (int ci = 0; ci < kC; ++ci) {
        const float4 wv = *reinterpret_cast<const float4*>(&ws[ci][4 * g]);
        s[ci] += d[4 * g] * wv.x;
        s[ci] += d[4 * g + 1] * wv.y;
        s[ci] += d[4 * g + 2] * wv.z;
        s[ci] += d[4 * g + 3] * wv.w;
      }
    }
  }
  bf16x8 outv[4], outy[4];
#pragma unroll
  for (int c4 = 0; c4 < 4; ++c4) {
    const bf16x8 av = reinterpret_cast<const bf16x8*>(a16 + q * kC)[c4];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int ci = c4 * 8 + e;
      outv[c4][e] = f2bf(s[ci] * (bf2f(av[e]) > 0.f ? 1.f : 0.01f));
      outy[c4][e] = f2bf(d[ci]);
    }
  }
#pragma unroll
  for (int c4 = 0; c4 < 4; ++c4) {
    reinterpret_cast<bf16x8*>(dz16 + q * kC)[c4] = outv[c4];
    reinterpret_cast<bf16x8*>(dYb + q * kC)[c4] = outy[c4];
  }
}

// ------------------------------------------------------------ wgrad MFMA --
// Weight gradient of the 1x1 head: dW[co][ci] = sum_p A[p][ci] * dZ[p][co],
// db[co] = sum_p dZ[p][co].  Persistent blocks over tiles of kWgRows rows x 64
// pixels; wave w owns the output block (co-block w & 1, ci-block w >> 1).
// LDS holds the tile's dZ and activation rows transposed ([channel][pixel]),
// written as packed 2-pixel dwords.  A block loads its next tile into
// registers before the current tile's MFMAs.
// partials: [gridDim.x][1024 + 32] fp32.
constexpr int kWgRows = 4;  // rows per tile

__global__ void __launch_bounds__(256)
wgrad1x1_kernel(const bf16* __restrict__ act, const bf16* __restrict__ dz,
                const int32_t* __restrict__ ext, int B, int H, int W, int accumulate,
                float* __restrict__ partials) {
  __shared__ __attribute__((aligned(16))) uint32_t lds_dz[kWgRows][kC][kChStride / 2];
  __shared__ __attribute__((aligned(16))) uint32_t lds_act[kWgRows][kC][kChStride / 2];
  __shared__ float dbred[256][8];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int cb = wave & 1, cib = wave >> 1;
  const int ntx = (W + kTileW - 1) / kTileW;
  const int nty = (H + kWgRows - 1) / kWgRows;
  const int ntiles = B * nty * ntx;  // < 2^25: activations below 2 GiB

  f32x4 acc = {0.f, 0.f, 0.f, 0.f};
  // accumulate: this block's partial sums of the previous sub-batches, loaded
  // now so that their latency hides behind the tiles (added at the end)
  float* P = partials + (int64_t)blockIdx.x * (kC * kC + kC);
  const int ci = cib * 16 + (lane & 15);
  f32x4 prev;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int co = cb * 16 + 4 * (lane >> 4) + e;
    prev[e] = accumulate ? P[co * kC + ci] : 0.f;
  }
  float dba[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) dba[e] = 0.f;

  // Staging of a tile: rows y0 .. y0 + kWgRows - 1 of both operands, each as
  // 16-B channel chunks of pixel pairs, in registers; masked lanes (outside
  // the entry's extent, or no next tile) read zeros.
  constexpr int kItems = kWgRows * 32 * 4;
  constexpr int kPer = kItems / 256;
  const uint32_t vbytes = (uint32_t)((int64_t)B * H * W * kC * 2);
  const rsrc_t rdz = make_rsrc(dz, vbytes), ract = make_rsrc(act, vbytes);
  uint4 sdz[kPer][2], sact[kPer][2];
  struct Tile {
    int b, y0, x0, ny, nx;
    bool valid;
  };
  auto tile_of = [&](int t) {
    Tile r;
    r.b = t / (nty * ntx);
    r.y0 = ((t / ntx) % nty) * kWgRows;
    r.x0 = (t % ntx) * kTileW;
    extent_of(ext, r.b, H, W, r.ny, r.nx);
    r.valid = r.y0 < r.ny && r.x0 < r.nx;
    return r;
  };
  auto ld16 = [&](rsrc_t r, bool ok, int64_t pix, int chunk) {
    const uint32_t off = ok ? (uint32_t)((pix * kC + chunk * 8) * 2) : kOOB;
    const auto v = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
    return uint4{v[0], v[1], v[2], v[3]};
  };
  auto issue_loads = [&](const Tile& t, bool live) {
    const int64_t img = (int64_t)t.b * H * W;
    const bool on = live && t.valid;
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int c = tid + 256 * k;
      const int chunk = c & 3, q = (c >> 2) & 31, row = c >> 7;
      const int y = t.y0 + row, xa = t.x0 + 2 * q;
      const bool rok = on && y < t.ny;
      const int64_t pix = img + (int64_t)y * W + xa;
      sdz[k][0] = ld16(rdz, rok && xa < t.nx, pix, chunk);
      sdz[k][1] = ld16(rdz, rok && xa + 1 < t.nx, pix + 1, chunk);
      sact[k][0] = ld16(ract, rok && xa < t.nx, pix, chunk);
      sact[k][1] = ld16(ract, rok && xa + 1 < t.nx, pix + 1, chunk);
    }
  };
  // staged registers -> LDS, channel-major with pixel pairs per dword; thread
  // tid always takes channel chunk tid & 3, and sums its dZ channels into the
  // bias gradient
  auto store_tile = [&]() {
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
      const int c = tid + 256 * k;
      const int chunk = c & 3, q = (c >> 2) & 31, row = c >> 7;
      const uint32_t a[4] = {sdz[k][0].x, sdz[k][0].y, sdz[k][0].z, sdz[k][0].w};
      const uint32_t c2[4] = {sdz[k][1].x, sdz[k][1].y, sdz[k][1].z, sdz[k][1].w};
      const uint32_t u[4] = {sact[k][0].x, sact[k][0].y, sact[k][0].z, sact[k][0].w};
      const uint32_t u2[4] = {sact[k][1].x, sact[k][1].y, sact[k][1].z, sact[k][1].w};
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        // channel 2i: low halves; channel 2i+1: high halves (bf16 bit patterns)
        lds_dz[row][chunk * 8 + 2 * i][q] = (a[i] & 0xFFFFu) | (c2[i] << 16);
        lds_dz[row][chunk * 8 + 2 * i + 1][q] = (a[i] >> 16) | (c2[i] & 0xFFFF0000u);
        dba[2 * i] += __uint_as_float(a[i] << 16) + __uint_as_float(c2[i] << 16);
        dba[2 * i + 1] += __uint_as_float(a[i] & 0xFFFF0000u) + __uint_as_float(c2[i] & 0xFFFF0000u);
        lds_act[row][chunk * 8 + 2 * i][q] = (u[i] & 0xFFFFu) | (u2[i] << 16);
        lds_act[row][chunk * 8 + 2 * i + 1][q] = (u[i] >> 16) | (u2[i] & 0xFFFF0000u);
      }
    }
  };

  int tile = blockIdx.x;
  Tile cur = tile_of(tile < ntiles ? tile : 0);
  issue_loads(cur, tile < ntiles);
  for (; tile < ntiles; tile += gridDim.x) {
    const bool valid = cur.valid;  // block-uniform
    if (valid) {
      __syncthreads();  // the previous tile's fragment reads are done
      store_tile();
      __syncthreads();
    }
    const int nt = tile + gridDim.x;
    cur = tile_of(nt < ntiles ? nt : tile);
    issue_loads(cur, nt < ntiles);
    if (!valid) continue;
#pragma unroll
    for (int rr = 0; rr < kWgRows; ++rr) {
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        const int base = (ks * 32 + 8 * (lane >> 4)) / 2;  // dword index of the 8-pixel group
        const u32x4 a4 = *reinterpret_cast<const u32x4*>(&lds_dz[rr][cb * 16 + (lane & 15)][base]);
        const u32x4 b4 = *reinterpret_cast<const u32x4*>(&lds_act[rr][cib * 16 + (lane & 15)][base]);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a4), as_bf16x8(b4), acc, 0, 0, 0);
      }
    }
  }
  // partial dW: D[co][ci], lane: ci = cib*16 + lane%16, co = cb*16 + 4*(lane/16) + e
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int co = cb * 16 + 4 * (lane >> 4) + e;
    P[co * kC + ci] = accumulate ? prev[e] + acc[e] : acc[e];
  }
  // partial db: thread t holds channels (t&3)*8 .. +8
#pragma unroll
  for (int e = 0; e < 8; ++e) dbred[tid][e] = dba[e];
  __syncthreads();
  if (tid < kC) {
    const int chunk = tid >> 3, e = tid & 7;
    float s = 0.f;
    for (int t = chunk; t < 256; t += 4) s += dbred[t][e];
    P[kC * kC + tid] = accumulate ? P[kC * kC + tid] + s : s;
  }
}

// Deterministic reduction of one layer's per-block partials P[nblk][stride], in
// two stages, for the calls that ask for one layer (igm_conv_wgrad_bf16,
// igm_conv_in_wgrad, igm_conv_wgrad_reduce_f32); a network's layers go through
// wgrad_reduce_layers_kernel.  Stage 1 (partials_group_sum_kernel): group g of R rows,
// rows g*R .. min(nblk, (g+1)*R) - 1, is summed in row order into its first
// row, in place; each (group, column) belongs to one thread, so the write
// races with nothing, and the loads are issued 8 at a time.  Stage 2 sums
// the group rows in group order.  The fixed order makes the result
// independent of scheduling.
__global__ void __launch_bounds__(256)
partials_group_sum_kernel(float* __restrict__ P, int nblk, int stride, int ncols, int R) {
  const int c = blockIdx.x * 256 + threadIdx.x;
  const int r0 = blockIdx.y * R;
  if (c >= ncols || r0 >= nblk) return;
  const int n = min(nblk, r0 + R) - r0;
  float* p = P + (int64_t)r0 * stride + c;
  float s = 0.f;
  int r = 0;
  for (; r + 8 <= n; r += 8) {
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = p[(int64_t)(r + i) * stride];
#pragma unroll
    for (int i = 0; i < 8; ++i) s += v[i];
  }
  for (; r < n; ++r) s += p[(int64_t)r * stride];
  p[0] = s;
}

// Position of entry src of a layer's partial sums in its HWIO kernel of cout
// output channels, or -1 past them; entries from taps * 1024 on are the bias.
__device__ __forceinline__ int wgrad_kernel_pos(int taps, int src, int cout) {
  const int tap = src / (kC * kC), r = src % (kC * kC);
  int ci = r % kC, co = r / kC;
  if (taps == 9) {  // wgrad3x3_kernel's layout: ((tap * 4 + block) * 64 + lane) * 4 + e
    const int block = r >> 8, lane = (r >> 2) & 63;
    co = 16 * (block >> 1) + 4 * (lane >> 4) + (r & 3);
    ci = 16 * (block & 1) + (lane & 15);
  }
  return co < cout ? (tap * kC + ci) * cout + co : -1;
}

// Stage 2 for a 3x3 or 1x1 layer: the group sums of each entry, in the order of
// wgrad_kernel_pos (then the 32 bias entries), scattered to dW (HWIO, cout
// output channels) and db.
__global__ void __launch_bounds__(256)
wgrad_reduce_kernel(const float* __restrict__ P, int ngroups, int R, int taps, int cout,
                    int accumulate, float* __restrict__ dW, float* __restrict__ db) {
  const int stride = taps * kC * kC + kC;
  const int src = blockIdx.x * 256 + threadIdx.x;
  if (src >= stride) return;
  float t = 0.f;
  for (int g = 0; g < ngroups; ++g) t += P[(int64_t)g * R * stride + src];
  if (src < taps * kC * kC) {
    const int pos = wgrad_kernel_pos(taps, src, cout);
    if (pos >= 0) dW[pos] = accumulate ? dW[pos] + t : t;
  } else {
    const int co = src - taps * kC * kC;
    if (co < cout) db[co] = accumulate ? db[co] + t : t;
  }
}

// The partial sums of every layer of a network into its flat gradient, in one
// launch: a block takes 64 consecutive entries of one layer's rows, each of its
// four waves every fourth row, in order, and wave 0 adds the four sums in order:
// rows of zeros at the end, of blocks without work, change nothing.  Layer by
// layer in two stages these were 34 launches of 4 to 6 us for 16 layers, which
// read 140 MB in all.
struct ReduceArgs {
  const float* part[3];  // layer 1, the 3x3 layers one after the other, the head
  int rows[3];
  int n3x3, cout, accumulate;
  const int64_t* offs;   // kernel of layer l at g + offs[2 l], its bias at g + offs[2 l + 1]
  float* g;
};
constexpr int reduce_blocks(int entries) { return (entries + 63) / 64; }
__global__ void __launch_bounds__(256)
wgrad_reduce_layers_kernel(const ReduceArgs a) {
  int blk = blockIdx.x, layer = 0, kind = 0;
  if (blk >= reduce_blocks(kWgIn)) {
    blk -= reduce_blocks(kWgIn);
    const int l = blk / reduce_blocks(kWg9);
    kind = l < a.n3x3 ? 1 : 2;
    layer = kind == 1 ? 1 + l : 1 + a.n3x3;
    blk -= (kind == 1 ? l : a.n3x3) * reduce_blocks(kWg9);
  }
  const int entries = kind == 0 ? kWgIn : (kind == 1 ? kWg9 : kWg1);
  const int rows = a.rows[kind];
  const int quarter = threadIdx.x >> 6, src = blk * 64 + (threadIdx.x & 63);
  float s = 0.f;
  if (src < entries) {
    const float* p = a.part[kind] + (kind == 1 ? (int64_t)(layer - 1) * rows * entries : 0) + src;
    int r = quarter;
    for (; r + 28 < rows; r += 32) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = p[(int64_t)(r + 4 * i) * entries];
#pragma unroll
      for (int i = 0; i < 8; ++i) s += v[i];
    }
    for (; r < rows; r += 4) s += p[(int64_t)r * entries];
  }
  __shared__ float red[4][64];
  red[quarter][threadIdx.x & 63] = s;
  __syncthreads();
  if (quarter != 0 || src >= entries) return;
  s = ((red[0][src & 63] + red[1][src & 63]) + red[2][src & 63]) + red[3][src & 63];
  const int cout = kind == 2 ? a.cout : kC;
  const int nk = entries - kC;  // the bias entries are the last 32
  float* d = nullptr;
  if (src >= nk) {
    if (src - nk < cout) d = a.g + a.offs[2 * layer + 1] + (src - nk);
  } else {
    const int pos = kind == 0 ? src : wgrad_kernel_pos(kind == 1 ? 9 : 1, src, cout);
    if (pos >= 0) d = a.g + a.offs[2 * layer] + pos;
  }
  if (d) *d = a.accumulate ? *d + s : s;
}

// Stage 1 + 2 on the host side: G groups of R rows, G <= kMaxGroups.
constexpr int kMaxGroups = 16;
inline void group_rows(int nblk, int* R, int* G) {
  *G = nblk < kMaxGroups ? nblk : kMaxGroups;
  *R = (nblk + *G - 1) / *G;
  *G = (nblk + *R - 1) / *R;
}

// Stage 2 as a plain column sum: out[i] = sum over the group rows of P[.][i],
// i < count
__global__ void __launch_bounds__(256)
sum_partials_kernel(const float* __restrict__ P, int ngroups, int R, int stride, int count,
                    int accumulate, float* __restrict__ out) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= count) return;
  float t = 0.f;
  for (int g = 0; g < ngroups; ++g) t += P[(int64_t)g * R * stride + i];
  out[i] = accumulate ? out[i] + t : t;
}

// ------------------------------------------------------------ optimizer --
// Per-tensor sum of squares (one block per tensor), deterministic.
__global__ void __launch_bounds__(256)
sqnorm_kernel(const float* __restrict__ g, const int64_t* __restrict__ offs, float* __restrict__ sq) {
  const int t = blockIdx.x;
  const int64_t a = offs[t], e = offs[t + 1];
  __shared__ float red[256];
  float s = 0.f;
  for (int64_t i = a + threadIdx.x; i < e; i += 256) s += g[i] * g[i];
  red[threadIdx.x] = s;
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
    __syncthreads();
  }
  if (threadIdx.x == 0) sq[t] = red[0];
}

// tf.clip_by_norm per tensor, then legacy Adam on the fp32 master weights.
__global__ void __launch_bounds__(256)
adam_clip_kernel(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                 float* __restrict__ v, int64_t n, const int64_t* __restrict__ offs, int ntens,
                 const float* __restrict__ sq, float clipnorm, float alpha, float omb1, float omb2,
                 float eps) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  int lo = 0, hi = ntens;  // offs[lo] <= i < offs[hi]
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (offs[mid] <= i) lo = mid; else hi = mid;
  }
  float gi = g[i];
  if (clipnorm > 0.f) {
    const float l2sum = sq[lo];
    const float l2norm = l2sum > 0.f ? sqrtf(l2sum) : l2sum;
    gi = gi * clipnorm / fmaxf(l2norm, clipnorm);
  }
  float mi = m[i], vi = v[i];
  mi += (gi - mi) * omb1;
  vi += (gi * gi - vi) * omb2;
  m[i] = mi;
  v[i] = vi;
  w[i] -= (mi * alpha) / (sqrtf(vi) + eps);
}

// bf16 MFMA operands from the fp32 HWIO master weights of the 3x3 layers:
// fwd[L][tap][co][ci] = W[tap][ci][co];  dgrad[L][tap][ci][co] = W[8 - tap][ci][co].
__global__ void __launch_bounds__(256)
pack3x3_kernel(const float* __restrict__ w, const int64_t* __restrict__ offs, int nlayers,
               bf16* __restrict__ fwd, bf16* __restrict__ dgr) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int per = 9 * kC * kC;
  if (i >= (int64_t)nlayers * per) return;
  const int L = (int)(i / per), r = (int)(i % per);
  const int tap = r / (kC * kC), a = (r / kC) % kC, c = r % kC;
  const float* W = w + offs[L];
  // fwd element [tap][co=a][ci=c]
  fwd[i] = f2bf(W[(tap * kC + c) * kC + a]);
  // dgrad element [tap][out=ci=a][in=co=c] = W[8-tap][ci=a][co=c]
  dgr[i] = f2bf(W[((8 - tap) * kC + a) * kC + c]);
}

// head operand [32 co (zero-padded)][32 ci] from HWIO [ci][cout].
__global__ void pack_head_kernel(const float* __restrict__ w, int cout, bf16* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= kC * kC) return;
  const int co = i / kC, ci = i % kC;
  out[i] = f2bf(co < cout ? w[ci * cout + co] : 0.f);
}

inline int grid_for(int64_t n, int b = 256) { return (int)((n + b - 1) / b); }

}  // namespace igm

// =================================================================== C-ABI ==
using namespace igm;

extern "C" {

int igm_conv1x1_head_fwd(const void* in, const void* wpacked, const float* bias,
                         const int32_t* extents, int32_t B, int32_t H, int32_t W, int32_t cout,
                         float* Y, void* stream) {
  IGM_CHECK_ARG(in && wpacked && bias && Y, "null pointer");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC, "cout must be in [1, 32]");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535, "bad sizes");
  const int64_t npx = (int64_t)H * W;
  dim3 grid((unsigned)((npx + 255) / 256), B);
  hipLaunchKernelGGL(head_mfma_kernel, grid, dim3(256), 0, (hipStream_t)stream, (const bf16*)in,
                     (const bf16*)wpacked, bias, extents, H, W, cout, Y);
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_conv1x1_head_bwd(const float* dY, const void* a16, const float* w_hwio,
                         const int32_t* extents, int32_t B, int32_t H, int32_t W, int32_t cout,
                         void* dz16, void* dY_bf16, void* stream) {
  IGM_CHECK_ARG(dY && a16 && w_hwio && dz16 && dY_bf16, "null pointer");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC, "cout must be in [1, 32]");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535, "bad sizes");
  const int64_t npx = (int64_t)H * W;
  dim3 grid((unsigned)((npx + 255) / 256), B);
  hipLaunchKernelGGL(head_bwd_kernel, grid, dim3(256), 0, (hipStream_t)stream, dY,
                     (const bf16*)a16, w_hwio, extents, H, W, cout, (bf16*)dz16, (bf16*)dY_bf16);
  IGM_CHECK_LAUNCH();
  return 0;
}

int64_t igm_wgrad_workspace_floats(int32_t taps, int32_t nblocks) {
  if (taps == 9) return (int64_t)nblocks * kWg9;
  if (taps == 1) return (int64_t)nblocks * kWg1;
  if (taps == 0) return (int64_t)nblocks * kWgIn;  // layer 1
  return 0;
}

int igm_conv_wgrad_partials_bf16(int32_t taps, const void* act, const void* dz,
                                 const int32_t* extents, int32_t B, int32_t H, int32_t W,
                                 int32_t nblocks, float* partials, int32_t accumulate,
                                 void* stream) {
  IGM_CHECK_ARG(act && dz && partials, "null pointer");
  IGM_CHECK_ARG(taps == 9 || taps == 1, "taps must be 9 or 1");
  IGM_CHECK_ARG(nblocks >= 1 && B >= 1 && H >= 1 && W >= 1, "bad sizes");
  IGM_CHECK_ARG((int64_t)B * H * W * kC * 2 < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  hipStream_t st = (hipStream_t)stream;
  const int acc = accumulate ? 1 : 0;
  if (taps == 9) return wgrad3x3_launch(act, dz, extents, B, H, W, nblocks, partials, acc, st);
  hipLaunchKernelGGL(wgrad1x1_kernel, dim3(nblocks), dim3(256), 0, st, (const bf16*)act, (const bf16*)dz,
                     extents, B, H, W, acc, partials);
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_conv_wgrad_reduce_f32(int32_t taps, int32_t cout, int32_t nblocks, float* partials,
                              int32_t accumulate, float* dW_hwio, float* db, void* stream) {
  IGM_CHECK_ARG(partials && dW_hwio && db, "null pointer");
  IGM_CHECK_ARG(taps == 9 || taps == 1 || taps == 0, "taps must be 9, 1 or 0 (layer 1)");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC, "cout must be in [1, 32]");
  IGM_CHECK_ARG(taps != 0 || cout == kC, "layer 1 has 32 outputs");
  IGM_CHECK_ARG(nblocks >= 1, "bad sizes");
  hipStream_t st = (hipStream_t)stream;
  int R, G;
  group_rows(nblocks, &R, &G);
  if (taps == 0) {
    // the layer-1 partial layout is [blk][1440 + 32] = [blk][n]: a plain column sum
    const int n = kWgIn;
    hipLaunchKernelGGL(partials_group_sum_kernel, dim3((n + 255) / 256, G), dim3(256), 0, st,
                       partials, nblocks, n, n, R);
    IGM_CHECK_LAUNCH();
    hipLaunchKernelGGL(sum_partials_kernel, dim3((9 * kCin * kC + 255) / 256), dim3(256), 0, st,
                       partials, G, R, n, 9 * kCin * kC, accumulate, dW_hwio);
    IGM_CHECK_LAUNCH();
    hipLaunchKernelGGL(sum_partials_kernel, dim3(1), dim3(256), 0, st, partials + 9 * kCin * kC,
                       G, R, n, kC, accumulate, db);
    IGM_CHECK_LAUNCH();
    return 0;
  }
  const int entries = taps * kC * kC + kC;
  hipLaunchKernelGGL(partials_group_sum_kernel, dim3((entries + 255) / 256, G), dim3(256), 0, st,
                     partials, nblocks, entries, entries, R);
  IGM_CHECK_LAUNCH();
  hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((entries + 255) / 256), dim3(256), 0, st, partials,
                     G, R, taps, cout, accumulate, dW_hwio, db);
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_wgrad_reduce_layers_f32(int32_t nlayers3x3, int32_t cout, int32_t nblocks_in,
                                int32_t nblocks_3x3, int32_t nblocks_head, const float* part_in,
                                const float* part_3x3, const float* part_head, int32_t accumulate,
                                const int64_t* offs, float* g, void* stream) {
  IGM_CHECK_ARG(part_in && part_head && offs && g, "null pointer");
  IGM_CHECK_ARG(nlayers3x3 >= 0 && (nlayers3x3 == 0 || part_3x3), "null part_3x3");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC, "cout must be in [1, 32]");
  IGM_CHECK_ARG(nblocks_in >= 1 && nblocks_head >= 1 && (nlayers3x3 == 0 || nblocks_3x3 >= 1), "bad sizes");
  ReduceArgs a{};
  a.part[0] = part_in; a.part[1] = part_3x3; a.part[2] = part_head;
  a.rows[0] = nblocks_in; a.rows[1] = nblocks_3x3; a.rows[2] = nblocks_head;
  a.n3x3 = nlayers3x3; a.cout = cout; a.accumulate = accumulate ? 1 : 0;
  a.offs = offs; a.g = g;
  const int blocks = reduce_blocks(kWgIn) + nlayers3x3 * reduce_blocks(kWg9) + reduce_blocks(kWg1);
  hipLaunchKernelGGL(wgrad_reduce_layers_kernel, dim3(blocks), dim3(256), 0, (hipStream_t)stream, a);
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_conv_wgrad_bf16(int32_t taps, const void* act, const void* dz, const int32_t* extents,
                        int32_t B, int32_t H, int32_t W, int32_t cout, int32_t nblocks,
                        float* workspace, int32_t accumulate, float* dW_hwio, float* db,
                        void* stream) {
  IGM_CHECK_ARG(act && dz && workspace && dW_hwio && db, "null pointer");
  IGM_CHECK_ARG(taps == 9 || taps == 1, "taps must be 9 or 1");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC, "cout must be in [1, 32]");
  if (const int rc = igm_conv_wgrad_partials_bf16(taps, act, dz, extents, B, H, W, nblocks, workspace,
                                                  0, stream))
    return rc;
  return igm_conv_wgrad_reduce_f32(taps, cout, nblocks, workspace, accumulate, dW_hwio, db, stream);
}

int igm_conv_in_wgrad(const float* f0, const float* f1, const float* f2, const float* f3,
                      const float* f4, int64_t fb, int64_t fr, int64_t fc, const int32_t* extents,
                      int32_t B, int32_t H, int32_t W, const void* dz1, int32_t nblocks,
                      float* workspace, int32_t accumulate, float* dW_hwio, float* db,
                      void* stream) {
  IGM_CHECK_ARG(f0 && f1 && f2 && f3 && f4 && dz1 && workspace && dW_hwio && db, "null pointer");
  if (const int rc = igm_conv_in_wgrad_partials(f0, f1, f2, f3, f4, fb, fr, fc, extents, B, H, W,
                                                dz1, nblocks, workspace, 0, stream))
    return rc;
  return igm_conv_wgrad_reduce_f32(0, kC, nblocks, workspace, accumulate, dW_hwio, db, stream);
}

int igm_conv_in_dgrad(const void* dz1, const float* w_hwio, const int32_t* extents, int32_t B,
                      int32_t H, int32_t W, float* dX, void* stream) {
  IGM_CHECK_ARG(dz1 && w_hwio && dX, "null pointer");
  IGM_CHECK_ARG(B >= 1 && H >= 1 && W >= 1 && B <= 65535 && H <= 65535, "bad sizes");
  hipLaunchKernelGGL(conv_in_dgrad_kernel, dim3((W + 255) / 256, H, B), dim3(256), 0,
                     (hipStream_t)stream, (const bf16*)dz1, extents, H, W, w_hwio, dX);
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_adam_clip_f32(float* w, const float* g, float* m, float* v, int64_t n, const int64_t* offs,
                      int32_t ntens, float* sq_workspace, double clipnorm, const IgmAdam* adam,
                      void* stream) {
  IGM_CHECK_ARG(w && g && m && v && offs && sq_workspace && adam, "null pointer");
  IGM_CHECK_ARG(ntens >= 1 && n >= 1, "bad sizes");
  hipStream_t st = (hipStream_t)stream;
  hipLaunchKernelGGL(sqnorm_kernel, dim3(ntens), dim3(256), 0, st, g, offs, sq_workspace);
  IGM_CHECK_LAUNCH();
  hipLaunchKernelGGL(adam_clip_kernel, dim3(grid_for(n)), dim3(256), 0, st, w, g, m, v, n, offs,
                     ntens, sq_workspace, (float)clipnorm, (float)adam->alpha,
                     (float)(1.0 - adam->beta1), (float)(1.0 - adam->beta2), (float)adam->epsilon);
  IGM_CHECK_LAUNCH();
  return 0;
}

int igm_pack_conv_weights(const float* w, const int64_t* offs3x3, int32_t nlayers3x3,
                          const float* w_head, int32_t cout, void* fwd, void* dgrad, void* head,
                          void* stream) {
  IGM_CHECK_ARG(w && w_head && fwd && dgrad && head, "null pointer");
  IGM_CHECK_ARG(nlayers3x3 == 0 || offs3x3, "null offs3x3");
  IGM_CHECK_ARG(cout >= 1 && cout <= kC && nlayers3x3 >= 0, "bad sizes");
  hipStream_t st = (hipStream_t)stream;
  if (nlayers3x3 > 0) {
    hipLaunchKernelGGL(pack3x3_kernel, dim3(grid_for((int64_t)nlayers3x3 * 9 * kC * kC)), dim3(256),
                       0, st, w, offs3x3, nlayers3x3, (bf16*)fwd, (bf16*)dgrad);
    IGM_CHECK_LAUNCH();
  }
  hipLaunchKernelGGL(pack_head_kernel, dim3(grid_for(kC * kC)), dim3(256), 0, st, w_head, cout,
                     (bf16*)head);
  IGM_CHECK_LAUNCH();
  return 0;
}

}  // extern "C"
