// Weight gradients of the emulator's 3x3 layers on gfx950 (layer 1, which reads
// float32 fields: below).  32 -> 32 layers:
//   dW[tap][co][ci] = sum_p dz[p][co] * act[p + delta_tap][ci],  db[co] = sum_p dz[p][co]
// (the tape through Conv2D, emulate/emulate.py:252).
//
// K is the pixels: a product takes 16 co x 16 ci over 32 pixels, so both
// operands have to be transposed, 8 pixels of one channel per lane where NHWC
// rows hold 8 channels of one pixel.  A wave owns a strip of 32 columns, walks
// down its rows and keeps the whole 9 x 32 x 32 gradient in its accumulators
// (144 registers per lane).  Each row of either operand is read from memory
// once, written to LDS as it is and read back transposed (ds_read_b64_tr_b16):
// the three x-shifts of the activation are three reads at other pixels, and
// their fragments stay in registers for the three rows that use them.  The
// wave's LDS is its own, so nothing waits for a barrier, and no VALU work is
// left.  db is a product with ones.
//
// What bounds it: 1000 x 1000 takes 25.5 us, 128 MB at 5.0 TB/s, a copy's
// rate (36 products of 16 cycles per 32 pixels are 7.5 us); 8 x 496 x 496
// padded patches 40 us, with 256 blocks, one wave per SIMD (512: 1000 x 1000
// 32.6 us).  The earlier kernel transposed with VALU packing into
// block-wide LDS tiles, read by all waves between barriers: 39 and 62 us.
//
// wgrad3x3_kernel is the weight gradient alone and serves igm_conv_wgrad_bf16 and
// igm_conv_wgrad_partials_bf16; the network's backward pass runs bwd3x3_kernel.
#include "conv_common.hpp"

namespace igm {

constexpr int kWgPx = 32;                 // columns of a wave's strip: the K of one product
constexpr int kWgRows = 4;                // rows of a round of the march

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;

// Transposed operand from LDS rows of kCh channels per pixel: 32 pixels, from
// pixel p on, of channel 16 cb + lane % 16; with g = lane / 16, slot 8 g + j
// is pixel 4 g + j (j < 4) or 16 + 4 g + j - 4.
template <int kCh>
__device__ __forceinline__ bf16x8 transposed(const bf16* s, int p, int cb) {
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const bf16* q = s + (p + 4 * g + (n >> 2)) * kCh + 16 * cb + 4 * (n & 3);
  const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)q);
  const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(q + 16 * kCh));
  return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// The sums of a block's four waves, in order, in the lanes' own layout: entry
// ((tap * 4 + block) * 64 + lane) * 4 + e, then the bias.
__device__ __forceinline__ void wave_sums(const f32x4 (&acc)[9][2][2], const f32x4 (&accb)[2],
                                          f32x4 (&sums)[4][kWg9 / 4], int blk, int accumulate, float* partials) {
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4, wave = threadIdx.x >> 6;
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) sums[wave][(t * 4 + i) * 64 + lane] = acc[t][i >> 1][i & 1];
  if (n == 0) {
#pragma unroll
    for (int c = 0; c < 2; ++c) sums[wave][9 * kC * kC / 4 + 4 * c + g] = accb[c];
  }
  __syncthreads();
  f32x4* P = reinterpret_cast<f32x4*>(partials + (int64_t)blk * kWg9);
  constexpr int kPer = (kWg9 / 4 + 255) / 256;
  f32x4 prev[kPer];
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int q = threadIdx.x + 256 * k;
    prev[k] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (accumulate) prev[k] = P[q < kWg9 / 4 ? q : 0];
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int q = threadIdx.x + 256 * k;
    if (q < kWg9 / 4) {
      const f32x4 v = ((sums[0][q] + sums[1][q]) + sums[2][q]) + sums[3][q];
      P[q] = accumulate ? prev[k] + v : v;
    }
  }
}

__global__ void __launch_bounds__(256, 1)
wgrad3x3_kernel(const bf16* __restrict__ act, const bf16* __restrict__ dz, const int32_t* __restrict__ ext,
                int B, int H, int W, int chunks, int accumulate, float* __restrict__ partials) {
  constexpr int kRing = 4;  // rows of each operand in flight from memory
  // rows in transposition, later the waves' sums
  constexpr int kStage = (kWgPx + 16 + kWgPx) * kC;
  __shared__ __attribute__((aligned(16))) union {
    bf16 rows[4][kStage];
    f32x4 sums[4][kWg9 / 4];
  } sm;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = xcd_remap(blockIdx.x, gridDim.x), wid = blk * 4 + wave, nw = gridDim.x * 4;
  bf16* sa = sm.rows[wave];                       // activation row: pixels x0 - 1 .. x0 + 32
  bf16* sz = sa + (kWgPx + 16) * kC;       // dz row: pixels x0 .. x0 + 31
  const uint32_t bytes = (uint32_t)((int64_t)B * H * W * kC * 2);
  const uint32_t rowbytes = (uint32_t)W * kC * 2;

  f32x4 acc[9][2][2], accb[2];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[t][i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  accb[0] = accb[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = f2bf(1.f);

  StripShare<kWgPx, kWgRows> share(ext, B, H, W, chunks, wid, nw);
  while (share.more()) {
    const StripRange sr = share.next();
    const int b = sr.b, x0 = sr.x0, y0 = sr.y0, y1 = sr.y1, ny = sr.ny, nx = sr.nx;
    if (y0 >= y1) continue;
    const uint32_t img = (uint32_t)b * H * rowbytes;
    // a lane's 16 B of a row: pixel lane / 4 of 16, chunk lane % 4
    const int px = lane >> 2;
    auto off = [&](int x, bool ok) { return (ok & (x >= 0) & (x < nx)) ? (uint32_t)(x * kC * 2 + (lane & 3) * 16) : kOOB; };
    const uint32_t oz[2] = {off(x0 + px, true), off(x0 + 16 + px, true)};
    const uint32_t oa[3] = {off(x0 - 1 + px, true), off(x0 + 15 + px, true), off(x0 + 31 + px, px < 2)};
    u32x4 stz[kRing][2], sta[kRing][3];
    // feed j: activation row y0 - 1 + j and dz row y0 - 2 + j
    auto load = [&](int s, int j) {
      const int ya = y0 - 1 + j, yz = y0 - 2 + j;
      const bool oka = (ya >= 0) & (ya < ny) & (ya <= y1), okz = (yz >= y0) & (yz < y1);
      const rsrc_t ra = make_rsrc(act, oka ? bytes : 0u), rz = make_rsrc(dz, okz ? bytes : 0u);
      const uint32_t pa = oka ? img + (uint32_t)ya * rowbytes : 0u, pz = okz ? img + (uint32_t)yz * rowbytes : 0u;
#pragma unroll
      for (int i = 0; i < 3; ++i) sta[s][i] = __builtin_amdgcn_raw_buffer_load_b128(ra, oa[i], pa, 0);
#pragma unroll
      for (int i = 0; i < 2; ++i) stz[s][i] = __builtin_amdgcn_raw_buffer_load_b128(rz, oz[i], pz, 0);
    };
    bf16x8 F[4][3][2], D[2][2];
    auto feed = [&](int s, int f, int d, int j) {
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(sa + i * 16 * kC + lane * 8) = sta[s][i];
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(sz + i * 16 * kC + lane * 8) = stz[s][i];
      load(s, j + kRing);
#pragma unroll
      for (int t = 0; t < 3; ++t)
#pragma unroll
        for (int c = 0; c < 2; ++c) F[f][t][c] = transposed<kC>(sa, t, c);
#pragma unroll
      for (int c = 0; c < 2; ++c) D[d][c] = transposed<kC>(sz, 0, c);
    };
    // products of dz row y0 + j - 3, whose operands feeds j - 3 .. j - 1 read
    auto mult = [&](int j) {
#pragma unroll
      for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          acc[t][i >> 1][i & 1] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              D[(j + 1) & 1][i >> 1], F[(j + 1 + t / 3) & 3][t % 3][i & 1], acc[t][i >> 1][i & 1], 0, 0, 0);
#pragma unroll
      for (int c = 0; c < 2; ++c)
        accb[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(D[(j + 1) & 1][c], ones, accb[c], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < kRing; ++s) load(s, s);
#pragma unroll
    for (int j = 0; j < 3; ++j) feed(j % kRing, j & 3, j & 1, j);
    const int end = y1 - y0 + 3;
    // four steps at a time (the rings' period); rows past the last feed zeros
    for (int j = 3; j < end; j += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        feed((3 + k) % kRing, (3 + k) & 3, (3 + k) & 1, j + k);
        mult(3 + k);
      }
    }
  }

  wave_sums(acc, accb, sm.sums, blk, accumulate, partials);
}

// The weight gradient and the data gradient, below = conv(dz, wt) * (act > 0 ?
// 1 : 0.01) with the taps-reversed weights wt, in one pass over act and dz: 192
// B per pixel where the two kernels move 320.  The same march; both operands'
// rows go to LDS four deep.  The data gradient reads its dz operand from there
// as it is, the weights from LDS too, and the activation's signs.  Two rows of
// both gradients are interleaved in twelve slots of 8 to 14 products, one per
// dz row and tap column: a slot's operands are read one slot ahead, a dz row's
// fragments serve both output rows, a tap's weights are kept for the second.
//
// What bounds it: at 1000 x 1000 the memory, 192 MB in 46 us, 4.2 TB/s (the two
// kernels: 57); 256 x 319 11.4 us (15.8), where a wave has four rows and as many
// steps to fill and drain.  With one row per step, the weights read for every
// row and operands in registers that spilled, 1000 x 1000 took 69 us.
//
// Batches of uneven patches take as long as the wave with the most rows, about
// 1 us a row and 8 us more.  Split by StripShare, 8 patches of 197 .. 294 cells
// take 37 us and of 302 .. 394 cells 50 us; with equal blocks of rows of the
// padded batch, dealt out in turn, 58 and 75.  At 410 .. 496 cells memory bounds
// it again, and neighbouring strips out of step cost 6 us: 88, where the padded
// blocks took 82.
template <int ST>
__global__ void __launch_bounds__(256, 1)
bwd3x3_kernel(const bf16* __restrict__ act, const bf16* __restrict__ dz, const bf16* __restrict__ wt,
              const int32_t* __restrict__ ext, int B, int H, int W, int chunks, int accumulate,
              bf16* __restrict__ below, float* __restrict__ partials) {
  constexpr int kRowPx = kWgPx + 16;  // an LDS row: pixels x0 - 1 .. x0 + 32 (and 14 unused)
  // four rows of each operand and the weights, later the waves' sums
  __shared__ __attribute__((aligned(16))) union {
    struct {
      bf16 act[4][4][kRowPx * kC], dz[4][4][kRowPx * kC];
      u32x4 w[18][64];
    } in;
    f32x4 sums[4][kWg9 / 4];
  } sm;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = xcd_remap(blockIdx.x, gridDim.x), wid = blk * 4 + wave, nw = gridDim.x * 4;
  const uint32_t bytes = (uint32_t)((int64_t)B * H * W * kC * 2);
  const uint32_t rowbytes = (uint32_t)W * kC * 2;
  for (int f = threadIdx.x >> 6; f < 18; f += 4) sm.in.w[f][lane] = *conv_weight_frag(wt, n, g, f >> 1, f & 1);
  __syncthreads();

  f32x4 acc[9][2][2], accb[2];
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[t][i >> 1][i & 1] = f32x4{0.f, 0.f, 0.f, 0.f};
  accb[0] = accb[1] = f32x4{0.f, 0.f, 0.f, 0.f};
  bf16x8 ones;
#pragma unroll
  for (int e = 0; e < 8; ++e) ones[e] = f2bf(1.f);

  if (ext != nullptr) {  // zeros outside the extents' strips, a row at a time
    const rsrc_t ro = make_rsrc(below, bytes);
    for (int r = wid; r < B * H; r += nw) {
      int ny, nx;
      extent_of(ext, r / H, H, W, ny, nx);
      const int x0 = r % H < ny ? (max(nx, 0) + kWgPx - 1) / kWgPx * kWgPx : 0;
      for (int x = x0 + (lane >> 2); x < W; x += 16)
        store_b128(u32x4{0, 0, 0, 0}, ro, (uint32_t)r * rowbytes + (uint32_t)(x * kC * 2 + (lane & 3) * 16));
    }
  }
  StripShare<kWgPx, kWgRows> share(ext, B, H, W, chunks, wid, nw);
  while (share.more()) {
    const StripRange sr = share.next();
    const int b = sr.b, x0 = sr.x0, y0 = sr.y0, y1 = sr.y1, ny = sr.ny, nx = sr.nx;
    if (y0 >= y1) continue;
    const uint32_t img = (uint32_t)b * H * rowbytes;
    uint32_t oo[2];  // data gradient: pixel x0 + 16 q + n, channels 8 g .. 8 g + 7
    bool xin[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      const int x = x0 + 16 * q + n;
      oo[q] = x < W ? (uint32_t)(x * kC + 8 * g) * 2 : kOOB;
      xin[q] = x < nx;
    }
    // a lane's 16 B of a row: pixel lane / 4 of 16, chunk lane % 4
    const int px = lane >> 2;
    auto off = [&](int x, bool ok) { return (ok & (x >= 0) & (x < nx)) ? (uint32_t)(x * kC * 2 + (lane & 3) * 16) : kOOB; };
    const uint32_t oi[3] = {off(x0 - 1 + px, true), off(x0 + 15 + px, true), off(x0 + 31 + px, px < 2)};
    struct Rows {
      u32x4 a[3], z[3];
    };
    // feed j: activation row y0 - 1 + j and dz row y0 - 2 + j
    auto load = [&](Rows& st, int j) {
      const int ya = y0 - 1 + j, yz = y0 - 2 + j;
      const bool oka = (ya >= 0) & (ya < ny) & (ya <= y1), okz = (yz >= 0) & (yz >= y0 - 1) & (yz < ny) & (yz <= y1);
      const rsrc_t ra = make_rsrc(act, oka ? bytes : 0u), rz = make_rsrc(dz, okz ? bytes : 0u);
      const uint32_t pa = oka ? img + (uint32_t)ya * rowbytes : 0u, pz = okz ? img + (uint32_t)yz * rowbytes : 0u;
#pragma unroll
      for (int i = 0; i < 3; ++i) st.a[i] = __builtin_amdgcn_raw_buffer_load_b128(ra, oi[i], pa, 0);
#pragma unroll
      for (int i = 0; i < 3; ++i) st.z[i] = __builtin_amdgcn_raw_buffer_load_b128(rz, oi[i], pz, 0);
    };
    auto put = [&](const Rows& st, int f) {
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(sm.in.act[wave][f] + i * 16 * kC + lane * 8) = st.a[i];
#pragma unroll
      for (int i = 0; i < 3; ++i) *reinterpret_cast<u32x4*>(sm.in.dz[wave][f] + i * 16 * kC + lane * 8) = st.z[i];
    };
    Rows st[2];
    bf16x8 F[4][3][2], D[2][2];
    auto readF = [&](int f, int t) {  // tap column t of the activation row in slot f
#pragma unroll
      for (int c = 0; c < 2; ++c) F[f][t][c] = transposed<kC>(sm.in.act[wave][f], t, c);
    };
    auto readD = [&](int f) {
#pragma unroll
      for (int c = 0; c < 2; ++c) D[f & 1][c] = transposed<kC>(sm.in.dz[wave][f], 1, c);
    };
    auto maskD = [&](int f, int j) {  // zero outside the wave's own rows
      const int yz = y0 - 2 + j;
      const uint32_t mask = ((yz >= y0) & (yz < y1)) ? ~0u : 0u;
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        u32x4 v = __builtin_bit_cast(u32x4, D[f & 1][c]);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] &= mask;
        D[f & 1][c] = as_bf16x8(v);
      }
    };
    // products 2 p and 2 p + 1 of dz row y0 + j - 3, from feeds j - 3 .. j - 1
    auto mult = [&](int j, int p) {
      if (p == 18) {
#pragma unroll
        for (int c = 0; c < 2; ++c)
          accb[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(D[(j + 1) & 1][c], ones, accb[c], 0, 0, 0);
        return;
      }
      const int t = p >> 1, c = p & 1;
#pragma unroll
      for (int i = 0; i < 2; ++i)
        acc[t][c][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(D[(j + 1) & 1][c], F[(j + 1 + t / 3) & 3][t % 3][i],
                                                               acc[t][c][i], 0, 0, 0);
    };
    // Rows y = y0 + j - 3 and y + 1 of the data gradient, from dz rows r = 0 ..
    // 3 of feeds j - 2 .. j + 1: tap row r of the first, r - 1 of the second.
    bf16x8 Z[2][2], Wt[3][2], Wn[2][2];
    f32x4 o[2][2][2];
    auto readZW = [&](int jj, int i) {  // operands of slot i = 3 r + s
      const int r = i / 3, s = i % 3;
#pragma unroll
      for (int q = 0; q < 2; ++q)
        Z[i & 1][q] = as_bf16x8(*reinterpret_cast<const u32x4*>(sm.in.dz[wave][(jj + 2 + r) & 3] + (16 * q + n + s) * kC + 8 * g));
      if (r < 3) {
#pragma unroll
        for (int c = 0; c < 2; ++c) Wn[i & 1][c] = as_bf16x8(sm.in.w[2 * (3 * r + s) + c][lane]);
      }
    };
    auto finish = [&](int jj, int k, int y) {  // row y + k
      const rsrc_t ro = make_rsrc(below, y + k < y1 ? bytes : 0u);
#pragma unroll
      for (int q = 0; q < 2; ++q) {
        const u32x4 av = *reinterpret_cast<const u32x4*>(sm.in.act[wave][(jj + 2 + k) & 3] + (16 * q + n + 1) * kC + 8 * g);
        bf16x8 h;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const uint32_t w = av[e >> 1];
          h[e] = f2bf(o[k][q][e >> 2][e & 3] *
                      (__uint_as_float((e & 1) ? (w & 0xFFFF0000u) : (w << 16)) > 0.f ? 1.f : 0.01f));
        }
        u32x4 v = __builtin_bit_cast(u32x4, h);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = xin[q] ? v[i] : 0u;
        store_b128<ST>(v, ro, oo[q] + img + (uint32_t)(y + k) * rowbytes);
      }
    };
    // Two rows of both gradients in twelve slots.
    auto step = [&](int jj, int j) {
      put(st[jj & 1], jj & 3);
      load(st[jj & 1], j + 2);
      readZW(jj, 0);
#pragma unroll
      for (int i = 0; i < 12; ++i) {
        if (i + 1 < 12) readZW(jj, i + 1);
        if (i == 0) readD(jj & 3);
        if (i == 3) maskD(jj & 3, j);
        if (i >= 1 && i < 4) readF(jj & 3, i - 1);
        if (i == 5) {
          put(st[(jj + 1) & 1], (jj + 1) & 3);
          load(st[(jj + 1) & 1], j + 3);
        }
        if (i == 6) readD((jj + 1) & 3);
        if (i == 9) maskD((jj + 1) & 3, j + 1);
        if (i >= 7 && i < 10) readF((jj + 1) & 3, i - 7);
        __builtin_amdgcn_sched_barrier(0);
        const int r = i / 3, s = i % 3;
#pragma unroll
        for (int q = 0; q < 2; ++q)
#pragma unroll
          for (int c = 0; c < 2; ++c) {
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
            if (r < 3)
              o[0][q][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Wn[i & 1][c], Z[i & 1][q], i == 0 ? zero : o[0][q][c], 0, 0, 0);
            if (r > 0)
              o[1][q][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(Wt[s][c], Z[i & 1][q], i == 3 ? zero : o[1][q][c], 0, 0, 0);
          }
        if (r < 3) {
#pragma unroll
          for (int c = 0; c < 2; ++c) Wt[s][c] = Wn[i & 1][c];
        }
#pragma unroll
        for (int p = 0; p < 3; ++p) mult(jj + i / 6, 3 * (i % 6) + p);
        if (i % 6 == 5) mult(jj + i / 6, 18);
        if (i == 10) finish(jj, 0, y0 + j - 3);
        if (i < 11) __builtin_amdgcn_sched_barrier(0);
      }
      finish(jj, 1, y0 + j - 3);
    };
    load(st[0], 0);
    load(st[1], 1);
#pragma unroll
    for (int j = 0; j < 3; ++j) {
      put(st[j & 1], j & 3);
      load(st[j & 1], j + 2);
#pragma unroll
      for (int t = 0; t < 3; ++t) readF(j & 3, t);
    }
    readD(2);
    maskD(2, 2);
    const int end = y1 - y0 + 3;
    // four rows at a time (the rings' period); rows past the last feed zeros
    for (int j = 3; j < end; j += 4) {
      step(3, j);
      step(5, j + 2);
    }
  }
  wave_sums(acc, accb, sm.sums, blk, accumulate, partials);
}

// Layer 1 (5 float32 fields -> 32): dW1[tap][ci][co] = sum_p X[p + delta_tap][ci] * dz1[p][co].
//
// The same march on the matrix units, with every float32 input split into
// three bf16 parts, x = h + m + l: 8 + 8 + 8 significant bits are all 24 of
// them, so the parts' products with the bf16 dz1 are exact and the sums stay
// float32, one per part.  The 5 fields' parts and a one are the 16 rows of a
// product: two products per tap and 32 pixels, the bias with them.  Channel
// 4 i + e of a pixel: part e (h, m, l) of field i for e < 3; e = 3: field 4's
// h, m, l, then the one.
//
// A part is zero where x has no bits left for it, and zero times an infinite
// dz1 is NaN.  h is zero only where x is (below 2^-133 aside), so its sum alone
// says what becomes of infinities and NaN: where it is not finite it is the
// result (split_sum).
//
// What bounds it: 1000 x 1000 takes 21 us (512 blocks, 23 with 256), 84 MB at
// 4.0 TB/s; 8 x 496 x 496 padded patches 30 us.  Float32 FMAs from LDS tiles
// took 90 and 168 us, with twice the rounding error.
constexpr int kXc = 16;  // channels of a split pixel

__device__ __forceinline__ float split_sum(float h, float m, float l) {
  return __builtin_isfinite(h) ? (l + m) + h : h;
}

__global__ void __launch_bounds__(256, 2)
conv_in_wgrad_kernel(const float* __restrict__ f0, const float* __restrict__ f1, const float* __restrict__ f2,
                     const float* __restrict__ f3, const float* __restrict__ f4, int64_t fb, int64_t fr, int64_t fc,
                     const bf16* __restrict__ dz, const int32_t* __restrict__ ext, int B, int H, int W, int chunks, int accumulate,
                     float* __restrict__ partials) {
  constexpr int kRing = 4;         // rows of each operand in flight from memory
  constexpr int kXpx = kWgPx + 2;  // pixels x0 - 1 .. x0 + 32
  constexpr int kStage = (kXpx * kXc + kWgPx * kC);
  __shared__ __attribute__((aligned(16))) union {
    bf16 rows[4][kStage];
    float sums[4][9][8][kC];
  } sm;
  const int lane = threadIdx.x & 63, n = lane & 15, g = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int blk = xcd_remap(blockIdx.x, gridDim.x), wid = blk * 4 + wave, nw = gridDim.x * 4;
  bf16* sx = sm.rows[wave];
  bf16* sz = sx + kXpx * kXc;
  const uint32_t bytes = (uint32_t)((int64_t)B * H * W * kC * 2);
  const uint32_t rowbytes = (uint32_t)W * kC * 2;
  const float* fs[kCin] = {f0, f1, f2, f3, f4};

  f32x4 acc[9][2];
#pragma unroll
  for (int t = 0; t < 9; ++t) acc[t][0] = acc[t][1] = f32x4{0.f, 0.f, 0.f, 0.f};

  StripShare<kWgPx, kWgRows> share(ext, B, H, W, chunks, wid, nw);
  while (share.more()) {
    const StripRange sr = share.next();
    const int b = sr.b, x0 = sr.x0, y0 = sr.y0, y1 = sr.y1, ny = sr.ny, nx = sr.nx;
    if (y0 >= y1) continue;
    const uint32_t img = (uint32_t)b * H * rowbytes;
    // dz: 16 B of a row per lane, pixel lane / 4 of 16; X: pixel x0 - 1 + lane.
    // X's addresses are clamped into the extent, its values masked when split.
    auto off = [&](int x) { return x < nx ? (uint32_t)(x * kC * 2 + (lane & 3) * 16) : kOOB; };
    const uint32_t oz[2] = {off(x0 + (lane >> 2)), off(x0 + 16 + (lane >> 2))};
    const int xx = x0 - 1 + lane;
    const bool okx = (xx >= 0) & (xx < nx);
    const int64_t ox = (int64_t)b * fb + (int64_t)min(max(xx, 0), nx - 1) * fc;
    u32x4 stz[kRing][2];
    float stx[kRing][kCin];
    // feed j: X row y0 - 1 + j and dz row y0 - 2 + j
    auto load = [&](int s, int j) {
      const int yx = y0 - 1 + j, yz = y0 - 2 + j;
      const bool okz = (yz >= y0) & (yz < y1);
      const rsrc_t rz = make_rsrc(dz, okz ? bytes : 0u);
      const uint32_t pz = okz ? img + (uint32_t)yz * rowbytes : 0u;
      const int64_t oy = (int64_t)min(max(yx, 0), ny - 1) * fr + ox;
#pragma unroll
      for (int ci = 0; ci < kCin; ++ci) stx[s][ci] = fs[ci][oy];
#pragma unroll
      for (int i = 0; i < 2; ++i) stz[s][i] = __builtin_amdgcn_raw_buffer_load_b128(rz, oz[i], pz, 0);
    };
    bf16x8 F[4][3], D[2][2];
    auto feed = [&](int s, int f, int d, int j) {
      const int yx = y0 - 1 + j;
      const bool ok = okx & (yx >= 0) & (yx < ny) & (yx <= y1);
      uint32_t part[3][kCin];
#pragma unroll
      for (int ci = 0; ci < kCin; ++ci) {
        // (quiet: a NaN keeps its upper bits' NaN in h)
        const float x = ok ? __builtin_canonicalizef(stx[s][ci]) : 0.f;
        part[0][ci] = __float_as_uint(x) & 0xFFFF0000u;
        const float h = __uint_as_float(part[0][ci]);
        const float r = x == h ? 0.f : x - h;  // (an infinity has no remainder)
        part[1][ci] = __float_as_uint(r) & 0xFFFF0000u;
        part[2][ci] = __float_as_uint(r - __uint_as_float(part[1][ci]));
      }
      u32x4 c[2];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint32_t last = i < 3 ? part[i][4] : 0x3F800000u;
        c[i >> 1][2 * (i & 1)] = (part[0][i] >> 16) | part[1][i];
        c[i >> 1][2 * (i & 1) + 1] = (part[2][i] >> 16) | (last & 0xFFFF0000u);
      }
      if (lane < kXpx) {
        reinterpret_cast<u32x4*>(sx + lane * kXc)[0] = c[0];
        reinterpret_cast<u32x4*>(sx + lane * kXc)[1] = c[1];
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4*>(sz + i * 16 * kC + lane * 8) = stz[s][i];
      load(s, j + kRing);
#pragma unroll
      for (int t = 0; t < 3; ++t) F[f][t] = transposed<kXc>(sx, t, 0);
#pragma unroll
      for (int cb = 0; cb < 2; ++cb) D[d][cb] = transposed<kC>(sz, 0, cb);
    };
    // products of dz row y0 + j - 3, whose operands feeds j - 3 .. j - 1 read
    auto mult = [&](int j) {
#pragma unroll
      for (int t = 0; t < 9; ++t)
#pragma unroll
        for (int cb = 0; cb < 2; ++cb)
          acc[t][cb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(F[(j + 1 + t / 3) & 3][t % 3], D[(j + 1) & 1][cb],
                                                               acc[t][cb], 0, 0, 0);
    };
#pragma unroll
    for (int s = 0; s < kRing; ++s) load(s, s);
#pragma unroll
    for (int j = 0; j < 3; ++j) feed(j % kRing, j & 3, j & 1, j);
    const int end = y1 - y0 + 3;
    for (int j = 3; j < end; j += 4) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        feed((3 + k) % kRing, (3 + k) & 3, (3 + k) & 1, j + k);
        mult(3 + k);
      }
    }
  }

  // the parts' sums, small ones first, then the four waves' in order
  __syncthreads();
#pragma unroll
  for (int t = 0; t < 9; ++t)
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
      const f32x4 a = acc[t][cb];
      sm.sums[wave][t][g][cb * 16 + n] = split_sum(a[0], a[1], a[2]);
      sm.sums[wave][t][4 + g][cb * 16 + n] = a[3];
    }
  __syncthreads();
  float* P = partials + (int64_t)blk * kWgIn;
  constexpr int kPer = (kWgIn + 255) / 256;
  float prev[kPer];  // (all loads before the first store)
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = threadIdx.x + 256 * k;
    prev[k] = (accumulate && i < kWgIn) ? P[i] : 0.f;
  }
#pragma unroll
  for (int k = 0; k < kPer; ++k) {
    const int i = threadIdx.x + 256 * k;
    if (i >= kWgIn) continue;
    const int co = i % kC, m = i / kC, t = m < 9 * kCin ? m / kCin : 4, ci = m < 9 * kCin ? m % kCin : 7;
    float v = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      v += ci == 4 ? split_sum(sm.sums[w][t][4][co], sm.sums[w][t][5][co], sm.sums[w][t][6][co]) : sm.sums[w][t][ci][co];
    P[i] = accumulate ? prev[k] + v : v;
  }
}

// (a start of the march: three rows of operands before the first products)
inline int wgrad_chunks(const int32_t* ext, int B, int H, int W, int nblocks) {
  return strip_chunks(ext, B, H, W, kWgPx, kWgRows, 3, 4 * nblocks);
}

int wgrad3x3_launch(const void* act, const void* dz, const int32_t* ext, int B, int H, int W, int nblocks,
                    float* partials, int accumulate, hipStream_t st) {
  hipLaunchKernelGGL(wgrad3x3_kernel, dim3(nblocks), dim3(256), 0, st, (const bf16*)act, (const bf16*)dz, ext, B, H, W,
                     wgrad_chunks(ext, B, H, W, nblocks), accumulate, partials);
  IGM_CHECK_LAUNCH();
  return 0;
}

}  // namespace igm

extern "C" int igm_conv3x3_bwd_bf16(const void* act, const void* dz, const void* wpacked_dgrad, const int32_t* extents,
                                    int32_t B, int32_t H, int32_t W, int32_t nblocks, float* partials,
                                    int32_t accumulate, void* dz_below, void* stream) {
  using namespace igm;
  IGM_CHECK_ARG(act && dz && wpacked_dgrad && partials && dz_below, "null pointer");
  IGM_CHECK_ARG(dz != dz_below && act != dz_below, "in and out must differ");
  IGM_CHECK_ARG(nblocks >= 1 && B >= 1 && H >= 1 && W >= 1, "bad sizes");
  const int64_t bytes = (int64_t)B * H * W * kC * 2;
  IGM_CHECK_ARG(bytes < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  const int acc = accumulate ? 1 : 0, chunks = wgrad_chunks(extents, B, H, W, nblocks);
  hipStream_t st = (hipStream_t)stream;
  switch (conv_store_mode(bytes, true)) {
#define IGM_STORE_CASE(ST)                                                                                          \
  case ST:                                                                                                          \
    hipLaunchKernelGGL((bwd3x3_kernel<ST>), dim3(nblocks), dim3(256), 0, st, (const bf16*)act,              \
                       (const bf16*)dz, (const bf16*)wpacked_dgrad, extents, B, H, W, chunks, acc,                  \
                       (bf16*)dz_below, partials);                                                                  \
    break;
    IGM_STORE_CASE(kStoreCached)
    IGM_STORE_CASE(kStoreStream)
    IGM_STORE_CASE(kStoreThrough)
#undef IGM_STORE_CASE
  }
  IGM_CHECK_LAUNCH();
  return 0;
}

extern "C" int igm_conv_in_wgrad_partials(const float* f0, const float* f1, const float* f2, const float* f3,
                                          const float* f4, int64_t fb, int64_t fr, int64_t fc, const int32_t* extents,
                                          int32_t B, int32_t H, int32_t W, const void* dz1, int32_t nblocks,
                                          float* partials, int32_t accumulate, void* stream) {
  using namespace igm;
  IGM_CHECK_ARG(f0 && f1 && f2 && f3 && f4 && dz1 && partials, "null pointer");
  IGM_CHECK_ARG(nblocks >= 1 && B >= 1 && H >= 1 && W >= 1, "bad sizes");
  IGM_CHECK_ARG((int64_t)B * H * W * kC * 2 < (int64_t)kOOB, "activations above 2 GiB (32-bit buffer offsets)");
  hipLaunchKernelGGL(conv_in_wgrad_kernel, dim3(nblocks), dim3(256), 0, (hipStream_t)stream, f0, f1, f2, f3, f4, fb, fr,
                     fc, (const bf16*)dz1, extents, B, H, W, wgrad_chunks(extents, B, H, W, nblocks),
                     accumulate ? 1 : 0, partials);
  IGM_CHECK_LAUNCH();
  return 0;
}
