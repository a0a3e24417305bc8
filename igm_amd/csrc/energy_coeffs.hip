// Coefficients of the energy that do not depend on the velocity, on gfx950:
// 7 planes per cell, computed once per solve from the 5 input fields.
//
// Reference: igm/processes/iceflow/energy/cost_shear.py:103-179,
// cost_gravity.py:24-69, cost_sliding_weertman.py:23-43,
// utils/gradient/compute_gradient.py:3-16.
//
// Plane meaning for the cell with lower-left node (j, i) (S = number of cells):
//   0  q  = dx * damp / max(H, thr)        damp = 1, or 0.01 where stag4h(C) <= 0
//   1  w  = H * Bs / (p * S)               Bs = stag4h(2 A^(-1/n)), p = 1 + 1/n
//   2  gx = 0.25 * rho*g*1e-6 * H * sx / S (sx, sy: staggered slope of usurf)
//   3  gy = 0.25 * rho*g*1e-6 * H * sy / S
//   4  cs = stag4h(C) / (s * S)            s = 1 + 1/m
//   5  bx, 6 by: staggered slope of the bed usurf - thk
// The 0.25 factors absorb the 1/4 of the horizontal node average, which the
// pass keeps unscaled (sum of the 4 corner nodes); dx in q puts the vertical
// derivative in the pass's units of 1/(4 dx) (dx = dX[b, 0, 0], the scalar
// spacing of the velocity derivatives, cost_shear.py:113).
//
// A wave owns 63 cells of a row, lane l the node column 63 strip + l, and
// walks up its rows: a node's fields are loaded once and its A^(-1/n) raised
// once, an edge's slope is divided out once; the right neighbour's come from
// lane l + 1 (DPP), the lower row's are kept.
//
// What bounds it: 48 B per cell; 1500 x 1500 takes 25 us, 4.3 TB/s (float64 40
// us).  A thread per cell, with its four corners' loads, powers and slopes of
// its own, took 43 us (float64 80).
#include "energy_pass.hpp"

namespace igm {

constexpr int kCoefOut = 63;  // cells of a wave's row

template <typename T>
__global__ void __launch_bounds__(256)
energy_coeffs_kernel(const T* __restrict__ thk, const T* __restrict__ usurf, const T* __restrict__ arrh,
                     const T* __restrict__ slid, const T* __restrict__ dX, int64_t fb, int64_t fr, int64_t fc,
                     const int32_t* __restrict__ extents, int Ny, int Nx, int nstrips, int nchunk, int rows, int ntask,
                     T inv_n, T inv_p, T inv_s, T thr, T rho_g, T* __restrict__ coef, T* __restrict__ hscale) {
  const int lane = threadIdx.x & 63;
  const int task = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (task >= ntask) return;
  const int strip = task % nstrips, chunk = (task / nstrips) % nchunk, b = task / (nstrips * nchunk);
  const int ny = extents ? min(extents[2 * b], Ny) : Ny;
  const int nx = extents ? min(extents[2 * b + 1], Nx) : Nx;
  const int i = strip * kCoefOut + lane;
  const int j0 = chunk * rows, j1 = min(j0 + rows, Ny);
  const int64_t plane = (int64_t)Ny * Nx;
  const int64_t base = (int64_t)b * fb, col = base + (int64_t)min(i, Nx - 1) * fc;
  const bool own = (lane < kCoefOut) & (i < Nx), cell = i < nx - 1;
  T* cb = coef + (int64_t)b * kPlanes * plane + (int64_t)j0 * Nx + i;
  const T dx = dX[base];
  if (task % (nstrips * nchunk) == 0 && lane == 0) hscale[b] = T(1) / (T(4) * dx);
  const T inv_S = T(1) / (T(ny - 1) * T(nx - 1));

  struct Raw {
    T t, s, d, a, c;
  };
  auto load = [&](int j) {
    const int64_t o = col + (int64_t)min(j, Ny - 1) * fr;
    return Raw{thk[o], usurf[o], dX[o], arrh[o], slid[o]};
  };
  // a node row: its fields, those of the right neighbours (r), the slopes of
  // the edges to them (ex: surface, eb: bed)
  struct Row {
    T t, s, d, a, c, b, tr, ar, cr, ex, eb;
  };
  auto node = [&](const Raw& x) {
    Row r{x.t, x.s, x.d, T(2) * T(pow(x.a, -inv_n)), x.c, x.s - x.t};
    r.tr = lane_from_right(r.t);
    r.ar = lane_from_right(r.a);
    r.cr = lane_from_right(r.c);
    const T d = lane_from_right(r.d) + r.d;
    r.ex = T(2) * (lane_from_right(r.s) - r.s) / d;
    r.eb = T(2) * (lane_from_right(r.b) - r.b) / d;
    return r;
  };
  auto st4 = [](T a11, T a10, T a01, T a00) { return (a11 + a10 + a01 + a00) / T(4); };

  const int jc = min(j1, ny - 1);  // cell rows below this one
  if (j0 < jc) {
    const Raw first = load(j0);
    Raw next = load(j0 + 1);
    Row lo = node(first);
    for (int j = j0; j < jc; ++j) {
      const Raw cur = next;
      next = load(j + 2);
      const Row hi = node(cur);
      const T H = st4(hi.tr, hi.t, lo.tr, lo.t);
      const T Bs = st4(hi.ar, hi.a, lo.ar, lo.a);
      const T Cs = st4(hi.cr, hi.c, lo.cr, lo.c);
      // compute_gradient.py:10-14 on the surface and on the bed
      const T d = hi.d + lo.d;
      const T ey = T(2) * (hi.s - lo.s) / d, fy = T(2) * (hi.b - lo.b) / d;
      const T sx = T(0.5) * (hi.ex + lo.ex), sy = T(0.5) * (lane_from_right(ey) + ey);
      const T bx = T(0.5) * (hi.eb + lo.eb), by = T(0.5) * (lane_from_right(fy) + fy);
      const T damp = Cs > T(0) ? T(1) : T(0.01);
      const T Hc = H > thr ? H : thr;
      const T v[kPlanes] = {dx * damp / Hc,
                            H * Bs * inv_p * inv_S,
                            T(0.25) * rho_g * H * sx * inv_S,
                            T(0.25) * rho_g * H * sy * inv_S,
                            Cs * inv_s * inv_S,
                            bx,
                            by};
      if (own) {
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) cb[p * plane] = cell ? v[p] : T(0);
      }
      cb += Nx;
      lo = hi;
    }
  }
  for (int j = max(j0, jc); j < j1; ++j, cb += Nx)
    if (own) {
#pragma unroll
      for (int p = 0; p < kPlanes; ++p) cb[p * plane] = T(0);
    }
}

template <typename T>
int coeffs_impl(const T* thk, const T* usurf, const T* arrh, const T* slid, const T* dX, int64_t fb, int64_t fr,
                int64_t fc, const int32_t* extents, int nbatch, int Ny, int Nx, const IgmPhysics* phys, T* coef,
                T* hscale, void* stream) {
  IGM_CHECK_ARG(thk && usurf && arrh && slid && dX && coef && hscale && phys, "null pointer");
  IGM_CHECK_ARG(nbatch >= 1 && Ny >= 2 && Nx >= 2, "need nbatch >= 1 and a grid of at least 2 x 2");
  IGM_CHECK_ARG(Ny <= 65535, "Ny must be <= 65535");
  IGM_CHECK_ARG(phys->force_negative_gravitational_energy == 0,
                "force_negative_gravitational_energy is not supported");
  const T inv_n = T(1.0 / phys->exp_glen);
  const T p = T(1.0 + 1.0 / phys->exp_glen);
  const T s = T(1.0 + 1.0 / phys->exp_weertman);
  const T rho_g = T(phys->ice_density * phys->gravity_cst * 1e-6);
  const int nstrips = (Nx + kCoefOut - 1) / kCoefOut;
  // four waves per SIMD, with equal shares of the strips' rows (1500 x 1500: 25
  // us; 27 with two waves, 27 with eight)
  int64_t rows = ((int64_t)nbatch * nstrips * Ny + 4095) / 4096;
  const int nchunk = (int)((Ny + rows - 1) / rows);
  const int64_t ntask = (int64_t)nbatch * nstrips * nchunk;
  hipLaunchKernelGGL(energy_coeffs_kernel<T>, dim3((unsigned)((ntask + 3) / 4)), dim3(256), 0, (hipStream_t)stream, thk,
                     usurf, arrh, slid, dX, fb, fr, fc, extents, Ny, Nx, nstrips, nchunk, (int)rows, (int)ntask, inv_n,
                     T(1) / p, T(1) / s, T(phys->thr_ice_thk), rho_g, coef, hscale);
  IGM_CHECK_LAUNCH();
  return 0;
}

}  // namespace igm

extern "C" {

int igm_energy_coeffs_f32(const float* thk, const float* usurf, const float* arrhenius, const float* slidingco,
                          const float* dX, int64_t fb, int64_t fr, int64_t fc, const int32_t* extents, int32_t nbatch,
                          int32_t Ny, int32_t Nx, const IgmPhysics* phys, float* coef, float* hscale, void* stream) {
  return igm::coeffs_impl<float>(thk, usurf, arrhenius, slidingco, dX, fb, fr, fc, extents, nbatch, Ny, Nx, phys, coef,
                                 hscale, stream);
}
int igm_energy_coeffs_f64(const double* thk, const double* usurf, const double* arrhenius, const double* slidingco,
                          const double* dX, int64_t fb, int64_t fr, int64_t fc, const int32_t* extents, int32_t nbatch,
                          int32_t Ny, int32_t Nx, const IgmPhysics* phys, double* coef, double* hscale, void* stream) {
  return igm::coeffs_impl<double>(thk, usurf, arrhenius, slidingco, dX, fb, fr, fc, extents, nbatch, Ny, Nx, phys, coef,
                                  hscale, stream);
}

}  // extern "C"
