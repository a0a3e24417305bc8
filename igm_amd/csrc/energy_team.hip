// Two iterations of IGM's energy solver in one pass over a small grid on gfx950
// (float32, planar layout, one field): what energy_pair.hip does, by teams.
//
// Reference: igm/processes/iceflow/solve/solve.py:45-84 and
// energy/cost_shear.py:103-179, cost_gravity.py:24-69,
// cost_sliding_weertman.py:23-43.
//
// The two-iteration pass marches: a wave of R rows runs R + 3 sweeps of the
// first iteration and R + 1 of the second, one after the other, and on a grid
// with a row per wave that chain of six is the launch's time, while most of
// the chip waits.  Here the four waves of a block take four consecutive cell
// rows at once: in a step, the sweep of the first iteration at U0, the first
// update, the sweep of the second iteration at U1 one row below, the second
// update, with the upper corners' contributions, U1 and the moments passed from
// wave to wave, and from the last wave to the first one's next step, through
// LDS.  The first step completes one row for both iterations, each further one
// four.
//
// A sweep without the row below keeps X and Z of its gradient (SplitRow), so
// that (carry - Z) + X rounds as in the march: the same results, bit for bit.
//
// What bounds it: the chain of a step, two sweeps and two updates of Nz levels
// in one wave per SIMD, about 4 us, and the launch, the prologue and the first
// loads before it: 10.9 us a launch at 100 x 100, Nz 10, where the march took
// 19.1; further steps take 6.5 to 8 us for four rows each.
#include "energy_pass.hpp"

namespace igm {

template <int NZ, int LAYOUT>
__global__ void __launch_bounds__(kPassBlock, 1)
energy_team_kernel(const PassArgs<float> a) {
  constexpr bool kInIL = (LAYOUT & kInInterleaved) != 0;
  constexpr bool kOutIL = (LAYOUT & kOutInterleaved) != 0;
  constexpr uint32_t ES = 4;
  const int lane = threadIdx.x & (kWave - 1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lblk = xcd_remap(blockIdx.x, gridDim.x);
  double e1_sh = 0.0, e1_sl = 0.0, e1_gr = 0.0;  // energy at U0 (first iteration)
  double e2_sh = 0.0, e2_sl = 0.0, e2_gr = 0.0;  // energy at U1 (second iteration)
  // From wave w to wave w + 1, slot w; from wave 3 to wave 0's next step, slot
  // 3 or 4 by the step's parity.  The upper corners' contributions of the
  // sweeps A and B, U1 and the moments m1: 125 KB at Nz 10, 150 KB at Nz 12.
  __shared__ float2 carry_a[5][NZ][kWave], carry_b[5][NZ][kWave], lds_q[5][NZ][kWave];
  __shared__ float4 lds_m[5][NZ][kWave];
  bool stopped = (a.stop != nullptr) && (*a.stop != 0);
  bool pair = true;  // two iterations (else one)
  float alpha1 = a.alpha, alpha2 = a.alpha2;
  if (a.alpha_tab != nullptr) {
    int it0;
    const int n = solve_prologue(a, lblk == 0, &it0);
    stopped = stopped || n == 0;
    pair = n == 2;
    if (n > 0) {
      alpha1 = a.alpha_tab[it0];
      alpha2 = pair ? a.alpha_tab[it0 + 1] : 0.0f;
    }
  } else if (a.prev_partials != nullptr) {
    const bool st = finalize_previous(a, lblk == 0);
    stopped = stopped || st;
  }

  if (!stopped) {
    const int strip = lblk % a.nstrips;
    const int rblk = lblk / a.nstrips;
    const int ic = strip * kPairOut - 2 + lane;
    const bool col_ok = (ic >= 0) & (ic < a.Nx);
    const bool own = (lane >= 2) & (lane <= kPairOut + 1) & col_ok;
    // node rows [j0, j1) of this block: the Ny rows split evenly over nrowblk
    const int j0 = (int)(((int64_t)rblk * a.Ny) / a.nrowblk);
    const int j1 = (int)(((int64_t)(rblk + 1) * a.Ny) / a.nrowblk);
    // (an interleaved buffer holds twice the bytes of a planar one; its V
    // resource is unused)
    const rsrc_t rU = make_rsrc(a.U, kInIL ? 2u * a.vel_bytes : a.vel_bytes);
    const rsrc_t rV = make_rsrc(kInIL ? a.U : a.V, a.vel_bytes);
    const rsrc_t rUo = make_rsrc(a.Uo, kOutIL ? 2u * a.vel_bytes : a.vel_bytes);
    const rsrc_t rVo = make_rsrc(kOutIL ? a.Uo : a.Vo, a.vel_bytes);
    const rsrc_t rC = make_rsrc(a.coef, a.coef_bytes);
    // no input moments (a fresh optimizer): every read returns 0; no output
    // moments (the last pass of a solve): every store is dropped
    const rsrc_t rMi = make_rsrc(a.mom, a.mom != nullptr ? a.mom_bytes : 0u);
    const rsrc_t rMo = make_rsrc(a.mom_out, a.mom_out != nullptr ? a.mom_bytes : 0u);
    const uint32_t kstep = (uint32_t)a.plane * ES;  // bytes between levels
    const uint32_t mstep = 4u * kstep;              // moments: 4 slots per node and level
    const float hh = a.hscale[0];
    const float hh2 = hh * hh;
    const float h05 = 0.5f * hh2, h025 = 0.25f * hh2;

    auto node_off = [&](int row, bool extra) -> uint32_t {
      const bool ok = extra & col_ok & (row >= 0) & (row < a.Ny);
      const uint32_t o = (uint32_t)(row * a.Nx + ic) * ES;
      return ok ? o : kOOB;
    };
    // a wave's inputs of a step: node rows c and c + 1 of U0 and V0 (rows j0-2
    // .. j1+1 are read), the coefficients of cell rows c (to j1) and c - 1, the
    // moments of node row c (j0-1 .. j1)
    struct In {
      float u[2][NZ], v[2][NZ], k[2][kPlanes], m[NZ][4];
    };
    auto load = [&](In& in, int c) {
#pragma unroll
      for (int r = 0; r < 2; ++r) {
        const uint32_t o = node_off(c + r, c + r <= j1 + 1);
#pragma unroll
        for (int k = 0; k < NZ; ++k) {
          if constexpr (kInIL) {
            const auto w = __builtin_amdgcn_raw_buffer_load_b64(rU, o == kOOB ? kOOB : 2u * o, 2u * k * kstep, 0);
            in.u[r][k] = __uint_as_float(w[0]);
            in.v[r][k] = __uint_as_float(w[1]);
          } else {
            in.u[r][k] = bload(rU, o, k * kstep, 0.f);
            in.v[r][k] = bload(rV, o, k * kstep, 0.f);
          }
        }
        const uint32_t co = node_off(c - r, c - r <= j1);
#pragma unroll
        for (int p = 0; p < kPlanes; ++p) in.k[r][p] = bload(rC, co, p * kstep, 0.f);
      }
      const uint32_t o = node_off(c, (c >= j0 - 1) & (c <= j1)), om = o == kOOB ? kOOB : 4u * o;
#pragma unroll
      for (int k = 0; k < NZ; ++k) mload(rMi, om, k * mstep, in.m[k]);
    };
    auto store = [&](int k, float u, float v, const float (&m)[4], uint32_t o) {
      if constexpr (kOutIL) {
        typedef unsigned int u2 __attribute__((ext_vector_type(2)));
        u2 w;
        w[0] = __float_as_uint(u);
        w[1] = __float_as_uint(v);
        __builtin_amdgcn_raw_buffer_store_b64(w, rUo, o == kOOB ? kOOB : 2u * o, 2u * k * kstep, 0);
      } else {
        bstore(u, rUo, o, k * kstep);
        bstore(v, rVo, o, k * kstep);
      }
      mstore(m, rMo, (o == kOOB ? kOOB : 4u * o) + k * mstep);
    };
    const auto none = [](int, float, float) {};

    In cur, next;
    load(cur, j0 - 2 + wave);
    for (int c = j0 - 2 + wave, s = 0; c - wave <= j1; c += 4, ++s) {
      if (c - wave + 4 <= j1) load(next, c + 4);
      __builtin_amdgcn_sched_barrier(0);
      const int put = wave < 3 ? wave : 3 + (s & 1), get = wave > 0 ? wave - 1 : 4 - (s & 1);
      const bool below = (wave > 0) | (s > 0);  // there is a row below
      // A: cell row c at U0
      SplitRow<float, NZ> ru, rv;
      {
        LevelSweep<float, NZ> sw(a, hh2, h05, h025, cur.k[0]);
#pragma unroll
        for (int k = 0; k < NZ; ++k)
          sw.level(k, cur.u[0][k], cur.v[0][k], cur.u[1][k], cur.v[1][k], ru, rv, none);
        const CellEnergy<float> e = sw.finish(ru, rv, none);
        const bool own_c = own & (c >= j0) & (c < j1);
        e1_sh += own_c ? (double)e.sh : 0.0;
        e1_sl += own_c ? (double)e.sl : 0.0;
        e1_gr += own_c ? (double)e.gr : 0.0;
      }
#pragma unroll
      for (int k = 0; k < NZ; ++k) carry_a[put][k][lane] = make_float2(ru.carry(k), rv.carry(k));
      __syncthreads();
      // first update: U1 and m1 of node row c
      float q_u[NZ], q_v[NZ];
      const uint32_t o1 = node_off(c, own & (c >= j0) & (c < j1) & !pair);
#pragma unroll
      for (int k = 0; k < NZ; ++k) {
        const float2 t = carry_a[get][k][lane];
        adam_step(cur.m[k], ru.gradient(k, below ? t.x : 0.f), rv.gradient(k, below ? t.y : 0.f), a.omb1, a.omb2,
                  alpha1, a.eps, cur.u[0][k], cur.v[0][k], q_u[k], q_v[k]);
      }
      if (!pair) {
#pragma unroll
        for (int k = 0; k < NZ; ++k) store(k, q_u[k], q_v[k], cur.m[k], o1);
        __syncthreads();  // (the contributions are read before the next step's overwrite them)
      } else {
#pragma unroll
        for (int k = 0; k < NZ; ++k) {
          lds_q[put][k][lane] = make_float2(q_u[k], q_v[k]);
          lds_m[put][k][lane] = make_float4(cur.m[k][0], cur.m[k][1], cur.m[k][2], cur.m[k][3]);
        }
        __syncthreads();
        // B: cell row c - 1 at U1
        float p_u[NZ], p_v[NZ];
        {
          LevelSweep<float, NZ> sw(a, hh2, h05, h025, cur.k[1]);
#pragma unroll
          for (int k = 0; k < NZ; ++k) {
            const float2 t = lds_q[get][k][lane];
            p_u[k] = below ? t.x : 0.f;
            p_v[k] = below ? t.y : 0.f;
            sw.level(k, p_u[k], p_v[k], q_u[k], q_v[k], ru, rv, none);
          }
          const CellEnergy<float> e = sw.finish(ru, rv, none);
          const bool own_c = own & (c - 1 >= j0) & (c - 1 < j1);
          e2_sh += own_c ? (double)e.sh : 0.0;
          e2_sl += own_c ? (double)e.sl : 0.0;
          e2_gr += own_c ? (double)e.gr : 0.0;
        }
#pragma unroll
        for (int k = 0; k < NZ; ++k) carry_b[put][k][lane] = make_float2(ru.carry(k), rv.carry(k));
        __syncthreads();
        // second update: node row c - 1
        const uint32_t o2 = node_off(c - 1, own & (c - 1 >= j0) & (c - 1 < j1));
#pragma unroll
        for (int k = 0; k < NZ; ++k) {
          const float2 t = carry_b[get][k][lane];
          const float4 m = lds_m[get][k][lane];
          float mk[4] = {m.x, m.y, m.z, m.w}, un, vn;
          adam_step(mk, ru.gradient(k, t.x), rv.gradient(k, t.y), a.omb1, a.omb2, alpha2, a.eps, p_u[k], p_v[k], un, vn);
          store(k, un, vn, mk, o2);
        }
      }
      cur = next;
    }
  }

  // deterministic block reduction: 6 doubles per block, the three energy
  // terms of each iteration
  __shared__ double red[kWavesPerBlock][6];
  double e[6] = {e1_sh, e1_sl, e1_gr, e2_sh, e2_sl, e2_gr};
#pragma unroll
  for (int t = 0; t < 6; ++t) e[t] = wave_sum(e[t]);
  if (lane == 0) {
#pragma unroll
    for (int t = 0; t < 6; ++t) red[threadIdx.x >> 6][t] = e[t];
  }
  __syncthreads();
  if (threadIdx.x == 0 && !stopped) {
    double* o = a.partials + 6 * (int64_t)lblk;
#pragma unroll
    for (int t = 0; t < 6; ++t) {
      double s = 0;
#pragma unroll
      for (int wv = 0; wv < kWavesPerBlock; ++wv) s += red[wv][t];
      o[t] = s;
    }
  }
}

int team_launch(int nz, int layout, int blocks, const PassArgs<float>& a, hipStream_t st) {
  switch (nz) {
#define IGM_TEAM_CASE(N)                                                                                            \
  case N:                                                                                                           \
    switch (layout) {                                                                                               \
      case 0: hipLaunchKernelGGL((energy_team_kernel<N, 0>), dim3(blocks), dim3(kPassBlock), 0, st, a); break;      \
      case 1: hipLaunchKernelGGL((energy_team_kernel<N, 1>), dim3(blocks), dim3(kPassBlock), 0, st, a); break;      \
      case 2: hipLaunchKernelGGL((energy_team_kernel<N, 2>), dim3(blocks), dim3(kPassBlock), 0, st, a); break;      \
      default: hipLaunchKernelGGL((energy_team_kernel<N, 3>), dim3(blocks), dim3(kPassBlock), 0, st, a); break;     \
    }                                                                                                               \
    break;
    IGM_TEAM_CASE(2)
    IGM_TEAM_CASE(3)
    IGM_TEAM_CASE(4)
    IGM_TEAM_CASE(5)
    IGM_TEAM_CASE(6)
    IGM_TEAM_CASE(8)
    IGM_TEAM_CASE(10)
    IGM_TEAM_CASE(12)
#undef IGM_TEAM_CASE
    default:
      set_error("igm_energy_pass2_f32: nz not compiled (supported: 2,3,4,5,6,8,10,12)");
      return -1;
  }
  IGM_CHECK_LAUNCH();
  return 0;
}

}  // namespace igm
