"""The moments and velocities that the fused pass writes with its gradient, on
grids of two waves per SIMD at few levels and one at ten.

The gradient is the energy + gradient pass's (the same sweep: equal bits), so a
moment m + (g - m) w is three roundings away from 64 bits, of which none is
more than 2^-24 (|g| + |m|) in float32, 2^-53 in float64 (twice that is asked,
for a fused one instead), and so is v with g^2.  An update alpha m / (sqrt(v) +
eps) is a handful of roundings from that of the moments it is made with, and
the reciprocal and square root are good to 1 ulp: 16 of the update's size, and
one of the result's."""
import pytest
import torch

from igm_amd import _lib as L
from igm_amd.energy import EnergyOperator
from oracle import energy as E
from tests.helpers import dzeta_for, small_glacier, smooth_velocity, to_dev
from tests.test_gpu_pair import random_moments

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("ny,nx,nz", [(1000, 1000, 2), (999, 1001, 3), (1000, 900, 4), (500, 700, 6), (300, 257, 10),
                                      (7, 61, 12)])
def test_fused_update_of_the_moments(dev, ny, nx, nz, dtype):
    print(f"case fused Adam {ny} x {nx} x {nz} {dtype}", flush=True)
    g = small_glacier(ny, nx, seed=nz)
    fields = {k: to_dev(g[k], dev, dtype) for k in ("thk", "usurf", "arrhenius", "slidingco", "dX")}
    op = EnergyOperator(dzeta_for(nz), E.DEFAULT_PHYSICS, fields=fields, dtype=dtype)
    U, V = (to_dev(a, dev, dtype) for a in smooth_velocity(nz, ny, nx, seed=nz))
    m0 = random_moments(nz, ny, nx, nz, dev).to(dtype)
    _, gU, gV = op.energy_grad(U, V)
    mom, Uo, Vo = m0.clone(), torch.full_like(U, float("nan")), torch.full_like(V, float("nan"))
    op.run_pass(2, U, V, Uo=Uo, Vo=Vo, moments=mom, adam=L.IgmAdam(alpha=0.5, beta1=0.9, beta2=0.999, epsilon=1e-7))
    one = torch.ones((), dtype=dtype)
    w1, w2 = float(one - torch.tensor(0.9, dtype=dtype)), float(one - torch.tensor(0.999, dtype=dtype))
    ulp = 2.0**-24 if dtype == torch.float32 else 2.0**-53
    for c, (x, gx, xo) in enumerate(((U, gU, Uo), (V, gV, Vo))):
        m, v, gd = m0[..., 2 * c].double(), m0[..., 2 * c + 1].double(), gx.double()
        mn, vn = mom[..., 2 * c].double(), mom[..., 2 * c + 1].double()
        assert bool(((mn - (m + (gd - m) * w1)).abs() <= 6 * ulp * (gd.abs() + m.abs())).all())
        assert bool(((vn - (v + (gd * gd - v) * w2)).abs() <= 6 * ulp * (gd * gd + v)).all())
        step = 0.5 * mn / (vn.sqrt() + 1e-7)
        assert bool(((xo.double() - (x.double() - step)).abs() <= ulp * (16 * step.abs() + 2 * x.double().abs())).all())
