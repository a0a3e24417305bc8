"""The energy's coefficients at the edges of their 63-cell strips and row
blocks, in every layout, and the powers of the float64 passes.

Tolerances: a coefficient is a handful of roundings away from the float64
formula, 4e-6 of its size in float32 (1e-13 in float64); slopes are
differences of elevations of up to 4000 m over 100 m, whose roundings are
2^-24 * 4000 / 100 = 2.4e-6 (4e-6 and 1e-13 are asked of an elevation over
100 m).  The float64 passes are held to the oracle as elsewhere, 1e-11."""
import ctypes as C

import numpy as np
import pytest
import torch

from igm_amd import _lib as L
from igm_amd.energy import EnergyOperator
from oracle import energy as E
from tests.helpers import dzeta_for, rel, small_glacier, smooth_velocity, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("layout", ["planar", "nhwc"])
@pytest.mark.parametrize("B,H,W,ext", [(1, 2, 2, None), (1, 3, 63, None), (1, 2, 64, None), (1, 7, 65, None),
                                       (1, 5, 127, None), (1, 700, 500, None),
                                       (3, 66, 130, [(66, 130), (40, 64), (2, 2)])])
def test_coefficients_against_float64(dev, B, H, W, ext, layout, dtype):
    gen = torch.Generator().manual_seed(H * W)
    X = torch.rand((B, H, W, 5), generator=gen, dtype=torch.float64)
    X = (X * torch.tensor([800.0, 3000.0, 100.0, 0.05, 1.0]) + torch.tensor([-200.0, 500.0, 20.0, -0.01, 99.5])).to(dtype)
    X[..., 0].clamp_(min=0.0)
    Xd = X.to(dev)
    if layout == "nhwc":
        fs, strides = [Xd[..., i] for i in range(5)], (H * W * 5, W * 5, 5)
    else:
        fs, strides = [Xd[..., i].contiguous() for i in range(5)], (H * W, W, 1)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    ph = L.IgmPhysics(exp_glen=3.0, exp_weertman=3.0, thr_ice_thk=0.1, ice_density=910.0, gravity_cst=9.81,
                      min_sr=1e-20, max_sr=1e20, regu_glen=1e-5, regu_weertman=1e-10)
    coef = torch.full((B, 7, H, W), float("nan"), dtype=dtype, device=dev)
    hs = torch.empty(B, dtype=dtype, device=dev)
    L.call("igm_energy_coeffs_f32" if dtype == torch.float32 else "igm_energy_coeffs_f64", *[L.ptr(f) for f in fs],
           *strides, L.ptr(e), B, H, W, C.addressof(ph), L.ptr(coef), L.ptr(hs), L.stream_ptr())
    got, eps = coef.cpu().double(), 4e-6 if dtype == torch.float32 else 1e-13
    for b in range(B):
        ny, nx = (H, W) if ext is None else ext[b]
        t, s, A, c, d = X[b, :ny, :nx].double().unbind(-1)
        st4 = lambda a: (a[1:, 1:] + a[1:, :-1] + a[:-1, 1:] + a[:-1, :-1]) / 4
        avg = lambda a, dim: (a.narrow(dim, 1, a.shape[dim] - 1) + a.narrow(dim, 0, a.shape[dim] - 1)) / 2
        def slope(a, dim):
            n = a.shape[dim] - 1
            return avg((a.narrow(dim, 1, n) - a.narrow(dim, 0, n)) / avg(d, dim), 1 - dim)
        Hh, Bs, Cs, S = st4(t), st4(2 * A ** (-1 / 3)), st4(c), (ny - 1) * (nx - 1)
        g = 0.25 * 910.0 * 9.81e-6 * Hh / S
        damp = (Cs > 0).double() * 0.99 + 0.01
        q = float(d[0, 0]) * damp / Hh.clamp(min=0.1)
        one, steep = torch.zeros_like(q), torch.full_like(q, 40.0)
        ref = [(q, one), (Hh * Bs / (4 / 3 * S), one), (g * slope(s, 1), g * steep), (g * slope(s, 0), g * steep),
               (Cs / (4 / 3 * S), one + 0.05 / S), (slope(s - t, 1), steep), (slope(s - t, 0), steep)]
        sure = Cs.abs() > 1e-8  # (the sign of the mean sliding coefficient picks the damping)
        for p, (r, scale) in enumerate(ref):
            d_ = (got[b, p, :ny - 1, :nx - 1] - r).abs()
            assert bool((d_ <= eps * (r.abs() + scale))[sure if p == 0 else slice(None)].all()), (b, p, float(d_.max()))
        rest = got[b].clone()
        rest[:, :ny - 1, :nx - 1] = 0
        assert not bool(rest.any())
        assert float(hs[b]) == pytest.approx(1 / (4 * float(d[0, 0])), rel=eps)


@pytest.mark.parametrize("n,m", [(3.0, 3.0), (3.0, 4.0), (4.0, 3.0)])
def test_float64_powers_against_the_oracle(dev, n, m):
    """Both exponents -1/3 take the short power, any other pair pow."""
    nz, ny, nx = 5, 40, 125
    g = small_glacier(ny, nx, seed=3)
    U, V = smooth_velocity(nz, ny, nx, seed=4)
    phys = dict(E.DEFAULT_PHYSICS, exp_glen=n, exp_weertman=m)
    fin = E.fieldin_tensors(g["thk"], g["usurf"], g["arrhenius"], g["slidingco"], g["dX"], torch.float64)
    c, _, gU, gV = E.energy_and_grad(torch.as_tensor(U), torch.as_tensor(V), fin, torch.as_tensor(dzeta_for(nz)), phys)
    fields = {k: to_dev(g[k], dev, torch.float64) for k in ("thk", "usurf", "arrhenius", "slidingco", "dX")}
    op = EnergyOperator(dzeta_for(nz), phys, fields=fields, dtype=torch.float64)
    e, hU, hV = op.energy_grad(to_dev(U, dev, torch.float64), to_dev(V, dev, torch.float64))
    assert abs(float(e[0, 3]) - float(c)) <= 1e-11 * abs(float(c))
    assert rel(torch.stack([hU.cpu(), hV.cpu()]), torch.stack([gU, gV])) <= 1e-11
