"""The power -1/3 of the float64 passes, value by value, against 50 digits.

A 2 x 2 field with one uniform velocity u has one cell with the sliding energy
csl N N^e, N = u^2 + r (a flat bed) and nothing else; with slidingco = s, csl =
s (1/s) is one.  u has 26 bits, so u^2 is exact; r is the smallest double, which
the half-speed cells around the field, of weight zero, need: 0 x 0^(-1/3) is NaN.
The energy is N t with one rounding, t the power as computed: within 2^-53 of N t.
A t that is the nearest double to N^e is within 2^-53 of it, so 2 x 2^-53 in
all; 2.1 are asked.  (pow, for comparison, may be further off.)"""
import decimal
import random
from fractions import Fraction

import pytest
import torch

from igm_amd.energy import EnergyOperator
from oracle import energy as E

pytestmark = pytest.mark.gpu

S = 1.0 + 1.0 / 3.0
REGU = 2.0**-537  # its square is the smallest double


def speeds():
    """26-bit numbers whose squares cover the doubles, subnormal ones too (with
    as many bits as those have), and the ends of every binade of the cube root's
    period."""
    r = random.Random(11)
    out = [(r.getrandbits(25) + 2**25) * 2.0**(r.randint(-505, 505) - 26) for _ in range(1500)]
    out += [(r.getrandbits(25) + 2**25) * 2.0**(r.randint(-17, 6) - 26) for _ in range(1500)]  # N of 1e-10 .. 1e3
    out += [m * 2.0**k for k in range(-536, -512) for m in (1.0, 1.25, 1.5, 1.75)]
    for k in (-33, -32, -31, -2, -1, 0, 1, 2, 3, 4, 40, 41, 42):
        out += [2.0**k, 2.0**k * (1 + 2.0**-25), 2.0**k * (1 - 2.0**-26), 2.0**k * (1 - 2.0**-25), 2.0**k * 1.4142135,
                2.0**k * 1.41421354]
    return [float(torch.tensor(u, dtype=torch.float64)) for u in out]


def test_power_minus_one_third(dev):
    us = speeds()
    assert S * (1.0 / S) == 1.0
    us = [u for u in us if Fraction(u) ** 2 == Fraction(u * u)]
    assert len(us) > 3100
    X = torch.tensor([0.0, 1000.0, 100.0, S, 100.0], dtype=torch.float64, device=dev).expand(len(us), 2, 2, 5).contiguous()
    op = EnergyOperator([1.0], dict(E.DEFAULT_PHYSICS, regu_weertman=REGU), X=X, dtype=torch.float64)
    U = torch.tensor(us, dtype=torch.float64, device=dev)[:, None, None, None].expand(-1, 2, 2, 2).contiguous()
    e = op.energy(U, torch.zeros_like(U)).cpu()
    assert bool((e[:, 0] == 0).all()) and bool((e[:, 2] == 0).all()) and torch.equal(e[:, 1], e[:, 3])
    worst = decimal.Decimal(0)
    with decimal.localcontext(decimal.Context(prec=50, Emin=-999999, Emax=999999)):
        x = decimal.Decimal(S / 2.0 - 1.0)
        for u, got in zip(us, e[:, 1].tolist()):
            N = decimal.Decimal(u * u + REGU * REGU)
            ref = N * (x * N.ln()).exp()
            err = abs(decimal.Decimal(got) / ref - 1) * 2**53
            worst = max(worst, err)
            assert err <= decimal.Decimal("2.1"), (u, got, float(err))
    print(f"largest error of N^(2/3): {float(worst):.3f} x 2^-53")


def test_power_of_zero_is_infinite(dev):
    """0^(-1/3) is infinite, as pow's: without regularisation a cell at rest has the sliding energy 0 x inf."""
    X = torch.tensor([0.0, 1000.0, 100.0, S, 100.0], dtype=torch.float64, device=dev).expand(1, 2, 2, 5).contiguous()
    for m in (3.0, 3.0 + 1e-9):  # the short power, pow
        op = EnergyOperator([1.0], dict(E.DEFAULT_PHYSICS, regu_weertman=0.0, exp_weertman=m), X=X, dtype=torch.float64)
        z = torch.zeros((1, 2, 2, 2), dtype=torch.float64, device=dev)
        assert bool(torch.isnan(op.energy(z, z)[0, 1]))
