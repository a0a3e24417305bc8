"""Infinities and NaN in layer 1's weight gradient, which sums the parts of a
split float32 input: every entry is finite, infinite (with its sign) or NaN as
the plain float32 sum of its products is."""
import math
import struct

import pytest
import torch

from igm_amd import _lib as L

pytestmark = pytest.mark.gpu


def wgrad(X, dz, nblocks, dev):
    _, H, W, _ = X.shape
    Xd, zd = X.to(dev), dz.to(torch.bfloat16).to(dev)
    ws = torch.empty(L.load().igm_wgrad_workspace_floats(0, nblocks), device=dev)
    dW, db = torch.empty((9, 5, 32), device=dev), torch.empty(32, device=dev)
    L.call("igm_conv_in_wgrad", *[Xd.data_ptr() + 4 * i for i in range(5)], H * W * 5, W * 5, 5, None, 1, H, W, L.ptr(zd),
           nblocks, L.ptr(ws), 0, L.ptr(dW), L.ptr(db), L.stream_ptr())
    return dW.cpu(), db.cpu()


def reference(X, dz):
    """The products of every tap, summed (float64 keeps what is infinite and NaN, and the finite sums)."""
    H, W = X.shape[1:3]
    xp = torch.nn.functional.pad(X[0].double(), (0, 0, 1, 1, 1, 1))
    z = dz[0].to(torch.bfloat16).double()
    return torch.stack([(xp[t // 3:t // 3 + H, t % 3:t % 3 + W, :, None] * z[:, :, None, :]).sum((0, 1)) for t in range(9)])


def same_kind(a, b):
    return (torch.equal(torch.isnan(a), torch.isnan(b)) and torch.equal(torch.isposinf(a), torch.isposinf(b))
            and torch.equal(torch.isneginf(a), torch.isneginf(b)))


@pytest.mark.parametrize("nblocks", [1, 7])
def test_infinite_gradients(dev, nblocks):
    """Inputs of one, two and three bf16 parts, negative ones and a zero, under
    gradients that are infinite at one pixel, infinite with both signs at two,
    and NaN; one channel is finite.  (13 rows and 45 columns: ragged strips.)"""
    gen = torch.Generator().manual_seed(3)
    X = torch.rand((1, 13, 45, 5), generator=gen) + 0.5
    X[..., 0] = 2.0                                    # one part
    X[..., 1] = 1.0 + 2.0**-9                          # two
    X[..., 2] = -(1.0 + 2.0**-9 + 2.0**-20)            # three
    X[..., 4] = torch.where(X[..., 4] > 1.0, 3000.0, -0.75)
    X[0, 6, 20, 3] = 0.0
    dz = torch.randn((1, 13, 45, 32), generator=gen)
    inf = float("inf")
    dz[0, 6, 20, 1], dz[0, 6, 20, 2] = inf, -inf
    dz[0, 6, 20, 3], dz[0, 8, 33, 3] = inf, -inf
    dz[0, 4, 31, 4], dz[0, 4, 32, 5] = inf, inf        # on either side of a strip's edge
    dz[0, 9, 9, 6] = float("nan")
    dW, db = wgrad(X, dz, nblocks, dev)
    ref = reference(X, dz)
    assert same_kind(dW, ref), [(int(i), float(dW.view(-1)[i]), float(ref.view(-1)[i]))
                                for i in (~torch.isclose(dW.double(), ref, equal_nan=True)).view(-1).nonzero()[:5]]
    assert same_kind(db, dz[0].sum((0, 1)))
    # chains of at most 13 * 45 float32 sums: 585 * 2^-24 * sum |x dz| at the very worst
    fin = torch.isfinite(ref)
    mag = reference(X.abs(), dz.abs())
    assert bool(((dW - ref).abs()[fin] <= 585 * 2.0**-24 * mag[fin]).all())


@pytest.mark.parametrize("bits", [0x7FC00000, 0x7F800001, 0xFF80FFFF])
def test_nan_inputs(dev, bits):
    """A NaN, quiet or signalling, whichever of its bits are set."""
    X, dz = torch.ones((1, 8, 40, 5)), torch.ones((1, 8, 40, 32))
    raw = X.view(torch.int32)
    raw[0, 3, 33, 2] = struct.unpack("<i", struct.pack("<I", bits))[0]
    assert math.isnan(float(X[0, 3, 33, 2]))
    dW, db = wgrad(X, dz, 3, dev)
    assert bool(torch.isnan(dW[:, 2]).all()) and bool(torch.isfinite(dW[:, [0, 1, 3, 4]]).all())
    assert bool(torch.isfinite(db).all())
