"""The 3x3 layers' kernels of large batches, whose outputs are stored cached
(above 80 MB) or non-temporally (from 120 MB): the one-pass backward and the
last layer with the output layer.  Their products are the single launches', in
the same order: equal bits.  (The single launches are held to float64 at such
sizes in test_gpu_conv3x3.)"""
import pytest
import torch

from igm_amd import _lib as L
from tests.test_gpu_conv3x3 import case

pytestmark = pytest.mark.gpu

# cached; non-temporal; the sizes on either side of both lines (80 and 120 MiB)
SIZES = [(1, 1201, 1250, None), (8, 512, 490, [(512 - 60 * i, 490 - 55 * i) for i in range(8)]), (1, 1280, 1024, None),
         (1, 1281, 1024, None), (1, 1920, 1023, None), (1, 1920, 1024, None)]


@pytest.mark.parametrize("B,H,W,ext", SIZES)
def test_backward_in_one_pass_of_large_batches(dev, B, H, W, ext):
    print(f"case backward {B} x {H} x {W}", flush=True)
    act, (w, _), _ = case(B, H, W, dev)
    dz = torch.randn((B, H, W, 32), generator=torch.Generator(dev).manual_seed(H), device=dev).to(torch.bfloat16)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    n, st = L.load().igm_wgrad_workspace_floats(9, 256), L.stream_ptr()
    p1, p2 = (torch.full((n,), float("nan"), device=dev) for _ in range(2))
    o1, o2 = (torch.full_like(act, float("nan")) for _ in range(2))
    L.call("igm_conv_wgrad_partials_bf16", 9, L.ptr(act), L.ptr(dz), L.ptr(e), B, H, W, 256, L.ptr(p1), 0, st)
    L.call("igm_conv3x3_dgrad_bf16", L.ptr(dz), L.ptr(w), L.ptr(act), L.ptr(e), B, H, W, L.ptr(o1), st)
    L.call("igm_conv3x3_bwd_bf16", L.ptr(act), L.ptr(dz), L.ptr(w), L.ptr(e), B, H, W, 256, L.ptr(p2), 0, L.ptr(o2), st)
    assert torch.equal(o1, o2) and torch.equal(p1, p2)


@pytest.mark.parametrize("cout", [20, 7])
@pytest.mark.parametrize("B,H,W,ext", SIZES[:4])
def test_last_layer_of_large_batches(dev, B, H, W, ext, cout):
    print(f"case last layer {B} x {H} x {W}", flush=True)
    x, (w, w2), (b, b2) = case(B, H, W, dev)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    head, hb, st = w2[0].contiguous(), b2[:cout].contiguous(), L.stream_ptr()
    Ys = [torch.full((B, H, W, cout), float("nan"), device=dev) for _ in range(3)]
    a, a2 = (torch.full_like(x, float("nan")) for _ in range(2))
    L.call("igm_conv3x3_fwd_bf16", L.ptr(x), L.ptr(w), L.ptr(b), L.ptr(e), B, H, W, L.ptr(a), st)
    L.call("igm_conv1x1_head_fwd", L.ptr(a), L.ptr(head), L.ptr(hb), L.ptr(e), B, H, W, cout, L.ptr(Ys[0]), st)
    for out, Y in ((a2, Ys[1]), (None, Ys[2])):
        L.call("igm_conv3x3_head_fwd_bf16", L.ptr(x), L.ptr(w), L.ptr(b), L.ptr(head), L.ptr(hb), L.ptr(e), B, H, W,
               cout, L.ptr(out), L.ptr(Y), st)
    assert torch.equal(a, a2) and torch.equal(Ys[0], Ys[1]) and torch.equal(Ys[0], Ys[2])
