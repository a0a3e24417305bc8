"""The 3x3 layer kernels (igm_conv3x3_fwd_bf16, igm_conv3x3_dgrad_bf16,
igm_conv3x3_pair_fwd_bf16) element by element against float64 sums of the
same bf16 operands, at the edges of their 62- and 64-column strips and row
blocks, on padded batches, and where two blocks share a compute unit.

Tolerance of an element: half a bf16 step of the result, 2^-9 |ref| (2^-8 is
asked), and the float32 accumulation of 288 products, at most 288 * 2^-24 *
sum |w x| ~ 288 * 6e-8 * 14 = 2.4e-4 (3e-4).  Two layers in one launch run
the same instructions as two launches: equal bits."""
import pytest
import torch

from igm_amd import _lib as L

pytestmark = pytest.mark.gpu

# (B, H, W, extents): one pixel, strips of 62 and 64 columns and one more,
# 1 to 8 rows, batches with uneven and empty entries, and grids of more than
# 1024 waves (blocks of at most 32 rows: 8 x 600 x 700) and of long waves
CASES = [(1, 1, 1, None), (1, 2, 62, None), (1, 3, 63, None), (1, 4, 64, None), (1, 5, 65, None), (1, 7, 125, None),
         (1, 8, 129, None), (1, 131, 124, None), (3, 37, 131, [(37, 131), (20, 64), (1, 1)]),
         (2, 65, 70, [(65, 5), (33, 70)]), (8, 600, 700, [(600 - 61 * i, 700 - 83 * i) for i in range(8)]),
         (1, 1100, 1300, None)]


def case(B, H, W, dev):
    g = torch.Generator().manual_seed(B + 7 * H + W)
    x = torch.randn((B, H, W, 32), generator=g).to(torch.bfloat16).to(dev)
    ws = [(torch.randn((9, 32, 32), generator=g) * 0.06).to(torch.bfloat16).to(dev) for _ in range(2)]
    bs = [(torch.randn(32, generator=g) * 0.1).to(dev) for _ in range(2)]
    return x, ws, bs


def conv64(x, w):
    """"Same" correlation, float64: w [tap][out][in]."""
    B, H, W, C = x.shape
    xp = torch.nn.functional.pad(x.double(), (0, 0, 1, 1, 1, 1))
    out = torch.zeros((B, H, W, C), dtype=torch.float64, device=x.device)
    for t in range(9):
        r, s = t // 3, t % 3
        out += (xp[:, r:r + H, s:s + W].reshape(-1, C) @ w[t].double().t().contiguous()).view(B, H, W, C)
    return out


def masked(x, ext):
    """x with zeros outside each entry's extent."""
    if ext is None:
        return x
    y = torch.zeros_like(x)
    for b, (ny, nx) in enumerate(ext):
        y[b, :ny, :nx] = x[b, :ny, :nx]
    return y


def check(out, ref):
    d = (out.double() - ref).abs() - (2.0 ** -8 * ref.abs() + 3e-4)
    assert bool(torch.isfinite(out.float()).all())
    assert float(d.max()) <= 0, (float(d.max()), int((d > 0).sum()))


@pytest.mark.parametrize("B,H,W,ext", CASES)
def test_layers_against_float64(dev, B, H, W, ext):
    print(f"case conv3x3 {B} x {H} x {W}", flush=True)
    x, (w1, w2), (b1, b2) = case(B, H, W, dev)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    st = L.stream_ptr()
    one, two, both, dg = (torch.full_like(x, float("nan")) for _ in range(4))
    L.call("igm_conv3x3_fwd_bf16", L.ptr(x), L.ptr(w1), L.ptr(b1), L.ptr(e), B, H, W, L.ptr(one), st)
    L.call("igm_conv3x3_fwd_bf16", L.ptr(one), L.ptr(w2), L.ptr(b2), L.ptr(e), B, H, W, L.ptr(two), st)
    L.call("igm_conv3x3_pair_fwd_bf16", L.ptr(x), L.ptr(w1), L.ptr(b1), L.ptr(w2), L.ptr(b2), L.ptr(e), B, H, W,
           L.ptr(both), st)
    L.call("igm_conv3x3_dgrad_bf16", L.ptr(x), L.ptr(w1), L.ptr(two), L.ptr(e), B, H, W, L.ptr(dg), st)
    torch.cuda.synchronize()
    xm = masked(x, ext)
    z = conv64(xm, w1)
    check(one, masked(torch.nn.functional.leaky_relu(z + b1.double(), 0.01), ext))
    check(dg, masked(z * torch.where(two.float() > 0, 1.0, 0.01), ext))
    assert torch.equal(both.view(torch.int16), two.view(torch.int16))


def test_network_forward_equals_layer_by_layer(dev):
    """CNN.forward in launches of two layers gives the bits of the pass that
    keeps every activation, for even and odd counts of 3x3 layers."""
    from igm_amd import emulator as EM
    for nl in (1, 2, 3, 4, 5):
        cnn = EM.CNN(nz=5, nb_layers=nl, device=dev, seed=nl)
        X = torch.randn((2, 33, 71, 5), generator=torch.Generator().manual_seed(nl)).to(dev)
        fields = EM.nhwc_fields(X)
        Y, acts = cnn.forward(fields, keep=True)
        assert len(acts) == nl
        assert torch.equal(cnn.forward(fields), Y)


@pytest.mark.parametrize("nblocks,accumulate", [(1, 0), (3, 1), (256, 0), (512, 1)])
@pytest.mark.parametrize("B,H,W,ext", [(1, 1, 1, None), (1, 5, 33, None), (2, 13, 64, [(13, 31), (7, 64)]),
                                       (3, 66, 70, [(65, 70), (66, 5), (1, 1)]), (1, 300, 257, None)])
def test_weight_gradient_against_float64(dev, B, H, W, ext, nblocks, accumulate):
    """igm_conv_wgrad_bf16 for any number of partial-sum rows, fewer and more
    than there is work for.  Tolerance: products of 32 pixels are added in
    float32 chains of at most 77,100 / 32 / 4 = 600 links (one block of four
    waves); if every rounding went the same way, 600 * 2^-24 = 3.6e-5 of the
    terms' size, as a random walk 1.5e-6: 1e-5 of the result's norm."""
    x, (w, z2), (b, _) = case(B, H, W, dev)
    dz = torch.randn((B, H, W, 32), generator=torch.Generator().manual_seed(H)).to(torch.bfloat16).to(dev)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    ws = torch.full((L.load().igm_wgrad_workspace_floats(9, nblocks),), float("nan"), device=dev)
    dW, db = torch.ones((3, 3, 32, 32), device=dev), torch.ones(32, device=dev)
    L.call("igm_conv_wgrad_bf16", 9, L.ptr(x), L.ptr(dz), L.ptr(e), B, H, W, 32, nblocks, L.ptr(ws), accumulate,
           L.ptr(dW), L.ptr(db), L.stream_ptr())
    torch.cuda.synchronize()
    xp = torch.nn.functional.pad(masked(x, ext).double(), (0, 0, 1, 1, 1, 1))
    zm = masked(dz, ext).double().reshape(-1, 32)
    for t in range(9):
        ref = xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(-1, 32).t().contiguous() @ zm + accumulate
        d = torch.linalg.vector_norm(dW[t // 3, t % 3].double() - ref)
        assert float(d) <= 1e-5 * max(float(torch.linalg.vector_norm(ref)), 1.0), (t, float(d))
    ref = zm.sum(0) + accumulate
    assert float(torch.linalg.vector_norm(db.double() - ref)) <= 1e-5 * max(float(torch.linalg.vector_norm(ref)), 1.0)


@pytest.mark.parametrize("nblocks,accumulate", [(1, 0), (3, 1), (512, 0)])
@pytest.mark.parametrize("layout", ["planar", "nhwc", "transposed"])
@pytest.mark.parametrize("B,H,W,ext", [(1, 1, 1, None), (2, 13, 64, [(13, 31), (7, 64)]),
                                       (3, 66, 70, [(65, 70), (66, 5), (1, 1)]), (1, 300, 257, None)])
def test_layer1_weight_gradient_against_float64(dev, B, H, W, ext, layout, nblocks, accumulate):
    """igm_conv_in_wgrad on raw magnitudes for every layout of the fields; the
    tolerance is the 3x3 layers' (the same chains), per field."""
    gen = torch.Generator().manual_seed(H * W)
    scale = torch.tensor([800.0, 3000.0, 100.0, 0.05, 100.0])
    X = (torch.rand((B, H, W, 5), generator=gen) * scale).to(dev)
    dz = torch.randn((B, H, W, 32), generator=gen).to(torch.bfloat16).to(dev)
    if layout == "nhwc":
        fs, strides = [X[..., i] for i in range(5)], (H * W * 5, W * 5, 5)
    elif layout == "planar":
        fs, strides = [X[..., i].contiguous() for i in range(5)], (H * W, W, 1)
    else:
        fs, strides = [X[..., i].transpose(1, 2).contiguous() for i in range(5)], (H * W, 1, H)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    ws = torch.full((L.load().igm_wgrad_workspace_floats(0, nblocks),), float("nan"), device=dev)
    dW, db = torch.ones((3, 3, 5, 32), device=dev), torch.ones(32, device=dev)
    L.call("igm_conv_in_wgrad", *[L.ptr(f) for f in fs], *strides, L.ptr(e), B, H, W, L.ptr(dz), nblocks, L.ptr(ws),
           accumulate, L.ptr(dW), L.ptr(db), L.stream_ptr())
    torch.cuda.synchronize()
    xp = torch.nn.functional.pad(masked(X, ext).double(), (0, 0, 1, 1, 1, 1))
    zm = masked(dz, ext).double().reshape(-1, 32)
    ref = torch.stack([xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(-1, 5).t().contiguous() @ zm for t in range(9)])
    d = (dW.reshape(9, 5, 32).double() - ref - accumulate).transpose(0, 1).reshape(5, -1)
    n = ref.transpose(0, 1).reshape(5, -1)
    assert (d.norm(dim=1) <= 1e-5 * n.norm(dim=1).clamp(min=1.0)).all(), d.norm(dim=1) / n.norm(dim=1)
    rb = zm.sum(0) + accumulate
    assert float((db.double() - rb).norm()) <= 1e-5 * max(float(rb.norm()), 1.0)


def test_layer1_weight_gradient_of_an_infinite_input(dev):
    """An infinity or NaN among the inputs reaches the entries it multiplies,
    as a float32 product would carry it, and no others."""
    X = torch.ones((1, 8, 8, 5), device=dev)
    X[0, 4, 4, 1], X[0, 2, 6, 3] = float("inf"), float("nan")
    dz = torch.ones((1, 8, 8, 32), dtype=torch.bfloat16, device=dev)
    ws = torch.empty(L.load().igm_wgrad_workspace_floats(0, 4), device=dev)
    dW, db = torch.empty((3, 3, 5, 32), device=dev), torch.empty(32, device=dev)
    L.call("igm_conv_in_wgrad", *[X.data_ptr() + 4 * i for i in range(5)], 320, 40, 5, None, 1, 8, 8, L.ptr(dz), 4,
           L.ptr(ws), 0, L.ptr(dW), L.ptr(db), L.stream_ptr())
    assert torch.isposinf(dW[:, :, 1]).all() and torch.isnan(dW[:, :, 3]).all()
    assert torch.isfinite(dW[:, :, [0, 2, 4]]).all() and torch.isfinite(db).all()


@pytest.mark.parametrize("layout", ["planar", "nhwc", "transposed"])
@pytest.mark.parametrize("B,H,W,ext", [(1, 1, 1, None), (1, 2, 63, None), (1, 5, 64, None), (1, 3, 65, None),
                                       (3, 66, 70, [(65, 70), (66, 5), (1, 1)]), (2, 300, 130, [(300, 128), (7, 64)]),
                                       (1, 700, 600, None)])
def test_layer1_against_float64(dev, B, H, W, ext, layout):
    """igm_conv_in_fwd element by element: half a bf16 step of the result, and
    the float32 rounding of a chain of 45 FMAs, at most 46 * 2^-24 * (|b| + sum
    |w x|) (2^-8 and 3e-6 of it are asked); zeros outside the extents."""
    gen = torch.Generator().manual_seed(H * W)
    X = (torch.rand((B, H, W, 5), generator=gen) * torch.tensor([800.0, 3000.0, 100.0, 0.05, 100.0])).to(dev)
    w, b = torch.randn((9, 5, 32), generator=gen).to(dev), torch.randn(32, generator=gen).to(dev)
    if layout == "nhwc":
        fs, strides = [X[..., i] for i in range(5)], (H * W * 5, W * 5, 5)
    elif layout == "planar":
        fs, strides = [X[..., i].contiguous() for i in range(5)], (H * W, W, 1)
    else:
        fs, strides = [X[..., i].transpose(1, 2).contiguous() for i in range(5)], (H * W, 1, H)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    out = torch.full((B, H, W, 32), float("nan"), dtype=torch.bfloat16, device=dev)
    L.call("igm_conv_in_fwd", *[L.ptr(f) for f in fs], *strides, L.ptr(e), B, H, W, L.ptr(w), L.ptr(b), L.ptr(out),
           L.stream_ptr())
    torch.cuda.synchronize()
    xp = torch.nn.functional.pad(masked(X, ext).double(), (0, 0, 1, 1, 1, 1))
    ref = b.double().expand(B, H, W, 32).clone()
    mag = ref.abs()
    for t in range(9):
        part = xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(-1, 5)
        ref += (part @ w[t].double()).view(B, H, W, 32)
        mag += (part.abs() @ w[t].double().abs()).view(B, H, W, 32)
    ref = masked(torch.where(ref > 0, ref, 0.01 * ref), ext)
    assert ((out.double() - ref).abs() <= 2.0**-8 * ref.abs() + masked(3e-6 * mag, ext)).all()


def test_layer1_of_an_infinite_input(dev):
    """An infinity reaches the 3x3 pixels around it and no others."""
    X = torch.ones((1, 9, 80, 5), device=dev)
    X[0, 4, 70, 1] = float("inf")
    w, b = torch.ones((9, 5, 32), device=dev), torch.zeros(32, device=dev)
    out = torch.zeros((1, 9, 80, 32), dtype=torch.bfloat16, device=dev)
    L.call("igm_conv_in_fwd", *[X.data_ptr() + 4 * i for i in range(5)], 3600, 400, 5, None, 1, 9, 80, L.ptr(w),
           L.ptr(b), L.ptr(out), L.stream_ptr())
    near = torch.zeros((9, 80), dtype=torch.bool, device=dev)
    near[3:6, 69:72] = True
    assert torch.isposinf(out[0, near]).all() and torch.isfinite(out[0, ~near]).all()


@pytest.mark.parametrize("nblocks,accumulate", [(1, 0), (3, 1), (256, 0), (300, 1)])
@pytest.mark.parametrize("B,H,W,ext", [(1, 1, 1, None), (1, 5, 33, None), (1, 64, 32, None),
                                       (2, 13, 64, [(13, 31), (7, 64)]), (3, 66, 70, [(65, 70), (66, 5), (1, 1)]),
                                       (1, 300, 257, None), (2, 700, 600, [(700, 600), (31, 599)])])
def test_backward_in_one_pass_equals_two(dev, B, H, W, ext, nblocks, accumulate):
    """igm_conv3x3_bwd_bf16 runs the products of igm_conv_wgrad_partials_bf16
    and igm_conv3x3_dgrad_bf16 in their order: equal bits."""
    act, (w, _), _ = case(B, H, W, dev)
    dz = torch.randn((B, H, W, 32), generator=torch.Generator().manual_seed(H)).to(torch.bfloat16).to(dev)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    n, st = L.load().igm_wgrad_workspace_floats(9, nblocks), L.stream_ptr()
    p1, p2 = torch.ones(n, device=dev), torch.ones(n, device=dev)
    o1, o2 = torch.full_like(act, float("nan")), torch.full_like(act, float("nan"))
    L.call("igm_conv_wgrad_partials_bf16", 9, L.ptr(act), L.ptr(dz), L.ptr(e), B, H, W, nblocks, L.ptr(p1), accumulate,
           st)
    L.call("igm_conv3x3_dgrad_bf16", L.ptr(dz), L.ptr(w), L.ptr(act), L.ptr(e), B, H, W, L.ptr(o1), st)
    L.call("igm_conv3x3_bwd_bf16", L.ptr(act), L.ptr(dz), L.ptr(w), L.ptr(e), B, H, W, nblocks, L.ptr(p2), accumulate,
           L.ptr(o2), st)
    assert torch.equal(o1, o2) and torch.equal(p1, p2)


@pytest.mark.parametrize("rows,n3x3,cout", [((1, 1, 1), 1, 2), ((3, 8, 5), 2, 20), ((33, 32, 31), 3, 32),
                                            ((512, 256, 100), 1, 6), ((7, 9, 4), 0, 20)])
def test_reduction_of_all_layers(dev, rows, n3x3, cout):
    """igm_wgrad_reduce_layers_f32 against the layers' own reductions: two
    orders of at most 512 float32 sums, each within 512 * 2^-24 * sum |p| at
    worst, together 6.2e-5 of it (2e-6 are asked: 23 roundings' random walk
    with room); rows of zeros after the last change no bit."""
    lib, st = L.load(), L.stream_ptr()
    kinds = [0] + [9] * n3x3 + [1]
    nr = {0: rows[0], 9: rows[1], 1: rows[2]}
    gen = torch.Generator().manual_seed(7)
    parts = [torch.randn(lib.igm_wgrad_workspace_floats(t, nr[t]), generator=gen).to(dev) for t in kinds]
    shapes = []
    for i, t in enumerate(kinds):
        co = cout if t == 1 else 32
        shapes += [(max(t, 1) if t else 9) * (5 if t == 0 else 32) * co, co]
    offs = torch.tensor([0] + list(torch.tensor(shapes).cumsum(0)), dtype=torch.int64, device=dev)
    def reduce(extra):
        ps = [torch.cat([p, torch.zeros(lib.igm_wgrad_workspace_floats(t, extra), device=dev)])
              for p, t in zip(parts, kinds)]
        mid = torch.cat(ps[1:-1]) if n3x3 else None
        g = torch.ones(int(offs[-1]), device=dev)
        L.call("igm_wgrad_reduce_layers_f32", n3x3, cout, nr[0] + extra, nr[9] + extra, nr[1] + extra, L.ptr(ps[0]),
               L.ptr(mid), L.ptr(ps[-1]), 1, L.ptr(offs), L.ptr(g), st)
        return g
    g = reduce(0)
    assert torch.equal(g, reduce(5))
    for i, t in enumerate(kinds):
        k, b = [torch.empty(shapes[2 * i + j], device=dev) for j in range(2)]
        ka, ba = torch.empty_like(k), torch.empty_like(b)
        for src, dk, db in ((parts[i].clone(), k, b), (parts[i].abs(), ka, ba)):
            L.call("igm_conv_wgrad_reduce_f32", t, cout if t == 1 else 32, nr[t], L.ptr(src), 0, L.ptr(dk), L.ptr(db), st)
        o = [int(v) for v in offs[2 * i:2 * i + 3]]
        assert ((g[o[0]:o[1]] - 1 - k).abs() <= 2e-6 * (ka + 1)).all()
        assert ((g[o[1]:o[2]] - 1 - b).abs() <= 2e-6 * (ba + 1)).all()


@pytest.mark.parametrize("cout,shift", [(20, 0), (32, 0), (2, 0), (7, 0), (20, 1)])
@pytest.mark.parametrize("B,H,W,ext", [(1, 1, 1, None), (1, 5, 65, None), (2, 13, 64, [(13, 31), (7, 64)]),
                                       (3, 66, 130, [(65, 130), (66, 5), (1, 1)]), (1, 300, 257, None)])
def test_last_layer_with_the_output_layer(dev, B, H, W, ext, cout, shift):
    """igm_conv3x3_head_fwd_bf16 runs the products of the two layers' launches:
    equal bits, with Y on and off 16 bytes, with and without the activations."""
    x, (w, w2), (b, b2) = case(B, H, W, dev)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    head, hb = w2[0].contiguous(), torch.cat([b2, b2])[:cout].contiguous()
    st, n = L.stream_ptr(), B * H * W * cout
    Ys = [torch.full((n + 1,), float("nan"), device=dev)[shift:shift + n] for _ in range(3)]
    a, a2 = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    L.call("igm_conv3x3_fwd_bf16", L.ptr(x), L.ptr(w), L.ptr(b), L.ptr(e), B, H, W, L.ptr(a), st)
    L.call("igm_conv1x1_head_fwd", L.ptr(a), L.ptr(head), L.ptr(hb), L.ptr(e), B, H, W, cout, L.ptr(Ys[0]), st)
    for out, Y in ((a2, Ys[1]), (None, Ys[2])):
        L.call("igm_conv3x3_head_fwd_bf16", L.ptr(x), L.ptr(w), L.ptr(b), L.ptr(head), L.ptr(hb), L.ptr(e), B, H, W,
               cout, L.ptr(out), L.ptr(Y), st)
    assert torch.equal(a, a2) and torch.equal(Ys[0], Ys[1]) and torch.equal(Ys[0], Ys[2])


@pytest.mark.parametrize("nl", [1, 2, 3, 4])
def test_network_passes_equal_their_launches(dev, nl):
    """igm_cnn_fwd and igm_cnn_bwd make the launches of every layer in order:
    the bits of the calls made one by one, for odd and even numbers of layers."""
    from igm_amd import emulator as EM
    B, H, W, nz = 2, 21, 70, 3
    gen = torch.Generator().manual_seed(nl)
    X = torch.rand((B, H, W, 5), generator=gen).to(dev)
    ext = torch.tensor([[21, 70], [9, 33]], dtype=torch.int32, device=dev)
    cnn, fields, st = EM.CNN(nz, nl, seed=3), EM.nhwc_fields(X), L.stream_ptr()
    fp, (fb, fr, fc) = fields[0], fields[1]
    Y, acts = cnn.forward(fields, extents=ext, keep=True)
    ref = [torch.empty((B, H, W, 32), dtype=torch.bfloat16, device=dev) for _ in range(nl)]
    L.call("igm_conv_in_fwd", *fp, fb, fr, fc, L.ptr(ext), B, H, W, L.ptr(cnn.kernel(0)), L.ptr(cnn.bias(0)),
           L.ptr(ref[0]), st)
    for i in range(1, nl):
        L.call("igm_conv3x3_fwd_bf16", L.ptr(ref[i - 1]), L.ptr(cnn.fwd[i - 1]), L.ptr(cnn.bias(i)), L.ptr(ext), B, H,
               W, L.ptr(ref[i]), st)
    Yr = torch.empty_like(Y)
    L.call("igm_conv1x1_head_fwd", L.ptr(ref[-1]), L.ptr(cnn.head), L.ptr(cnn.bias(nl)), L.ptr(ext), B, H, W, 2 * nz,
           L.ptr(Yr), st)
    assert torch.equal(Y, Yr) and torch.equal(cnn.forward(fields, extents=ext), Yr)
    assert all(torch.equal(a, r) for a, r in zip(acts, ref))

    dY, gX, g = torch.randn(Y.shape, generator=gen).to(dev), torch.empty_like(X), torch.empty_like(X)
    got = cnn.backward(dY, acts, fields, extents=ext, input_grad=gX, nblocks=8).clone()
    dz, below = torch.empty_like(ref[0]), torch.empty_like(ref[0])
    kinds = [0] + [9] * (nl - 1) + [1]
    parts = [torch.empty(L.load().igm_wgrad_workspace_floats(t, 8), device=dev) for t in kinds]
    L.call("igm_conv1x1_head_bwd", L.ptr(dY), L.ptr(ref[-1]), L.ptr(cnn.kernel(nl)), L.ptr(ext), B, H, W, 2 * nz,
           L.ptr(dz), L.ptr(below), st)
    L.call("igm_conv_wgrad_partials_bf16", 1, L.ptr(ref[-1]), L.ptr(below), L.ptr(ext), B, H, W, 8, L.ptr(parts[nl]), 0,
           st)
    for i in range(nl - 1, 0, -1):
        L.call("igm_conv3x3_bwd_bf16", L.ptr(ref[i - 1]), L.ptr(dz), L.ptr(cnn.dgr[i - 1]), L.ptr(ext), B, H, W, 8,
               L.ptr(parts[i]), 0, L.ptr(below), st)
        dz, below = below, dz
    L.call("igm_conv_in_wgrad_partials", *fp, fb, fr, fc, L.ptr(ext), B, H, W, L.ptr(dz), 8, L.ptr(parts[0]), 0, st)
    L.call("igm_conv_in_dgrad", L.ptr(dz), L.ptr(cnn.kernel(0)), L.ptr(ext), B, H, W, L.ptr(g), st)
    mid = torch.cat(parts[1:nl]) if nl > 1 else None
    out = torch.empty_like(cnn.g)
    L.call("igm_wgrad_reduce_layers_f32", nl - 1, 2 * nz, 8, 8, 8, L.ptr(parts[0]), L.ptr(mid), L.ptr(parts[nl]), 0,
           L.ptr(cnn.offs), L.ptr(out), st)
    assert torch.equal(got, out) and torch.equal(gX, g)
