"""How the 3x3 layers' backward kernel splits the rows of a batch over its waves
(StripShare): every row of every entry once, whatever the extents and the number
of blocks.  Weight gradient and data gradient against float64, with the
tolerances of test_gpu_conv3x3.py: an element of the data gradient to half a
bf16 step and the rounding of 288 products; the weight gradient's chains are at
most 2,000 links here (one block), which as a random walk is 2.7e-6 of its norm
(1e-5 are asked)."""
import pytest
import torch

from igm_amd import _lib as L
from tests.test_gpu_conv3x3 import case, check, conv64, masked

pytestmark = pytest.mark.gpu


def uneven(B, H, W):
    """Extents of B entries, every fourth empty in one or both directions."""
    return [(0 if b % 4 == 1 else 1 + (7 * b) % H, 0 if b % 8 > 4 else 1 + (13 * b) % W) for b in range(B)]


# entries past the 64 of a wave's lanes, the first and the last ones empty; all
# empty; ranges that run over many strips and entries (one block) and units
# fewer than waves; no extents with strips that the waves don't divide evenly
@pytest.mark.parametrize("nblocks", [1, 3, 256])
@pytest.mark.parametrize("B,H,W,ext", [(1, 9, 70, [(9, 70)]), (3, 8, 40, [(0, 40), (5, 0), (0, 0)]),
                                       (64, 6, 65, uneven(64, 6, 65)), (131, 13, 67, [(0, 9)] + uneven(129, 13, 67) + [(7, 0)]),
                                       (6, 61, 190, [(61, 1), (1, 190), (60, 33), (4, 64), (5, 65), (61, 190)]),
                                       (3, 21, 160, None), (1, 130, 96, None)])
def test_split_rows_of_a_batch(dev, B, H, W, ext, nblocks):
    print(f"case split {B} x {H} x {W}, {nblocks} blocks", flush=True)
    act, (w, _), _ = case(B, H, W, dev)
    dz = torch.randn((B, H, W, 32), generator=torch.Generator().manual_seed(H)).to(torch.bfloat16).to(dev)
    e = None if ext is None else torch.tensor(ext, dtype=torch.int32, device=dev)
    P = torch.full((L.load().igm_wgrad_workspace_floats(9, nblocks),), float("nan"), device=dev)
    below = torch.full_like(act, float("nan"))
    dW, db = torch.empty((3, 3, 32, 32), device=dev), torch.empty(32, device=dev)
    L.call("igm_conv3x3_bwd_bf16", L.ptr(act), L.ptr(dz), L.ptr(w), L.ptr(e), B, H, W, nblocks, L.ptr(P), 0, L.ptr(below),
           L.stream_ptr())
    L.call("igm_conv_wgrad_reduce_f32", 9, 32, nblocks, L.ptr(P), 0, L.ptr(dW), L.ptr(db), L.stream_ptr())
    torch.cuda.synchronize()
    am, zm = masked(act, ext), masked(dz, ext)
    check(below, masked(conv64(zm, w) * torch.where(am.float() > 0, 1.0, 0.01), ext))
    xp = torch.nn.functional.pad(am.double(), (0, 0, 1, 1, 1, 1))
    z = zm.double().reshape(-1, 32)
    for t in range(9):
        ref = xp[:, t // 3:t // 3 + H, t % 3:t % 3 + W].reshape(-1, 32).t().contiguous() @ z
        d = torch.linalg.vector_norm(dW[t // 3, t % 3].double() - ref)
        assert float(d) <= 1e-5 * max(float(torch.linalg.vector_norm(ref)), 1.0), (t, float(d))
    assert float((db.double() - z.sum(0)).norm()) <= 1e-5 * max(float(z.sum(0).norm()), 1.0)
