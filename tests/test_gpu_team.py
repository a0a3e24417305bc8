"""The two forms of the two-iteration pass on either side of the line between
them: teams of four waves on grids of up to three steps, the march of single
waves on larger ones.  The checks are the pass's own: bits equal to two
one-iteration passes, and a solve's to one on single iterations, with and
without early stopping (test_gpu_pair)."""
import numpy as np
import pytest
import torch

from igm_amd.solver import LegacyAdamState, solve
from tests.helpers import small_glacier
from tests.test_gpu_pair import first_mismatch, gpu_op
from tests.test_gpu_pair import test_pair_equals_two_single_passes as check_pair

pytestmark = pytest.mark.gpu


# one strip: 256 blocks at once; two strips: 128; 17: 15.  Rows per team: 1, 2,
# 5, 6, 9; then the march
@pytest.mark.parametrize("ny,nx,nz", [(255, 60, 2), (258, 59, 3), (640, 61, 2), (641, 61, 3), (1152, 120, 2),
                                      (135, 1000, 3), (1153, 120, 2), (136, 1000, 3), (460, 300, 10), (2400, 60, 4)])
def test_pair_on_both_sides_of_the_line(dev, ny, nx, nz):
    check_pair(dev, ny, nx, nz)


@pytest.mark.parametrize("ny,nx", [(150, 70), (470, 300)])
@pytest.mark.parametrize("nit,patience,delta", [(5, 0, 0.0), (40, 2, 5e-3), (40, 1, 2e-2)])
def test_solve_on_both_sides_of_the_line(dev, ny, nx, nit, patience, delta):
    op = gpu_op(small_glacier(ny, nx, seed=5), 4, dev)
    z = torch.zeros((4, ny, nx), device=dev)
    kw = dict(early_stopping=patience > 0)
    if patience:
        kw |= dict(relative_min_delta=delta, patience=patience, check_every=4)
    r1 = solve(op, z, z.clone(), nit, LegacyAdamState(lr=1.0), pairs=False, **kw)
    r2 = solve(op, z, z.clone(), nit, LegacyAdamState(lr=1.0), pairs=True, **kw)
    assert (r2.iterations, r2.stopped) == (r1.iterations, r1.stopped)
    assert first_mismatch(r2.U, r1.U) is None and first_mismatch(r2.V, r1.V) is None
    c1, c2 = np.asarray(r1.costs), np.asarray(r2.costs)
    assert c1.shape == c2.shape and np.all(np.abs(c2 - c1) <= 1e-12 * np.abs(c1))
