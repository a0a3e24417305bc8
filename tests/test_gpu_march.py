"""The march of single waves (energy_pair_kernel), the two-iteration pass of
every grid that teams of four waves don't take: each number of levels it is
compiled for, each layout, absent moments and early stopping, with the checks
of test_gpu_pair, whose grids are the teams'.

Which kernel a grid takes is read from the workspace: 6 doubles per block of
the two-iteration pass, more than 3 per block of the one-iteration pass on
these grids; the teams would be fewer blocks.

IGM_PAIR_WAVES, which a process reads once, keeps small grids on the march too:
a child process with it set takes the grids of test_gpu_pair through it."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

from igm_amd import _lib as L
from igm_amd.solver import LegacyAdamState, solve
from tests.helpers import small_glacier
from tests.test_gpu_pair import CASES as SMALL
from tests.test_gpu_pair import first_mismatch, gpu_op
from tests.test_gpu_pair import test_pair_equals_two_single_passes as check_pair
from tests.test_gpu_pair import test_pair_interleaved_layouts as check_layouts
from tests.test_gpu_pair import test_pair_without_input_moments_is_a_fresh_optimizer as check_fresh

pytestmark = pytest.mark.gpu

NZ = [2, 3, 4, 5, 6, 8, 10, 12]
# blocks of the march: 5, 17, 2 and 1 strips in the most row blocks that run at once
BLOCKS = {(460, 300): 255, (136, 1000): 255, (1153, 120): 256, (2400, 60): 256}


def marches(ny, nx):
    assert L.load().igm_energy_workspace_doubles(1, ny, nx) == 6 * BLOCKS[ny, nx], "not the march's split"


@pytest.mark.parametrize("nz", NZ)
@pytest.mark.parametrize("ny,nx", BLOCKS)
def test_march_equals_two_single_passes(dev, ny, nx, nz):
    marches(ny, nx)
    check_pair(dev, ny, nx, nz)


@pytest.mark.parametrize("nz", NZ)
def test_march_in_every_layout_and_without_moments(dev, nz):
    ny, nx = [(460, 300), (136, 1000)][nz % 4 // 2]
    marches(ny, nx)
    check_layouts(dev, ny, nx, nz)
    check_fresh(dev, ny, nx, nz)


@pytest.mark.parametrize("nz,nit,patience,delta", [(10, 33, 0, 0.0), (10, 60, 1, 2e-2), (10, 60, 3, 2e-3), (5, 40, 2, 5e-3),
                                                   (12, 7, 10, 2e-4)])
def test_solve_on_the_march(dev, nz, nit, patience, delta):
    ny, nx = 460, 300
    marches(ny, nx)
    op = gpu_op(small_glacier(ny, nx, seed=nz), nz, dev)
    z = torch.zeros((nz, ny, nx), device=dev)
    kw = dict(early_stopping=patience > 0)
    if patience:
        kw |= dict(relative_min_delta=delta, patience=patience, check_every=4)
    r1 = solve(op, z, z.clone(), nit, LegacyAdamState(lr=1.0), pairs=False, **kw)
    r2 = solve(op, z, z.clone(), nit, LegacyAdamState(lr=1.0), pairs=True, **kw)
    assert (r2.iterations, r2.stopped) == (r1.iterations, r1.stopped)
    assert first_mismatch(r2.U, r1.U) is None and first_mismatch(r2.V, r1.V) is None
    c1, c2 = np.asarray(r1.costs), np.asarray(r2.costs)
    assert c1.shape == c2.shape and np.all(np.abs(c2 - c1) <= 1e-12 * np.abs(c1))


SMALL_GRIDS = """
import torch
from igm_amd import _lib as L
from tests import test_gpu_march as M
dev = torch.device("cuda:0")
# 100 x 100: 2 strips of 100 row blocks, 50 blocks; the teams take 200
assert L.load().igm_energy_workspace_doubles(1, 100, 100) == 6 * 50
for ny, nx, nz in M.SMALL:
    M.check_pair(dev, ny, nx, nz)
for ny, nx, nz in ((100, 100, 10), (37, 131, 5), (5, 7, 4), (61, 60, 12)):
    M.check_layouts(dev, ny, nx, nz)
    M.check_fresh(dev, ny, nx, nz)
"""


def test_small_grids_on_the_march(dev):
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    path = os.pathsep.join(p for p in (root, os.environ.get("PYTHONPATH")) if p)
    r = subprocess.run([sys.executable, "-c", SMALL_GRIDS], cwd=root, timeout=100, capture_output=True, text=True,
                       env=dict(os.environ, IGM_PAIR_WAVES="1024", PYTHONPATH=path))
    assert r.returncode == 0, r.stdout[-1000:] + r.stderr[-3000:]
