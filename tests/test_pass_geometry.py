"""The row split of the energy passes (host code only), read from the
workspace size: 3 doubles per block of the one-iteration passes, 6 per block
of the two-iteration pass, the larger of both.  A pass runs in one round: at
most 512 blocks of the one-iteration passes and 256 of the two-iteration
pass, except where one row block per strip needs more.  Small grids run the
two-iteration pass in teams, one block per strip and 1, 5 or 9 rows (team)."""
import pytest

from igm_amd import _lib as L


def blocks(strips, rows):
    return (strips * rows + 3) // 4


# (batch, ny, nx, row blocks of a strip: one iteration, two iterations)
CASES = [
    (1, 500, 500, 113, 113),    # 9 strips: 113 row blocks are 1017 waves, 114 would be 257 blocks of two-iteration passes
    (1, 757, 1203, 102, 48),    # 20 and 21 strips
    (1, 1500, 1500, 81, 40),    # 25 strips of either: 2025 and 1000 waves
    (1, 100, 100, 100, "team 100"),    # one row per wave; one per team
    (1, 2, 2, 2, "team 2"),
    (1, 257, 61, 257, "team 52"),      # 1 and 2 strips; 128 blocks of 3 rows would take two steps, as 52 of 5 do
    (1, 256, 300, 204, "team 29"),     # short waves: 1024 of them, not 2048; 51 blocks of 6: three steps, as 29 of 9
    (1, 307, 300, 204, "team 35"),     # 5 strips: 51 blocks of 7 rows
    (1, 460, 300, 204, 204),           # 51 of 10 rows: four steps
    (3, 150, 260, 68, "team 30"),      # a batch: 15 strips
    (2100, 64, 62, 1, "team 64"),      # more entries than blocks of a round: one row block each
]


@pytest.mark.parametrize("batch,ny,nx,one,two", CASES)
def test_one_round(batch, ny, nx, one, two):
    n1, n2 = (nx + 61) // 62, (nx + 59) // 60
    pair = n2 * int(two.split()[1]) if isinstance(two, str) else blocks(n2, two)
    want = max(3 * batch * blocks(n1, one), 6 * pair)
    assert L.load().igm_energy_workspace_doubles(batch, ny, nx) == want
    assert pair <= 256
    if batch * blocks(n1, 1) <= 512:
        assert batch * blocks(n1, one) <= 512
