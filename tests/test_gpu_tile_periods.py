"""Staggered tiles whose region ends on the last face of a periodic direction (n = 12, 22, 32 along z, y
and x in 3-D; 28 and 54 in 2-D), against the FP64 oracle as in test_gpu_tile_sweeps."""
import pytest

import test_gpu_tile_sweeps as T
from lowmachfhd_amd.grid import Grid

pytestmark = pytest.mark.gpu

GRIDS = {
    "z12": lambda: Grid((48, 48, 24), 1 / 48),
    "y22_x12": lambda: Grid((12, 22, 16), 1 / 16),
    "x32": lambda: Grid((32, 8, 12), 1 / 32),
    "2d_y28": lambda: Grid((112, 56), 1 / 112),
    "2d_y54": lambda: Grid((60, 54), 1 / 60),
}


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("vt", [-1, 1])
def test_regions_ending_on_a_period(gname, vt, monkeypatch):
    monkeypatch.setitem(T.GRIDS, gname, GRIDS[gname])
    T.test_stag_tiles(gname, vt, 1)
