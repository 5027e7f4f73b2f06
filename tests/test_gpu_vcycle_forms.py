"""The V-cycles' launch forms against the FP64 oracle where their rules turn: sweep counts of zero and
one (the first step from zero, the half residual and the prolongation inside a sweep each need
a sweep to belong to), omega other than 1 (no half residual), levels of odd size, walls of both
kinds (a face beside one reads its own reflection) and several V-cycles.  Sums of the same terms:
1e-12 for the V-cycle, ten times that for the preconditioner (a quotient of h^2 on top)."""
import numpy as np
import pytest

from lowmachfhd_amd.grid import NO_SLIP_WALL, PERIODIC, SLIP_WALL, Grid
from test_gpu_parity import consistent_u, pair, rel

pytestmark = pytest.mark.gpu

W, Q, P = NO_SLIP_WALL, SLIP_WALL, PERIODIC
GRIDS = {
    "periodic": lambda: Grid((32, 32, 32), 1 / 32),
    "walls_odd_levels": lambda: Grid((36, 20, 44), 1 / 44, bc_lo=(W, Q, W), bc_hi=(Q, W, W)),
    "long_rows": lambda: Grid((72, 32, 34), 1 / 72, bc_lo=(P, P, Q), bc_hi=(P, P, W)),
    "2d_walls": lambda: Grid((128, 72), 1 / 128, bc_lo=(P, W), bc_hi=(P, Q)),
}
KNOBS = {
    "default": {},
    "no_down": dict(stag_mg_nsmooths_down=0, mg_nsmooths_down=0),
    "no_up": dict(stag_mg_nsmooths_up=0, mg_nsmooths_up=0),
    "one_each": dict(stag_mg_nsmooths_down=1, stag_mg_nsmooths_up=1, mg_nsmooths_down=1, mg_nsmooths_up=1),
    "omega": dict(stag_mg_omega=0.9),
    "two_cycles": dict(stag_mg_max_vcycles=2, mg_max_vcycles=2, stag_mg_rel_tol=0.0),
}


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("vt", [-1, 1])
@pytest.mark.parametrize("kname", list(KNOBS))
def test_vcycle_forms(gname, vt, kname):
    g = GRIDS[gname]()
    rng = np.random.default_rng(21)
    o, s = pair(g, vt, 5.0, rng, **KNOBS[kname])
    bu = consistent_u(g, [rng.standard_normal(g.face_shape(a)) for a in range(g.dm)])
    bp = rng.standard_normal(g.cc_shape())
    bp -= bp.mean()
    assert rel(s.stag_mg_solver(bu), o.stag_mg_solve(bu)) < 1e-12
    xu, xp = s.apply_precon(bu, bp)
    ru, rp = o.apply_precon(bu, bp)
    assert rel(xu, ru) < 1e-11 and rel([xp], [rp]) < 1e-11
    s.close()
