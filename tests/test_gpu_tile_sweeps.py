"""The sweeps of a multigrid level in one launch (tiles) against the FP64 oracle where the tiles'
shapes turn: levels of one tile and of several whose last is cut, levels smaller than the layers
around a tile (their periodic images appear several times in it), walls, 2-D, a second V-cycle
(which starts from values, not from its first half sweep) and the level sizes on both sides of the
rule.  The one-workgroup coarse kernel is kept to levels of extents up to 4, so that tiles run below
it.  FP64: sums of the same terms in the same order, 1e-12; FP32: 6e-8 a rounding, some 40 sweeps of
it and an inverse Laplacian of rough data (condition about 1 relative to its own norm): 2e-5."""
import numpy as np
import pytest

from lowmachfhd_amd.grid import NO_SLIP_WALL, PERIODIC, SLIP_WALL, Grid
from test_gpu_parity import _solver_mod, consistent_u, pair, rel

pytestmark = pytest.mark.gpu

W, Q, P = NO_SLIP_WALL, SLIP_WALL, PERIODIC
GRIDS = {
    "one_and_a_cut_tile": lambda: Grid((20, 12, 8), 1 / 20),
    "small": lambda: Grid((8, 8, 8), 1 / 8),
    "walls": lambda: Grid((28, 20, 24), 1 / 28, bc_lo=(W, Q, P), bc_hi=(Q, W, P)),
    "all_walls": lambda: Grid((16, 24, 12), 1 / 24, bc_lo=(W, W, Q), bc_hi=(W, Q, W)),
    "most_tiles": lambda: Grid((32, 32, 32), 1 / 32),
    "one_too_many": lambda: Grid((32, 32, 34), 1 / 32, bc_lo=(P, P, W), bc_hi=(P, P, W)),
    "odd_below": lambda: Grid((20, 12, 14), 1 / 20, bc_lo=(P, W, P), bc_hi=(P, W, P)),
    "2d": lambda: Grid((120, 60), 1 / 120),
    "2d_walls": lambda: Grid((72, 100), 1 / 72, bc_lo=(P, W), bc_hi=(P, Q)),
}


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("cycles", [1, 2])
def test_mac_tiles(gname, cycles):
    S = _solver_mod()
    g = GRIDS[gname]()
    rng = np.random.default_rng(31)
    small = {"coarse_n": 4, "mac_coarse_n": 4}
    forms = (dict(precision=S.FP64, krylov=S.GMRES_LEFT), dict(precision=S.MIXED, krylov=S.FGMRES))
    default = [S.get_tune(g, visc_type=-1, **kn) for kn in forms]
    try:
        for kn in forms:
            S.set_tune(g, small, visc_type=-1, **kn)
        o, s = pair(g, -1, 5.0, rng, mg_max_vcycles=cycles)
        bp = rng.standard_normal(g.cc_shape())
        bp -= bp.mean()
        ref = o.mac_mg_solve(bp)
        for kn, tol in zip(forms, (1e-12, 2e-5)):
            if kn["precision"] == S.MIXED:
                s = S.StokesSolver(g, visc_type=-1, mg_max_vcycles=cycles, **kn)
                s.set_coeffs(*o.coeffs)
            assert s.tune["mac_coarse_n"] == 4
            assert rel([s.mac_mg_solver(bp)], [ref]) < tol
            s.close()
    finally:
        for kn, d in zip(forms, default):
            S.set_tune(g, {k: d[k] for k in small}, visc_type=-1, **kn)


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("vt", [-1, 1])
@pytest.mark.parametrize("cycles", [1, 2])
def test_stag_tiles(gname, vt, cycles):
    S = _solver_mod()
    g = GRIDS[gname]()
    rng = np.random.default_rng(32)
    small = {"coarse_n": 4, "mac_coarse_n": 4}
    forms = (dict(precision=S.FP64, krylov=S.GMRES_LEFT), dict(precision=S.MIXED, krylov=S.FGMRES))
    default = [S.get_tune(g, visc_type=vt, **kn) for kn in forms]
    more = dict(stag_mg_max_vcycles=cycles, stag_mg_rel_tol=0.0)
    try:
        for kn in forms:
            S.set_tune(g, small, visc_type=vt, **kn)
        o, s = pair(g, vt, 5.0, rng, **more)
        bu = consistent_u(g, [rng.standard_normal(g.face_shape(a)) for a in range(g.dm)])
        ref = o.stag_mg_solve(bu)
        for kn, tol in zip(forms, (1e-12, 2e-5)):
            if kn["precision"] == S.MIXED:
                s = S.StokesSolver(g, visc_type=vt, **more, **kn)
                s.set_coeffs(*o.coeffs)
            assert s.tune["coarse_n"] == 4
            assert rel(s.stag_mg_solver(bu), ref) < tol
            s.close()
    finally:
        for kn, d in zip(forms, default):
            S.set_tune(g, {k: d[k] for k in small}, visc_type=vt, **kn)
