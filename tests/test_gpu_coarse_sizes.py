"""The coarse V-cycles' one-workgroup kernels over the sizes where their rule turns: levels that fill
one, two or more slots of a thread, sizes that are no power of two, odd levels (two-phase colour
steps), walls, 2-D, and workgroups too small to hold a level in registers -- against the FP64
oracle.  Tolerances: FP64 sums of the same terms in the same order differ from the oracle's by
its own order of evaluation only (1e-12, as for the split levels); the mixed form runs the
multigrid in FP32 (2e-6)."""
import numpy as np
import pytest

from lowmachfhd_amd.grid import NO_SLIP_WALL, PERIODIC, SLIP_WALL, Grid
from test_gpu_parity import _solver_mod, consistent_u, pair, rel

pytestmark = pytest.mark.gpu

GRIDS = {
    "bottom_10x6x7": lambda: Grid((40, 24, 28), 1 / 40),
    "from_12": lambda: Grid((24, 24, 24), 1 / 24, bc_lo=(PERIODIC, PERIODIC, NO_SLIP_WALL),
                            bc_hi=(PERIODIC, PERIODIC, NO_SLIP_WALL)),
    "from_8": lambda: Grid((16, 16, 16), 1 / 16),
    "bottom_9x5x3": lambda: Grid((36, 20, 12), 1 / 36, bc_lo=(NO_SLIP_WALL, SLIP_WALL, PERIODIC),
                                 bc_hi=(SLIP_WALL, NO_SLIP_WALL, PERIODIC)),
    "2d_from_48": lambda: Grid((96, 48), 1 / 96),
    "2d_from_32": lambda: Grid((64, 64), 1 / 64, bc_lo=(PERIODIC, NO_SLIP_WALL), bc_hi=(PERIODIC, SLIP_WALL)),
}


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("vt", [-1, 1, -2, 3])
@pytest.mark.parametrize("nt", [1024, 256])
def test_coarse_sizes(gname, vt, nt):
    S = _solver_mod()
    g = GRIDS[gname]()
    rng = np.random.default_rng(11)
    forms = (dict(precision=S.FP64, krylov=S.GMRES_LEFT), dict(precision=S.MIXED, krylov=S.FGMRES))
    for kn in forms:
        S.set_tune(g, {"coarse_threads": nt}, visc_type=vt, **kn)
    try:
        o, s = pair(g, vt, 5.0, rng)
        bu = consistent_u(g, [rng.standard_normal(g.face_shape(a)) for a in range(g.dm)])
        bp = rng.standard_normal(g.cc_shape())
        bp -= bp.mean()
        ref_u, (ref_pu, ref_pp) = o.stag_mg_solve(bu), o.apply_precon(bu, bp)
        for kn, tol in zip(forms, (1e-12, 2e-6)):
            if kn["precision"] == S.MIXED:
                s = S.StokesSolver(g, visc_type=vt, **kn)
                s.set_coeffs(*o.coeffs)
            assert s.tune["coarse_threads"] == nt
            assert rel(s.stag_mg_solver(bu), ref_u) < tol
            xu, xp = s.apply_precon(bu, bp)
            assert rel(xu, ref_pu) < 10 * tol and rel([xp], [ref_pp]) < 10 * tol  # a quotient of h^2 on top
            s.close()
    finally:
        for kn in forms:
            S.set_tune(g, {"coarse_threads": 1024}, visc_type=vt, **kn)
