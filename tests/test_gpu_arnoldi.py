"""The Arnoldi step's sweeps where they can go wrong: vectors of odd length (their last element has
no pair), short cycles, cycles past the 15 vectors the fused sweeps take, and a step that loses
all of w (the norm is then formed instead of taken by Pythagoras).  GMRES is run against the
oracle's modified Gram-Schmidt: the same iterations, solutions that agree to 1e-9 at a tolerance
of 1e-11 (the residual each leaves, times a condition of about 100)."""
import numpy as np
import pytest

from lowmachfhd_amd.grid import NO_SLIP_WALL, PERIODIC, Grid
from test_gpu_parity import _solver_mod, consistent_u, pair, rel

pytestmark = pytest.mark.gpu

GRIDS = {
    "odd_length": lambda: Grid((7, 5, 3), 1 / 7),
    "odd_length_walls": lambda: Grid((14, 7, 9), 1 / 14, bc_lo=(PERIODIC, PERIODIC, NO_SLIP_WALL),
                                     bc_hi=(PERIODIC, PERIODIC, NO_SLIP_WALL)),
    "2d": lambda: Grid((10, 9), 1 / 10),
    "even_length": lambda: Grid((16, 12, 8), 1 / 16),
}


def _rhs(g, rng):
    return consistent_u(g, [rng.standard_normal(g.face_shape(a)) for a in range(g.dm)]), np.zeros(g.cc_shape())


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("m", [3, 15, 16, 40])
@pytest.mark.parametrize("flexible", [0, 1])
def test_gmres_cycles(gname, m, flexible):
    S = _solver_mod()
    g = GRIDS[gname]()
    rng = np.random.default_rng(5)
    kn = dict(gmres_rel_tol=1e-11, gmres_max_inner=m, gmres_max_outer=40, gmres_max_iter=120)
    o, s = pair(g, -1, 5.0, rng, **kn)
    bu, bp = _rhs(g, rng)
    xu1, xp1, st1, rc = o.gmres(bu, bp)
    assert rc == 0
    if flexible:
        s.close()
        s = S.StokesSolver(g, visc_type=-1, krylov=S.FGMRES, **kn)
        s.set_coeffs(*o.coeffs)
    xu2, xp2, st2 = s.gmres(bu, bp)
    assert st2.converged == 1
    if not flexible:
        assert abs(st2.iters - st1.total_iter) <= 1
    assert rel(xu2, xu1) < 1e-9 and rel(xp2, xp1) < 1e-9
    s.close()


@pytest.mark.parametrize("flexible", [0, 1])
def test_step_that_loses_w(flexible):
    """Twelve more steps than the tolerance needs: the residual estimate falls to rounding and w lies
    in the span of the basis.  Further steps cannot raise the residual that the tolerance's steps
    left, except to its rounding floor."""
    S = _solver_mod()
    g = Grid((4, 4, 4), 1 / 4)
    rng = np.random.default_rng(6)
    kn = dict(visc_type=1, krylov=S.FGMRES if flexible else S.GMRES_LEFT, gmres_rel_tol=1e-11, gmres_max_inner=30)
    o, s = pair(g, 1, 5.0, rng, gmres_rel_tol=1e-11, gmres_max_inner=30)
    bu, bp = _rhs(g, rng)
    s.close()
    s = S.StokesSolver(g, **kn)
    s.set_coeffs(*o.coeffs)
    xu, xp, st1 = s.gmres(bu, bp)
    r1 = st1.true_rel_resid
    s.close()
    s = S.StokesSolver(g, gmres_min_iter=st1.iters + 12, gmres_max_outer=2, **kn)
    s.set_coeffs(*o.coeffs)
    xu, xp, st2 = s.gmres(bu, bp)
    print(f"flexible={flexible}: {st1.iters} then {st2.iters} steps, residual {r1:.2e} then {st2.true_rel_resid:.2e}")
    assert st2.iters > st1.iters
    assert np.isfinite(st2.true_rel_resid) and st2.true_rel_resid <= max(r1, 1e-13)
    s.close()
