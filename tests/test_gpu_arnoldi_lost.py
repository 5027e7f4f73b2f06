"""Steps that lose all of w, in one GMRES cycle on the device.  A periodic 2 x 2 grid has 12 unknowns
(4 of each velocity component, 4 pressures), so by step 13 at the latest w lies in the span of the
basis: what the first pass leaves is its rounding, within that span, and the step is repaired.  Steps
past 15 take the path that forms the norm.  The extra steps act on the rounding of a solution that
step 6 has to 1e-11: velocities and pressure differences stay within 1e-9 of the oracle's (the
tolerance times a condition of about 100).  In the left form the constant pressure, which the operator
does not see, grows out of the rounding of the extra steps; only the velocities are compared there."""
import numpy as np
import pytest

from lowmachfhd_amd.grid import Grid
from test_gpu_parity import _solver_mod, consistent_u, pair, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vt", [1, -1])
@pytest.mark.parametrize("steps", [13, 15, 16, 20, 28])
@pytest.mark.parametrize("flexible", [0, 1])
def test_exhausted_space(flexible, steps, vt):
    S = _solver_mod()
    g = Grid((2, 2), 1 / 2)
    rng = np.random.default_rng(6)
    kn = dict(gmres_rel_tol=1e-11, gmres_max_inner=30)
    o, s = pair(g, vt, 5.0, rng, **kn)
    s.close()
    bu = consistent_u(g, [rng.standard_normal(g.face_shape(a)) for a in range(g.dm)])
    bp = np.zeros(g.cc_shape())
    xu1, xp1, _, rc = o.gmres(bu, bp)
    assert rc == 0
    s = S.StokesSolver(g, visc_type=vt, krylov=S.FGMRES if flexible else S.GMRES_LEFT, gmres_min_iter=steps,
                       gmres_max_outer=1, **kn)
    s.set_coeffs(*o.coeffs)
    xu2, xp2, st = s.gmres(bu, bp)
    assert st.iters == steps
    est = np.array(list(st.resid_hist)[:steps])
    assert np.all(np.isfinite(est)) and np.all(est[1:] <= est[:-1])  # each rotation multiplies it by |sn| <= 1
    assert est[-1] <= 1e-16 * est[0]
    assert rel(xu2, xu1) < 1e-9
    if flexible:
        assert rel([xp2 - xp2.mean()], [xp1 - xp1.mean()]) < 1e-9
    s.close()
