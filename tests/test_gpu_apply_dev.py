"""lmfhd_apply_matrix_dev on the caller's vectors as they are: wall faces of x count as zero whatever
they hold and stay untouched, x and b may be the same vector, and odd sizes, 2-D and cross terms
give the oracle's result (sums of the same terms: 1e-13)."""
import numpy as np
import pytest

from lowmachfhd_amd.grid import NO_SLIP_WALL, PERIODIC, SLIP_WALL, Grid
from test_gpu_parity import pair, rel

pytestmark = pytest.mark.gpu

W, Q, P = NO_SLIP_WALL, SLIP_WALL, PERIODIC
GRIDS = {
    "odd_periodic": lambda: Grid((9, 7, 5), 1 / 9),
    "walls": lambda: Grid((17, 12, 10), 1 / 17, bc_lo=(W, Q, W), bc_hi=(Q, W, W)),
    "row_over_256": lambda: Grid((260, 3, 4), 1 / 260, bc_lo=(P, P, W), bc_hi=(P, P, W)),
    "2d_walls": lambda: Grid((31, 18), 1 / 31, bc_lo=(W, P), bc_hi=(W, P)),
}


@pytest.mark.parametrize("gname", list(GRIDS))
@pytest.mark.parametrize("vt", [-1, -3, 2])
@pytest.mark.parametrize("in_place", [0, 1])
def test_apply_matrix_dev(gname, vt, in_place):
    import torch

    g = GRIDS[gname]()
    rng = np.random.default_rng(8)
    o, s = pair(g, vt, 5.0, rng)
    u = [rng.standard_normal(g.face_shape(a)) for a in range(g.dm)]  # walls hold values too
    p = rng.standard_normal(g.cc_shape())
    ref_u, ref_p = o.apply_matrix(u, p)
    x0 = torch.from_numpy(s.pack(u, p)).to("cuda:0")
    x = x0.clone()
    b = x if in_place else torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    s.apply_matrix_dev(x.data_ptr(), b.data_ptr())
    s.sync()
    bu, bp = s.unpack(b.cpu().numpy())
    assert rel(bu, ref_u) < 1e-13 and rel([bp], [ref_p]) < 1e-13
    if not in_place:
        assert torch.equal(x, x0)
    s.close()
