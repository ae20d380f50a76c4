"""Degree 4, whose workgroups take two tiles of 16 x 4 cells on grids of more tiles than CUs (256): odd tile
counts (the last workgroup has one), tiles cut on the right and above, the counts beside the rule's line,
single cells; against the CPU oracle."""
import pytest

from frhip import ics
from test_gpu_fr2d import RES_TOL, STATE_TOL, rel_inf, rel_l2, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,flux,bc", [(1, 1, "hll", "ghost"), (16, 4, "rusanov", "periodic"),
                                           (17, 4, "roe", "ghost"), (33, 3, "hll", "periodic"),
                                           (15, 9, "rusanov", "ghost"), (529, 2, "hll", "ghost"),
                                           (270, 65, "hll", "ghost"), (272, 68, "roe", "periodic"),
                                           (257, 61, "rusanov", "ghost"), (240, 68, "rusanov", "periodic"),
                                           (256, 64, "hll", "periodic")])
def test_two_tiles_per_workgroup(nx, ny, flux, bc):
    ps, u, s, orc = setup(nx, ny, 4, flux, bc, seed=nx + ny)
    assert rel_inf(s.rhs(u), orc.rhs(u)) <= RES_TOL
    dt, _ = ics.cfl_steps(u, 1.4, min(ps.dx0, 10.0 / ny), 0.05, 1.0)
    for scheme in ("ssprk3", "rk4"):
        s.set_state(u)
        s.step(dt, 2, scheme)
        uc = u.copy(order="F")
        getattr(orc, scheme)(uc, dt, 2)
        assert rel_l2(s.get_state(), uc) <= STATE_TOL
    s.close()
