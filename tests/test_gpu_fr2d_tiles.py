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


# 17 x 17 = 289 tiles, an odd number above 256: workgroups of two tiles, the last with one
@pytest.mark.parametrize("cells", ["parallelogram", "polar"])
@pytest.mark.parametrize("flux,bc", [("hll", "ghost"), ("rusanov", "periodic"), ("roe", "ghost")])
def test_two_tiles_per_workgroup_on_general_cells(cells, flux, bc):
    import frhip
    from oracle import oracle as O
    from test_gpu_fr2d import _sheared_geometry
    from test_oracle_metrics import G, oracle_for, polar_space, smooth_state

    nx, ny, deg = 270, 65, 4
    if cells == "polar":
        ps = polar_space(nx, ny, deg)
        u = smooth_state(ps, seed=3)
        s, orc = frhip.FREuler2D(ps, G, flux, bc), oracle_for(ps, flux, bc)
    else:
        ps, u, s, _ = setup(nx, ny, deg, flux, bc, seed=3)
        dx, dy, iJ, n1, n2 = _sheared_geometry(nx, ny)
        s.set_geometry(iJ)
        orc = O.Fr2d(nx, ny, deg, dx, dy, 1.4, flux, bc, iJ=iJ, n1=n1, n2=n2)
    assert rel_inf(s.rhs(u), orc.rhs(u)) <= RES_TOL
    for scheme in ("ssprk3", "rk4"):  # RK4 on polar cells keeps one tile
        s.set_state(u)
        s.step(1e-5, 2, scheme)
        uc = u.copy(order="F")
        getattr(orc, scheme)(uc, 1e-5, 2)
        assert rel_l2(s.get_state(), uc) <= STATE_TOL
    s.close()
