"""Register-resident 1D stepping at the edges of its chunks, and the sensor's comparison against the
cut of the switch."""
import numpy as np
import pytest

import frhip

pytestmark = pytest.mark.gpu


def state(ncell, deg, eq, seed):
    ps = frhip.FRPSpace1D(0.0, 1.0, ncell, deg)
    rng = np.random.default_rng(seed)
    x = ps.xpg + 0.0
    if eq == "advection":
        return ps, np.asfortranarray(np.sin(2 * np.pi * x) + 0.01 * rng.uniform(-1, 1, x.shape))
    rho = 1 + 0.2 * np.sin(2 * np.pi * x) + 0.01 * rng.uniform(-1, 1, x.shape)
    u, p = 0.3 * np.cos(2 * np.pi * x), 1 + 0.1 * np.sin(4 * np.pi * x)
    return ps, np.asfortranarray(np.stack([rho, rho * u, p / 0.4 + 0.5 * rho * u * u], -1))


# one chunk (up to 256 cells), the first size with halos, chunk lengths of 160 cells and one off
@pytest.mark.parametrize("ncell", [2, 3, 63, 64, 65, 255, 256, 257, 319, 320, 321, 1000])
@pytest.mark.parametrize("scheme,nsteps", [("ssprk3", 33), ("rk4", 25), ("midpoint", 1), ("euler", 97)])
@pytest.mark.parametrize("eq,bc", [("euler", "period"), ("euler", "dirichlet"), ("advection", "period")])
def test_chunks_equal_a_launch_per_stage(ncell, scheme, nsteps, eq, bc):
    ps, u0 = state(ncell, 2, eq, ncell)
    out = []
    for path in ("batched", "auto"):
        g = frhip.FREulerProblem(ps, 1.4, bc, "hll") if eq == "euler" else frhip.FRAdvectionProblem(ps, 1.0, bc)
        g.set_path(path)
        g.set_state(u0)
        g.step(0.02 / ncell, nsteps, scheme)
        out.append(g.get_state())
        g.close()
    assert np.all(np.isfinite(out[0]))
    assert np.array_equal(*out)


@pytest.mark.parametrize("limit", [False, True])
@pytest.mark.parametrize("nsteps", [1, 2, 9])
def test_many_chunks_equal_a_launch_per_stage(nsteps, limit):
    """More than 256 chunks of 160 cells: the chunks of 232 cells with 12 halo cells."""
    ncell = np.array([2048, 232, 233, 256, 257, 464, 465, 64] * 24)
    deg = np.array([2, 3, 4, 1] * 48)
    members = [state(int(n), int(d), "euler", b)[1] for b, (n, d) in enumerate(zip(ncell, deg))]
    out = []
    for path, graph in (("batched", False), ("auto", False), ("auto", True)):
        e = frhip.Ensemble1D(ncell, deg, 1.0 / ncell, 1.4, "rusanov", "period")
        e.set_path(path)
        e.set_state(e.pack(members))
        run = e.run_graph if graph else e.run
        if graph:
            e.run_graph(1e-5, nsteps, 0, filter=True, limit=limit)
        counts = run(1e-5, nsteps, filter=True, limit=limit)
        out.append((counts, e.get_state()))
        e.close()
    assert out[0][0] == out[1][0] == out[2][0] and out[0][0][0] > 0
    assert np.all(np.isfinite(out[0][1]))
    assert np.array_equal(out[0][1], out[1][1]) and np.array_equal(out[0][1], out[2][1])


@pytest.mark.parametrize("deg", [2, 3, 5, 7])
def test_sensor_flags_by_the_cut(deg):
    """Cells whose top mode lies a relative 1e-11 ... 1e-3 of the energy ratio above or below the cut
    of the switch (sigma = 0.99: Se = S0 - kappa (2 / pi) asin 0.98): flagged above, not below.  The
    nodal values carry the ratio to about 1e-13 (1e-16 over a top mode of 1e-3 of the mean)."""
    cut = 10.0 ** (-3 * np.log10(deg) - 4.0 * 2 / np.pi * np.arcsin(0.98))
    delta = np.geomspace(1e-11, 1e-3, 400)
    r, _ = np.polynomial.legendre.leggauss(deg + 1)
    V = np.polynomial.legendre.legvander(r, deg) * np.sqrt((2 * np.arange(deg + 1) + 1) / 2)
    for sign in (1.0, -1.0):
        q = cut * (1 + sign * delta)
        c0 = 1.3
        top = np.sqrt(q * (c0 * c0 + 1e-6) / (1 - q))  # su = top^2 / (c0^2 + top^2 + 1e-6)
        rho = c0 * V[:, 0][None, :] + top[:, None] * V[:, deg][None, :]
        ps = frhip.FRPSpace1D(0.0, 1.0, delta.size, deg)
        g = frhip.FREulerProblem(ps, 1.4, "period", "hll")
        g.set_state(np.asfortranarray(np.stack([rho, 0 * rho, 2.5 + 0 * rho], -1)))
        assert g.sensor_filter(1e-4) == (delta.size if sign > 0 else 0)
        g.close()
