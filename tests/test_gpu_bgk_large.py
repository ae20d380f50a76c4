"""The 2D BGK stage kernel of states above 64 MiB (a tile walked through a group of velocities, the
moments summed on the way) against the CPU oracle, on grids with partial tiles of every width."""
import numpy as np
import pytest

from frhip import bgk
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,deg,nu,nv,nmem", [(67, 61, 1, 23, 24, 1), (37, 29, 2, 21, 22, 2),
                                                  (130, 5, 3, 31, 29, 1), (21, 23, 4, 26, 27, 1),
                                                  (8, 9, 2, 124, 123, 1)])
def test_large_state_step_parity(nx, ny, deg, nu, nv, nmem):
    u, wu = bgk.velocity_grid(nu)
    v, wv = bgk.velocity_grid(nv)
    taus = np.array([1e-2, 1e-1])[:nmem]
    f0 = bgk.maxwellian_state(nx, ny, deg, u, v, amp=0.1, nmem=nmem)
    f0 = f0 * (1.0 + 0.02 * np.random.default_rng(nx).uniform(-1, 1, size=f0.size))
    assert f0.nbytes > 64 << 20
    dt = 0.1 / (deg + 1) / max(nx, ny) / np.abs(u).max()
    g = bgk.BGK2D(nx, ny, deg, u, wu, v, wv, taus)
    g.set_state(f0)
    g.step(dt, 1)
    out = g.get_state().reshape(nmem, -1)
    # one step: dt L is below f, and L agrees to 1e-12 of its largest value
    for f, got, tau in zip(f0.reshape(nmem, -1), out, taus):
        L = lambda x: O.bgk2d_rhs(x, nx, ny, deg, u, wu, v, wv, tau).ravel()  # noqa: E731
        a = f + dt * L(f)
        b = 0.75 * f + 0.25 * a + 0.25 * dt * L(a)
        ref = f / 3 + 2 / 3 * b + 2 / 3 * dt * L(b)
        assert np.linalg.norm(got - ref) <= 1e-12 * np.linalg.norm(ref)
    # the sums of a state and those of the stage that made it agree: a split call gives the same bits
    g.step(dt, 1)
    two = g.get_state()
    g.set_state(f0)
    g.step(dt, 2)
    assert np.array_equal(g.get_state(), two)


@pytest.mark.parametrize("nx,ny,deg,nv", [(67, 61, 1, 23), (37, 29, 2, 31), (20, 33, 2, 16)])
def test_steps_of_one_call_and_of_several(nx, ny, deg, nv):
    # odd and even step counts end in different buffers; partial tiles read u^n for cells stored elsewhere
    u, wu = bgk.velocity_grid(nv)
    f0 = bgk.maxwellian_state(nx, ny, deg, u, u, amp=0.1)
    dt = 0.1 / (deg + 1) / max(nx, ny) / np.abs(u).max()
    g = bgk.BGK2D(nx, ny, deg, u, wu, u, wu, [1e-2])
    g.set_state(f0)
    outs = []
    for _ in range(3):
        g.step(dt, 1)
        outs.append(g.get_state())
    for n in (1, 2, 3):
        g.set_state(f0)
        g.step(dt, n)
        assert np.array_equal(g.get_state(), outs[n - 1])


@pytest.mark.parametrize("nx,ny,deg,nv,nmem", [(1, 1, 2, 12, 7000), (3, 5, 1, 16, 600), (4, 4, 3, 16, 170), (6, 6, 3, 16, 115),
                                               (14, 14, 2, 16, 20), (2, 2, 1, 49, 230)])
def test_many_members_of_few_cells(nx, ny, deg, nv, nmem):
    """States above 64 MiB on either side of the line that the share of lanes with a cell draws: the first
    and the last members against the oracle."""
    u, wu = bgk.velocity_grid(nv)
    taus = np.geomspace(1e-2, 1e-1, nmem)
    one = bgk.maxwellian_state(nx, ny, deg, u, u, amp=0.1)
    rng = np.random.default_rng(nmem)
    f0 = (one[None, :] * (1.0 + 0.02 * rng.uniform(-1, 1, (nmem, 1)))).ravel()
    assert f0.nbytes > 64 << 20
    dt = 0.1 / (deg + 1) / max(nx, ny) / np.abs(u).max()
    g = bgk.BGK2D(nx, ny, deg, u, wu, u, wu, taus)
    g.set_state(f0)
    g.step(dt, 1)
    out = g.get_state().reshape(nmem, -1)
    for b in (0, 1, nmem // 2, nmem - 1):
        f = f0.reshape(nmem, -1)[b]
        L = lambda x: O.bgk2d_rhs(x, nx, ny, deg, u, wu, u, wu, taus[b]).ravel()  # noqa: B023, E731
        a = f + dt * L(f)
        c = 0.75 * f + 0.25 * a + 0.25 * dt * L(a)
        ref = f / 3 + 2 / 3 * c + 2 / 3 * dt * L(c)
        assert np.linalg.norm(out[b] - ref) <= 1e-12 * np.linalg.norm(ref)


def test_sums_and_moments_share_their_memory():
    """A new context holds the state, the moments (four per point, or per velocity group: here one) and the
    Maxwellian factors; moments and right-hand sides between steps leave no trace in them."""
    torch = pytest.importorskip("torch")
    u, wu = bgk.velocity_grid(2)
    torch.zeros(1, device="cuda")
    g = bgk.BGK2D(8, 8, 1, u, wu, u, wu, [1e-2])  # the library's code is on the device
    free = torch.cuda.mem_get_info()[0]
    big = bgk.BGK2D(2048, 2048, 1, u, wu, u, wu, [1e-2])
    state = 2048 * 2048 * 4 * 4 * 8
    assert big.len * 8 == state
    assert free - torch.cuda.mem_get_info()[0] <= 3 * state + (64 << 20)
    big.close()
    g.close()
    u, wu = bgk.velocity_grid(24)
    f0 = bgk.maxwellian_state(57, 43, 2, u, u, amp=0.1)
    g = bgk.BGK2D(57, 43, 2, u, wu, u, wu, [1e-2])
    out = []
    for between in (lambda: None, lambda: (g.moments(), g.rhs(f0))):
        g.set_state(f0)
        g.step(1e-4, 1)
        between()
        g.step(1e-4, 1)
        out.append((g.get_state(), g.moments()))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
    g.close()
