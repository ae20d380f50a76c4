"""The work that users of frhip have it do, as cases that can be timed and checked.

Families (the `path` of a case) and what they stand for:

    rhs2d   the drop-in right-hand side dudt!(du, u, p, t) on device arrays, as an ODE package calls it
    step2d  n explicit steps of the device-resident 2D Euler solver, the state put in and read back
    loop2d  n iterations of the shock-vortex host loop (limiter, step, sensor + filter, ghost copy)
    fr1d    n steps of one 1D problem (Euler or advection) from a host state to a host state
    ens1d   n steps of many uneven 1D Euler problems together, sensor + filter before every step
    bgk2d   n SSP-RK3 steps of the 2D discrete-velocity BGK model, its moments read back
    bgk1d   n steps of the 1D BGK model from a host state to a host state
    mol1d   mol!(du, u, p, t) of the 1D BGK model on device arrays

listed() holds the sizes of this repository's benchmark, scripts and tests beside odd ones; draw()
spreads the sizes, degrees, fluxes, boundary modes, cells and schemes of the same families.
exact() restates each path array-at-a-time in 64 bits with torch and numpy alone.
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "fluxreconstruction.jl_amd"))

import frhip  # noqa: E402
from frhip import sensor  # noqa: E402

GAMMA = 1.4
TAU = 1e-2
STAGES = {"ssprk3": 3, "rk4": 4, "midpoint": 2, "euler": 1}


def listed():
    return [
        # one dudt! call of an ODE package at the benchmark's grid, with the reference's flux and ghost layer
        dict(name="rhs_256x256_p3", path="rhs2d", nx=256, ny=256, deg=3, flux="hll", bc="ghost", cells="rect"),
        # the headline benchmark's stepping: vortex grid, Rusanov, periodic
        dict(name="step_256x256_p3", path="step2d", nx=256, ny=256, deg=3, flux="rusanov", bc="periodic", cells="rect",
             scheme="ssprk3", steps=20),
        # a production grid, too large for the last-level cache and ragged against the kernels' tiles
        dict(name="step_1000x600_p3", path="step2d", nx=1000, ny=600, deg=3, flux="rusanov", bc="periodic", cells="rect",
             scheme="ssprk3", steps=4),
        # higher degree on an odd grid, the reference's flux and ghost layer as data
        dict(name="step_201x133_p4", path="step2d", nx=201, ny=133, deg=4, flux="hll", bc="ghost", cells="rect",
             scheme="ssprk3", steps=10),
        # curvilinear cells (a polar mesh), the metric of every solution point read beside the state
        dict(name="step_polar_256x256_p3", path="step2d", nx=256, ny=256, deg=3, flux="rusanov", bc="ghost",
             cells="polar", scheme="ssprk3", steps=10),
        # example/shock-vortex.jl at its own size: launches and latency count
        dict(name="loop_100x50_p2", path="loop2d", nx=100, ny=50, deg=2, mode="modal", scheme="midpoint", steps=10),
        # the learned-sensor run of the shock-vortex case
        dict(name="loop_512x256_p3_learned", path="loop2d", nx=512, ny=256, deg=3, mode="learned", scheme="ssprk3",
             steps=10),
        # the smallest work: 1D advection, 100 cells, p = 2, RK4
        dict(name="advection_100_p2", path="fr1d", eq="advection", ncell=100, deg=2, flux="hll", bc="period",
             scheme="rk4", steps=100),
        # 512 uneven Riemann problems of 64 to 2048 cells, p in {2, 3, 4}
        dict(name="riemann_512", path="ens1d", members=512, lo=64, hi=2048, dlo=2, dhi=4, scheme="ssprk3", steps=100),
        # the kinetic benchmark: 128 x 128 cells x 24 x 24 velocities
        dict(name="bgk_128x128_p2_24x24", path="bgk2d", nx=128, ny=128, deg=2, nu=24, nv=24, members=1, steps=4),
        # example/bgk_wave.jl at its own size
        dict(name="bgk1d_20x100_p2", path="bgk1d", nx=20, nu=100, deg=2, members=1, scheme="midpoint", steps=100),
        # mol! of a large 1D kinetic state
        dict(name="mol_8192x256_p2", path="mol1d", nx=8192, nu=256, deg=2, members=1),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, points, deg):
    """nx, ny >= lo with at most `points` solution points, over the logarithm of the size."""
    most = points / (deg + 1) ** 2
    cells = math.exp(rng.uniform(math.log(lo * lo), math.log(most)))
    nx = max(lo, min(int(cells / lo), int(math.sqrt(cells) * math.exp(rng.uniform(-0.7, 0.7)))))
    return nx, max(lo, int(cells / nx))


def draw(rng):
    path = rng.choice(["rhs2d", "step2d", "step2d", "loop2d", "fr1d", "ens1d", "bgk2d", "bgk1d", "mol1d"])
    c = dict(path=path)
    if path in ("rhs2d", "step2d"):
        c["deg"] = rng.choice([1, 2, 3, 3, 4, 5])
        c["nx"], c["ny"] = _grid(rng, 8, 2.5e6, c["deg"])
        c.update(flux=rng.choice(["hll", "rusanov", "rusanov", "roe"]), bc=rng.choice(["ghost", "periodic"]),
                 cells=rng.choice(["rect", "rect", "affine", "polar"]))
        if path == "step2d":
            c.update(scheme=rng.choice(["ssprk3", "ssprk3", "midpoint", "rk4"]), steps=rng.randint(2, 10))
    elif path == "loop2d":
        c["mode"] = rng.choice(["modal", "modal", "learned", "off"])
        c["deg"] = 3 if c["mode"] == "learned" else rng.choice([2, 3, 4])
        c["nx"], c["ny"] = _grid(rng, 24, 2.0e6, c["deg"])
        c.update(scheme=rng.choice(["ssprk3", "midpoint"]), steps=rng.randint(3, 10))
    elif path == "fr1d":
        c.update(eq=rng.choice(["euler", "advection"]), ncell=_log(rng, 16, 4000), deg=rng.randint(1, 7),
                 flux=rng.choice(["hll", "rusanov", "roe"]), bc=rng.choice(["dirichlet", "period"]),
                 scheme=rng.choice(["ssprk3", "rk4", "midpoint", "euler"]), steps=_log(rng, 10, 100))
    elif path == "ens1d":
        lo = _log(rng, 16, 128)
        dlo = rng.randint(1, 3)
        c.update(members=_log(rng, 8, 256), lo=lo, hi=lo * rng.randint(2, 10), dlo=dlo, dhi=rng.randint(dlo, 4),
                 scheme=rng.choice(["ssprk3", "midpoint"]), steps=_log(rng, 10, 60))
    elif path == "bgk2d":
        c.update(nx=_log(rng, 8, 72), ny=_log(rng, 8, 72), deg=rng.randint(1, 3), nu=rng.randint(8, 24),
                 nv=rng.randint(8, 24), members=rng.choice([1, 1, 2]), steps=rng.randint(1, 3))
    elif path == "bgk1d":
        c.update(nx=_log(rng, 8, 400), nu=rng.randint(16, 128), deg=rng.randint(1, 4), members=rng.choice([1, 1, 8]),
                 scheme=rng.choice(["ssprk3", "midpoint", "euler"]), steps=_log(rng, 10, 60))
    else:
        c.update(nx=_log(rng, 100, 8192), nu=rng.randint(32, 256), deg=rng.randint(1, 4), members=rng.choice([1, 1, 2]))
    return c


# ------------------------------------------------------------------ operators, in 64 bits, from numpy
@functools.lru_cache(maxsize=None)
def _ops(deg):
    P = np.polynomial.legendre
    n = deg + 1
    r, w = P.leggauss(n)
    norm = np.sqrt((2.0 * np.arange(n) + 1.0) / 2.0)
    V = P.legvander(r, deg) * norm  # orthonormal Legendre modes at the points
    iV = np.linalg.inv(V)
    end = [(P.legvander(np.array([x]), deg) * norm)[0] @ iV for x in (-1.0, 1.0)]
    dV = np.stack([P.legval(r, P.legder(np.eye(n)[q])) if q else np.zeros(n) for q in range(n)], 1) * norm
    d = [P.legval(r, P.legder(np.eye(n + 1)[q])) if q else np.zeros(n) for q in (deg, deg + 1)]
    return dict(r=r, w=w, V=V, iV=iV, ll=end[0], lr=end[1], dl=dV @ iV, dhl=(-1.0) ** deg * 0.5 * (d[0] - d[1]),
                dhr=0.5 * (d[0] + d[1]))


def _dev(a):
    return torch.as_tensor(np.asarray(a, dtype=np.float64), device="cuda")


def _devops(deg):
    return {k: _dev(v) for k, v in _ops(deg).items()}


# ------------------------------------------------------------------ inputs, from the seed alone
def _waves(rng, x, y=None):
    """A smooth periodic field on [0, 1] (x [0, 1]) in [-1, 1]: three sine modes."""
    s = 0.0
    for _ in range(3):
        kx, ky, ph = int(rng.integers(1, 4)), int(rng.integers(-2, 3)), float(rng.uniform(0, 2 * np.pi))
        arg = 2 * np.pi * kx * x + ph if y is None else 2 * np.pi * (kx * x + ky * y) + ph
        s = s + (torch.sin(arg) if isinstance(arg, torch.Tensor) else np.sin(arg)) / 3.0
    return s


def _conserve(rho, U, V, p):
    return torch.stack(torch.broadcast_tensors(rho, rho * U, rho * V, p / (GAMMA - 1) + 0.5 * rho * (U * U + V * V)))


def _points(c):
    """Unit-square coordinates of every solution point, ghost cells included: x over (k, j, i) broadcast
    shapes of a (l, k, ny+2, nx+2) field."""
    r = _dev(_ops(c["deg"])["r"])
    x = (torch.arange(c["nx"] + 2, device="cuda", dtype=torch.float64)[None, :] - 0.5 + 0.5 * r[:, None]) / c["nx"]
    y = (torch.arange(c["ny"] + 2, device="cuda", dtype=torch.float64)[None, :] - 0.5 + 0.5 * r[:, None]) / c["ny"]
    return x[None, :, None, :], y[:, None, :, None]


def _state2d(c, seed):
    """(4, l, k, ny+2, nx+2): the column-major state u(i, j, k, l, m) of the solvers."""
    rng = np.random.default_rng([seed, 2])
    x, y = _points(c)
    if c["path"] != "loop2d":  # smooth flow with sub- and supersonic parts
        f = [_waves(rng, x, y) for _ in range(4)]
        u0, v0 = rng.uniform(-1.0, 1.0, 2)
        return _conserve(1 + 0.2 * f[0], u0 + 0.3 * f[1], v0 + 0.3 * f[2], 1 + 0.2 * f[3]).contiguous()
    # a stationary normal shock and a vortex upstream of it, on [0, 2] x [0, 1]
    mach = rng.uniform(1.05, 1.3)
    rc, xc, yc = 0.075 * rng.uniform(0.8, 1.2), 0.25 * rng.uniform(0.8, 1.2), 0.5 * rng.uniform(0.8, 1.2)
    amp = rng.uniform(0.3, 0.6)
    X, Y = 2.0 * x, y
    s = ((X - xc) ** 2 + (Y - yc) ** 2) / rc ** 2
    e = amp * torch.exp(0.5 * (1 - s))
    T = 1 - (GAMMA - 1) / (2 * GAMMA) * e * e
    rho, u1 = T ** (1 / (GAMMA - 1)), mach * math.sqrt(GAMMA)
    r2 = (GAMMA + 1) * mach ** 2 / ((GAMMA - 1) * mach ** 2 + 2)
    p2 = 1 + 2 * GAMMA / (GAMMA + 1) * (mach ** 2 - 1)
    up = (X <= 0.5) & (Y > -1)
    pick = lambda a, b: torch.where(up, a, torch.full((), b, dtype=torch.float64, device="cuda"))  # noqa: E731
    return _conserve(pick(rho, r2), pick(u1 - e * (Y - yc) / rc, u1 / r2), pick(e * (X - xc) / rc, 0.0),
                     pick(rho * T, p2)).contiguous()


def _lengths(c):
    return (2.0, 1.0) if c["path"] == "loop2d" else (10.0, 10.0)


def _iJ(c):
    """Inverse Jacobian entries r_x, r_y, s_x, s_y: numbers, or (l, k, ny+2, nx+2) on the polar mesh."""
    Lx, Ly = _lengths(c)
    dx, dy = Lx / c["nx"], Ly / c["ny"]
    if c["cells"] == "rect":
        return 2 / dx, 0.0, 0.0, 2 / dy
    if c["cells"] == "affine":
        m = np.linalg.inv(np.array([[dx / 2, 0.4 * dx / 2], [0.0, dy / 2]]))
        return tuple(float(v) for v in m.ravel())
    dr, dt = 5.0 / c["nx"], math.pi / c["ny"]
    rr = 1.0 + (np.arange(c["nx"] + 2) - 0.5) * dr
    tt = (np.arange(c["ny"] + 2) - 0.5) * dt
    P, q = _ops(c["deg"])["r"], {}
    for d, f in enumerate((np.cos, np.sin)):
        v = [(rr + sr * dr / 2)[None, :] * f(tt + st * dt / 2)[:, None] for sr, st in ((-1, -1), (1, -1), (1, 1), (-1, 1))]
        k, l = P[None, :, None, None], P[:, None, None, None]
        q[d, 0] = 0.25 * ((1 - l) * (v[1] - v[0]) + (1 + l) * (v[2] - v[3]))
        q[d, 1] = 0.25 * ((1 - k) * (v[3] - v[0]) + (1 + k) * (v[2] - v[1]))
    q = {a: np.broadcast_to(b, (P.size, P.size, c["ny"] + 2, c["nx"] + 2)) for a, b in q.items()}
    det = q[0, 0] * q[1, 1] - q[0, 1] * q[1, 0]
    return _dev(q[1, 1] / det), _dev(-q[0, 1] / det), _dev(-q[1, 0] / det), _dev(q[0, 0] / det)


def _dt2d(c, U):
    rho, p = U[0], _pressure(U)
    lam = (torch.sqrt(GAMMA * p / rho) + torch.maximum(U[1].abs(), U[2].abs()) / rho).max().item()
    Lx, Ly = _lengths(c)
    # the reference's face terms are not upwind everywhere on the polar mesh: short steps stay finite
    h = 0.1 * min(5.0 / c["nx"], math.pi / c["ny"]) if c["cells"] == "polar" else min(Lx / c["nx"], Ly / c["ny"])
    return 0.15 / (c["deg"] + 1) * h / lam


def _loop_case(c):
    return dict(c, cells="rect", flux="hll", bc="ghost")


def _riemann(c, seed):
    """ncell, deg and the (ncell, nsp, 3) states of uneven Riemann problems, the jump on a cell face."""
    rng = np.random.default_rng([seed, 1])
    shape = np.random.default_rng(c["members"])  # the sizes belong to the case, the data to the seed
    n = shape.integers(c["lo"], c["hi"] + 1, c["members"])
    d = shape.integers(c["dlo"], c["dhi"] + 1, c["members"])
    out = []
    for b in range(c["members"]):
        rho, p = rng.uniform(0.5, 1.0, (2, 2))
        vel = rng.uniform(-0.2, 0.2, 2)
        right = ((np.arange(n[b]) + 0.5) / n[b] > rng.uniform(0.3, 0.7)).astype(int)
        w = np.stack([rho, rho * vel, p / (GAMMA - 1) + 0.5 * rho * vel * vel], -1)[right]
        out.append(np.asfortranarray(np.repeat(w[:, None, :], d[b] + 1, axis=1)))
    return n, d, out


def _ens_dt(n):
    return 0.05 / float(n.max()) / 2.5


def _state1d(c, seed):
    rng = np.random.default_rng([seed, 3])
    x = ((np.arange(c["ncell"]) + 0.5)[:, None] + 0.5 * _ops(c["deg"])["r"][None, :]) / c["ncell"]
    if c["eq"] == "advection":
        k, ph = int(rng.integers(1, 3)), rng.uniform(0, 2 * np.pi)
        return np.asfortranarray(rng.uniform(0.5, 1.5) * np.sin(2 * np.pi * k * x + ph))
    rho, u, p = 1 + 0.2 * _waves(rng, x), rng.uniform(-0.5, 0.5) + 0.2 * _waves(rng, x), 1 + 0.2 * _waves(rng, x)
    return np.asfortranarray(np.stack([rho, rho * u, p / (GAMMA - 1) + 0.5 * rho * u * u], -1))


def _dt1d(c):
    return 0.1 / (c["deg"] + 1) / c["ncell"] / (1.0 if c["eq"] == "advection" else 3.0)


def _taus(c):
    return np.geomspace(TAU, 10 * TAU, c["members"])


def _hermite(n):
    x, w = np.polynomial.hermite.hermgauss(n)
    return x, w * np.exp(x * x)


def _bgk2d_state(c, seed):
    """(members, b, a, l, k, ny, nx): Maxwellians of a smooth flow."""
    rng = np.random.default_rng([seed, 4])
    x, y = _points(c)
    x, y = x[..., 1:-1], y[:, :, 1:-1]
    a, b = _dev(_hermite(c["nu"])[0]), _dev(_hermite(c["nv"])[0])
    fs = []
    for _ in range(c["members"]):
        rho, lam = 1 + 0.1 * _waves(rng, x, y), 1 + 0.1 * _waves(rng, x, y)
        U, V = 0.1 * _waves(rng, x, y), 0.1 * _waves(rng, x, y)
        ea = torch.exp(-lam * (a[:, None, None, None, None] - U) ** 2)
        eb = rho * lam / math.pi * torch.exp(-lam * (b[:, None, None, None, None] - V) ** 2)
        fs.append(eb[:, None] * ea[None])
    return torch.stack(fs).contiguous()


def _bgk2d_dt(c):
    return 0.1 / (c["deg"] + 1) / max(c["nx"], c["ny"]) / float(np.abs(_hermite(max(c["nu"], c["nv"]))[0]).max())


def _vgrid(c):
    du = 10.0 / c["nu"]
    return -5.0 + (np.arange(c["nu"]) + 0.5) * du, np.full(c["nu"], du)


def _bgk1d_state(c, seed):
    """(nx, nu, nsp, members), column-major: the Maxwellians of bgk_wave.jl's kind of wave."""
    rng = np.random.default_rng([seed, 5])
    x = ((np.arange(c["nx"]) + 0.5)[:, None] + 0.5 * _ops(c["deg"])["r"][None, :]) / c["nx"]
    u = _vgrid(c)[0][None, :, None]
    f = []
    for _ in range(c["members"]):
        rho, lam, U = (v[:, None, :] for v in (1 + 0.1 * _waves(rng, x), 1 + 0.1 * _waves(rng, x), 0.5 + 0.2 * _waves(rng, x)))
        f.append(rho * np.sqrt(lam / np.pi) * np.exp(-lam * (u - U) ** 2))
    return np.asfortranarray(np.stack(f, -1))


def _bgk1d_dt(c):
    return 0.1 / (c["deg"] + 1) / c["nx"] / 5.0


# ------------------------------------------------------------------ what a user's program holds, and one pass
@functools.lru_cache(maxsize=2)
def _space2d(cells, nx, ny, deg, Lx, Ly):
    if cells == "polar":
        return frhip.FRPSpace2D(frhip.CSpace2D(1.0, 6.0, nx, 0.0, math.pi, ny, 1, 1), deg)
    return frhip.FRPSpace2D(0.0, Lx, nx, 0.0, Ly, ny, deg, 1, 1)


def prepare(case, seed):
    path = case["path"]
    if path in ("rhs2d", "step2d", "loop2d"):
        c = _loop_case(case) if path == "loop2d" else case
        solver = frhip.FREuler2D(_space2d(c["cells"], c["nx"], c["ny"], c["deg"], *_lengths(c)), GAMMA, c["flux"], c["bc"])
        if c["cells"] == "affine":
            solver.set_geometry(np.reshape(_iJ(c), (2, 2)))
        solver.use_torch_stream()
        if path == "loop2d" and c["mode"] == "learned":
            sensor.attach(solver, sensor.SensorMLP.load())
        U = _state2d(c, seed)
        return dict(case=c, solver=solver, u=U, out=torch.empty_like(U), dt=_dt2d(c, U))
    if path == "fr1d":
        ps = frhip.FRPSpace1D(0.0, 1.0, case["ncell"], case["deg"])
        if case["eq"] == "euler":
            pr = frhip.FREulerProblem(ps, GAMMA, case["bc"], case["flux"])
        else:
            pr = frhip.FRAdvectionProblem(ps, 1.0, case["bc"])
        return dict(case=case, solver=pr, u=_state1d(case, seed), dt=_dt1d(case))
    if path == "ens1d":
        n, d, members = _riemann(case, seed)
        e = frhip.Ensemble1D(n, d, 1.0 / n, GAMMA, "rusanov", "dirichlet")
        return dict(case=case, solver=e, u=e.pack(members), dt=_ens_dt(n))
    if path == "bgk2d":
        (u, wu), (v, wv) = _hermite(case["nu"]), _hermite(case["nv"])
        g = frhip.BGK2D(case["nx"], case["ny"], case["deg"], u, wu, v, wv, _taus(case))
        return dict(case=case, solver=g, u=_bgk2d_state(case, seed).reshape(-1), dt=_bgk2d_dt(case))
    g = frhip.BGK1D(frhip.FRPSpace1D(0.0, 1.0, case["nx"], case["deg"]), frhip.VSpace1D(-5.0, 5.0, case["nu"]), _taus(case))
    f = _bgk1d_state(case, seed)
    if path == "mol1d":
        u = _dev(f.ravel(order="F"))
        return dict(case=case, solver=g, u=u, out=torch.empty_like(u))
    return dict(case=case, solver=g, u=f, dt=_bgk1d_dt(case))


def _read2d(state):
    s = state["solver"]
    rc = frhip.lib().fr2d_get_state_dev(s.h, state["out"].data_ptr())
    if rc:
        raise RuntimeError("fr2d_get_state_dev: %d" % rc)
    return state["out"]


def run(state):
    c, s = state["case"], state["solver"]
    path = c["path"]
    if path == "rhs2d":
        s.dudt(state["out"], state["u"])
        return state["out"]
    if path == "step2d":
        s.set_state(state["u"])
        s.step(state["dt"], c["steps"], c["scheme"])
        return _read2d(state)
    if path == "loop2d":
        s.set_state(state["u"])
        n = s.run_host_loop(state["dt"], c["steps"], c["mode"], scheme=c["scheme"])
        return dict(state=_read2d(state), filtered=n)
    if path == "fr1d":
        s.set_state(state["u"])
        s.step(state["dt"], c["steps"], c["scheme"])
        return s.get_state()
    if path == "ens1d":
        s.set_state(state["u"])
        n, _ = s.run(state["dt"], c["steps"], filter=True, scheme=c["scheme"])
        return dict(state=s.get_state(), filtered=n)
    if path == "bgk2d":
        s.set_state(state["u"])
        s.step(state["dt"], c["steps"])
        return s.moments()
    if path == "bgk1d":
        s.set_state(state["u"])
        s.step(state["dt"], c["steps"], c["scheme"])
        return s.get_state()
    return s.mol(state["out"], state["u"])


def work(case):
    """A right-hand side reads its state and writes du; a stage reads the state it differentiates (and,
    after the first, the step's start) and writes its result; a filter pass reads the state and writes it.
    The metric of curvilinear cells is read by each.  The host states' way over the bus is not counted.
    Operations: the two sides' contractions, fluxes and Riemann problems per value, in round numbers."""
    p = case["path"]
    n = case["deg"] + 1 if "deg" in case else (case["dlo"] + case["dhi"]) / 2 + 1
    steps, stages = case.get("steps", 1), STAGES.get(case.get("scheme"), 3 if p == "bgk2d" else 1)
    if p in ("rhs2d", "step2d", "loop2d"):
        dof = case["nx"] * case["ny"] * n * n * 4
    elif p == "fr1d":
        dof = case["ncell"] * n * (3 if case["eq"] == "euler" else 1)
    elif p == "ens1d":
        sizes, degs, _ = _riemann(case, 0)
        dof = 3 * int((sizes * (degs + 1)).sum())
    elif p == "bgk2d":
        dof = case["nx"] * case["ny"] * n * n * case["nu"] * case["nv"] * case["members"]
    else:
        dof = case["nx"] * n * case["nu"] * case["members"]
    flops = (4 * n + 40) if p in ("rhs2d", "step2d", "loop2d", "fr1d", "ens1d") else (4 * n + 20)
    if p in ("rhs2d", "mol1d"):
        return dict(bytes=dof * (16 + (8 if case.get("cells") == "polar" else 0)), flops=dof * flops)
    per = 24 * stages - 8 + (8 * stages if case.get("cells") == "polar" else 0)
    if p in ("loop2d", "ens1d") and case.get("mode") != "off":
        per, flops = per + 16, flops + (4 * n * n if p == "loop2d" else 4 * n) / stages
    return dict(bytes=dof * steps * per, flops=dof * steps * stages * flops)


# ------------------------------------------------------------------ the same in 64 bits, array at a time
def _pressure(U):
    return (GAMMA - 1) * (U[-1] - 0.5 * sum(m * m for m in U[1:-1]) / U[0])


def _flux(U, d=1):
    """Flux along momentum component d of states (variables first), and the pressure."""
    p, v = _pressure(U), U[d] / U[0]
    F = [m * v for m in U[:-1]] + [(U[-1] + p) * v]
    F[0], F[d] = U[d], F[d] + p
    return torch.stack(F), p


def _interface(kind, L, R):
    (FL, pL), (FR, pR) = _flux(L), _flux(R)
    uL, uR = L[1] / L[0], R[1] / R[0]
    cL, cR = torch.sqrt(GAMMA * pL / L[0]), torch.sqrt(GAMMA * pR / R[0])
    if kind == "rusanov":
        return 0.5 * (FL + FR) - 0.5 * torch.maximum(uL.abs() + cL, uR.abs() + cR) * (R - L)
    if kind == "hll":
        lo, hi = torch.minimum(uL - cL, uR - cR), torch.maximum(uL + cL, uR + cR)
        mid = (hi * FL - lo * FR + hi * lo * (R - L)) / (hi - lo)
        return torch.where(lo >= 0, FL, torch.where(hi <= 0, FR, mid))
    sL, sR = torch.sqrt(L[0]), torch.sqrt(R[0])
    mean = lambda a, b: (sL * a + sR * b) / (sL + sR)  # noqa: E731
    two = L.shape[0] == 4
    vL, vR = (L[2] / L[0], R[2] / R[0]) if two else (0 * uL, 0 * uR)
    u, v, H = mean(uL, uR), mean(vL, vR), mean((L[-1] + pL) / L[0], (R[-1] + pR) / R[0])
    a2 = (GAMMA - 1) * (H - 0.5 * (u * u + v * v))
    a, rt = torch.sqrt(a2), sL * sR
    dp, du = pR - pL, uR - uL
    w1, w5 = (dp - rt * a * du) / (2 * a2), (dp + rt * a * du) / (2 * a2)
    w2, w3 = R[0] - L[0] - dp / a2, rt * (vR - vL)
    l1, l2, l5 = (u - a).abs(), u.abs(), (u + a).abs()
    D = [l1 * w1 + l2 * w2 + l5 * w5, l1 * w1 * (u - a) + l2 * w2 * u + l5 * w5 * (u + a),
         l1 * w1 * v + l2 * (w2 * v + w3) + l5 * w5 * v,
         l1 * w1 * (H - u * a) + l2 * (w2 * 0.5 * (u * u + v * v) + w3 * v) + l5 * w5 * (H + u * a)]
    return 0.5 * (FL + FR) - 0.5 * torch.stack(D if two else [D[0], D[1], D[3]])


def _turn(U, c, s):
    return torch.stack([U[0], c * U[1] + s * U[2], c * U[2] - s * U[1], U[3]])


def _wrap(U):
    U = U.clone()
    U[..., 0], U[..., -1] = U[..., -2].clone(), U[..., 1].clone()
    U[..., 0, :], U[..., -1, :] = U[..., -2, :].clone(), U[..., 1, :].clone()
    return U


def _rhs2d(c, o, iJ, U):
    """du of a (4, l, k, j, i) state, zero on the ghost layer."""
    if c["bc"] == "periodic":
        U = _wrap(U)
    rx, ry, sx, sy = iJ
    if c["cells"] == "affine":
        h1, h2 = math.hypot(rx, ry), math.hypot(sx, sy)
        n1, n2, q1, q2 = (rx / h1, ry / h1), (sx / h2, sy / h2), h1, h2
    else:
        n1, n2, q1, q2 = (1.0, 0.0), (0.0, 1.0), rx, sy
    if torch.is_tensor(q1):
        q1, q2 = q1[..., 1:-1, 1:-1], q2[..., 1:-1, 1:-1]
    F, G = _flux(U, 1)[0], _flux(U, 2)[0]
    f1, f2 = rx * F + ry * G, sx * F + sy * G
    F = G = None
    k = lambda A, w: torch.einsum("mlkji,k->mlji", A, w)  # noqa: E731
    l = lambda A, w: torch.einsum("mlkji,l->mkji", A, w)  # noqa: E731
    A, B = k(U, o["lr"])[:, :, 1:-1, :-1], k(U, o["ll"])[:, :, 1:-1, 1:]
    X = _turn(_interface(c["flux"], _turn(A, *n1), _turn(B, *n1)), n1[0], -n1[1])
    A, B = l(U, o["lr"])[:, :, :-1, 1:-1], l(U, o["ll"])[:, :, 1:, 1:-1]
    Y = _turn(_interface(c["flux"], _turn(A, *n2), _turn(B, *n2)), n2[0], -n2[1])
    f1, f2 = f1[..., 1:-1, 1:-1], f2[..., 1:-1, 1:-1]
    d = torch.einsum("kq,mlqji->mlkji", o["dl"], f1) + torch.einsum("lq,mqkji->mlkji", o["dl"], f2)
    gl, gr = o["dhl"][None, None, :, None, None], o["dhr"][None, None, :, None, None]
    d += (q1 * X[:, :, None, :, :-1] - k(f1, o["ll"])[:, :, None]) * gl
    d += (q1 * X[:, :, None, :, 1:] - k(f1, o["lr"])[:, :, None]) * gr
    gl, gr = o["dhl"][None, :, None, None, None], o["dhr"][None, :, None, None, None]
    d += (q2 * Y[:, None, :, :-1, :] - l(f2, o["ll"])[:, None]) * gl
    d += (q2 * Y[:, None, :, 1:, :] - l(f2, o["lr"])[:, None]) * gr
    du = torch.zeros_like(U)
    du[..., 1:-1, 1:-1] = -d
    return du


def _step(f, u, dt, scheme):
    if scheme == "ssprk3":
        a = u + dt * f(u)
        b = 0.75 * u + 0.25 * a + 0.25 * dt * f(a)
        return u / 3 + 2 / 3 * b + 2 / 3 * dt * f(b)
    if scheme == "midpoint":
        return u + dt * f(u + 0.5 * dt * f(u))
    if scheme == "euler":
        return u + dt * f(u)
    k1 = f(u)
    k2 = f(u + 0.5 * dt * k1)
    k3 = f(u + 0.5 * dt * k2)
    return u + dt / 6 * (k1 + 2 * k2 + 2 * k3 + f(u + dt * k3))


def _switch(Se, S0, kappa):
    """Cells of the Persson-Peraire sensor: sigma < 0.99."""
    mid = 0.5 * (1 - torch.sin(0.5 * math.pi * (Se - S0) / kappa))
    return torch.where(Se < S0 - kappa, 1.0, torch.where(Se < S0 + kappa, mid, 0.0)) < 0.99


def _strength(modes):
    """The learned sensor's output per cell: BF16 operands, otherwise 64 bits."""
    with np.load(os.path.join(ROOT, "fluxreconstruction.jl_amd", "frhip", "data", "sensor_mlp.npz")) as z:
        p = torch.as_tensor(z["params"], device="cuda")
    bf = lambda a: a.to(torch.float32).to(torch.bfloat16).double()  # noqa: E731
    W1, b1, W2, b2, W3, b3 = torch.split(p, [512, 32, 1024, 32, 32, 1])
    x = bf(modes / torch.sqrt((modes * modes).sum(0) + 1e-300)).reshape(16, -1)
    h = torch.relu(bf(W1).reshape(32, 16) @ x + b1.double()[:, None])
    h = torch.relu(bf(W2).reshape(32, 32) @ bf(h) + b2.double()[:, None])
    return torch.relu(W3.double() @ h + b3.double()).reshape(modes.shape[1:])


def _filter2d(c, o, U):
    if c["mode"] == "off":
        return U
    n = c["deg"] + 1
    M = torch.einsum("ak,bl,mlkji->mabji", o["iV"], o["iV"], U).reshape(4, n * n, *U.shape[3:])
    if c["mode"] == "modal":
        Se = torch.log10(M[0, -1] ** 2 / (M[0] ** 2).sum(0))
        lam = 5e-4 * _switch(Se, -3 * math.log10(c["deg"]), 9.0).double()
    else:
        lam = 5e-4 * _strength(M[0])
    q = torch.arange(n * n, device="cuda", dtype=torch.float64)[:, None, None]
    M = (M / (1 + lam * ((q + 1) * q) ** 2)).reshape(4, n, n, *U.shape[3:])
    return torch.where(lam > 0, torch.einsum("ka,lb,mabji->mlkji", o["V"], o["V"], M), U)


def _limit2d(o, U):
    """The limiter's density part; None where its pressure part would act."""
    I = U[..., 1:-1, 1:-1]
    mean = torch.einsum("mlkji,k,l->mji", I, o["w"] / 2, o["w"] / 2)
    ends = [torch.einsum("mlkji,%s->m%sji" % ax, I, o[e]) for ax in (("k", "l"), ("l", "k")) for e in ("ll", "lr")]
    low = torch.stack([e[0].amin(0) for e in ends] + [I[0].amin((0, 1))]).amin(0)
    if not bool((mean[0] > 0).all()) or any(not bool((_pressure(e) > 1e-12).all()) for e in ends + [I]):
        return None
    t = torch.clamp((mean[0] - 1e-13) / (mean[0] - low + 1e-8), max=1.0)
    U = U.clone()
    U[0, ..., 1:-1, 1:-1] = torch.where(t < 1, t * (I[0] - mean[0]) + mean[0], I[0])
    return U


def _inflow_left(U):
    U = U.clone()
    U[..., 0, :], U[..., -1, :] = U[..., 1, :].clone(), U[..., -2, :].clone()
    U[..., -1] = U[..., -2].clone()
    return U


def _exact2d(case, seed):
    c = _loop_case(case) if case["path"] == "loop2d" else case
    U, o, iJ = _state2d(c, seed), _devops(c["deg"]), _iJ(c)
    f = functools.partial(_rhs2d, c, o, iJ)
    if c["path"] == "rhs2d":
        return f(U)
    dt = _dt2d(c, U)
    if c["path"] == "step2d":
        for _ in range(c["steps"]):
            U = _step(f, U, dt, c["scheme"])
        return _wrap(U) if c["bc"] == "periodic" else U
    for _ in range(c["steps"]):
        U = _limit2d(o, U)
        if U is None:
            return None
        U = _inflow_left(_filter2d(c, o, _step(f, U, dt, c["scheme"])))
    return dict(state=U, filtered=None)


def _rhs1d(c, o, iJ, ends, U):
    """du of a (variables, p, cells) state; `ends` marks cells that are held (Dirichlet)."""
    if c["eq"] == "euler":
        f = _flux(U)[0] * iJ
    else:
        f = U * iJ
    k = lambda A, w: torch.einsum("mpi,p->mi", A, w)  # noqa: E731
    fL, fR, uL, uR = k(f, o["ll"]), k(f, o["lr"]), k(U, o["ll"]), k(U, o["lr"])
    if c["eq"] == "euler":
        X = _interface(c["flux"], uR.roll(1, -1), uL) * iJ
    else:
        eps = torch.full_like(uL, 1e-8)
        eps[:, 0] = 1e-6  # the wrap-around face
        a = (fL - fR.roll(1, -1)) / (uL - uR.roll(1, -1) + eps)
        X = 0.5 * (fL + fR.roll(1, -1)) - 0.5 * a.abs() * (uL - uR.roll(1, -1))
    d = torch.einsum("pq,mqi->mpi", o["dl"], f) + (X - fL)[:, None] * o["dhl"][None, :, None]
    d += (X.roll(-1, -1) - fR)[:, None] * o["dhr"][None, :, None]
    return -d if ends is None else torch.where(ends, 0.0, -d)


def _filter1d(deg, o, dt, U):
    M = torch.einsum("ap,mpi->mai", o["iV"], U)
    Se = torch.log10(M[0, -1] ** 2 / ((M[0] ** 2).sum(0) + 1e-6))
    lam = dt * math.exp(0.875 * deg) * 0.15
    q = torch.arange(deg + 1, device="cuda", dtype=torch.float64)[None, :, None]
    G = torch.einsum("pa,mai->mpi", o["V"], M / (1 + lam * ((q + 1) * q) ** 2))
    return torch.where(_switch(Se, -3 * math.log10(deg), 4.0), G, U)


def _exact1d(c, seed):
    u = _state1d(c, seed)
    U = _dev(u.reshape(u.shape + (1,) * (3 - u.ndim))).permute(2, 1, 0)
    ends = None
    if c["bc"] == "dirichlet":
        ends = torch.zeros(c["ncell"], dtype=torch.bool, device="cuda")
        ends[0] = ends[-1] = True
    f = functools.partial(_rhs1d, c, _devops(c["deg"]), 2.0 * c["ncell"], ends)
    for _ in range(c["steps"]):
        U = _step(f, U, _dt1d(c), c["scheme"])
    return U.permute(2, 1, 0).cpu().numpy().reshape(u.shape)


def _exact_ens(c, seed):
    n, d, members = _riemann(c, seed)
    done = [None] * len(members)
    dt = _ens_dt(n)
    for deg in sorted(set(d)):
        own = [b for b in range(len(members)) if d[b] == deg]  # end to end: their end cells are held
        U = _dev(np.concatenate([members[b] for b in own])).permute(2, 1, 0)
        first = np.concatenate([[0], np.cumsum(n[own])])
        ends = torch.zeros(first[-1], dtype=torch.bool, device="cuda")
        ends[first[:-1]] = True
        ends[first[1:] - 1] = True
        o = _devops(int(deg))
        f = functools.partial(_rhs1d, dict(eq="euler", flux="rusanov"), o, _dev(np.repeat(2.0 * n[own], n[own])), ends)
        for _ in range(c["steps"]):
            U = _step(f, _filter1d(int(deg), o, dt, U), dt, c["scheme"])
        U = U.permute(2, 1, 0).cpu().numpy()
        for q, b in enumerate(own):
            done[b] = U[first[q]:first[q + 1]].ravel(order="F")
    return dict(state=np.concatenate(done), filtered=None)


def _moments2d(f, u, wu, v, wv):
    fw = f * (wv[:, None] * wu[None, :])[None, :, :, None, None, None, None]
    s = fw.sum((1, 2))
    su = torch.einsum("mbalkji,a->mlkji", fw, u)
    sv = torch.einsum("mbalkji,b->mlkji", fw, v)
    e = torch.einsum("mbalkji,ba->mlkji", fw, 0.5 * (u * u + (v * v)[:, None]))
    return s, su, sv, e


def _exact_bgk2d(c, seed):
    f, o, gamma = _bgk2d_state(c, seed), _devops(c["deg"]), 2.0
    (u, wu), (v, wv) = ([_dev(q) for q in _hermite(c[k])] for k in ("nu", "nv"))
    tau = _dev(_taus(c)).reshape(-1, 1, 1, 1, 1, 1, 1)
    jx, jy = 2.0 * c["nx"], 2.0 * c["ny"]

    def rhs(f):
        s, su, sv, e = _moments2d(f, u, wu, v, wv)
        lam = 0.5 * s / (gamma - 1) / (e - 0.5 * (su * su + sv * sv) / s)
        ea = torch.exp(-lam[:, None] * (u[None, :, None, None, None, None] - (su / s)[:, None]) ** 2)
        eb = (s * lam / math.pi)[:, None] * torch.exp(-lam[:, None] * (v[None, :, None, None, None, None] - (sv / s)[:, None]) ** 2)
        r = (eb[:, :, None] * ea[:, None] - f) / tau
        for ax, (vel, j, dim) in enumerate(((u, jx, -1), (v, jy, -2))):
            shape = (1, 1, -1) if ax == 0 else (1, -1, 1)
            g = f * (vel * j).reshape(*shape, 1, 1, 1, 1)
            sub = ("mbalkji", "k", "mbalji") if ax == 0 else ("mbalkji", "l", "mbakji")
            L, R = (torch.einsum("%s,%s->%s" % sub, g, o[q]) for q in ("ll", "lr"))
            pos = (vel > 0).reshape(*shape, 1, 1, 1)
            X = torch.where(pos, R.roll(1, dim), L)  # left (bottom) face of every cell
            at = 4 if ax == 0 else 3
            r -= torch.einsum("kq,mbalqji->mbalkji" if ax == 0 else "lq,mbaqkji->mbalkji", o["dl"], g)
            w = [1] * 7
            w[at] = -1
            r -= (X - L).unsqueeze(at) * o["dhl"].reshape(w) + (X.roll(-1, dim) - R).unsqueeze(at) * o["dhr"].reshape(w)
        return r

    for _ in range(c["steps"]):
        f = _step(rhs, f, _bgk2d_dt(c), "ssprk3")
    return torch.stack([q.reshape(c["members"], -1) for q in _moments2d(f, u, wu, v, wv)], 1).cpu().numpy()


def _exact_bgk1d(c, seed):
    f0 = _bgk1d_state(c, seed)
    f, o, gamma = _dev(f0).permute(3, 2, 1, 0), _devops(c["deg"]), 3.0  # (member, point, velocity, cell)
    u, w = (_dev(q)[:, None] for q in _vgrid(c))
    tau, j = _dev(_taus(c)).reshape(-1, 1, 1, 1), 2.0 * c["nx"]

    def rhs(f):
        m = [(w * f * q).sum(2, keepdim=True) for q in (1.0, u, 0.5 * u * u)]
        U, lam = m[1] / m[0], 0.5 * m[0] / (gamma - 1) / (m[2] - 0.5 * m[1] * m[1] / m[0])
        g = f * u * j
        L, R = (torch.einsum("mkui,k->mui", g, o[q]) for q in ("ll", "lr"))
        X = torch.where(u > 0, R.roll(1, -1), L)
        d = torch.einsum("kq,mqui->mkui", o["dl"], g) + (X - L)[:, None] * o["dhl"][None, :, None, None]
        d += (X.roll(-1, -1) - R)[:, None] * o["dhr"][None, :, None, None]
        return (m[0] * torch.sqrt(lam / math.pi) * torch.exp(-lam * (u - U) ** 2) - f) / tau - d

    if c["path"] == "mol1d":
        return rhs(f).reshape(-1)
    for _ in range(c["steps"]):
        f = _step(rhs, f, _bgk1d_dt(c), c["scheme"])
    f = f.permute(3, 2, 1, 0).cpu().numpy()
    return np.asfortranarray(f if c["members"] > 1 else f[..., 0])


def exact(case, seed):
    path = case["path"]
    if path in ("rhs2d", "step2d", "loop2d"):
        return _exact2d(case, seed)
    fn = {"fr1d": _exact1d, "ens1d": _exact_ens, "bgk2d": _exact_bgk2d}.get(path, _exact_bgk1d)
    return fn(case, seed)
