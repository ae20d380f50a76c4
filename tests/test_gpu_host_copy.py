"""Host states large enough for the pinned chunks (whole chunks, a remainder, one value over) come back
from the device as they went in, and again after a step count of zero."""
import numpy as np
import pytest

import frhip

pytestmark = pytest.mark.gpu

CHUNK, FROM = 2 << 20, 24 << 20


@pytest.mark.parametrize("nbytes", [FROM - 8, FROM, FROM + 8, FROM + CHUNK - 8, 13 * CHUNK + 24, 17 * CHUNK])
def test_large_host_state_round_trip(nbytes):
    # advection cells of degree 1: two values per cell, and one member of an odd count where needed
    ncell = -(-nbytes // 16)
    pr = frhip.FRAdvectionProblem(frhip.FRPSpace1D(0.0, 1.0, ncell, 1), 1.0, "period")
    u = np.asfortranarray(np.random.default_rng(nbytes).standard_normal((ncell, 2)))
    assert u.nbytes - nbytes in (0, 8)
    for _ in range(2):
        pr.set_state(u)
        assert np.array_equal(pr.get_state(), u)
        u = -u[::-1]


@pytest.mark.parametrize("stream", ["own", "null", "per_thread", "torch"])
def test_large_host_state_behind_queued_steps(stream):
    """Steps are queued and not waited for: a state read back holds them, a state put in comes after them
    (hipStreamPerThread is handle 2, another stream in every thread)."""
    import ctypes as C

    torch = pytest.importorskip("torch")
    ncell = FROM // 16 + 3 * CHUNK // 16 + 5
    pr = frhip.FRAdvectionProblem(frhip.FRPSpace1D(0.0, 1.0, ncell, 1), 1.0, "period")
    u = np.asfortranarray(np.random.default_rng(0).standard_normal((ncell, 2)))
    steps = (0.1 / ncell, 400, "ssprk3")
    pr.set_state(u)
    pr.step(*steps)
    torch.cuda.synchronize()
    ref = pr.get_state()
    side = torch.cuda.Stream()
    if stream != "own":
        handle = {"null": 0, "per_thread": 2, "torch": side.cuda_stream}[stream]
        assert frhip.lib().fr1d_set_stream(pr.h, C.c_void_p(handle)) == 0
    for _ in range(2):
        pr.set_state(u)
        pr.step(*steps)
        assert np.array_equal(pr.get_state(), ref)
        pr.step(*steps)
        pr.set_state(u)
        torch.cuda.synchronize()
        pr.step(0.1 / ncell, 0)
        assert np.array_equal(pr.get_state(), u)
    pr.close()


def test_large_pinned_state_round_trip():
    import ctypes as C

    torch = pytest.importorskip("torch")
    ncell = FROM // 16 + 77
    pr = frhip.FRAdvectionProblem(frhip.FRPSpace1D(0.0, 1.0, ncell, 1), 1.0, "period")
    u = torch.empty(2 * ncell, dtype=torch.float64, pin_memory=True)
    out = torch.zeros(2 * ncell, dtype=torch.float64, pin_memory=True)
    u.copy_(torch.from_numpy(np.random.default_rng(1).standard_normal(2 * ncell)))
    ptr = lambda t: C.cast(t.data_ptr(), C.POINTER(C.c_double))  # noqa: E731
    assert frhip.lib().fr1d_set_state(pr.h, ptr(u)) == 0
    assert frhip.lib().fr1d_get_state(pr.h, ptr(out)) == 0
    assert torch.equal(out, u)
    assert np.array_equal(pr.get_state().ravel(order="F"), u.numpy())
    pr.close()
