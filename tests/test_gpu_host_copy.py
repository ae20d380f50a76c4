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
