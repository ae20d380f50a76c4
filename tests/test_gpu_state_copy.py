"""The device copies of a 2D state between the reference layout and the padded one: every value at
its place, at row lengths around the 64-element pieces and the 512-element runs a wavefront takes."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,deg", [(1, 1, 1), (5, 3, 5), (61, 2, 2), (62, 7, 1), (63, 4, 3), (126, 5, 1), (510, 3, 1),
                                       (511, 2, 1), (1023, 2, 2)])
def test_state_device_round_trip(nx, ny, deg):
    import frhip

    s = frhip.FREuler2D(frhip.FRPSpace2D(0.0, 1.0, nx, 0.0, 1.0, ny, deg, 1, 1))
    s.use_torch_stream()
    u = torch.arange(s.len, dtype=torch.float64, device="cuda")
    s.set_state(u)
    out = torch.full_like(u, -1.0)
    assert frhip.lib().fr2d_get_state_dev(s.h, out.data_ptr()) == 0
    assert torch.equal(out, u)
    assert np.array_equal(s.get_state().ravel(order="F"), u.cpu().numpy())
    s.set_state(s.get_state() + 1.0)
    assert frhip.lib().fr2d_get_state_dev(s.h, out.data_ptr()) == 0
    assert torch.equal(out, u + 1.0)
    s.close()


# rows of 3 to 33 values: 16, 8, 4 and 2 of them side by side in a wavefront, and the first that has one to
# itself; row counts that end inside a group
@pytest.mark.parametrize("nx,ny,deg", [(1, 77, 1), (2, 1, 1), (3, 130, 2), (6, 41, 1), (7, 9, 3), (14, 33, 2), (15, 5, 1),
                                       (30, 18, 1), (31, 6, 2), (1, 3000, 5)])
def test_narrow_state_device_round_trip(nx, ny, deg):
    test_state_device_round_trip(nx, ny, deg)
