"""A reset brings every held view up to date, whichever arrays are held, masked or not."""
import numpy as np
import pytest

from tests.parity import make_pair

pytestmark = pytest.mark.gpu

VIEWS = ("body_positions", "body_quaternions", "body_velocities", "body_angular_velocities", "body_accelerations",
         "joint_positions", "joint_velocities", "joint_forces", "observations", "contacts")


@pytest.mark.parametrize("held", [("observations",), ("body_positions", "joint_velocities"), VIEWS], ids=len)
@pytest.mark.parametrize("masked", [False, True])
def test_held_views_after_reset(held, masked):
    g, o, acts = make_pair("ant", 13, 4, seed=4)
    late, _, _ = make_pair("ant", 13, 4, seed=4)  # hands out nothing until the end
    views = {v: getattr(g, "get_" + v)(zero_copy=True) for v in held}
    mask = (np.arange(13) % 3 == 1).astype(np.uint8) if masked else None
    for k in range(4):
        if k % 2:
            g.reset(mask)
            late.reset(mask)
            o.reset(mask)
        else:
            g.step(acts[k])
            late.step(acts[k])
            o.step(acts[k])
    for v, view in views.items():
        assert view.tobytes() == getattr(late, "get_" + v)(zero_copy=False).tobytes(), v
    np.testing.assert_array_equal(g.get_contact_counts(), o.contact_counts)
    g.step(acts[0])
    o.step(acts[0])
    np.testing.assert_array_equal(g.get_body_positions().view(np.uint32), o.positions.view(np.uint32))
