"""FEEngine operators on element lists longer than one launch has threads (2^24):
every thread goes on with a stride."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm

pytestmark = pytest.mark.gpu

COUNT = 2 ** 22 + 777  # quadrangles of four points each


def test_lists_longer_than_a_launch():
    m = akm.rectangle_quad4(3, 2, 1.0, 1.0)
    model = akx.SolidMechanicsModel(m)
    model.add_material(E=1.0, nu=0.3, rho=1.0)
    model.init_full()
    fe = model.get_fe_engine()
    rng = np.random.default_rng(3)
    u = rng.normal(size=(m.nb_nodes, 1))
    D = rng.normal(size=(m.nb_elements * 4, 2))
    E = m.nb_elements
    ids = (np.arange(COUNT) % E).astype(np.uint32)
    whole, rest = COUNT // E, COUNT % E

    def rows(few):  # the six elements' rows over and over
        r = few.reshape(E, -1)
        return np.concatenate([np.tile(r, (whole, 1)), r[:rest]]).reshape(-1, few.shape[1])

    for op, operand in ((fe.gradient_on_integration_points, u),
                        (fe.interpolate_on_integration_points, u)):
        assert np.array_equal(op(operand, elements=ids), rows(op(operand)))
    assert np.array_equal(fe.compute_btd(rows(D), ids), rows(fe.compute_btd(D)))
    b = D[:, :1].copy()
    assert np.array_equal(fe.compute_ntb(rows(b), ids), rows(fe.compute_ntb(b)))
