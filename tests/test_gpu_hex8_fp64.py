"""The FP64 hexahedron kernel (one lane per quadrature point) at the edges of
its waves of 8 elements and blocks of 32, on every law, on element- and
node-ordered slots, and on two laws in one mesh (element lists)."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm
from tests import gpu_helpers as gh

pytestmark = pytest.mark.gpu

LAWS = {"elastic": akx.ELASTIC, "neohookean": akx.NEOHOOKEAN, "damage": akx.NEOHOOKEAN_DAMAGE}


def _material(law, m):
    mat = dict(kind=LAWS[law], E=1e7, nu=0.4, rho=1000.0)
    if law == "damage":
        mat.update(Sd=2e4, Yd=np.random.default_rng(1).uniform(10., 3e3, size=m.nb_elements * 8))
    return mat


def _check(m, materials, elem_mat=None, launch=None):
    p = gh.Pair(m, materials, elem_mat)
    X, rng = m.nodes, np.random.default_rng(7)
    p.set_nodal("displacement", 1e-2 * rng.normal(size=X.shape) * (X[1] - X[0])[0])
    p.set_nodal("velocity", rng.normal(size=X.shape))
    p.set_time_step(0.3 * p.cpu.stable_time_step())
    if launch:
        p.gpu.set_launch(**launch)
    p.step(3)
    exact = all(mt["kind"] == akx.ELASTIC for mt in materials)
    for name, oname in (("displacement", "u"), ("velocity", "v"), ("internal_force", "f_int")):
        a, b = p.gpu.get(name), p.cpu.nodal(oname)
        # the finite-strain laws' logarithm may differ in its last bit
        assert np.array_equal(a, b) if exact else gh.rel(a, b) < 1e-12, name
    return p


# 1, 7, 8, 9, 31, 32, 33 elements and a few blocks
@pytest.mark.parametrize("shape", [(1, 1, 1), (7, 1, 1), (2, 2, 2), (3, 3, 1), (31, 1, 1),
                                   (4, 4, 2), (11, 3, 1), (9, 8, 7)])
@pytest.mark.parametrize("law", list(LAWS))
def test_wave_and_block_edges(law, shape):
    m = akm.jitter_interior(akm.box_hex8(*shape), 0.02 / max(shape), 3)
    p = _check(m, [_material(law, m)])
    if law == "damage":
        d = p.cpu.field("damage").reshape(-1)
        assert d.max() > 0 and gh.rel(p.gpu.get("damage"), d) < 1e-12


@pytest.mark.parametrize("layout", [0, 1, 6])
def test_slot_layouts_and_two_laws(layout):
    m = akm.box_hex8(5, 4, 3)
    em = np.random.default_rng(2).integers(0, 2, size=m.nb_elements)
    _check(m, [_material("elastic", m), _material("neohookean", m)], em,
           dict(slot_layout=layout, element_block=64))
    _check(m, [_material("elastic", m)], None, dict(slot_layout=layout, mixed_recompute=0))
