"""What a step runs with after the launch shape is set, queried or tuned."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm
from tests import gpu_helpers as gh

pytestmark = pytest.mark.gpu

STEEL = dict(E=210e9, nu=0.3, rho=7800.0)


def _pair(mesh, law=STEEL):
    p = gh.Pair(mesh, [law])
    p.set_nodal("velocity", np.random.default_rng(3).normal(size=mesh.nodes.shape))
    p.set_time_step(0.5 * p.cpu.stable_time_step())
    return p


@pytest.mark.parametrize("make,fp64", [(lambda: akm.rectangle_tri3(20, 11, 1.0, 1.0), 6),
                                       (lambda: akm.cube_tet4(4), 6),
                                       (lambda: akm.cube_hex8(3), 1)])
def test_tuning_one_path_leaves_the_fp64_layout(make, fp64):
    """The FP64 path keeps its default layout while the mixed path is tuned,
    and its own choice afterwards; its steps stay the oracle's."""
    p = _pair(make())
    q = p.gpu.query
    assert q("slot_layout_fp64") == fp64 and q("slot_layout_mixed") == 0
    shape, _ = p.gpu.autotune(akx.MIXED, 2)
    assert q("slot_layout_fp64") == fp64
    assert q("slot_layout") == shape["slot_layout"]
    for n in (1, 4):
        p.gpu.solve_step_graph(n, akx.FP64)
        p.cpu.solve_step(n)
        assert np.array_equal(p.gpu.get_displacement(), p.cpu.nodal("u"))
    own, _ = p.gpu.autotune(akx.FP64, 2)
    assert q("slot_layout") == own["slot_layout"] == q("slot_layout_fp64")
    p.gpu.autotune(akx.MIXED, 2)
    assert q("slot_layout_fp64") == own["slot_layout"]
    p.step(3)
    assert np.array_equal(p.gpu.get_displacement(), p.cpu.nodal("u"))


@pytest.mark.parametrize("layout", range(7))
def test_queried_layout_is_the_one_that_runs(layout):
    """A layout set holds for both paths, where it applies."""
    tet, hex8 = _pair(akm.cube_tet4(4)).gpu, _pair(akm.cube_hex8(3)).gpu
    for g in (tet, hex8):
        g.set_launch(slot_layout=layout)
        assert g.query("slot_layout") == layout
    assert tet.query("slot_layout_fp64") == (6 if layout == 6 else min(layout, 1))
    assert tet.query("slot_layout_mixed") == layout
    assert hex8.query("slot_layout_fp64") == min(layout, 1)
    assert hex8.query("slot_layout_mixed") == min(layout, 5)
