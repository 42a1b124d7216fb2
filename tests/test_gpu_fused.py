"""The fused FP64 step over node blocks (the FP64 path's default, slot layout
6): bit-identical to the oracle at the edges of its blocks and chunks, with the
blocks' nodes staged in LDS and without, and on meshes whose Jacobians leave
the range of the shared-divisor quotients."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm
from tests import gpu_helpers as gh

pytestmark = pytest.mark.gpu

MESHES = {
    # nodes below, at and just above a block of 64; several blocks and chunks
    "tri_one": lambda: akm.rectangle_tri3(1, 1, 1.0, 1.0),
    "tri_64": lambda: akm.rectangle_tri3(7, 7, 1.0, 1.0),
    "tri_65": lambda: akm.rectangle_tri3(12, 4, 1.0, 1.0),
    "tri_large": lambda: akm.rectangle_tri3(211, 167, 1.3, 1.0),
    "quad": lambda: akm.rectangle_quad4(37, 23, 1.5, 1.0),
    "tet_small": lambda: akm.cube_tet4(3),
    "tet": lambda: akm.cube_tet4(9),
    "tet_large": lambda: akm.cube_tet4(22),
}


def _run(mesh, materials, elem_mat=None, steps=(1, 4), scale=1.0, keep=False, fext=False,
         launch=None):
    m = akm.Mesh(mesh.elem_type, mesh.nodes * scale, mesh.conn)
    p = gh.Pair(m, materials, elem_mat, keep_numbering=keep)
    X, rng = m.nodes, np.random.default_rng(3)
    mask = np.zeros_like(X, dtype=bool)
    mask[np.isclose(X[:, 0] / scale, 0.0)] = True
    p.block(mask)
    p.set_nodal("displacement", 1e-3 * scale * rng.normal(size=X.shape) / 30 * ~mask)
    p.set_nodal("velocity", rng.normal(size=X.shape) * ~mask)
    if fext:
        p.set_nodal("external_force", rng.normal(size=X.shape))
    p.set_time_step(0.5 * p.cpu.stable_time_step())
    if launch:
        p.gpu.set_launch(**launch)
    for n in steps:
        p.step(n)
        for name, oname in (("displacement", "u"), ("velocity", "v"), ("acceleration", "a"),
                            ("internal_force", "f_int")):
            assert np.array_equal(p.gpu.get(name), p.cpu.nodal(oname)), (name, n)
    return p


STEEL = dict(E=210e9, nu=0.3, rho=7800.0)


@pytest.mark.parametrize("name", list(MESHES))
def test_default_fp64_step_bitwise(name):
    p = _run(MESHES[name](), [STEEL], fext=name in ("tri_65", "tet"))
    assert p.gpu.query("fused_staged_lds") > 0
    assert p.gpu.query("slot_layout") == 0  # nothing was set


@pytest.mark.parametrize("name", ["tri_large", "quad", "tet"])
def test_several_materials_bitwise(name):
    m = MESHES[name]()
    mats = [STEEL, dict(E=70e9, nu=0.33, rho=2700.0), dict(E=3e9, nu=0.4, rho=1200.0)]
    _run(m, mats, np.random.default_rng(5).integers(0, 3, size=m.nb_elements))


@pytest.mark.parametrize("scale", [1e-60, 1e-8, 1e6, 1e60])
@pytest.mark.parametrize("name", ["tri_65", "quad", "tet_small"])
def test_quotients_at_extreme_scales_bitwise(name, scale):
    """Jacobians far from 1: det(J) leaves 2^+-300 at scales of 1e+-60, where
    the step divides as the compiler does."""
    _run(MESHES[name](), [STEEL], scale=scale)


def test_numbering_without_locality_bitwise():
    """A shuffled numbering, kept: every block touches most of the mesh, so it
    owns few nodes."""
    m = MESHES["tet_large"]()
    rng = np.random.default_rng(2)
    perm = rng.permutation(m.nb_nodes)
    inv = np.argsort(perm)
    shuffled = akm.Mesh(m.elem_type, m.nodes[perm],
                        inv[m.conn.astype(np.int64)][rng.permutation(m.nb_elements)])
    p = _run(shuffled, [STEEL], keep=True, steps=(2, 3))
    assert p.gpu.query("fused_blocks") > 2 * m.nb_nodes / 256


def test_node_in_thousands_of_elements_runs_on_slots():
    """A fan of 3,000 triangles about one node: no block holds its nodes."""
    t = np.linspace(0, 2 * np.pi, 3000, endpoint=False)
    X = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], axis=1)])
    i = np.arange(3000)
    fan = akm.Mesh(akx.TRIANGLE_3, X, np.stack([0 * i, 1 + i, 1 + (i + 1) % 3000], axis=1))
    p = _run(fan, [STEEL], steps=(1, 2), launch=dict(slot_layout=6))
    assert p.gpu.query("fused_available") == 1 and p.gpu.query("fused_staged_lds") == 0


def test_layout_set_and_unset_capture_apart():
    """A graph captured on the default layout is not replayed once a layout is
    set, nor the other way round; results stay the oracle's."""
    p = _run(MESHES["tet"](), [STEEL], steps=(1,))
    for k, layout in enumerate((None, 0, 6, 1)):
        if layout is not None:
            p.gpu.set_launch(slot_layout=layout)
        for n in (3, 4, 3):
            p.gpu.solve_step_graph(n, akx.FP64)
            p.cpu.solve_step(n)
            assert np.array_equal(p.gpu.get_displacement(), p.cpu.nodal("u")), (layout, n)


@pytest.mark.parametrize("name", ["tri_one", "tri_64", "tri_65", "tri_large", "quad", "tet",
                                  "tet_large", "fan"])
def test_mixed_step_staged_and_not(name):
    """The mixed fused step with its nodes staged in LDS, on several materials,
    and on a fan whose nodes no block holds.  Differences are formed in FP64
    and rounded once (2^-24): 1e-5 covers the sums over an element; the fan's
    triangles are 477 times as long as wide, and their area as much less exact."""
    fan = name == "fan"
    if fan:
        t = np.linspace(0, 2 * np.pi, 3000, endpoint=False)
        X = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], axis=1)])
        i = np.arange(3000)
        m = akm.Mesh(akx.TRIANGLE_3, X, np.stack([0 * i, 1 + i, 1 + (i + 1) % 3000], axis=1))
    else:
        m = MESHES[name]()
    mats = [STEEL, dict(E=70e9, nu=0.33, rho=2700.0), dict(E=3e9, nu=0.4, rho=1200.0)]
    rng = np.random.default_rng(5)
    p = gh.Pair(m, mats, rng.integers(0, 3, size=m.nb_elements))
    p.set_nodal("displacement", 1e-5 * rng.normal(size=m.nodes.shape))
    p.set_nodal("velocity", rng.normal(size=m.nodes.shape))
    p.set_nodal("external_force", rng.normal(size=m.nodes.shape))
    p.set_time_step(0.5 * p.cpu.stable_time_step())
    p.gpu.set_launch(slot_layout=6)
    assert p.gpu.query("fused_records") == (0 if fan else 1)
    for n in (1, 3):
        p.step(n, akx.MIXED)
        for field, oname in (("displacement", "u"), ("velocity", "v"), ("internal_force", "f_int")):
            assert gh.rel(p.gpu.get(field), p.cpu.nodal(oname)) <= 1e-5 * (477 if fan else 1), \
                (field, n)
