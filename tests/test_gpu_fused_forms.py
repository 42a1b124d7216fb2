"""The mixed fused step with its nodes staged in LDS and through element ids: the
same bits.  A mesh steps alone (staged) and beside a disjoint fan about a node in
3,000 elements, whose blocks cannot hold their nodes, so that the whole mesh runs
through element ids; the fan's elements come last, and the other nodes see the
same contributions in the same order."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm

pytestmark = pytest.mark.gpu

K = 3000


def _fan(et):
    t = np.linspace(0, 2 * np.pi, K, endpoint=False)
    ring = np.stack([np.cos(t), np.sin(t)], axis=1)
    i, j = np.arange(K), (np.arange(K) + 1) % K
    if et == akx.TRIANGLE_3:
        return np.concatenate([[[0.0, 0.0]], ring]), np.stack([0 * i, 1 + i, 1 + j], axis=1)
    if et == akx.QUADRANGLE_4:
        h = np.pi / K
        outer = 1.5 * np.stack([np.cos(t + h), np.sin(t + h)], axis=1)
        return (np.concatenate([[[0.0, 0.0]], ring, outer]),
                np.stack([0 * i, 1 + i, 1 + K + i, 1 + j], axis=1))
    ring = np.concatenate([ring, np.zeros((K, 1))], axis=1)
    return (np.concatenate([[[0.0, 0, 0], [0, 0, 1.0]], ring]),
            np.stack([0 * i, 2 + i, 2 + j, 0 * i + 1], axis=1))


MESHES = {
    "tri_one": lambda: akm.rectangle_tri3(1, 1, 1.0, 1.0),
    "tri": lambda: akm.rectangle_tri3(61, 47, 1.3, 1.0),
    "quad": lambda: akm.rectangle_quad4(37, 23, 1.5, 1.0),
    "tet_one": lambda: akm.box_tet4(1, 1, 1),
    "tet": lambda: akm.cube_tet4(9),
}


@pytest.mark.parametrize("materials", [1, 3])
@pytest.mark.parametrize("kind", [akx.ELASTIC, akx.NEOHOOKEAN])
@pytest.mark.parametrize("name", list(MESHES))
def test_staged_step_equals_element_ids(name, kind, materials):
    alone = MESHES[name]()
    X, conn = _fan(alone.elem_type)
    both = akm.Mesh(alone.elem_type, np.concatenate([alone.nodes, X + 10.0]),
                    np.concatenate([alone.conn, conn + alone.nb_nodes]))
    rng = np.random.default_rng(8)
    N, E = alone.nb_nodes, alone.nb_elements
    em = rng.integers(0, materials, size=both.nb_elements)
    em[:materials] = np.arange(materials)  # every material is used in either mesh
    u, v, f = (s * rng.normal(size=both.nodes.shape) for s in (1e-6, 1.0, 1e3))
    u[N:], v[N:] = 0.0, 0.0  # the fan's flat elements stay as they are
    out = []
    for mesh, staged in ((alone, 1), (both, 0)):
        g = akx.SolidMechanicsModel(mesh)
        for k in range(materials):
            g.add_material(kind=kind, E=1e9 * (k + 1), nu=0.3, rho=1000.0 + k)
        if materials > 1:
            g.assign_materials(em[:mesh.nb_elements])
        g.init_full()
        g.set_launch(slot_layout=6)
        assert g.query("fused_available") == 1 and g.query("fused_records") == staged
        n = mesh.nb_nodes
        g.set("displacement", u[:n])
        g.set("velocity", v[:n])
        for steps, force in ((1, False), (4, True), (3, True)):
            g.set("external_force", f[:n] * force)
            g.set_time_step(1e-6)
            g.solve_step(steps, akx.MIXED)
            out.append([g.get(k)[:N] for k in ("displacement", "velocity", "acceleration",
                                               "internal_force")])
    assert E < both.nb_elements and np.abs(out[0][3]).max() > 0
    for a, b in zip(out[:3], out[3:]):
        for x, y in zip(a, b):
            assert np.isfinite(x).all() and np.array_equal(x, y)
