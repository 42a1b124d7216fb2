"""The mixed patch kernel at the edges of its three forms: up to 255 nodes per
patch, up to 511, and the general one (more nodes, or local node and rank too
wide for one 16-bit word), with one and with two materials of a law.

Node values are rounded to FP32 relative to one node of a patch that is at
most 127 elements long here, so an element's edge carries up to 127 * 2^-24 =
8e-6 of error; 1e-4 leaves a factor for the sum over the element."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm
from tests import gpu_helpers as gh

pytestmark = pytest.mark.gpu


def _fan(n):
    t = np.linspace(0, 2 * np.pi, n, endpoint=False)
    X = np.concatenate([[[0.0, 0.0]], np.stack([np.cos(t), np.sin(t)], axis=1)])
    i = np.arange(n)
    return akm.Mesh(akx.TRIANGLE_3, X, np.stack([0 * i, 1 + i, 1 + (i + 1) % n], axis=1))


def _fan_and_one(n):
    f = _fan(n)
    one = 3.0 + np.array([[0.0, 0.0], [0.1, 0.0], [0.0, 0.1]])
    return akm.Mesh(f.elem_type, np.concatenate([f.nodes, one]),
                    np.concatenate([f.conn, [[n + 1, n + 2, n + 3]]]))


# name: mesh, nodes of the largest patch (None: not checked), packed
MESHES = {
    "tet_one": (lambda: akm.box_tet4(1, 1, 1), 8, 1),
    "tet_blocks": (lambda: akm.box_tet4(5, 5, 4), None, 1),
    "quad_254": (lambda: akm.rectangle_quad4(126, 1, 126.0, 1.0), 254, 1),
    "quad_256": (lambda: akm.rectangle_quad4(127, 1, 127.0, 1.0), 256, 1),
    "hex_510": (lambda: akm.box_hex8(84, 1, 2, 84.0, 1.0, 2.0), 510, 1),
    "hex_516": (lambda: akm.box_hex8(85, 1, 2, 85.0, 1.0, 2.0), 516, 1),
    "hex_blocks": (lambda: akm.box_hex8(13, 7, 9, 13.0, 7.0, 9.0), None, 1),
    "fan_rank_253": (lambda: _fan(254), 255, 1),
    "fan_rank_254": (lambda: _fan(255), 256, 1),
    "fan_unpacked": (lambda: _fan_and_one(255), 259, 0),
}


@pytest.mark.parametrize("materials", [1, 2])
@pytest.mark.parametrize("name", list(MESHES))
def test_patch_forms(name, materials):
    make, nodes, packed = MESHES[name]
    m = make()
    law = [dict(kind=akx.NEOHOOKEAN, E=1e7, nu=0.4, rho=1000.0),
           dict(kind=akx.NEOHOOKEAN, E=3e7, nu=0.3, rho=2000.0)][:materials]
    rng = np.random.default_rng(5)
    em = rng.integers(0, materials, size=m.nb_elements) if materials > 1 else None
    X = m.nodes[m.conn]  # the shortest edge: nothing turns inside out
    h = min(np.linalg.norm(X[:, a] - X[:, b], axis=1).min() for a in range(1, X.shape[1])
            for b in range(a))
    u, v = 0.02 * h * rng.normal(size=m.nodes.shape), rng.normal(size=m.nodes.shape)
    out = {}
    for layout in (4, 5):  # the general form, and what the mixed path runs
        p = gh.Pair(m, law, em)
        p.set_nodal("displacement", u)
        p.set_nodal("velocity", v)
        p.set_time_step(0.2 * p.cpu.stable_time_step())
        p.gpu.set_launch(slot_layout=layout)
        p.step(3, akx.MIXED)
        out[layout] = [p.gpu.get(f) for f in ("displacement", "velocity", "internal_force")]
        assert p.gpu.query("patch_available") == 1
        assert p.gpu.query("patch_packed") == packed
        if nodes is not None:
            assert p.gpu.query("patch_max_nodes") == nodes
        for g, o in zip(out[layout], ("u", "v", "f_int")):
            assert gh.rel(g, p.cpu.nodal(o)) <= 1e-4, (layout, o)
    # the same FP32 partials in another place
    for a, b in zip(out[4], out[5]):
        assert gh.rel(a, b) <= 1e-6
