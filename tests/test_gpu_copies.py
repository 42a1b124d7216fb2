"""Copies between a caller's arrays and the device through the page-locked
slots: sizes at the edges of a slot and of two (1, 2 MB) and of the one- and
four-thread copies (8 MB), renumbered and not."""
import numpy as np
import pytest

from akantu_amd import akx
from akantu_amd import mesh as akm

pytestmark = pytest.mark.gpu


# nodes of 16 bytes each: 1 MB, a little more, 2 MB, more, 8 MB, more
@pytest.mark.parametrize("grid", [(2, 2), (256, 256), (257, 256), (512, 256), (513, 257),
                                  (1024, 512), (1025, 513)])
@pytest.mark.parametrize("keep", [False, True])
def test_nodal_fields_round_trip(grid, keep):
    m = akm.rectangle_quad4(grid[0] - 1, grid[1] - 1, 1.0, 1.0)
    model = akx.SolidMechanicsModel(m, keep_numbering=keep)
    model.add_material(E=210e9, nu=0.3, rho=7800.0)
    model.init_full()
    rng = np.random.default_rng(grid[0])
    u, v = rng.normal(size=(2, m.nb_nodes, 2))
    model.set("displacement", u)
    model.set("velocity", v)
    assert np.array_equal(model.get("displacement"), u)
    assert np.array_equal(model.get("velocity"), v)
    assert np.array_equal(model.get("current_position"), m.nodes + u)
    # the mass of a regular grid: one value per node, reported per component
    mass = model.get("mass")
    assert np.array_equal(mass[:, 0], mass[:, 1])
    assert mass[:, 0].sum() == pytest.approx(7800.0, rel=1e-12)


@pytest.mark.parametrize("n", [1, 37449, 37450, 74899, 299594, 299595])
def test_network_outputs_do_not_depend_on_the_copy(n):
    """28 bytes per point: 37,449.1 points per MB."""
    m = akm.box_tet4(1, 1, 1)
    model = akx.SolidMechanicsModel(m)
    model.add_material(kind=akx.NEOHOOKEAN_DAMAGE, E=1e9, nu=0.3, rho=1200.0, Sd=5e6,
                       Yd=np.full(m.nb_elements, 1e6))
    model.init_full()
    model.surrogate_setup(0, 0.05)
    x = np.random.default_rng(4).uniform(-1, 1, size=(n, 7)).astype(np.float32)
    y = model.surrogate_infer(x)
    parts = [model.surrogate_infer(x[k:k + 30000]) for k in range(0, n, 30000)]
    assert np.array_equal(y, np.concatenate(parts))


def _plate(keep):
    """1.07 million quadrangles of four points."""
    m = akm.rectangle_quad4(1050, 1020, 1.0, 1.0)
    model = akx.SolidMechanicsModel(m, keep_numbering=keep)
    model.add_material(E=210e9, nu=0.3, rho=7800.0)
    model.init_full()
    return m, model


def test_renumbered_copies_in_pieces():
    """Fields of more than 128 MiB go to and from the caller's numbering in
    pieces: the same values as without renumbering, and no more than a piece of
    device memory beside the field."""
    rng = np.random.default_rng(6)
    out = []
    u = a = f = None
    for keep in (True, False):
        m, model = _plate(keep)
        fe = model.get_fe_engine()
        if u is None:
            u = rng.normal(size=(m.nb_nodes, 2))
            a = rng.normal(size=(m.nb_nodes, 2))
            f = rng.normal(size=(m.nb_elements * 4, 4))  # 137 MB
        model.set("displacement", u)
        stress = model.get("stress")                     # 137 MB
        assert model.query("scratch_bytes") <= 128 << 20
        out.append((stress, fe.interpolate_on_integration_points(a, 2),
                    fe.assemble_field_lumped(f, np.tile(a, 2))))
        del model, fe
    for x, y in zip(*out):
        assert np.array_equal(x, y)


def test_scratch_kept_between_calls_is_bounded():
    """Operand and result of 229 MiB each, then a result of 131 MiB in a third
    buffer: a context keeps 512 MiB in all, nothing above 256 MiB."""
    m, model = _plate(True)
    fe = model.get_fe_engine()
    f = np.ones((m.nb_elements * 4, 7))
    per_point = fe.integrate_on_integration_points(f, 7)
    assert per_point[:, 0].sum() == pytest.approx(1.0, rel=1e-9)
    assert model.query("scratch_bytes") >= 2 * f.nbytes
    u = np.random.default_rng(7).normal(size=(m.nb_nodes, 2))
    ids = np.arange(m.nb_elements, dtype=np.uint32)[::-1].copy()
    g = fe.gradient_on_integration_points(u, 2, ids)
    assert model.query("scratch_bytes") <= 512 << 20
    first = fe.compute_btd(g)                       # 274 MB of results
    assert model.query("scratch_bytes") <= 512 << 20
    assert np.array_equal(fe.compute_btd(g[:4000], np.arange(1000)), first[:4000])


@pytest.mark.parametrize("kb", [1, 17, 126, 131, 520, 1020, 1030, 2600])
@pytest.mark.parametrize("keep", [False, True])
def test_successive_copies_share_the_slots(kb, keep):
    """Operands and results around the sizes where the copies change (128 KiB:
    host renumbering and uploads without an event, 1 MiB: one slot), several in
    a row without a wait of the caller's own."""
    n = max(2, int(round((kb * 1024 / 16) ** 0.5)))
    m = akm.rectangle_quad4(n - 1, n - 1, 1.0, 1.0)
    model = akx.SolidMechanicsModel(m, keep_numbering=keep)
    model.add_material(E=210e9, nu=0.3, rho=7800.0)
    model.init_full()
    fe = model.get_fe_engine()
    rng = np.random.default_rng(n)
    u, v = rng.normal(size=(2, m.nb_nodes, 2))
    blocked = rng.random(m.nodes.shape) < 0.3
    for k in range(3):
        model.set("displacement", u + k)
        model.set("velocity", v - k)
        model.set("blocked_dofs", np.roll(blocked, k))
        ids = rng.permutation(m.nb_elements).astype(np.uint32)
        g = fe.gradient_on_integration_points(u + k, 2, ids)
        assert np.array_equal(model.get("displacement"), u + k)
        assert np.array_equal(model.get("velocity"), v - k)
        assert np.array_equal(model.get("current_position"), m.nodes + (u + k))
        assert np.array_equal(model.get("blocked_dofs"), np.roll(blocked, k))
        whole = fe.gradient_on_integration_points(u + k, 2)
        rows = (ids[:, None].astype(np.int64) * 4 + np.arange(4)).reshape(-1)
        assert np.array_equal(g, whole[rows])
        mass = model.get("mass")
        assert np.array_equal(mass[:, 0], mass[:, 1]) and mass.min() > 0
