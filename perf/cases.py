"""Workloads of the explicit-dynamics engine as a user's program runs them: the
time step on every element type, law and precision, from a bar of 4,000
triangles to a cube of 6 M tetrahedra; the energies, stable time step and
output a driver asks for between steps; the FEEngine operators on a caller's
fields; the constitutive surrogate inside the step, evaluated on its own,
differentiated and trained.

    listed()             the fixed cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  inputs and the model a program keeps
    run(state)           one pass, through akantu_amd.akx
    work(case)           bytes and operations a pass cannot do without
    exact(case, seed)    the pass's results in 64 bits, by plain torch

The FP64 cases run as the plain drivers do, on the default launch shape; the
mixed cases on the shape the autotuner settles on for that kind of mesh (per
patch partial sums, or the fused step for triangles), set by hand so that
every run takes the same one.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

from akantu_amd import akx
from akantu_amd import mesh as akm

ELASTIC = dict(E=210e9, nu=0.3, rho=7800.0)
NEOHOOKEAN = dict(E=10e6, nu=0.45, rho=1000.0)
DAMAGE = dict(E=1e9, nu=0.3, rho=1200.0)
DAMAGE_SD, STRAIN_LIMIT = 5e6, 0.05  # Marigo slope, the surrogate's envelope
LAWS = {"elastic": (akx.ELASTIC, ELASTIC), "neohookean": (akx.NEOHOOKEAN, NEOHOOKEAN),
        "damage": (akx.NEOHOOKEAN_DAMAGE, DAMAGE)}
LAYERS = [(7, 128), (128, 128), (128, 128), (128, 128), (128, 7)]
NPARAM = sum(i * o + o for i, o in LAYERS)
ACT_K = 0.1666259765625  # slope of the network's smoothstep (the FP16 value next to 1/6)


# ----------------------------------------------------------------------------
# the cases
# ----------------------------------------------------------------------------
def _step(mesh, nx, ny, nz, law, precision, steps, per_call=0, graph=False, layout=-1,
          fext=False, moving=False, network=False):
    return dict(kind="step", mesh=mesh, nx=nx, ny=ny, nz=nz, law=law, precision=precision,
                steps=steps, per_call=per_call or steps, graph=graph, layout=layout, fext=fext,
                moving=moving, network=network)


def listed():
    return [
        # a small 2D bar stepped one solveStep() at a time, as the reference's
        # explicit driver loop does: launches and latency
        dict(_step("bar", 100, 20, 0, "elastic", "fp64", 40, per_call=1), name="bar_fp64"),
        # the bit-exact path on a 3D solid of ordinary size
        dict(_step("cube", 60, 60, 60, "elastic", "fp64", 20), name="cube_fp64"),
        # the large workload: 6 M tetrahedra, mixed precision
        dict(_step("cube", 100, 100, 100, "elastic", "mixed", 20, layout=5), name="cube_mixed"),
        # finite-strain hexahedra driven by a moving boundary, both precisions
        dict(_step("box", 64, 64, 64, "neohookean", "mixed", 40, layout=5, moving=True),
             name="hex8_neohookean_mixed"),
        dict(_step("box", 40, 41, 39, "neohookean", "fp64", 10, moving=True),
             name="hex8_neohookean_fp64"),
        # many independent specimens advanced together by one graph launch
        dict(_step("ensemble", 128, 0, 0, "elastic", "mixed", 50, graph=True, layout=6),
             name="ensemble_mixed"),
        # the notched plate with damage: the plain law, and its network
        dict(_step("plate", 81, 80, 16, "damage", "mixed", 40, layout=5, moving=True),
             name="plate_damage_mixed"),
        dict(_step("plate", 81, 80, 16, "damage", "mixed", 10, layout=5, moving=True,
                   network=True), name="plate_network_mixed"),
        # a few Adam iterations on the GPU's own training set
        dict(kind="train", paths=4000, path_steps=250, iterations=20, batch=8192,
             name="network_train"),
        # the network on a caller's points, and a batch's gradient
        dict(kind="network", points=200003, batch=8192, bf16=False, name="network_infer_gradient"),
        # what a driver asks for between steps: energies, stable step, dump
        dict(kind="output", mesh="cube", nx=40, ny=41, nz=39, law="elastic", dumps=True,
             name="energies_and_dump"),
        # FEEngine operators on a caller's fields
        dict(kind="operators", mesh="box", nx=31, ny=30, nz=29, part=1.0,
             name="operators_hex8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _sizes(rng, mesh, lo, hi):
    """nx, ny, nz of a mesh of about lo to hi elements (log-uniform), sides
    within about a factor two of each other."""
    E = _log(rng, lo, hi)
    if mesh in ("bar", "plane"):
        cells = E / (2 if mesh == "bar" else 1)
        nx = max(2, int(math.sqrt(cells * rng.uniform(0.5, 5))))
        return nx, max(2, int(cells / nx)), 0
    cells = E / (1 if mesh == "box" else 6)
    if mesh == "plate":
        n = max(8, int((cells * 5) ** (1 / 3)))
        return n, max(8, int(n * rng.uniform(0.8, 1.2))), max(2, n // 5)
    n = cells ** (1 / 3)
    nx, ny = (max(2, int(n * rng.uniform(0.7, 1.4))) for _ in range(2))
    return nx, ny, max(2, int(cells / (nx * ny)))


def draw(rng):
    kind = rng.choice(["step"] * 8 + ["network", "train", "output", "operators"])
    if kind == "train":
        return dict(kind="train", paths=_log(rng, 500, 4000), path_steps=rng.randint(100, 250),
                    iterations=rng.randint(5, 30), batch=256 * _log(rng, 4, 48))
    if kind == "network":
        return dict(kind="network", points=_log(rng, 1000, 400000), batch=256 * _log(rng, 1, 64),
                    bf16=rng.random() < 0.3)
    if kind == "output":
        mesh = rng.choice(["bar", "plane", "cube", "box"])
        nx, ny, nz = _sizes(rng, mesh, 2000, 100000 if mesh == "box" else 500000)
        return dict(kind="output", mesh=mesh, nx=nx, ny=ny, nz=nz,
                    law=rng.choice(["elastic", "neohookean", "damage"]), dumps=rng.random() < 0.7)
    if kind == "operators":
        mesh = rng.choice(["bar", "plane", "cube", "box"])
        nx, ny, nz = _sizes(rng, mesh, 2000, 40000 if mesh == "box" else 150000)
        return dict(kind="operators", mesh=mesh, nx=nx, ny=ny, nz=nz,
                    part=rng.choice([1.0, 0.5]))
    precision = rng.choice(["fp64", "mixed"])
    mesh = rng.choice(["bar", "plane", "cube", "cube", "box", "plate", "ensemble"])
    if mesh == "ensemble":
        nx, ny, nz = _log(rng, 8, 128), 0, 0
    else:
        nx, ny, nz = _sizes(rng, mesh, 2000, 200000 if mesh == "box" else 1500000)
    law = {"ensemble": "elastic", "plate": "damage"}.get(mesh) or rng.choice(
        ["elastic", "elastic", "neohookean"] + (["damage"] if mesh == "box" else []))
    layout = -1
    if precision == "mixed":
        layout = rng.choice([5, 5, 6] if mesh in ("bar", "ensemble") else [5])
    steps = rng.randint(5, 30)
    return _step(mesh, nx, ny, nz, law, precision, steps,
                 per_call=rng.choice([steps, steps, 1]), graph=rng.random() < 0.3, layout=layout,
                 fext=mesh != "ensemble" and rng.random() < 0.3,
                 moving=mesh != "ensemble" and rng.random() < 0.4,
                 network=mesh == "plate" and precision == "mixed" and rng.random() < 0.3)


# ----------------------------------------------------------------------------
# inputs
# ----------------------------------------------------------------------------
def _mesh(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    kind = case["mesh"]
    if kind == "bar":
        return akm.rectangle_tri3(nx, ny, 1.0, ny / nx)
    if kind == "plane":
        return akm.rectangle_quad4(nx, ny, 1.0, ny / nx)
    if kind == "cube":
        m = akm.box_tet4(nx, ny, nz, 1.0, ny / nx, nz / nx)
        return akm.jitter_interior(m, 0.01 / nx, seed)
    if kind == "box":
        m = akm.box_hex8(nx, ny, nz, 1.0, ny / nx, nz / nx)
        return akm.jitter_interior(m, 0.01 / nx, seed)
    return akm.notched_plate_tet4(nx, ny, nz, 0.1, 0.1 * ny / nx, 0.1 * nz / nx)


def _smooth(X, rng, strain):
    """A smooth displacement of about the given strain: three waves along the
    body with wave lengths of a half to twice its longest side."""
    L = float((X.max(axis=0) - X.min(axis=0)).max())
    out = np.zeros_like(X)
    for _ in range(3):
        k = rng.normal(size=X.shape[1])
        k *= 2 * np.pi / (L * rng.uniform(0.5, 2.0)) / np.linalg.norm(k)
        amp = rng.normal(size=X.shape[1])
        amp *= strain / 3 / np.linalg.norm(amp) / np.linalg.norm(k)
        out += np.sin(X @ k + rng.uniform(0, 2 * np.pi))[:, None] * amp
    return out


def _thresholds(count, rng):
    return 1e6 * rng.weibull(5.0, size=count)


def _inputs(case, seed):
    """Mesh, fields, boundary and law parameters of a model, from the seed."""
    rng = np.random.default_rng(seed)
    if case["mesh"] == "ensemble":
        # the specimens' sizes belong to the case, their materials to the seed
        ens = akm.concatenate_specimens(akm.ensemble_tri3(case["nx"]))
        par = np.array([[s.E, s.nu, s.rho] for s in ens.specimens])
        par[:, 0] *= rng.uniform(0.8, 1.25, size=len(par))
        u = _smooth(ens.mesh.nodes, rng, 1e-4)
        u[ens.blocked] = 0.0
        return dict(mesh=ens.mesh, material=ens.element_material, parameters=par,
                    specimen=ens.node_specimen(), blocked=ens.blocked, u=u, v=ens.velocity,
                    top=None, axis=0, speed=0.0, fext=None, Yd=None)
    m = _mesh(case, seed)
    X, law = m.nodes, case["law"]
    par = LAWS[law][1]
    axis = 1 if case["mesh"] == "plate" else m.dim - 1
    blocked = np.zeros_like(X, dtype=bool)
    blocked[np.isclose(X[:, axis], X[:, axis].min())] = True
    strain = {"elastic": 1e-3, "neohookean": 1e-2, "damage": 3e-2}[law]
    u = _smooth(X, rng, strain)
    v = _smooth(X, rng, strain) * math.sqrt(par["E"] / par["rho"]) * 4
    u[blocked] = v[blocked] = 0.0
    top = None
    if case.get("moving"):
        top = np.nonzero(np.isclose(X[:, axis], X[:, axis].max()))[0]
        v[top, axis] = 0.0
    fext = None
    if case.get("fext"):
        fext = rng.normal(size=X.shape) * 1e-6 * par["E"] / m.nb_nodes ** ((m.dim - 1) / m.dim)
    return dict(mesh=m, material=None, parameters=np.array([[par["E"], par["nu"], par["rho"]]]),
                specimen=None, blocked=blocked, u=u, v=v, top=top, axis=axis,
                speed=0.5 if case["mesh"] != "plate" else 20.0, fext=fext,
                Yd=_thresholds(m.nb_elements * m.nb_qp, rng) if law == "damage" else None)


def _parameters(seed):
    """A network of the surrogate's size with outputs of the size of a trained
    one: weights uniform with unit gain, a small last layer."""
    rng = np.random.default_rng(seed + 77)
    out = []
    for k, (i, o) in enumerate(LAYERS):
        a = math.sqrt(3.0 / i) * (0.02 if k == 4 else 1.0)
        out += [rng.uniform(-a, a, size=o * i), rng.uniform(-0.05, 0.05, size=o) * (k < 4)]
    return np.concatenate(out).astype(np.float32)


class _DeviceArray:
    def __init__(self, address, shape):
        self.__cuda_array_interface__ = dict(shape=shape, typestr="<f8", data=(address, False),
                                             version=2)


def _view(model, name):
    """The model's nodal field in place, in its own node numbering."""
    p = ctypes.c_void_p()
    model.ctx.check(akx.lib.akx_field_device_pointer(model.ctx.h, akx.FIELDS[name],
                                                     ctypes.byref(p)))
    return torch.as_tensor(_DeviceArray(p.value, (model.mesh.nb_nodes, model.dim)),
                           device="cuda")


class _Pinned:
    """Page-locked host memory for an asynchronous download, as a tensor (which
    keeps the memory alive for whoever holds the result)."""

    def __init__(self, shape, dtype):
        self.tensor = torch.empty(shape, dtype=torch.from_numpy(np.empty(0, dtype)).dtype,
                                  pin_memory=True)
        self.ptr = ctypes.c_void_p(self.tensor.data_ptr())
        self.nbytes = self.tensor.numel() * self.tensor.element_size()


def _numbering(model):
    """caller -> internal node numbers, and the same for the fields' entries."""
    perm = np.zeros(model.mesh.nb_nodes, dtype=np.int64)
    model.ctx.check(akx.lib.akx_node_numbering(model.ctx.h,
                                               perm.ctypes.data_as(ctypes.c_void_p)))
    inv = np.empty_like(perm)
    inv[perm] = np.arange(perm.size)
    inv = torch.from_numpy(inv).cuda()
    return inv, inv[:, None] * model.dim + torch.arange(model.dim, device="cuda")


def _model(case, inp):
    m = inp["mesh"]
    model = akx.SolidMechanicsModel(m)
    kind = LAWS[case["law"]][0]
    for E, nu, rho in inp["parameters"]:
        model.add_material(kind=kind, E=E, nu=nu, rho=rho, Sd=DAMAGE_SD, Yd=inp["Yd"])
    if inp["material"] is not None:
        model.assign_materials(inp["material"])
    model.init_full()
    model.set("blocked_dofs", inp["blocked"])
    if inp["specimen"] is not None:
        dt = model.get_stable_time_step_per_material()
        model.set_node_time_steps(0.8 * dt[inp["specimen"]])
        model.set_time_step(0.8 * float(dt.min()))
    else:
        dt = 0.8 * model.get_stable_time_step()
        model.set_time_step(dt)
        if inp["top"] is not None:
            model.set_dirichlet_increment(inp["top"], inp["axis"], inp["speed"] * dt)
    if inp["fext"] is not None:
        model.set("external_force", inp["fext"])
    return model


# ----------------------------------------------------------------------------
# prepare / run
# ----------------------------------------------------------------------------
def prepare(case, seed):
    return _KINDS[case["kind"]][0](case, seed)


def run(state):
    return _KINDS[state["case"]["kind"]][1](state)


def _prepare_step(case, seed):
    inp = _inputs(case, seed)
    model = _model(case, inp)
    if case["layout"] >= 0:
        model.set_launch(256, 256, 1, 1, case["layout"], 0)
    inv, entries = _numbering(model)
    start = {}
    for name, f in (("displacement", inp["u"]), ("velocity", inp["v"])):
        start[name] = torch.empty_like(_view(model, name))
        start[name][inv] = torch.from_numpy(np.ascontiguousarray(f)).cuda()
    state = dict(case=case, model=model, entries=entries, start=start, damage=None,
                 fields={n: _view(model, n) for n in ("displacement", "velocity", "acceleration")})
    if inp["Yd"] is not None:
        state["damage"] = _Pinned(*model.field_layout("damage"))
    if case["network"]:
        model.surrogate_setup(0, STRAIN_LIMIT)
        model.surrogate_params(_parameters(seed))
        model.surrogate_enable(True)
    return state


def _run_step(state):
    case, model, f = state["case"], state["model"], state["fields"]
    # a run starts from its own initial fields (a parameter study restarts)
    f["displacement"].copy_(state["start"]["displacement"])
    f["velocity"].copy_(state["start"]["velocity"])
    f["acceleration"].zero_()
    precision = akx.FP64 if case["precision"] == "fp64" else akx.MIXED
    step = model.solve_step_graph if case["graph"] else model.solve_step
    for _ in range(case["steps"] // case["per_call"]):
        step(case["per_call"], precision)
    out = {n: t.take(state["entries"]) for n, t in f.items()}
    if state["damage"] is not None:
        model.wait(model.get_async("damage", state["damage"]))
        out["damage"] = state["damage"].tensor
    return out


def _network_model():
    m = akm.box_tet4(2, 2, 2)
    model = akx.SolidMechanicsModel(m)
    model.add_material(kind=akx.NEOHOOKEAN_DAMAGE, Sd=DAMAGE_SD, Yd=np.full(m.nb_elements, 1e6),
                       **DAMAGE)
    model.init_full()
    model.surrogate_setup(0, STRAIN_LIMIT)
    return model


def _prepare_train(case, seed):
    model = _network_model()
    model.surrogate_generate(case["paths"], case["path_steps"], seed=seed)
    model.surrogate_params(_parameters(seed))
    return dict(case=case, model=model, seed=seed)


def _run_train(state):
    case, model = state["case"], state["model"]
    loss = model.surrogate_train(case["iterations"], batch=case["batch"], lr=2e-3,
                                 seed=state["seed"])
    return dict(loss=loss, parameters=model.surrogate_params())


def _samples(case, seed):
    rng = np.random.default_rng(seed)
    x, xb = (np.concatenate([rng.uniform(-1, 1, size=(n, 6)) * rng.uniform(0.02, 1, size=(n, 1)),
                             rng.uniform(0, 0.5, size=(n, 1))], axis=1).astype(np.float32)
             for n in (case["points"], case["batch"]))
    # targets of the size of the law's remainder: quadratic in the strain
    t = np.concatenate([0.5 * xb[:, :6] ** 2 - 0.2 * xb[:, [1]] * xb[:, [0]],
                        0.1 * xb[:, [0]] ** 3], axis=1).astype(np.float32)
    return x, xb, t


def _prepare_network(case, seed):
    model = _network_model()
    if case["bf16"]:
        model.surrogate_format("bf16")
    model.surrogate_params(_parameters(seed))
    x, xb, t = _samples(case, seed)
    return dict(case=case, model=model, x=x, xb=xb, t=t)


def _run_network(state):
    y = state["model"].surrogate_infer(state["x"])
    gradient, loss = state["model"].surrogate_gradients(state["xb"], state["t"])
    return dict(outputs=y, gradient=gradient, loss=loss)


def _prepare_output(case, seed):
    inp = _inputs(dict(case, fext=True), seed)
    model = _model(case, inp)
    model.set("external_force", inp["fext"])
    model.set("displacement", inp["u"])
    model.set("velocity", inp["v"])
    model.assemble_internal_forces(akx.FP64)
    buffers = {}
    if case["dumps"]:
        for name in ("displacement", "velocity", "stress"):
            buffers[name] = _Pinned(*model.field_layout(name))
    return dict(case=case, model=model, buffers=buffers)


def _run_output(state):
    model = state["model"]
    tickets = [model.get_async(name, b) for name, b in state["buffers"].items()]
    out = {k.replace(" ", "_"): model.get_energy(k)
           for k in ("kinetic", "potential", "external work")}
    out["stable_time_step"] = model.get_stable_time_step()
    for t in tickets:
        model.wait(t)
    out.update({name: b.tensor for name, b in state["buffers"].items()})
    return out


def _operands(case, seed, m):
    rng = np.random.default_rng(seed + 5)
    E, Q, d = m.nb_elements, m.nb_qp, m.dim
    ids = None
    if case["part"] < 1.0:
        ids = np.sort(rng.choice(E, size=int(E * case["part"]), replace=False)).astype(np.uint32)
    rows = (E if ids is None else ids.size) * Q
    return dict(ids=ids, u=_smooth(m.nodes, rng, 1e-2), D=rng.normal(size=(rows, d * d)),
                f=rng.normal(size=(rows, d)), s=rng.normal(size=rows),
                field=rng.uniform(0.5, 2.0, size=(E * Q, 2)))


def _prepare_operators(case, seed):
    m = _mesh(case, seed)
    model = akx.SolidMechanicsModel(m)
    model.add_material(kind=akx.ELASTIC, **ELASTIC)
    model.init_full()
    return dict(case=case, model=model, engine=model.get_fe_engine(), op=_operands(case, seed, m))


def _run_operators(state):
    fe, op = state["engine"], state["op"]
    ids = op["ids"]
    return dict(gradient=fe.gradient_on_integration_points(op["u"], elements=ids),
                values=fe.interpolate_on_integration_points(op["u"], elements=ids),
                btd=fe.compute_btd(op["D"], elements=ids),
                integral=fe.integrate(op["f"], elements=ids),
                total=fe.integrate_scalar(op["s"], elements=ids),
                lumped=fe.assemble_field_lumped(op["field"]))


# ----------------------------------------------------------------------------
# bytes and operations
# ----------------------------------------------------------------------------
def _counts(case):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["mesh"] == "ensemble":
        E = nx * 21000  # specimens of 2,000 to 40,000 elements
        return E, E * 0.52, 3, 1, 2
    if case["mesh"] == "bar":
        return 2 * nx * ny, (nx + 1) * (ny + 1), 3, 1, 2
    if case["mesh"] == "plane":
        return nx * ny, (nx + 1) * (ny + 1), 4, 4, 2
    N = (nx + 1) * (ny + 1) * (nz + 1)
    return (nx * ny * nz, N, 8, 8, 3) if case["mesh"] == "box" else (6 * nx * ny * nz, N, 4, 1, 3)


def work(case):
    net = 2.0 * sum(i * o for i, o in LAYERS)
    if case["kind"] == "train":
        return dict(bytes=case["iterations"] * (case["batch"] * 56.0 + NPARAM * 24.0),
                    flops=case["iterations"] * case["batch"] * 3 * net)
    if case["kind"] == "network":
        return dict(bytes=case["points"] * 56.0 + case["batch"] * 56.0 + NPARAM * 8.0,
                    flops=case["points"] * net + case["batch"] * 3 * net)
    E, N, n, Q, d = _counts(case)
    point = 2.0 * d * d * n * 3 + 4 * n * d + 60  # Jacobian, gradient, forces; inverse and law
    if case["kind"] == "operators":
        rows = E * Q * case["part"]
        per_row = d * d * 2 + 2 * d + 1 + d * n  # gradient, D, values, f, s, btd
        return dict(bytes=8.0 * (rows * per_row + 2 * N * d + rows / Q * d + E * Q * 2 + 4 * N)
                    + 4.0 * E * n, flops=rows * 2.0 * d * d * n * 2)
    if case["kind"] == "output":
        nbytes = 4.0 * E * n + 8.0 * N * (d * 5 + 1) + N * d
        if case["dumps"]:
            nbytes += 8.0 * (E * Q * d * d + 2 * N * d)
        return dict(bytes=nbytes, flops=E * Q * point * 2)
    # one step: connectivity, coordinates, u (and v, a or the previous u), mass
    # and flags; the damage and its threshold per point
    nodal = (2 + (3 if case["precision"] == "mixed" else 6)) * d * 8.0 + 8 + d
    per_step = 4.0 * E * n + N * nodal + (E * Q * 24.0 if case["law"] == "damage" else 0)
    flops = E * Q * (point + (net if case["network"] else 0))
    return dict(bytes=per_step * case["steps"], flops=flops * case["steps"])


# ----------------------------------------------------------------------------
# the same results in 64 bits
# ----------------------------------------------------------------------------
def exact(case, seed):
    if case["kind"] == "train":
        return None  # a path of many BF16 roundings
    return _KINDS[case["kind"]][2](case, seed)


def _corners(n, d):
    if n == 2 ** d and d == 2:
        return np.array([[-1, -1], [1, -1], [1, 1], [-1, 1]], dtype=float)
    return np.array([[-1, -1, -1], [1, -1, -1], [1, 1, -1], [-1, 1, -1],
                     [-1, -1, 1], [1, -1, 1], [1, 1, 1], [-1, 1, 1]], dtype=float)


def _reference_element(n, d):
    """Quadrature points: N (Q, n), dN/dxi (Q, n, d), weights (Q,)."""
    if n == d + 1:
        dn = np.concatenate([-np.ones((1, d)), np.eye(d)])
        return np.full((1, n), 1.0 / n), dn[None], np.array([1.0 / math.factorial(d)])
    c, Q, g = _corners(n, d), 2 ** d, 1 / math.sqrt(3)
    xi = np.array([[g if q >> k & 1 else -g for k in range(d)] for q in range(Q)])
    f = 0.5 * (1 + xi[:, None, :] * c[None])  # (Q, n, d)
    N = f.prod(axis=2)
    dn = np.stack([0.5 * c[None, :, k] * np.delete(f, k, axis=2).prod(axis=2) for k in range(d)],
                  axis=2)
    return N, dn, np.ones(Q)


class _Solid:
    """Gradients, forces, masses and energies of a mesh in torch float64."""

    def __init__(self, m):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.X = torch.from_numpy(np.ascontiguousarray(m.nodes)).to(dev)
        self.conn = torch.from_numpy(m.conn.astype(np.int64)).to(dev)
        self.E, self.n = self.conn.shape
        self.d = self.X.shape[1]
        N, dn, w = (torch.from_numpy(a).to(dev) for a in _reference_element(self.n, self.d))
        self.N, self.Q = N, N.shape[0]
        xe = self.X[self.conn]  # (E, n, d)
        self.B, self.J = [], []
        for q in range(self.Q):
            F = self._product(xe.transpose(1, 2), dn[q])  # dx_i / dxi_k
            self.J.append(torch.linalg.det(F) * w[q])
            self.B.append(self._product(dn[q].expand(self.E, -1, -1), torch.linalg.inv(F)))

    @staticmethod
    def _product(a, b):
        """Small matrix products, summed term by term."""
        return (a.unsqueeze(-1) * b.unsqueeze(-3)).sum(-2)

    def gradient(self, u, q):
        """du_i / dX_j, (E, i, j)."""
        return self._product(u[self.conn].transpose(1, 2).contiguous(), self.B[q])

    def scatter(self, values):  # (E, n, ...) -> (N, ...)
        out = torch.zeros((self.X.shape[0],) + values.shape[2:], dtype=values.dtype,
                          device=values.device)
        return out.index_add_(0, self.conn.reshape(-1), values.reshape((-1,) + values.shape[2:]))

    def lumped(self, field):  # (E, Q, k)
        return self.scatter(sum(field[:, q, None, :] * (self.J[q][:, None] * self.N[q])[..., None]
                                for q in range(self.Q)))


class _Body:
    """The explicit step of one case in float64."""

    def __init__(self, case, inp, network=None):
        self.case, self.inp, self.net = case, inp, network
        self.S = S = _Solid(inp["mesh"])
        dev = S.X.device
        par = inp["parameters"]
        lam, mu = par[:, 1] * par[:, 0] / ((1 + par[:, 1]) * (1 - 2 * par[:, 1])), \
            par[:, 0] / (2 * (1 + par[:, 1]))
        em = inp["material"] if inp["material"] is not None else np.zeros(S.E, dtype=np.int64)
        self.lam, self.mu, self.rho = (torch.from_numpy(np.ascontiguousarray(a[em])).to(dev)
                                       for a in (lam, mu, par[:, 2]))
        self.mass = S.lumped(self.rho[:, None, None].expand(-1, S.Q, 1))[:, 0]
        t = {k: torch.from_numpy(np.ascontiguousarray(inp[k])).to(dev)
             for k in ("u", "v", "blocked")}
        self.u, self.v, self.free = t["u"].clone(), t["v"].clone(), ~t["blocked"]
        self.moved = torch.zeros_like(self.u)
        self.a = torch.zeros_like(self.u)
        self.fext = torch.zeros_like(self.u) if inp["fext"] is None else \
            torch.from_numpy(inp["fext"]).to(dev)
        self.damage = None
        if inp["Yd"] is not None:
            self.Yd = torch.from_numpy(inp["Yd"]).to(dev).reshape(S.E, S.Q)
            self.damage = torch.zeros_like(self.Yd)
        self.dt = self._time_step()
        if inp["top"] is not None:
            top = torch.from_numpy(inp["top"]).to(dev)
            self.moved[top, inp["axis"]] = inp["speed"] * float(self.dt)
            self.free[top, inp["axis"]] = False

    def stable(self):
        """Stable step per element: inscribed size over the wave speed."""
        S = self.S
        x = (S.X + self.u)[S.conn] if self.case["kind"] == "output" else S.X[S.conn]

        def dist(a, b):
            return (x[:, a] - x[:, b]).norm(dim=1)

        def area(a, b, c):
            p = (dist(a, b) + dist(b, c) + dist(a, c)) / 2
            return (p * (p - dist(a, b)) * (p - dist(b, c)) * (p - dist(a, c))).sqrt(), p
        if S.n == 3:
            A, p = area(0, 1, 2)
            h = 2 * A / p
        elif S.n == 4 and S.d == 3:
            faces = sum(area(*f)[0] for f in ((0, 1, 2), (0, 1, 3), (0, 2, 3), (1, 2, 3)))
            vol = torch.linalg.det(x[:, 1:] - x[:, :1]).abs() / 6
            h = 6 * vol / faces
        else:
            edges = [(0, 1), (1, 2), (2, 3), (3, 0)]
            if S.n == 8:
                edges += [(a, a + 4) for a in range(4)] + [(a + 4, b + 4) for a, b in edges]
            h = torch.stack([dist(*e) for e in edges]).min(dim=0).values
        return h / ((self.lam + 2 * self.mu) / self.rho).sqrt()

    def _time_step(self):
        dt = self.stable()
        if self.inp["specimen"] is None:
            return 0.8 * dt.min()
        em = torch.from_numpy(self.inp["material"].astype(np.int64)).to(dt.device)
        best = torch.full((len(self.inp["parameters"]),), math.inf, dtype=dt.dtype,
                          device=dt.device)
        best.scatter_reduce_(0, em, dt, "amin")
        return (0.8 * best)[torch.from_numpy(self.inp["specimen"]).to(dt.device)][:, None]

    def law(self, G):
        """Second Piola-Kirchhoff (small strain: Cauchy) stress and energy."""
        eye = torch.eye(self.S.d, dtype=G.dtype, device=G.device)
        lam, mu = self.lam[:, None, None], self.mu[:, None, None]
        if self.case["law"] == "elastic":
            eps = (G + G.transpose(1, 2)) / 2
            S = lam * eps.diagonal(dim1=1, dim2=2).sum(1)[:, None, None] * eye + 2 * mu * eps
            return S, 0.5 * (S * eps).sum((1, 2))
        F = G + eye
        C = self.S._product(F.transpose(1, 2), F)
        lnJ = torch.linalg.det(F).log()
        Ci = torch.linalg.inv(C)
        S = mu * (eye - Ci) + lam * lnJ[:, None, None] * Ci
        W = 0.5 * self.lam * lnJ ** 2 + self.mu * (
            -lnJ + 0.5 * (C.diagonal(dim1=1, dim2=2).sum(1) - self.S.d))
        return S, W

    def network(self, G, q):
        """The law's stress and energy with the network's remainder."""
        Eg = 0.5 * (G + G.transpose(1, 2) + self.S._product(G.transpose(1, 2), G))
        Ev = torch.stack([Eg[:, i, j] for i, j in ((0, 0), (1, 1), (2, 2), (1, 2), (0, 2),
                                                   (0, 1))], dim=1)
        lam, mu = self.lam, self.mu
        tr = Ev[:, :3].sum(1)
        y = _evaluate(self.net, torch.cat([Ev / STRAIN_LIMIT, self.damage[:, q, None]], dim=1))
        size = (lam + 2 * mu) * STRAIN_LIMIT ** 2
        Sv = 2 * mu[:, None] * Ev + size[:, None] * y[:, :6]
        Sv[:, :3] += (lam * tr)[:, None]
        S = torch.stack([Sv[:, k] for k in (0, 5, 4, 5, 1, 3, 4, 3, 2)], dim=1).reshape(-1, 3, 3)
        W = 0.5 * lam * tr ** 2 + mu * (Eg * Eg).sum((1, 2)) + size * STRAIN_LIMIT * y[:, 6]
        plain, Wp = self.law(G)
        inside = (Ev.abs() <= STRAIN_LIMIT).all(1)
        return torch.where(inside[:, None, None], S, plain), torch.where(inside, W, Wp)

    def forces(self):
        S, out = self.S, 0
        for q in range(S.Q):
            G = S.gradient(self.u, q)
            P, W = self.network(G, q) if self.net is not None else self.law(G)
            if self.damage is not None:
                d = self.damage[:, q]
                d = torch.where(W - self.Yd[:, q] - DAMAGE_SD * d > 0,
                                (W - self.Yd[:, q]) / DAMAGE_SD, d).clamp(max=1.0)
                self.damage[:, q] = d
                P = (1 - d)[:, None, None] * P
            if self.case["law"] != "elastic":
                P = P + S._product(G, P)
            out = out - S._product(S.B[q], P.transpose(1, 2)) * S.J[q][:, None, None]
        return S.scatter(out)

    def step(self):
        free, dt = self.free, self.dt
        self.u += self.moved
        self.u += torch.where(free, dt * self.v + 0.5 * dt * dt * self.a, 0.0)
        self.v += torch.where(free, dt * self.a, 0.0)
        delta = (self.fext + self.forces() - self.mass[:, None] * self.a) / self.mass[:, None]
        self.v += torch.where(free, 0.5 * dt * delta, 0.0)
        self.a += torch.where(free, delta, 0.0)


def _evaluate(layers, x):
    h = x
    for k, (W, b) in enumerate(layers):
        h = h @ W.T + b
        if k < 4:
            t = (ACT_K * h + 0.5).clamp(0, 1)
            h = h * (t * t * (3 - 2 * t))
    return h


def _layers(seed, device):
    p = torch.from_numpy(_parameters(seed).astype(np.float64)).to(device)
    out, at = [], 0
    for i, o in LAYERS:
        out.append((p[at:at + i * o].reshape(o, i), p[at + i * o:at + i * o + o]))
        at += i * o + o
    return out


def _exact_step(case, seed):
    inp = _inputs(case, seed)
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    body = _Body(case, inp, _layers(seed, dev) if case["network"] else None)
    for _ in range(case["steps"]):
        body.step()
    out = dict(displacement=body.u, velocity=body.v, acceleration=body.a)
    if body.damage is not None:
        out["damage"] = body.damage.reshape(-1)
    return out


def _exact_network(case, seed):
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    x, xb, t = (torch.from_numpy(a.astype(np.float64)).to(dev) for a in _samples(case, seed))
    layers = [(W.clone().requires_grad_(), b.clone().requires_grad_())
              for W, b in _layers(seed, dev)]
    with torch.no_grad():
        y = torch.cat([_evaluate(layers, c) for c in x.split(100000)])
    loss = ((_evaluate(layers, xb) - t) ** 2).mean()
    loss.backward()
    return dict(outputs=y, gradient=torch.cat([g.grad.reshape(-1) for l in layers for g in l]),
                loss=float(loss))


def _exact_output(case, seed):
    inp = _inputs(dict(case, fext=True), seed)
    body = _Body(case, inp)
    S = body.S
    out = dict(kinetic=float((body.mass[:, None] * body.v ** 2).sum() / 2))
    stress, potential = [], 0.0
    for q in range(S.Q):
        P, W = body.law(S.gradient(body.u, q))
        potential += float((W * S.J[q]).sum())
        stress.append(P.transpose(1, 2).reshape(S.E, 1, -1))
    out["potential"] = potential
    fixed = ~body.free
    dt0 = float(_Body(dict(case, kind="step"), inp).dt)
    power = torch.where(fixed, -body.forces() * body.v, body.fext * body.v).sum()
    out["external_work"] = float(power) * dt0
    out["stable_time_step"] = float(body.stable().min())
    if case["dumps"]:
        out["displacement"], out["velocity"] = body.u, body.v
        # the output of a damage law is its current, undamaged state's stress
        out["stress"] = None if case["law"] == "damage" else \
            torch.cat(stress, dim=1).reshape(S.E * S.Q, -1)
    if case["law"] == "damage":
        # the assembly of prepare() has advanced the damage
        out["potential"] = None
    return out


def _exact_operators(case, seed):
    m = _mesh(case, seed)
    op, S = _operands(case, seed, m), _Solid(m)
    dev = S.X.device
    ids = torch.arange(S.E, device=dev) if op["ids"] is None else \
        torch.from_numpy(op["ids"].astype(np.int64)).to(dev)
    t = {k: torch.from_numpy(np.ascontiguousarray(op[k])).to(dev)
         for k in ("u", "D", "f", "s", "field")}
    d, Q, R = S.d, S.Q, ids.numel()
    D, f = t["D"].reshape(R, Q, d, d).transpose(2, 3), t["f"].reshape(R, Q, d)
    J = torch.stack(S.J, dim=1)[ids]
    grad = torch.stack([S.gradient(t["u"], q)[ids] for q in range(Q)], dim=1)
    btd = torch.stack([S._product(D[:, q], S.B[q][ids].transpose(1, 2)) for q in range(Q)], dim=1)
    ue = t["u"][S.conn[ids]]
    values = torch.stack([(ue * S.N[q][None, :, None]).sum(1) for q in range(Q)], dim=1)
    return dict(gradient=grad.transpose(2, 3).reshape(R * Q, d * d),
                values=values.reshape(R * Q, d),
                btd=btd.transpose(2, 3).reshape(R * Q, -1),
                integral=(f * J[..., None]).sum(1),
                total=float((t["s"].reshape(R, Q) * J).sum()),
                lumped=S.lumped(t["field"].reshape(S.E, Q, 2)))


_KINDS = {"step": (_prepare_step, _run_step, _exact_step),
          "train": (_prepare_train, _run_train, None),
          "network": (_prepare_network, _run_network, _exact_network),
          "output": (_prepare_output, _run_output, _exact_output),
          "operators": (_prepare_operators, _run_operators, _exact_operators)}
