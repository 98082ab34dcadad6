"""Timed workloads of the framework: what a program that uses it calls, through
its public entry points, at the sizes of its configurations and over the range
around them.

A case is a dict of plain values.  Its "kind" says what one pass does:

  demo       a short simulation from scratch: the full mesh at max_level, the
             initial field, the first adaptation, then adaptive time steps
  restart    adaptive time steps from a saved adapted mesh and its field; the
             scheme of both is upwind advection or the Burgers flux operator
  frozen     one time step on a mesh that is not adapted (update_ghost_mr,
             upwind, swap): the inner loop between two adaptations
  convection one flux-based operator (constant velocity, Burgers or a velocity
             field) on a mesh that is not adapted, as each stage of a
             multi-stage time scheme calls it
  weno5      the WENO5 operator on a mesh of one level
  batch      one adaptive step of many independent instances advanced together
  adjoint    the loss gradient through frozen steps of many instances: forward
             and backward through torch.autograd

Shapes follow the seeded fields of the benchmark: "boxes" indicator boxes and
"gauss" Gaussians in the unit box, eps 1e-4 (1e-3 in 3D), regularity 2,
Dirichlet 0, float64; "angle" is the direction of the velocity in degrees.  In
the runs that adapt, the seed places the shapes; where the mesh stays as it is,
the mesh belongs to the case and the seed scales the shapes on it.
"""
import math

import numpy as np
import torch

import samurai_amd as sa

_CTX = None


def _ctx():
    """One context per process: every object of a program lives on its stream."""
    global _CTX
    if _CTX is None:
        _CTX = sa.Context(0)
    return _CTX


# the shapes of the large 2D run, and of the 3D ones
_FLAT = {"boxes": 3, "gauss": 2, "angle": 36}
_SOLID = {"boxes": 1, "gauss": 1, "angle": 45}


def listed():
    return [
        # the smallest whole run (unit square, L2..8), ten time steps: meshes of
        # a few thousand cells, where launches and host work count
        {"name": "demo_2d_L8", "kind": "demo", "scheme": "upwind", "dim": 2, "lo": 2, "hi": 8, "s": 1, "steps": 10, **_FLAT},
        # the large 2D run (L4..12), continued for ten adaptive steps
        {"name": "restart_2d_L12", "kind": "restart", "scheme": "upwind", "dim": 2, "lo": 4, "hi": 12, "s": 1, "steps": 10, **_FLAT},
        # the 3D run (L2..8), continued for five adaptive steps
        {"name": "restart_3d_L8", "kind": "restart", "scheme": "upwind", "dim": 3, "lo": 2, "hi": 8, "s": 1, "steps": 5, **_SOLID},
        # one time step between adaptations: the smallest call
        {"name": "frozen_2d_L7", "kind": "frozen", "dim": 2, "lo": 2, "hi": 7, "s": 1, **_FLAT},
        # the same on the large 2D mesh
        {"name": "frozen_2d_L12", "kind": "frozen", "dim": 2, "lo": 4, "hi": 12, "s": 1, **_FLAT},
        # and in 3D
        {"name": "frozen_3d_L8", "kind": "frozen", "dim": 3, "lo": 2, "hi": 8, "s": 1, **_SOLID},
        # the same step on a uniform mesh of 16.8 M cells: the bandwidth-bound end
        {"name": "uniform_2d_L12", "kind": "frozen", "dim": 2, "lo": 12, "hi": 12, "s": 1, **_FLAT},
        # the linear flux-based operator on the large adapted mesh
        {"name": "convection_2d_L12", "kind": "convection", "op": "linear", "dim": 2, "lo": 4, "hi": 12, "s": 1, **_FLAT},
        # a Burgers run: the flux-based operator on a mesh that changes with every step
        {"name": "burgers_2d_L10", "kind": "restart", "scheme": "burgers", "dim": 2, "lo": 2, "hi": 10, "s": 1, "steps": 5, **_FLAT},
        # the fifth-order operator on 1024^2 cells
        {"name": "weno5_2d_L10", "kind": "weno5", "dim": 2, "lo": 10, "hi": 10, **_FLAT},
        # many uneven instances (max level 7..10) per step
        {"name": "batch_128", "kind": "batch", "n": 128, "lo": 7, "hi": 10},
        # gradients of 32 instances over 100 frozen steps, checkpoints every 10
        {"name": "adjoint_32", "kind": "adjoint", "n": 32, "hi": 10, "steps": 100, "every": 10},
    ]


def draw(rng):
    kind = rng.choice(["demo", "restart", "frozen", "frozen", "frozen", "uniform", "convection", "convection", "convection", "weno5", "weno5",
                       "batch", "adjoint"])
    if kind == "batch":
        hi = rng.randint(8, 10)
        return {"kind": "batch", "n": int(round(2 ** rng.uniform(5.5, 7))), "lo": rng.randint(6, hi - 1), "hi": hi}
    if kind == "adjoint":
        every = rng.randint(2, 12)
        return {"kind": "adjoint", "n": rng.randint(1, 32), "hi": rng.randint(6, 10), "steps": every * rng.randint(1, 6), "every": every}
    dim = rng.choice([2, 2, 3])
    boxes = rng.randint(0, 3 if dim == 2 else 2)
    shapes = {"boxes": boxes, "gauss": rng.randint(0 if boxes else 1, 3 if dim == 2 else 1), "angle": rng.randint(0, 359)}
    if kind == "weno5":
        hi = rng.randint(5, 11) if dim == 2 else rng.randint(4, 7)
        return {"kind": "weno5", "dim": dim, "lo": hi, "hi": hi, **shapes}
    if kind == "uniform":
        hi = rng.randint(6, 12) if dim == 2 else rng.randint(4, 8)
        return {"kind": "frozen", "dim": dim, "lo": hi, "hi": hi, "s": rng.choice([0, 1]), **shapes}
    case = {"kind": kind, "dim": dim, "s": rng.choice([0, 1, 1]), **shapes}
    if kind == "demo":
        case["hi"] = rng.randint(6, 10) if dim == 2 else rng.randint(4, 7)
    elif kind == "restart":
        case["hi"] = rng.randint(8, 12) if dim == 2 else rng.randint(5, 8)
    elif kind == "frozen":
        case["hi"] = rng.randint(6, 12) if dim == 2 else rng.randint(4, 8)
    else:
        case["hi"] = rng.randint(6, 12) if dim == 2 else rng.randint(4, 7)
        case["op"] = rng.choice(["linear", "burgers", "field"])
    case["lo"] = rng.randint(2, max(2, min(5, case["hi"] - 3)))
    if kind in ("demo", "restart"):
        case["steps"] = rng.randint(2, 10) if dim == 2 else rng.randint(2, 5)
        case["scheme"] = rng.choice(["upwind", "upwind", "burgers"])
        if case["scheme"] == "burgers":
            case["hi"] = min(case["hi"], 10 if dim == 2 else 7)
    return case


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
class _DeviceArray:
    """A field's storage for torch (no copy); keeps the field alive."""

    def __init__(self, field):
        self.field = field
        self.__cuda_array_interface__ = {"shape": (int(field.size()),), "typestr": "<f8", "data": (int(field.device_ptr()), False),
                                         "version": 3, "strides": None}


def _storage(field):
    return torch.as_tensor(_DeviceArray(field), device="cuda")


def _shapes(seed, dim, n_boxes, n_gauss):
    """Boxes (centre, half side) and Gaussians (centre, sigma, amplitude)."""
    r = np.random.default_rng(seed)
    lo, hi = (0.05, 0.2) if dim == 2 else (0.1, 0.2)
    boxes = [(r.uniform(0.2, 0.8, dim), 0.5 * r.uniform(lo, hi)) for _ in range(n_boxes)]
    gauss = [(r.uniform(0.2, 0.8, dim), r.uniform(0.02, 0.08), r.uniform(0.5, 1.0)) for _ in range(n_gauss)]
    return boxes, gauss


def _evaluate(axes, shapes):
    """The field at the product of the axes' coordinates (z, y, x order) as a
    sum of separable terms, on the GPU."""
    boxes, gauss = shapes
    dim = len(axes)
    out = torch.zeros([len(c) for c in reversed(axes)], dtype=torch.float64, device="cuda")
    for k, c in enumerate(list(boxes) + list(gauss)):
        f = []
        for d in range(dim):
            x = axes[d] - float(c[0][d])
            f.append((x.abs() <= c[1]).double() if k < len(boxes) else torch.exp(-x * x / (2.0 * c[1] * c[1])))
        amp = 1.0 if k < len(boxes) else float(c[2])
        term = f[1][:, None] * f[0][None, :]
        if dim == 3:
            term = f[2][:, None, None] * term[None]
        out += amp * term
    return out


def _box_values(dim, level, shapes):
    """The field on every cell of the full level, in traversal order (host)."""
    x = (torch.arange(1 << level, dtype=torch.float64, device="cuda") + 0.5) / (1 << level)
    return _evaluate([x] * dim, shapes).reshape(-1).cpu().numpy()


def _cell_values(cells, shapes, seed):
    """The shapes, each times a factor of the seed, at the centres of the cells
    (host rows of mesh.cells())."""
    scale = np.random.default_rng(seed).uniform(0.5, 1.5, len(shapes[0]) + len(shapes[1]))
    boxes, gauss = shapes
    dim = len((boxes + gauss)[0][0])
    h = np.ldexp(1.0, -cells[:, 0])
    x = [h * (cells[:, 1 + d] + 0.5) for d in range(dim)]
    u = np.zeros(len(cells))
    for k, (c, half) in enumerate(boxes):
        u += scale[k] * np.all([np.abs(x[d] - c[d]) <= half for d in range(dim)], axis=0)
    for k, (c, sigma, amp) in enumerate(gauss):
        u += scale[len(boxes) + k] * amp * np.exp(-sum((x[d] - c[d]) ** 2 for d in range(dim)) / (2.0 * sigma * sigma))
    return u


def _eps(dim):
    return 1e-4 if dim == 2 else 1e-3


def _velocity(case):
    t = math.radians(case["angle"])
    return np.array([math.cos(t), math.sin(t), math.cos(t)][: case["dim"]])


def _dt(dim, hi):
    return 0.5 * 2.0 ** -hi if dim == 2 else 0.4 * 2.0 ** -hi / 3


def _field_shapes(case, seed):
    return _shapes(seed, case["dim"], case["boxes"], case["gauss"])


def _new_field(mesh, values):
    u = sa.make_scalar_field("u", mesh)
    u.set_cells(values)
    sa.make_bc_dirichlet(u, 0.0)
    return u


#: the seed that places the shapes a case's own mesh is adapted to
_MESH_SEED = 20

#: a run's result has room for so many times the expected leaves
_ROOM = 4.0


def _adapted(case, seed):
    """A mesh adapted to the field of the seed, and the field on it."""
    dim, lo, hi = case["dim"], case["lo"], case["hi"]
    mesh = sa.make_mesh(_ctx(), sa.mesh_config(dim, lo, hi, case.get("s", 1)))
    u = _new_field(mesh, _box_values(dim, hi, _field_shapes(case, seed)))
    if lo < hi:
        sa.make_MRAdapt(u)(_eps(dim), 2.0)
    return mesh, u


def _on_its_mesh(case, seed):
    """The case's own mesh, and the seed's field on it."""
    if case["lo"] == case["hi"]:
        return _adapted(case, seed)
    mesh, u = _adapted(case, _MESH_SEED)
    u.set_cells(_cell_values(mesh.cells(), _field_shapes(case, _MESH_SEED), seed))
    return mesh, u


def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        return _prepare_batch(case, seed)
    if kind == "adjoint":
        return _prepare_adjoint(case, seed)
    dim, lo, hi = case["dim"], case["lo"], case["hi"]
    state = {"case": case, "a": _velocity(case), "dt": _dt(dim, hi), "eps": _eps(dim)}
    if kind == "demo":
        # what the program has before its run: its configuration and its initial condition
        state["config"] = sa.mesh_config(dim, lo, hi, case["s"])
        state["values"] = _box_values(dim, hi, _field_shapes(case, seed))
    elif kind == "restart":
        # what a restart file holds: the leaves and their values
        mesh, u = _adapted(case, seed)
        state["config"] = sa.mesh_config(dim, lo, hi, case["s"])
        state["cells"], state["values"] = np.ascontiguousarray(mesh.cells()[:, :4], dtype=np.int32), u.cells()
    if kind in ("demo", "restart"):
        room = int(min(_ROOM * _leaves(case), float(1 << (dim * hi))))
        state["result"] = (np.full((room, 5), -1, dtype=np.int64), np.full(room, -1.0))
    elif kind == "frozen":
        mesh, u = _on_its_mesh(case, seed)
        unp1 = sa.make_scalar_field("unp1", mesh)
        state.update(mesh=mesh, u=u, unp1=unp1, views=[_storage(u), _storage(unp1)])
    elif kind == "convection":
        mesh, u = _on_its_mesh(case, seed)
        out = sa.make_scalar_field("f", mesh)
        op = sa.make_convection_upwind(None if case["op"] == "burgers" else state["a"])
        if case["op"] == "field":  # solid rotation about the centre (and a rise in 3D)
            c = mesh.cells()
            x = (c[:, 1:4] + 0.5) * np.ldexp(1.0, -c[:, 0])[:, None]
            parts = []
            for d, v in enumerate([0.5 - x[:, 1], x[:, 0] - 0.5, x[:, 2]][:dim]):
                f = sa.make_scalar_field("v%d" % d, mesh)
                f.set_cells(v)
                sa.make_bc_dirichlet(f, 0.0)
                parts.append(f)
            op = sa.make_convection_upwind(parts)
        state.update(mesh=mesh, u=u, out=out, op=op, view=_storage(out))
    else:
        mesh = sa.make_mesh(_ctx(), sa.mesh_config(dim, lo, hi, 1, 3))
        u = _new_field(mesh, _box_values(dim, hi, _field_shapes(case, seed)))
        out = sa.make_scalar_field("f", mesh)
        state.update(mesh=mesh, u=u, out=out, op=sa.make_convection_weno5(state["a"]), view=_storage(out))
    return state


def _instance_level(k, lo, hi):
    return int(np.random.default_rng([k, 17]).integers(lo, hi + 1))


def _instance_shapes(k, seed):
    r = np.random.default_rng([k, 23])
    total = int(r.integers(1, 6))
    n_boxes = int(r.integers(0, total + 1))
    return _shapes([k, seed], 2, n_boxes, total - n_boxes)


def _instances(n, levels, seed, turn):
    """n adapted instances with a max_level in `levels` each: the seed places
    their shapes, `turn` sets their directions."""
    inst = []
    for k in range(n):
        hi = _instance_level(k, *levels)
        theta = np.random.default_rng([k, turn, 3]).uniform(0.0, 2.0 * math.pi)
        mesh = sa.make_mesh(_ctx(), sa.mesh_config(2, 2, hi, 1))
        u = _new_field(mesh, _box_values(2, hi, _instance_shapes(k, seed)))
        unp1 = sa.make_scalar_field("unp1", mesh)
        inst.append((u, unp1, np.array([math.cos(theta), math.sin(theta)]), 0.5 * 2.0 ** -hi))
    first = sa.Batch(_ctx(), inst)
    first.set_tuning(256, 0, sa.MODE_STAGES)
    first.adapt(1e-4, 2.0)
    first.close()
    return inst


def _prepare_batch(case, seed):
    inst = _instances(case["n"], (case["lo"], case["hi"]), seed, seed)
    batch = sa.Batch(_ctx(), inst)
    # the shape the autotuner settles on for this workload, without its timing runs
    batch.set_tuning(256, 0, sa.MODE_STAGES)
    # where a pass collects the fields of all instances, on the library's stream
    room = int(sum(100.0 * 2 ** u.mesh.max_level for u, _, _, _ in inst))
    return {"case": case, "inst": inst, "batch": batch, "fields": torch.zeros(room, dtype=torch.float64, device="cuda"),
            "stream": torch.cuda.ExternalStream(_ctx().stream())}


def _prepare_adjoint(case, seed):
    from samurai_amd.torch_adjoint import advect
    inst = _instances(case["n"], (case["hi"], case["hi"]), _MESH_SEED, seed)
    meshes = [u.mesh for u, _, _, _ in inst]
    n = case["n"]
    prob = sa.AdjointProblem(_ctx(), meshes, [i[3] for i in inst], bc=[0.0] * n, steps=case["steps"], checkpoint_every=case["every"])
    cells = [m.cells() for m in meshes]
    u0, target = (torch.tensor(np.concatenate([_cell_values(c, _instance_shapes(k, _MESH_SEED), [k, seed, j]) for k, c in enumerate(cells)]),
                               device="cuda") for j in (0, 1))
    area = torch.tensor(np.concatenate([np.ldexp(1.0, -2 * c[:, 0]) for c in cells]), device="cuda")
    return {"case": case, "prob": prob, "advect": advect, "u0": u0.requires_grad_(True), "area": area, "target": target,
            "a": torch.tensor(np.array([i[2] for i in inst]), requires_grad=True)}


# ---------------------------------------------------------------------------
# passes
# ---------------------------------------------------------------------------
def _time_steps(state, mesh, u, adapt_first):
    unp1 = sa.make_scalar_field("unp1", mesh)
    adapt = sa.make_MRAdapt(u)
    if adapt_first:
        adapt(state["eps"], 2.0)
    if state["case"]["scheme"] == "burgers":
        conv, f = sa.make_convection_upwind(), sa.make_scalar_field("f", mesh)
        for _ in range(state["case"]["steps"]):
            adapt(state["eps"], 2.0)
            unp1.resize()
            f.resize()
            conv(u, out=f)
            sa.sub_scaled(u, 0.15 * state["dt"], f, unp1)  # wave speeds up to 2 max|u|
            sa.swap(u, unp1)
    else:
        for _ in range(state["case"]["steps"]):
            adapt(state["eps"], 2.0)
            sa.update_ghost_mr(u)
            unp1.resize()
            sa.upwind(state["a"], state["dt"], u, unp1)
            sa.swap(u, unp1)
    # the program's result: the leaves and their values, in arrays of its own
    # (every pass on a state gives the same leaves)
    n = mesh.nb_cells()
    for of, got in zip(state["result"], (mesh.cells(), u.cells())):
        of[:n] = got
    return state["result"]


def run(state):
    kind = state["case"]["kind"]
    if kind == "demo":
        mesh = sa.make_mesh(_ctx(), state["config"])
        return _time_steps(state, mesh, _new_field(mesh, state["values"]), True)
    if kind == "restart":
        mesh = sa.make_mesh_from_cells(_ctx(), state["config"], state["cells"])
        return _time_steps(state, mesh, _new_field(mesh, state["values"]), False)
    if kind == "frozen":
        u, unp1 = state["u"], state["unp1"]
        sa.update_ghost_mr(u)
        sa.upwind(state["a"], state["dt"], u, unp1)
        sa.swap(u, unp1)
        state["views"].reverse()  # the storages were swapped
        return list(state["views"])
    if kind in ("convection", "weno5"):
        state["op"](state["u"], out=state["out"])
        return state["view"]
    if kind == "batch":
        state["batch"].step(1e-4, 2.0)
        fields = [_storage(u) for u, _, _, _ in state["inst"]]
        with torch.cuda.stream(state["stream"]):
            torch.cat(fields, out=state["fields"][: sum(f.numel() for f in fields)])
        return int(state["batch"].nb_cells()), state["fields"]
    u0, a = state["u0"], state["a"]
    u0.grad = a.grad = None
    uT = state["advect"](u0, a, state["prob"])
    loss = 0.5 * (state["area"] * (uT - state["target"]) ** 2).sum()
    loss.backward()
    return uT.detach(), u0.grad, a.grad


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: every leaf value read once and written once per step (and, where
    the mesh is adapted or rebuilt, one byte of tag per leaf and 16 bytes per
    64 cells of mesh); flops: the operator's on every leaf."""
    kind = case["kind"]
    if kind == "batch":
        n = sum(26.0 * 2 ** _instance_level(k, case["lo"], case["hi"]) for k in range(case["n"]))
        return {"bytes": 17.0 * n, "flops": 60.0 * n}
    if kind == "adjoint":
        # forward, recomputation and backward of every step
        n = 26.0 * case["n"] * 2 ** case["hi"]
        return {"bytes": 3 * 16.0 * n * case["steps"], "flops": 3 * 25.0 * n * case["steps"]}
    dim, n = case["dim"], _leaves(case)
    if kind == "weno5":
        # the flux of every interface once
        return {"bytes": 16.0 * n, "flops": 75.0 * dim * n}
    if kind == "demo":
        first = float(1 << (dim * case["hi"]))
        return {"bytes": 8.0 * first + 17.0 * n * case["steps"], "flops": 20.0 * first + 30.0 * dim * n * case["steps"]}
    if kind == "restart":
        return {"bytes": 17.0 * n * case["steps"], "flops": 30.0 * dim * n * case["steps"]}
    if kind == "convection" and case["op"] == "field":
        return {"bytes": 8.0 * (dim + 2) * n, "flops": 8.0 * dim * n}
    return {"bytes": 16.0 * n, "flops": 10.0 * dim * n}


def _leaves(case):
    """Leaves of the seeded fields' meshes, as measured: with the prediction of
    order 1 a band along the shapes' edges, of order 0 their inside as well."""
    dim, hi = case["dim"], case["hi"]
    full = float(1 << (dim * hi))
    if case["lo"] == hi:
        return full
    if case["s"] == 0:
        return (0.2 if dim == 2 else 0.045) * full
    return min(full, 38.0 * 2.0 ** hi if dim == 2 else 3.9 * 4.0 ** hi)


def tolerance(case):
    # Meshes are whole numbers: they have to be the same.  Another order of
    # the handful of terms of a cell moves its value by a unit or two in the
    # last place (1.3e-16 against exact() on uniform meshes), the divisions of
    # the WENO5 weights by up to 3e-14, the gradients' long sums by 1e-13.
    if case["kind"] == "adjoint":
        return {"rel": 1e-12, "max": 1e-10}
    if case["kind"] == "weno5":
        return {"rel": 1e-13, "max": 1e-11}
    return {"rel": 1e-15, "max": 1e-13, "differ": 0.0}


# ---------------------------------------------------------------------------
# the uniform meshes in plain torch
# ---------------------------------------------------------------------------
def exact(case, seed):
    """The operators on meshes of one level.  On adapted meshes the result is
    defined by the mesh's own projections and predictions, which the framework
    computes in 64 bits already."""
    if case["kind"] not in ("frozen", "weno5") or case["lo"] != case["hi"]:
        return None
    dim, n = case["dim"], 1 << case["hi"]
    u = torch.tensor(_box_values(dim, case["hi"], _field_shapes(case, seed)), device="cuda").reshape([n] * dim)
    a, h = _velocity(case), 1.0 / n
    if case["kind"] == "weno5":
        return None if dim == 3 and case["hi"] > 6 else _exact_weno5(u, a, h)
    # u with a layer of ghosts: Dirichlet 0 reflects the sign, corners mirror twice
    g = u
    for d in range(dim):
        first, last = g.narrow(d, 0, 1), g.narrow(d, n - 1, 1)
        g = torch.cat([-first, g, -last], d)
    new = u.clone()
    for d in range(dim):
        v, axis = float(a[d]), dim - 1 - d
        sel = g
        for o in range(dim):
            if o != axis:
                sel = sel.narrow(o, 1, n)
        left, right = sel.narrow(axis, 0, n + 1), sel.narrow(axis, 1, n + 1)
        flux = max(v, 0.0) * left + min(v, 0.0) * right
        new -= _dt(dim, case["hi"]) / h * (flux.narrow(axis, 1, n) - flux.narrow(axis, 0, n))
    out = torch.zeros([n + 2] * dim, dtype=torch.float64, device="cuda")
    out[tuple(slice(1, n + 1) for _ in range(dim))] = new
    return [out.reshape(-1), g.reshape(-1)]


def _exact_weno5(u, a, h):
    dim, n = u.dim(), u.shape[0]
    res = torch.zeros_like(u)
    for d in range(dim):
        v, axis = float(a[d]), dim - 1 - d
        w = u.movedim(axis, 0)
        # three ghost layers: Dirichlet 0, then the polynomials through the three
        # and the five values next to the layer
        low, high = [-w[0]], [-w[-1]]
        for c in ((3.0, -3.0, 1.0), (5.0, -10.0, 10.0, -5.0, 1.0)):
            kl = (low[::-1] + [w[j] for j in range(3)])[: len(c)]
            kh = (high[::-1] + [w[n - 1 - j] for j in range(3)])[: len(c)]
            low.append(sum(ck * x for ck, x in zip(c, kl)))
            high.append(sum(ck * x for ck, x in zip(c, kh)))
        e = torch.cat([torch.stack(low[::-1]), w, torch.stack(high)])
        f = v * e
        s = [f[k: k + n + 1] for k in range(6)]  # cells -2..3 about each interface
        q = s[:5] if v >= 0 else s[:0:-1]
        b = [13 / 12 * (q[0] - 2 * q[1] + q[2]) ** 2 + 0.25 * (q[0] - 4 * q[1] + 3 * q[2]) ** 2,
             13 / 12 * (q[1] - 2 * q[2] + q[3]) ** 2 + 0.25 * (q[1] - q[3]) ** 2,
             13 / 12 * (q[2] - 2 * q[3] + q[4]) ** 2 + 0.25 * (3 * q[2] - 4 * q[3] + q[4]) ** 2]
        w3 = [wk / (1e-6 + bk) ** 2 for wk, bk in zip((0.1, 0.6, 0.3), b)]
        c3 = [(2 * q[0] - 7 * q[1] + 11 * q[2]) / 6, (-q[1] + 5 * q[2] + 2 * q[3]) / 6, (2 * q[2] + 5 * q[3] - q[4]) / 6]
        flux = sum(x * y for x, y in zip(w3, c3)) / sum(w3)
        res += ((flux[1:] - flux[:-1]) / h).movedim(0, axis)
    out = torch.zeros([n + 6] * dim, dtype=torch.float64, device="cuda")
    out[tuple(slice(3, n + 3) for _ in range(dim))] = res
    return out.reshape(-1)
