"""The flux-based operators where they run on term lists (meshes that are not
graduated or do not tile the box), against the host's lists evaluated in numpy,
bit for bit: jumps of several levels, a missing leaf, and a leaf missing while
another is covered twice (the volume of the box all the same).  One mesh object
takes them in turn, so lists kept from the mesh before would show."""
import numpy as np
import pytest

import samurai_amd as sa
from oracle_lib import OracleSim
from test_ghost_flow import random_mesh
from test_ghost_holes import holed

pytestmark = pytest.mark.gpu


def jumps(dim, lmax, seed):
    """Leaves of a tree refined at random, not graduated."""
    rng = np.random.default_rng(seed)
    todo, leaves = [(0, 0, 0, 0)], []
    while todo:
        l, x, y, z = todo.pop()
        if l < 2 or (l < lmax and rng.random() < 0.35):
            todo += [(l + 1, 2 * x + (k & 1), 2 * y + ((k >> 1) & 1), 2 * z + (k >> 2)) for k in range(1 << dim)]
        else:
            leaves.append((l, x, y, z))
    return np.array(leaves)


def twice(host_ctx, dim, lmax, s, seed):
    """A leaf missing at a level, another one of it under its own children."""
    base = random_mesh(host_ctx, dim, 2, lmax, s, 1, seed).cells()[:, :4]
    at = np.flatnonzero(base[:, 0] == lmax - 1)
    over = base[at[0]]
    kids = np.array([[lmax, 2 * over[1] + (k & 1), 2 * over[2] + ((k >> 1) & 1), 2 * over[3] + (k >> 2)] for k in range(1 << dim)])
    return np.concatenate([np.delete(base, at[len(at) // 2], 0), kids])


@pytest.mark.parametrize("dim,lmax,s", [(2, 6, 0), (2, 5, 1), (3, 4, 0), (3, 4, 1)])
def test_operators_match_the_lists(gpu_ctx, host_ctx, dim, lmax, s):
    cfg = sa.mesh_config(dim, 2, lmax, s)
    mesh = None
    for kind in ("hole", "jumps", "twice", "hole again"):
        if kind == "jumps" and (dim, s) == (2, 1):
            continue  # predictions of radius 1 reach past the ghosts of such meshes
        cells = jumps(dim, lmax, 3) if kind == "jumps" else (twice(host_ctx, dim, lmax, s, 2) if kind == "twice" else holed(host_ctx, dim, 2, lmax, s, len(kind)))
        print("terms", dim, lmax, s, kind, len(cells), flush=True)
        host = sa.make_mesh_from_cells(host_ctx, cfg, cells)
        assert host.validate() == 0 and host.ghost_form() == (1 if kind == "jumps" else 0)
        if mesh is None:
            mesh = sa.make_mesh_from_cells(gpu_ctx, cfg, cells)
            fields = [sa.make_scalar_field("f%d" % k, mesh) for k in range(3 + dim)]
            for f in fields:
                sa.make_bc_dirichlet(f, 0.25)
        else:
            mesh.assign_cells(cells)
            for f in fields:
                f.resize()
        rng = np.random.default_rng(lmax)
        u, w, out, vel = fields[0], fields[1], fields[2], fields[3:]
        for f in fields:
            f.set_storage(rng.standard_normal(f.size()))

        def want(f, velocity):
            st = f.storage()  # ghosts updated
            row, ptr, src, coef = sa.convection_terms(host, velocity)
            l, r = st[src[0::2]], st[src[1::2]]
            if velocity is None:
                term = np.where(0.5 * (l + r) >= 0, l * l, r * r) * coef
            else:
                term = np.where(src[1::2] < 0, coef * l, coef * l + coef * r)
            total, n = np.zeros(len(st)), np.diff(ptr)
            for k in range(n.max()):  # the k-th term of every row, in order
                rows = n > k
                total[row[rows]] += term[ptr[:-1][rows] + k]
            return total

        # the velocity changes and comes back, on two fields
        for f, a in ((u, [0.3, -1.1, 0.7]), (w, [0.3, -1.1, 0.7]), (u, [-0.4, 0.0, 2.0]), (u, [0.3, -1.1, 0.7])):
            got = sa.make_convection_upwind(a[:dim])(f, out=out).storage()
            assert np.array_equal(got, want(f, np.array(a[:dim]))), kind
        for f in (u, w):
            assert np.array_equal(sa.make_convection_upwind()(f, out=out).storage(), want(f, None)), kind
        # the velocity field against the oracle, every slot known to both at first
        values = [rng.standard_normal(len(cells)) for _ in range(dim + 1)]
        for f, x in zip([u] + vel, values):
            st = np.zeros(f.size())
            st[mesh.cells()[:, 4]] = x
            f.set_storage(st)
        o = OracleSim(dim, 2, lmax, pred_s=s, cells=cells)
        o.set_poison(False)
        o.set_dirichlet(0.25)
        o.set_values(values[0])
        ref = o.convection_upwind_heterogeneous([o.ghost_updated(x, 0.25) for x in values[1:]])
        got = sa.make_convection_upwind(vel)(u, out=out).storage()
        # at most 24 terms of |2^level w u| in another order: 24 additions of 24 terms
        bound = 24 * 24 * 2.0 ** -53 * 2.0 ** lmax * max(np.abs(p.storage()).max() for p in vel) * np.abs(u.storage()).max()
        known = ~np.isnan(ref)  # the oracle marks the slots no ghost update writes
        assert known.mean() > 0.95 and np.abs(got - ref)[known].max() <= bound, kind
