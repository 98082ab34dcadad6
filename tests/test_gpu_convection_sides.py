"""The flux-based operators by side kinds, against the ordered term lists the host
builds from its interface walk (evaluated in numpy, bit for bit) and, for the
velocity field, the oracle: random graded meshes (jumps at every kind of face,
refined up to the boundary), one-level meshes, both prediction radii, zero and
negative velocities, values of both signs, and a mesh that changes between two
calls."""
import numpy as np
import pytest

import samurai_amd as sa
from oracle_lib import OracleSim
from test_ghost_flow import random_mesh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,lmin,lmax,s", [(2, 1, 2, 1), (2, 1, 5, 0), (2, 2, 6, 1), (2, 5, 5, 1), (2, 3, 7, 1), (3, 1, 3, 1), (3, 2, 4, 0),
                                             (3, 2, 5, 1), (3, 3, 3, 1)])
def test_operators_match_oracle(gpu_ctx, host_ctx, dim, lmin, lmax, s):
    mesh = None
    for seed in (1, 2):
        host = random_mesh(host_ctx, dim, lmin, lmax, s, 1, seed)
        cells = host.cells()
        print("sides", dim, lmin, lmax, s, len(cells), flush=True)
        o = OracleSim(dim, lmin, lmax, pred_s=s, cells=cells)
        o.set_poison(False)
        o.set_dirichlet(0.0)
        if mesh is None:
            mesh = sa.make_mesh_from_cells(gpu_ctx, sa.mesh_config(dim, lmin, lmax, s), cells)
            u, out = sa.make_scalar_field("u", mesh), sa.make_scalar_field("f", mesh)
            sa.make_bc_dirichlet(u, 0.0)
            parts = [sa.make_scalar_field("v%d" % d, mesh) for d in range(dim)]
            for p in parts:
                sa.make_bc_dirichlet(p, 0.0)
        else:
            mesh.assign_cells(cells)
            for f in (u, out, *parts):
                f.resize()
        rng = np.random.default_rng(seed)
        v = rng.standard_normal(len(cells))
        o.set_values(v)
        u.set_cells(v)

        def check(op, velocity):
            got = op(u, out=out).storage()
            st = u.storage()  # ghosts updated
            row, ptr, src, coef = sa.convection_terms(host, velocity)
            l, r = st[src[0::2]], st[src[1::2]]
            if velocity is None:
                term = np.where(0.5 * (l + r) >= 0, l * l, r * r) * coef
            else:
                term = np.where(src[1::2] < 0, coef * l, coef * l + coef * r)
            want, n = np.zeros(len(st)), np.diff(ptr)
            for k in range(n.max() if len(n) else 0):  # the k-th term of every row, in order
                rows = n > k
                want[row[rows]] += term[ptr[:-1][rows] + k]
            assert np.array_equal(got.view(np.uint64), want.view(np.uint64))

        for a in ([0.3, -1.1, 0.7], [-0.4, 0.0, 2.0], [0.0, 0.5, -0.1]):
            check(sa.make_convection_upwind(a[:dim]), np.array(a[:dim]))
        check(sa.make_convection_upwind(), None)
        w = [rng.standard_normal(len(cells)) for _ in range(dim)]
        for p, x in zip(parts, w):
            p.set_cells(x)
        ref = o.convection_upwind_heterogeneous([o.ghost_updated(x, 0.0) for x in w])
        got = sa.make_convection_upwind(parts)(u, out=out).storage()
        # at most 24 terms of |2^level w u| in another order: 24 additions of 24 terms
        bound = 24 * 24 * 2.0 ** -53 * 2.0 ** lmax * max(np.abs(p.storage()).max() for p in parts) * np.abs(u.storage()).max()
        known = ~np.isnan(ref)  # the oracle marks the slots no ghost update writes
        assert known.mean() > 0.99 and np.abs(got - ref)[known].max() <= bound
