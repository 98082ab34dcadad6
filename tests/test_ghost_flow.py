"""The dataflow form of update_ghost_mr: its recipes against the staged ones on
the host, and the launch against the oracle on the GPU."""
import numpy as np
import pytest

import samurai_amd as sa
from oracle_lib import OracleSim

# smallest meshes, both prediction radii, several levels, 3D, wide ghost layers
MESHES = [(2, 1, 2, 1, 1), (2, 1, 4, 0, 1), (2, 2, 6, 1, 1), (2, 3, 7, 1, 1), (3, 1, 3, 1, 1), (3, 2, 4, 0, 1), (3, 2, 5, 1, 1), (2, 4, 4, 1, 3),
          (3, 3, 3, 1, 2)]


def random_mesh(ctx, dim, lmin, lmax, s, r, seed):
    """A graded mesh with random refinement up to the boundary, and its cells."""
    m = sa.make_mesh(ctx, sa.mesh_config(dim, lmin, lmax, s, r))
    rng = np.random.default_rng(seed)
    for _ in range(lmax - lmin):
        cells, tags = m.cells(), np.zeros(m.nb_cells(sa.REFERENCE), dtype=np.uint8)
        keys = np.column_stack([cells[:, 0], cells[:, 1:4] // 2])
        _, group, size = np.unique(keys, axis=0, return_inverse=True, return_counts=True)
        coarsen = (rng.random(len(size)) < 0.7) & (size == 1 << dim)  # whole sibling groups
        tags[cells[:, 4]] = np.where(coarsen[group.ravel()], sa.COARSEN, sa.KEEP)
        m.rebuild_from_tags(tags)
    return m


@pytest.mark.parametrize("dim,lmin,lmax,s,r", MESHES)
def test_recipe_flow_is_the_staged_recipes(host_ctx, dim, lmin, lmax, s, r):
    for seed in range(3):
        assert random_mesh(host_ctx, dim, lmin, lmax, s, r, seed).validate() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dim,lmin,lmax,s,r", MESHES)
def test_ghosts_with_any_value_match_oracle(gpu_ctx, host_ctx, dim, lmin, lmax, s, r):
    """Several updates in a row, with infinities, NaN and the bits the launch
    marks its ghosts with among the cells: every slot as the oracle's, bit for
    bit where it is a number."""
    cells = random_mesh(host_ctx, dim, lmin, lmax, s, r, 5).cells()
    o = OracleSim(dim, lmin, lmax, pred_s=s, radius=r, cells=cells)
    o.set_poison(False)
    o.set_dirichlet(0.75)
    mesh = sa.make_mesh_from_cells(gpu_ctx, sa.mesh_config(dim, lmin, lmax, s, r), cells)
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.75)
    rng = np.random.default_rng(8)
    for step in range(4):
        print("ghosts", dim, lmin, lmax, s, r, "step", step, flush=True)
        v = rng.standard_normal(len(cells))
        if step >= 2:
            v[rng.integers(0, len(v), 3)] = [np.inf, -np.inf, np.nan]
        if step == 3:
            v[0] = np.array([0x7FF05A3C96E1D2B4], dtype=np.uint64).view(np.float64)[0]
        st = np.zeros(u.size())
        st[cells[:, 4]] = v
        o.set_storage(st)
        u.set_storage(st)
        o.update_ghost_mr()
        sa.update_ghost_mr(u)
        a, b = o.storage(), u.storage()
        assert np.array_equal(np.isnan(a), np.isnan(b))
        k = ~np.isnan(a)
        assert np.array_equal(a[k].view(np.uint64), b[k].view(np.uint64))
