"""The dataflow form of update_ghost_mr: its recipes against the staged ones on
the host, and both forms against the oracle on the GPU (left to itself an update
takes the cheaper one, which for most of these meshes is the staged one)."""
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


@pytest.mark.parametrize("dim,lmin,lmax,s,r", MESHES)
def test_flow_exists(host_ctx, dim, lmin, lmax, s, r):
    for seed in range(3):
        assert random_mesh(host_ctx, dim, lmin, lmax, s, r, seed).ghost_form() == 1


@pytest.fixture
def form_ctx(gpu_ctx):
    yield gpu_ctx
    gpu_ctx.set_ghost_form(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("form", [0, 1])
@pytest.mark.parametrize("dim,lmin,lmax,s,r", MESHES)
def test_both_forms_match_oracle(form_ctx, host_ctx, dim, lmin, lmax, s, r, form):
    """Every mesh in either form, every slot, from storages of old values."""
    form_ctx.set_ghost_form(form)
    for seed in (0, 7):
        cells = random_mesh(host_ctx, dim, lmin, lmax, s, r, seed).cells()
        print("form", form, dim, lmin, lmax, s, r, len(cells), flush=True)
        o = OracleSim(dim, lmin, lmax, pred_s=s, radius=r, cells=cells)
        o.set_poison(False)
        o.set_dirichlet(-0.5)
        mesh = sa.make_mesh_from_cells(form_ctx, sa.mesh_config(dim, lmin, lmax, s, r), cells)
        assert mesh.ghost_form() == (2 if form else 0)
        u = sa.make_scalar_field("u", mesh)
        sa.make_bc_dirichlet(u, -0.5)
        rng = np.random.default_rng(seed)
        for step in range(3):
            st = rng.standard_normal(u.size())
            o.set_storage(st)
            u.set_storage(st)
            o.update_ghost_mr()
            sa.update_ghost_mr(u)
            assert np.array_equal(o.storage().view(np.uint64), u.storage().view(np.uint64)), (seed, step)


@pytest.mark.gpu
@pytest.mark.parametrize("dim,s", [(2, 0), (2, 1), (3, 0), (3, 1)])
@pytest.mark.parametrize("n", [1, 3, 70])
def test_batched_flow_matches_staged(form_ctx, host_ctx, dim, s, n):
    """Frozen steps of few and of more than 64 instances, the smallest meshes
    among them, against the plain calls in the staged form."""
    print("batched flow", dim, s, n, flush=True)
    levels = [(1, 2), (1, 4), (2, 5), (3, 3)] if dim == 2 else [(1, 2), (1, 3), (2, 4), (2, 2)]
    kinds = [random_mesh(host_ctx, dim, *levels[k % 4], s, 1, k).cells() for k in range(8)]
    a, dt = np.array([0.6, -0.8, 0.3][:dim]), 0.01
    sets = []
    for _ in range(2):
        inst = []
        for k in range(n):
            mesh = sa.make_mesh_from_cells(form_ctx, sa.mesh_config(dim, *levels[k % 4], s), kinds[k % 8])
            u, unp1 = sa.make_scalar_field("u", mesh), sa.make_scalar_field("v", mesh)
            for f in (u, unp1):
                sa.make_bc_dirichlet(f, 0.1 * k)
            u.set_cells(np.random.default_rng(k).standard_normal(mesh.nb_cells()))
            inst.append((u, unp1, a, dt))
        sets.append(inst)
    assert all(i[0].mesh.ghost_form() >= 1 for i in sets[0])
    b = sa.Batch(form_ctx, sets[0])
    for step in range(4):
        form_ctx.set_ghost_form(-1)
        b.advance()
        form_ctx.set_ghost_form(0)
        for (u, unp1, _, _), (v, _, _, _) in zip(sets[1], sets[0]):
            sa.update_ghost_mr(u)
            sa.upwind(a, dt, u, unp1)
            sa.swap(u, unp1)
            assert np.array_equal(u.cells(), v.cells()), step
