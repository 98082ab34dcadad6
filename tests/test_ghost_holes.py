"""Meshes whose leaves do not tile the box (make_mesh_from_cells accepts them):
a missing child is predicted from the very cell that projects it, an order only
the staged ghost update has, so none of the dataflow forms may take them."""
import numpy as np
import pytest

import samurai_amd as sa
from oracle_lib import OracleSim
from test_ghost_flow import random_mesh

MESHES = [(2, 2, 5, 0), (2, 2, 6, 1), (2, 3, 7, 1), (3, 1, 3, 1), (3, 2, 4, 0), (3, 2, 4, 1)]


def holed(host_ctx, dim, lmin, lmax, s, seed, refined=True):
    """Leaves with one missing whose siblings remain, at a level with coarser and
    (if refined) finer ones."""
    cells = random_mesh(host_ctx, dim, lmin, lmax, s, 1, seed).cells()
    level = lmax if not refined else min(lmax - 1, max(lmin + 1, lmax - 2))
    at = np.flatnonzero(cells[:, 0] == level)
    return np.delete(cells, at[len(at) // 2], 0)


def leaves(cells):
    return {tuple(c[:4]) for c in np.asarray(cells)}


@pytest.mark.parametrize("dim,lmin,lmax,s", MESHES)
def test_holes_have_no_flow(host_ctx, dim, lmin, lmax, s):
    cfg = sa.mesh_config(dim, lmin, lmax, s)
    for seed in range(3):
        full = random_mesh(host_ctx, dim, lmin, lmax, s, 1, seed)
        assert full.ghost_form() == 1 and full.validate() == 0
        assert sa.make_mesh_from_cells(host_ctx, cfg, full.cells()).ghost_form() == 1
        for refined in (False, True):
            m = sa.make_mesh_from_cells(host_ctx, cfg, holed(host_ctx, dim, lmin, lmax, s, seed, refined))
            assert m.ghost_form() == 0 and m.validate() == 0
            # the hole stays when the mesh changes around it, and goes with a new mesh
            tags = np.zeros(m.nb_cells(sa.REFERENCE), dtype=np.uint8)
            c = m.cells()
            tags[c[:, 4]] = np.where(c[:, 0] < lmax, sa.REFINE, sa.KEEP)
            m.rebuild_from_tags(tags)
            assert leaves(m.cells()) != leaves(c) and m.ghost_form() == 0
            m.assign_cells(full.cells())
            assert m.ghost_form() == 1


@pytest.mark.parametrize("dim", [2, 3])
def test_overlaps_and_leaves_outside_have_no_flow(host_ctx, dim):
    """The right volume is not enough: a leaf missing and another one covered
    twice, and a leaf moved out of the box."""
    lmin, lmax = 2, 4
    base = random_mesh(host_ctx, dim, lmin, lmax, 1, 1, 1).cells()[:, :4]
    at = np.flatnonzero(base[:, 0] == 3)
    assert len(at) > 2
    gone, twice = at[len(at) // 2], base[at[0]]
    rest = np.delete(base, gone, 0)
    kids = np.array([[4, *(2 * twice[1:3] + (k & 1, (k >> 1) & 1)), 2 * twice[3] + (k >> 2)] for k in range(1 << dim)])
    outside = base[gone].copy()
    outside[1] += 8
    for cells in (np.concatenate([rest, kids]), np.concatenate([rest, outside[None]])):
        volume = (2.0 ** (-dim * cells[:, 0].astype(float))).sum()
        assert volume == 1.0
        assert sa.make_mesh_from_cells(host_ctx, sa.mesh_config(dim, lmin, lmax), cells).ghost_form() == 0


def test_partial_families_have_no_flow(host_ctx):
    """Flags that coarsen one child of a family leave a leaf over its siblings."""
    m = sa.make_mesh(host_ctx, sa.mesh_config(2, 2, 4))
    tags = np.zeros(m.nb_cells(sa.REFERENCE), dtype=np.uint8)
    c = m.cells()
    tags[c[:, 4]] = sa.KEEP
    tags[c[0, 4]] = sa.COARSEN
    m.rebuild_from_tags(tags)
    assert len(leaves(m.cells())) == 256 and (3, 0, 0, 0) in leaves(m.cells())
    assert m.ghost_form() == 0


def partial_flags(m, dim):
    """Flags on a mesh of 16^dim cells that coarsen the first child of one family
    (its parent then lies over the others) and, of as many families as make up for
    that, another child (which leaves a hole)."""
    c = m.cells()
    at = {tuple(x[1:1 + dim]): x[4] for x in c}
    tags = np.zeros(m.nb_cells(sa.REFERENCE), dtype=np.uint8)
    tags[c[:, 4]] = sa.KEEP
    tags[at[(4,) * dim]] = sa.COARSEN
    for f in range(1, 1 << dim):
        tags[at[(1 + 2 * (f % 4), 9, 1 + 2 * (f // 4))[:dim]]] = sa.COARSEN
    return tags


@pytest.mark.parametrize("dim", [2, 3])
def test_holes_and_overlaps_of_one_volume_have_no_flow(host_ctx, dim):
    m = sa.make_mesh(host_ctx, sa.mesh_config(dim, 2, 4))
    assert m.ghost_form() == 1
    m.rebuild_from_tags(partial_flags(m, dim))
    assert (2.0 ** (-dim * m.cells()[:, 0].astype(float))).sum() == 1.0
    assert m.ghost_form() == 0 and m.validate() == 0


@pytest.mark.gpu
@pytest.mark.parametrize("dim", [2, 3])
def test_holes_from_device_flags_have_no_flow(gpu_ctx, dim):
    import torch
    print("device flags", dim, flush=True)
    m = sa.make_mesh(gpu_ctx, sa.mesh_config(dim, 2, 4))
    gpu_ctx.set_ghost_form(1)
    try:
        assert m.ghost_form() == 2
        tags = torch.tensor(partial_flags(m, dim), device="cuda")
        torch.cuda.synchronize()
        assert m.rebuild_from_device_tags(tags.data_ptr(), tags.numel()) == 0
        assert (2.0 ** (-dim * m.cells()[:, 0].astype(float))).sum() == 1.0
        assert m.ghost_form() == 0
    finally:
        gpu_ctx.set_ghost_form(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("dim,lmin,lmax,s", MESHES)
def test_holed_ghosts_match_oracle(gpu_ctx, host_ctx, dim, lmin, lmax, s):
    gpu_ctx.set_ghost_form(1)
    try:
        for seed, refined in ((0, True), (1, False)):
            cells = holed(host_ctx, dim, lmin, lmax, s, seed, refined)
            print("hole", dim, lmin, lmax, s, len(cells), flush=True)
            o = OracleSim(dim, lmin, lmax, pred_s=s, cells=cells)
            o.set_poison(False)
            o.set_dirichlet(0.75)
            mesh = sa.make_mesh_from_cells(gpu_ctx, sa.mesh_config(dim, lmin, lmax, s), cells)
            assert mesh.ghost_form() == 0
            u = sa.make_scalar_field("u", mesh)
            sa.make_bc_dirichlet(u, 0.75)
            st = np.random.default_rng(seed).standard_normal(u.size())
            o.set_storage(st)
            u.set_storage(st)
            for step in range(3):
                o.update_ghost_mr()
                sa.update_ghost_mr(u)
                assert np.isfinite(u.storage()).all()
                assert np.array_equal(o.storage().view(np.uint64), u.storage().view(np.uint64)), step
    finally:
        gpu_ctx.set_ghost_form(-1)


@pytest.mark.gpu
@pytest.mark.parametrize("dim,lmin,lmax,s", [(2, 2, 5, 0), (2, 2, 6, 1), (3, 2, 4, 1)])
def test_holed_batch_and_gradient(gpu_ctx, host_ctx, dim, lmin, lmax, s):
    """One instance with a hole among whole ones: frozen steps as the plain calls
    give them, and gradients as the stage programs'."""
    import torch
    print("hole batch", dim, lmin, lmax, s, flush=True)
    a, dt = np.array([0.6, -0.8, 0.3][:dim]), 0.2 * 2.0 ** -lmax
    sets = [random_mesh(host_ctx, dim, lmin, lmax, s, 1, 3).cells(), holed(host_ctx, dim, lmin, lmax, s, 4)]
    both = []
    for _ in range(2):
        inst = []
        for k, cells in enumerate(sets):
            mesh = sa.make_mesh_from_cells(gpu_ctx, sa.mesh_config(dim, lmin, lmax, s), cells)
            u, unp1 = sa.make_scalar_field("u", mesh), sa.make_scalar_field("v", mesh)
            for f in (u, unp1):
                sa.make_bc_dirichlet(f, 0.5)
            u.set_storage(np.random.default_rng(k).standard_normal(u.size()))
            unp1.set_storage(np.zeros(u.size()))
            inst.append((u, unp1, a, dt))
        both.append(inst)
    b = sa.Batch(gpu_ctx, both[0])
    for step in range(3):
        b.advance()
        for (u, unp1, _, _), (v, _, _, _) in zip(both[1], both[0]):
            sa.update_ghost_mr(u)
            sa.upwind(a, dt, u, unp1)
            sa.swap(u, unp1)
            assert np.isfinite(v.cells()).all() and np.array_equal(u.cells(), v.cells()), step

    u0 = torch.tensor(np.concatenate([i[0].cells() for i in both[0]]), device="cuda")
    gT = torch.tensor(np.random.default_rng(5).standard_normal(u0.numel()), device="cuda")
    got = []
    for tuning in (None, (256, 0, 1)):
        # a problem each: what a hole's parent reads is left by the step before
        p = sa.AdjointProblem(gpu_ctx, [i[0].mesh for i in both[0]], [dt] * 2, bc=[0.5, 0.25], steps=4, checkpoint_every=2)
        if tuning:
            p.set_tuning(*tuning)
        p.set_velocity(np.array([a, -a]))
        uT, g0 = torch.empty_like(u0), torch.empty_like(u0)
        torch.cuda.synchronize()
        p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        ga = p.backward_ptr(gT.data_ptr(), g0.data_ptr())
        got.append((uT.cpu().numpy(), g0.cpu().numpy(), ga))
        assert all(np.isfinite(x).all() for x in got[-1])
    for x, y in zip(*got):
        assert np.array_equal(x, y)


@pytest.mark.gpu
@pytest.mark.parametrize("dim,lmax,s", [(2, 6, 0), (3, 4, 0), (3, 4, 1)])
def test_jumps_of_several_levels_match_oracle(gpu_ctx, host_ctx, dim, lmax, s):
    """Leaves that tile the box but are not graduated have the flow: both forms."""
    from test_gpu_convection_terms import jumps
    cells = jumps(dim, lmax, 3)
    print("jumps", dim, lmax, s, len(cells), flush=True)
    o = OracleSim(dim, 2, lmax, pred_s=s, cells=cells)
    o.set_poison(False)
    o.set_dirichlet(0.75)
    mesh = sa.make_mesh_from_cells(gpu_ctx, sa.mesh_config(dim, 2, lmax, s), cells)
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.75)
    st = np.random.default_rng(1).standard_normal(u.size())
    o.set_storage(st)
    o.update_ghost_mr()
    try:
        for form in (0, 1):
            gpu_ctx.set_ghost_form(form)
            assert mesh.ghost_form() == 2 * form
            u.set_storage(st)
            sa.update_ghost_mr(u)
            assert np.array_equal(o.storage().view(np.uint64), u.storage().view(np.uint64)), form
    finally:
        gpu_ctx.set_ghost_form(-1)
