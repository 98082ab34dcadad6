"""A wave of a dataflow launch that goes on without a value of the launch says
so: with no rounds to wait (the kernels end as ever, at once) the next call that
waits for the context's work fails, and the context works on afterwards.  So
does a side table without room."""
import numpy as np
import pytest

import samurai_amd as sa
from test_ghost_flow import random_mesh

pytestmark = pytest.mark.gpu


@pytest.fixture
def ctx(gpu_ctx):
    c = sa.Context(0)
    yield c
    c.close()


def field(ctx, host_ctx, dim, lmin, lmax, s):
    cells = random_mesh(host_ctx, dim, lmin, lmax, s, 1, 5).cells()
    mesh = sa.make_mesh_from_cells(ctx, sa.mesh_config(dim, lmin, lmax, s), cells)
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.5)
    u.set_cells(np.random.default_rng(1).standard_normal(len(cells)))
    return mesh, u


@pytest.mark.parametrize("dim,lmin,lmax,s", [(2, 2, 7, 0), (2, 2, 7, 1), (3, 2, 5, 0), (3, 2, 5, 1)])
def test_ghosts(ctx, host_ctx, dim, lmin, lmax, s):
    print("ghost fault", dim, lmin, lmax, s, flush=True)
    mesh, u = field(ctx, host_ctx, dim, lmin, lmax, s)
    ctx.set_ghost_form(1)
    assert mesh.ghost_form() == 2
    sa.update_ghost_mr(u)
    want = u.storage()
    unp1 = sa.make_scalar_field("v", mesh)
    sa.make_bc_dirichlet(unp1, 0.5)
    values = u.cells()
    b = sa.Batch(ctx, [(u, unp1, [0.0] * dim, 0.0)])
    for update in (lambda: sa.update_ghost_mr(u), b.advance):
        ctx.set_wait_rounds(0)
        update()
        with pytest.raises(sa.SamuraiError, match="update_ghost_mr"):
            ctx.synchronize()
        ctx.set_wait_rounds(1 << 17)
        u.set_cells(values)
        update()
        sa.update_ghost_mr(u)
        assert np.array_equal(u.storage(), want)


@pytest.mark.parametrize("dim,lmin,lmax,s", [(2, 2, 6, 1), (3, 2, 4, 0)])
def test_gradient(ctx, host_ctx, dim, lmin, lmax, s):
    import torch
    print("gradient fault", dim, lmin, lmax, s, flush=True)
    mesh, u = field(ctx, host_ctx, dim, lmin, lmax, s)
    p = sa.AdjointProblem(ctx, [mesh], [0.2 * 2.0 ** -lmax], bc=[0.5], steps=4, checkpoint_every=2)
    p.set_velocity([[0.6, -0.8, 0.1][:dim]])
    u0 = torch.tensor(u.cells(), device="cuda")
    gT = torch.tensor(np.random.default_rng(2).standard_normal(u0.numel()), device="cuda")
    uT, g0 = torch.empty_like(u0), torch.empty_like(u0)
    torch.cuda.synchronize()

    def both():
        p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        p.backward_ptr(gT.data_ptr(), g0.data_ptr())
        return uT.cpu().numpy(), g0.cpu().numpy()

    want = both()
    ctx.set_wait_rounds(0)
    with pytest.raises(sa.SamuraiError, match="adjoint"):
        p.forward_ptr(u0.data_ptr(), uT.data_ptr())
    with pytest.raises(sa.SamuraiError, match="adjoint"):
        p.backward_ptr(gT.data_ptr(), g0.data_ptr())
    ctx.set_wait_rounds(1 << 17)
    for a, b in zip(want, both()):
        assert np.array_equal(a, b)
    # values with the bits the launches mark their slots with are only NaN
    u0[0] = gT[1] = torch.tensor([0x7FF05A3C96E1D2B4]).view(torch.float64)[0]
    torch.cuda.synchronize()
    got = both()
    p.set_tuning(256, 0, 1)
    for a, b in zip(got, both()):
        assert np.isnan(a).any() and np.array_equal(a, b, equal_nan=True)


def large_coarse_levels(mesh):
    """Levels whose maximum pass is a launch of its own in the staged form: two
    and the launch for the others are more than the dataflow form's."""
    c = mesh.cells()
    n = [len(np.unique(c[c[:, 0] == l][:, 1:4] // 2, axis=0)) for l in range(mesh.max_level + 1)]
    return sum(k > 2048 for k in n)


@pytest.mark.parametrize("dim,lmin,lmax", [(2, 7, 9), (3, 4, 6)])
def test_tags(ctx, host_ctx, dim, lmin, lmax):
    import torch
    print("tag fault", dim, lmin, lmax, flush=True)
    mesh, u = field(ctx, host_ctx, dim, lmin, lmax, 1)
    assert large_coarse_levels(mesh) >= 2
    ad = sa.make_MRAdapt(u)
    ctx.set_ghost_form(0)
    tags = [torch.zeros(mesh.nb_cells(sa.REFERENCE), dtype=torch.uint8, device="cuda") for _ in range(3)]
    torch.cuda.synchronize()
    for t, rounds in zip(tags, (1 << 17, 0, 1 << 17)):
        ctx.set_wait_rounds(rounds)
        ad.tags_into(0, 1e-1, 1.0, t.data_ptr())
        if rounds:
            ctx.synchronize()
        else:
            with pytest.raises(sa.SamuraiError, match="tag finalization"):
                ctx.synchronize()
    assert torch.equal(tags[0], tags[2])


@pytest.mark.parametrize("dim,lmin,lmax,s", [(2, 2, 6, 1), (3, 2, 4, 0)])
def test_side_table(ctx, host_ctx, dim, lmin, lmax, s):
    print("side table fault", dim, lmin, lmax, s, flush=True)
    ops = (sa.make_convection_upwind([0.6, -0.8, 0.3][:dim]), sa.make_convection_upwind())
    mesh, u = field(ctx, host_ctx, dim, lmin, lmax, s)
    out = sa.make_scalar_field("f", mesh)
    want = [op(u, out=out).storage() for op in ops]
    ctx.set_side_entries(8)
    mesh, u = field(ctx, host_ctx, dim, lmin, lmax, s)  # its table is built anew
    out = sa.make_scalar_field("f", mesh)
    with pytest.raises(sa.SamuraiError, match="side table"):
        ops[0](u, out=out).storage()
    for _ in range(2):
        for op, w in zip(ops, want):
            assert np.array_equal(op(u, out=out).storage(), w)
