"""The dataflow form of the frozen steps and their adjoint against the staged
programs (which set_tuning selects): the same bits for both prediction radii,
2D and 3D, one to many instances, and checkpoint intervals around the number of
adjoint steps of a launch."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def frozen(sa, ctx, dim, lmax, s, seed):
    mesh = sa.make_mesh(ctx, sa.mesh_config(dim, 1, lmax, s))
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.5)
    rng = np.random.default_rng(seed)
    x = (mesh.cells()[:, 1:1 + dim] + 0.5) * 2.0 ** -lmax
    c = rng.uniform(0.0, 1.0, dim)  # up to the boundary
    u.set_cells(np.where(np.abs(x - c).max(axis=1) < 0.15, 1.0, 0.2) + 0.3 * np.exp(-((x - 0.4) ** 2).sum(axis=1) / 0.02))
    sa.make_MRAdapt(u)(1e-2, 1.0)
    return mesh, u.cells()


@pytest.mark.parametrize("dim,lmax,s,n,steps,every", [(2, 4, 1, 1, 1, 1), (2, 6, 0, 3, 6, 3), (2, 6, 1, 2, 18, 18), (2, 5, 1, 2, 34, 17),
                                                      (3, 3, 1, 2, 4, 2), (3, 4, 0, 1, 3, 1), (3, 5, 1, 2, 4, 4)])
def test_flow_matches_stage_programs(gpu_ctx, dim, lmax, s, n, steps, every):
    import samurai_amd as sa
    import torch
    print("flow", dim, lmax, s, n, steps, every, flush=True)
    inst = [frozen(sa, gpu_ctx, dim, lmax, s, 10 + k) for k in range(n)]
    rng = np.random.default_rng(2)
    a = rng.uniform(-1.0, 1.0, (n, dim))
    p = sa.AdjointProblem(gpu_ctx, [m for m, _ in inst], [0.2 * 2.0 ** -lmax] * n, bc=list(rng.uniform(0, 1, n)), steps=steps, checkpoint_every=every)
    u0 = torch.tensor(np.concatenate([u for _, u in inst]), device="cuda")
    gT = torch.tensor(rng.standard_normal(u0.numel()), device="cuda")

    def both_ways():
        uT, g0 = torch.empty_like(u0), torch.empty_like(u0)
        torch.cuda.synchronize()
        p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        ga = p.backward_ptr(gT.data_ptr(), g0.data_ptr())
        return uT.cpu().numpy(), g0.cpu().numpy(), ga

    p.set_velocity(a)
    with pytest.raises(sa.SamuraiError):
        p.backward_ptr(gT.data_ptr(), torch.empty_like(u0).data_ptr())
    flow = [both_ways()]
    p.set_velocity(-a)
    flow.append(both_ways())
    p.set_tuning(256, 0, 1)
    staged = []
    for v in (a, -a):
        p.set_velocity(v)
        staged.append(both_ways())
    for got, want in zip(flow, staged):
        for g, w in zip(got, want):
            assert np.array_equal(g, w)


def test_tuning_between_forward_and_backward(gpu_ctx):
    """A launch shape set after a forward is used from the next one on: the
    backward of the one before still has its states."""
    import samurai_amd as sa
    import torch
    print("tuning in between", flush=True)
    mesh, u = frozen(sa, gpu_ctx, 2, 6, 1, 7)
    p = sa.AdjointProblem(gpu_ctx, [mesh], [0.2 / 64], bc=[0.5], steps=6, checkpoint_every=3)
    u0 = torch.tensor(u, device="cuda")
    gT = torch.tensor(np.random.default_rng(3).standard_normal(u0.numel()), device="cuda")
    uT, g0 = torch.empty_like(u0), torch.empty_like(u0)
    torch.cuda.synchronize()
    p.set_velocity([[0.7, -0.3]])
    got = []
    for shape in ((256, 0, 1), (512, 2, 0), None):
        p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        if shape:
            p.set_tuning(*shape)
        ga = p.backward_ptr(gT.data_ptr(), g0.data_ptr())
        got.append((uT.cpu().numpy(), g0.cpu().numpy(), ga))
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
    p.set_velocity([[0.1, -0.3]])
    with pytest.raises(sa.SamuraiError):
        p.backward_ptr(gT.data_ptr(), g0.data_ptr())


def test_less_room_means_fewer_steps_per_launch(gpu_ctx):
    """The arrays of a launch of 12 adjoint steps, of 2, and no room for those:
    the stage programs.  (A wait without rounds shows which form runs.)"""
    import samurai_amd as sa
    import torch
    print("less room", flush=True)
    ctx = sa.Context(0)
    mesh, u = frozen(sa, ctx, 2, 6, 1, 7)
    steps, every = 24, 12
    u0 = torch.tensor(u, device="cuda")
    gT = torch.tensor(np.random.default_rng(3).standard_normal(u0.numel()), device="cuda")
    uT, g0 = torch.empty_like(u0), torch.empty_like(u0)
    torch.cuda.synchronize()
    least = 8 * mesh.nb_cells(sa.REFERENCE) * (steps // every + every + 3)  # what the stage programs take
    got = []
    for room, flow in ((1 << 40, True), (least, True), (least - 1, False)):
        ctx.set_flow_bytes(room)
        p = sa.AdjointProblem(ctx, [mesh], [0.2 / 64], bc=[0.5], steps=steps, checkpoint_every=every)
        p.set_velocity([[0.7, -0.3]])
        p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        ga = p.backward_ptr(gT.data_ptr(), g0.data_ptr())
        got.append((uT.cpu().numpy(), g0.cpu().numpy(), ga))
        ctx.set_wait_rounds(0)
        if flow:
            with pytest.raises(sa.SamuraiError, match="adjoint"):
                p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        else:
            p.forward_ptr(u0.data_ptr(), uT.data_ptr())
        ctx.set_wait_rounds(1 << 17)
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
    ctx.close()
