"""The maximum pass of the tags as one dataflow launch (meshes with two and more
levels of over 2048 coarse cells): flags, details, meshes and transferred fields
of every harten call against the oracle, and the device half alone twice."""
import numpy as np
import pytest

from test_gpu_parity import test_harten_matches_oracle as harten_matches_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,lmin,lmax,s,ic", [(2, 2, 9, 1, "seeded"), (2, 5, 8, 0, "disc"), (3, 2, 6, 1, "disc")])
def test_tags_of_larger_meshes_match_oracle(gpu_ctx, dim, lmin, lmax, s, ic):
    harten_matches_oracle(gpu_ctx, dim, lmin, lmax, s, ic)


@pytest.mark.parametrize("dim,level", [(2, 11), (3, 7)])
def test_repeated_tags_are_the_same(gpu_ctx, dim, level):
    """Tags of one state, computed several times into arrays of old values."""
    import torch

    import samurai_amd as sa
    from initial_conditions import seeded_2d, sphere_3d
    print("repeated tags", dim, level, flush=True)
    mesh = sa.make_mesh(gpu_ctx, sa.mesh_config(dim, 2, level, 1))
    u = sa.make_scalar_field("u", mesh)
    u.set_cells(seeded_2d(mesh.cells(), 3) if dim == 2 else sphere_3d(mesh.cells()))
    sa.make_bc_dirichlet(u, 0.0)
    ad = sa.make_MRAdapt(u)
    ad(1e-4, 2.0)
    out = []
    for k in range(8):
        t = torch.full((mesh.nb_cells(sa.REFERENCE),), 0xEE, dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()
        ad.tags_into(0, 1e-4, 2.0, t.data_ptr())
        gpu_ctx.synchronize()
        out.append(t.cpu().numpy())
        assert out[-1].max() < 8
        assert np.array_equal(out[0], out[-1]), k


def random_cells(host_ctx, dim, lmin, lmax, coarsen):
    import samurai_amd as sa
    m = sa.make_mesh(host_ctx, sa.mesh_config(dim, lmin, lmax))
    rng = np.random.default_rng(3)
    for _ in range(lmax - lmin):
        cells, tags = m.cells(), np.zeros(m.nb_cells(sa.REFERENCE), dtype=np.uint8)
        keys = np.column_stack([cells[:, 0], cells[:, 1:4] // 2])
        _, group, size = np.unique(keys, axis=0, return_inverse=True, return_counts=True)
        take = (rng.random(len(size)) < coarsen) & (size == 1 << dim)
        tags[cells[:, 4]] = np.where(take[group.ravel()], sa.COARSEN, sa.KEEP)
        m.rebuild_from_tags(tags)
    return m.cells()


@pytest.mark.parametrize("dim,lmin,lmax,coarsen,flow", [(2, 1, 2, 0.5, False), (2, 1, 5, 0.5, False), (3, 1, 4, 0.6, False), (2, 7, 9, 0.7, True),
                                                        (3, 4, 6, 0.7, True), (2, 8, 10, 0.7, True), (2, 8, 10, 0.3, False)])
def test_both_forms_give_the_same_tags(host_ctx, dim, lmin, lmax, coarsen, flow):
    """The dataflow launch and the launches per level on one state, from a few
    coarse cells to both sides of the size from which the latter are cheaper;
    which one the rule takes shows when the waits get no rounds."""
    import torch

    import samurai_amd as sa
    ctx = sa.Context(0)
    cells = random_cells(host_ctx, dim, lmin, lmax, coarsen)
    print("both forms", dim, lmin, lmax, len(cells), flush=True)
    mesh = sa.make_mesh_from_cells(ctx, sa.mesh_config(dim, lmin, lmax), cells)
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.0)
    ad = sa.make_MRAdapt(u)
    ctx.set_ghost_form(0)
    for scale in (1.0, 1e-3):
        u.set_cells(np.where(np.random.default_rng(5).random(len(cells)) < 0.05, 1.0, scale))
        out = []
        for form in (0, 1, -1):
            ctx.set_tag_form(form)
            out.append(torch.full((mesh.nb_cells(sa.REFERENCE),), 0xEE, dtype=torch.uint8, device="cuda"))
            torch.cuda.synchronize()
            ad.tags_into(0, 1e-2, 1.0, out[-1].data_ptr())
            ctx.synchronize()
        assert torch.equal(out[0], out[1]) and torch.equal(out[0], out[2])
        assert len(torch.unique(out[0])) > 1
    ctx.set_wait_rounds(0)
    ad.tags_into(0, 1e-2, 1.0, out[0].data_ptr())
    if flow:
        with pytest.raises(sa.SamuraiError, match="tag finalization"):
            ctx.synchronize()
    else:
        ctx.synchronize()
    ctx.close()
