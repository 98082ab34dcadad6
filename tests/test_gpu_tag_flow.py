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
