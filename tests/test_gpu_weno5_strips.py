"""The WENO5 kernels of the larger one-level meshes (strips; tiles below) against
the kernel of one thread per cell, which the oracle checks: the same bits for
velocities of both signs and zero, and for values whose weights leave the range
of the shared-reciprocal divisions."""
import numpy as np
import pytest

import samurai_amd as sa

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,level", [(2, 6), (2, 9), (2, 10), (3, 6), (3, 7)])
@pytest.mark.parametrize("kind", ["smooth", "rough", "huge"])
def test_kernels_agree(gpu_ctx, dim, level, kind, monkeypatch):
    print("weno5 strips", dim, level, kind, flush=True)
    mesh = sa.make_mesh(gpu_ctx, sa.mesh_config(dim, level, level, 1, 3))
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.25)
    n = mesh.nb_cells()
    rng = np.random.default_rng(level)
    v = np.sin(np.arange(n) * 0.37) if kind == "smooth" else rng.standard_normal(n)
    if kind == "huge":
        v *= 10.0 ** rng.integers(-160, 160, n)
        v[rng.integers(0, n, 8)] = [np.inf, -np.inf, np.nan, 1e308, -1e308, 5e-324, 0.0, -0.0]
    u.set_cells(v)
    for a in ([1.5, -0.75, 0.5], [-1.0, 0.0, -2.0]):
        conv = sa.make_convection_weno5(a[:dim])
        got = conv(u).cells()
        monkeypatch.setenv("SMR_WENO5_UNTILED", "1")
        want = conv(u).cells()
        monkeypatch.delenv("SMR_WENO5_UNTILED")
        assert np.array_equal(np.isnan(got), np.isnan(want))
        k = ~np.isnan(want)
        assert np.array_equal(got[k].view(np.uint64), want[k].view(np.uint64))


@pytest.mark.parametrize("level", [8, 9, 10])
def test_weights_of_larger_meshes_match_plain_divisions(gpu_ctx, level):
    """The same where the divisions change to the shared reciprocals, and in strips."""
    weights_match_plain_divisions(gpu_ctx, level)


def test_weights_outside_the_range_match_plain_divisions(gpu_ctx):
    """One row of cells whose smoothness indicators grow past 2^300: the flux
    differences against the formula in numpy (IEEE divisions), bit for bit."""
    weights_match_plain_divisions(gpu_ctx, 6)


def weights_match_plain_divisions(gpu_ctx, level):
    n = 1 << level
    mesh = sa.make_mesh(gpu_ctx, sa.mesh_config(2, level, level, 1, 3))
    u = sa.make_scalar_field("u", mesh)
    sa.make_bc_dirichlet(u, 0.0)
    for scale in (1e-200, 1e-8, 1.0, 1e10, 1e37, 1e38, 1e60):
        row = scale * np.random.default_rng(3).standard_normal(n)
        u.set_cells(np.tile(row, n))
        got = sa.make_convection_weno5([1.0, 0.0])(u).cells().reshape(n, n)[n // 2]
        f = [row[k:n - 5 + k] for k in range(6)]  # cells -2..3 about interface i + 1/2, i = 2..n-4
        q = [1. / 3 * f[0] - 7. / 6 * f[1] + 11. / 6 * f[2], -1. / 6 * f[1] + 5. / 6 * f[2] + 1. / 3 * f[3],
             1. / 3 * f[2] + 5. / 6 * f[3] - 1. / 6 * f[4]]
        s = [13. / 12 * (b * b) + 1. / 4 * (c * c) for b, c in ((f[0] - 2 * f[1] + f[2], f[0] - 4 * f[1] + 3 * f[2]),
                                                                (f[1] - 2 * f[2] + f[3], f[1] - f[3]),
                                                                (f[2] - 2 * f[3] + f[4], 3 * f[2] - 4 * f[3] + f[4]))]
        a = [w / ((1e-6 + x) * (1e-6 + x)) for w, x in zip((0.1, 0.6, 0.3), s)]
        total = a[0] + a[1] + a[2]
        flux = a[0] / total * q[0] + a[1] / total * q[1] + a[2] / total * q[2]
        fa = float(n)
        want = (0.0 + flux[:-1] * -fa) + flux[1:] * fa
        assert np.array_equal(got[3:n - 3], want)
