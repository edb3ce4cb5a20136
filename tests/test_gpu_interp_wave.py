"""GPU: 3-D FP64 type 2 with wide kernels (W >= 9: a wave per point), and the
3-D interpolation's choice of threads: every support from 9 to 16, few and
many points per tile, smaller tiles than the default, plans, records, float32
coordinates and the offset check, against the direct sum; gradients and large
tiles on both sides of each line."""
import numpy as np
import pytest

from conftest import kernel_rows

pytestmark = pytest.mark.gpu
SHAPE = (18, 20, 23)


def eps_for(W, ofactor=2.0):
    """just above the table's epsilon for W: no smaller support reaches it"""
    return kernel_rows(ofactor, 3, False)[W][1] * 1.01


def points(M, rng):
    c = rng.uniform(-np.pi, np.pi, (M, 3))
    c[M // 2:] = 0.3 + 0.01 * c[M // 2:]  # more than one subproblem
    return c


@pytest.mark.parametrize("digits", [7, 8, 9, 10, 11, 12, 13])
@pytest.mark.parametrize("sigma", [(1.2, 1.5), (1.5, 2.5)])
def test_wide_3d(gpu, digits, sigma):
    """the supports that the cost model picks"""
    from ducc_amd import nufft
    if sigma[1] == 1.5 and digits > 10:
        pytest.skip("the table has no kernel of this accuracy")
    eps = 10.0 ** -digits
    rng = np.random.default_rng(digits)
    g = rng.standard_normal(SHAPE) + 1j * rng.standard_normal(SHAPE)
    for M in (1, 70, 3000):
        c = points(M, rng)
        v = nufft.u2nu(grid=g, coord=c, forward=False, epsilon=eps,
                       sigma_min=sigma[0], sigma_max=sigma[1])
        r = nufft.nudft_direct(2, c, g, SHAPE, False, np.arange(M))
        lim = 4 * eps * np.linalg.norm(g) * np.sqrt(M)
        assert np.linalg.norm(v - r) <= lim + 1e-12 * np.linalg.norm(r)


@pytest.mark.parametrize("W", range(9, 17))
@pytest.mark.parametrize("log2tile", [0, 2])
def test_every_support(gpu, W, log2tile):
    """W = 9 .. 16, in the default tiles and in 4^3 ones: unplanned, planned
    (points in tile order), as records, from float32 coordinates"""
    from ducc_amd import nufft
    eps = eps_for(W)
    rng = np.random.default_rng(W)
    g = rng.standard_normal(SHAPE) + 1j * rng.standard_normal(SHAPE)
    sig = dict(sigma_min=2.0, sigma_max=2.0, log2tile=log2tile)
    for M in (1, 70, 3000):
        c = points(M, rng)
        r = nufft.nudft_direct(2, c, g, SHAPE, False, np.arange(M))
        # (the direct sum of 8280 terms rounds at 1e-13)
        lim = 4 * eps * np.linalg.norm(g) * np.sqrt(M) + \
            1e-12 * np.linalg.norm(r)
        info = {}
        v = nufft.u2nu(grid=g, coord=c, forward=False, epsilon=eps,
                       info=info, check_offsets=True, **sig)
        assert info["W"] == W and info["fp64"]
        assert info["log2tile"] == (2 if log2tile or W > 13 else 3)
        assert np.linalg.norm(v - r) <= lim
        p = nufft.plan(nu2u=False, coord=c, grid_shape=SHAPE, epsilon=eps,
                       check_offsets=True, **sig)
        assert p.info()["W"] == W
        assert np.array_equal(p.u2nu(grid=g, forward=False), v)
        v2 = nufft.u2nu(grid=g, coord=c, forward=False, epsilon=eps,
                        point_records=True, **sig)
        assert np.array_equal(v2, v)
        c32 = c.astype(np.float32)
        r = nufft.nudft_direct(2, c32, g, SHAPE, False, np.arange(M))
        v = nufft.u2nu(grid=g, coord=c32, forward=False, epsilon=eps, **sig)
        # float32 coordinates are folded in plain double precision
        assert np.linalg.norm(v - r) <= lim + 1e-12 * np.linalg.norm(r)


@pytest.mark.parametrize("W", range(8, 15))
def test_gradient_threads(gpu, W):
    """coordinate gradients on both sides of the 512-thread rule (W = 10 to
    13; a hundred points a tile)"""
    from ducc_amd import nufft
    eps = eps_for(W)
    rng = np.random.default_rng(W)
    g = rng.standard_normal(SHAPE) + 1j * rng.standard_normal(SHAPE)
    k = [np.arange(n) - n // 2 for n in SHAPE]
    for M in (50, 5000, 200_000):
        c = rng.uniform(-np.pi, np.pi, (M, 3))
        d = nufft.u2nu_coord_grad(grid=g, coord=c, forward=False,
                                  epsilon=eps, sigma_min=2.0, sigma_max=2.0)
        sel = rng.integers(0, M, 40)
        E = [np.exp(1j * np.outer(c[sel, a], k[a])) for a in range(3)]
        for a in range(3):
            F = list(E)
            F[a] = E[a] * (1j * k[a])
            r = np.einsum("pa,pb,pc,abc->p", *F, g, optimize=True)
            # the derivative's error: the kernel's times its steepness
            lim = (20 * eps + 1e-12) * np.linalg.norm(r)
            assert np.linalg.norm(d[sel, a] - r) <= lim, (M, a)


@pytest.mark.parametrize("W,single", [(4, True), (6, True), (8, True),
                                      (5, False), (8, False)])
def test_large_tiles(gpu, W, single):
    """16^3 tiles where they fit (512 threads), 8^3 where they do not, W = 8
    in FP64 (256)"""
    from ducc_amd import nufft
    eps = kernel_rows(2.0, 3, single)[W][1] * 1.01
    rng = np.random.default_rng(W)
    dt = np.complex64 if single else np.complex128
    g = (rng.standard_normal(SHAPE) +
         1j * rng.standard_normal(SHAPE)).astype(dt)
    for M in (30, 60_000):
        c = points(M, rng)
        info = {}
        v = nufft.u2nu(grid=g, coord=c, forward=True, epsilon=eps,
                       sigma_min=2.0, sigma_max=2.0, log2tile=4, info=info,
                       precision="fp32" if single else "fp64")
        assert info["W"] == W
        assert info["log2tile"] == (3 if W == 8 else 4)
        sel = np.arange(0, M, max(1, M // 200))
        r = nufft.nudft_direct(2, c, g, SHAPE, True, sel)
        lim = 4 * eps + (2e-6 if single else 1e-12)
        assert np.linalg.norm(v[sel] - r) <= lim * np.linalg.norm(g) * \
            np.sqrt(len(sel))
