"""GPU: type-1 flush of a tile region by plain stores (cells that only one
subproblem reaches) beside atomics: on the periodic seam, on grids smaller
than a region, beside tiles of several subproblems, on both sides of the
support where it starts, against the direct sum over all modes."""
import numpy as np
import pytest

from conftest import kernel_rows

pytestmark = pytest.mark.gpu


def clouds(rng, nd, period=2 * np.pi):
    """name -> points"""
    u = rng.uniform(-np.pi, np.pi, (3000, nd))
    seam = np.where(rng.random((600, nd)) < 0.5, -np.pi, np.pi) + \
        rng.uniform(-0.05, 0.05, (600, nd))
    hot = np.concatenate([u[:500], 0.4 + 0.02 * u[:2500]])  # 3 subproblems
    edge = np.concatenate([seam, -np.pi + 0.01 * rng.random((1500, nd)),
                           u[:200]])  # a crowded tile on the seam
    return dict(one=u[:1], uniform=u, seam=seam, hot=hot, edge=edge)


# (ndim, shape, log2tile): grids below one region, of two tiles, of a few
# tiles with a partial last one; 64-cell tiles keep plain stores to W = 13
CASES = [(2, (5, 6), 0), (2, (9, 40), 0), (2, (60, 47), 0), (2, (75, 41), 6),
         (1, (7,), 0), (1, (300,), 0), (1, (1500,), 0)]


@pytest.mark.parametrize("nd,shape,log2tile", CASES)
@pytest.mark.parametrize("W,single", [(4, True), (6, True), (7, True),
                                      (8, True), (5, False), (7, False),
                                      (12, False), (14, False)])
@pytest.mark.parametrize("fp64_acc", [False, True])
def test_flush(gpu, nd, shape, log2tile, W, single, fp64_acc):
    from ducc_amd import nufft
    if fp64_acc and not single:
        pytest.skip("FP64 accumulates in FP64 as it is")
    idx, eps = kernel_rows(2.0, nd, single)[W]
    rng = np.random.default_rng(W)
    dt = np.complex64 if single else np.complex128
    n = int(np.prod(shape))
    for name, c in clouds(rng, nd).items():
        M = len(c)
        p = (rng.standard_normal(M) + 1j * rng.standard_normal(M)).astype(dt)
        out = np.empty(shape, dt)
        info = {}
        # (epsilon above 1e-5 selects fixed point on the single path)
        nufft.nu2u(points=p, coord=c, forward=True, epsilon=2e-5, out=out,
                   kernel_idx=idx, log2tile=log2tile, info=info,
                   fp64_accumulation=fp64_acc,
                   precision="fp32" if single else "fp64")
        assert info["W"] == W
        ref = nufft.nudft_direct(1, c, p, shape, True, np.arange(n))
        # eps of the transform's norm (2 in 2-D, 4 in 1-D; a mode is of size
        # sqrt(M)); fixed point rounds at 1e-6 of it
        lim = (4 * eps + (4e-6 if single else 1e-13)) * \
            np.linalg.norm(p) * np.sqrt(n)
        assert np.linalg.norm(out.reshape(-1) - ref) <= lim, name


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_nonfinite_value(gpu, bad):
    """one value that is not finite: no mode comes out finite, whichever
    cells its tile stores plainly"""
    from ducc_amd import nufft
    rng = np.random.default_rng(0)
    for W in (4, 6, 8):
        c = rng.uniform(-np.pi, np.pi, (4000, 2))
        p = np.ones(4000, np.complex64)
        p[17] = bad
        out = np.zeros((60, 50), np.complex64)
        nufft.nu2u(points=p, coord=c, forward=True, epsilon=2e-5, out=out,
                   kernel_idx=kernel_rows(2.0, 2, True)[W][0],
                   precision="fp32")
        assert not np.isfinite(out).any()
