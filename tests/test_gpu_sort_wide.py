"""GPU: the one-launch and the one-pass index builds at their edges (points
per workgroup, blocks, tiles up to and past what one pass takes): the order
bit for bit, and a transform that uses the subproblem list."""
import numpy as np
import pytest

from oracle import core as O

pytestmark = pytest.mark.gpu

# 4096 points: one workgroup; 2^19: blocks of 1024 / 4096 points; 3969 tiles
# take one pass up to 5.6e5 points
MS = [1, 63, 64, 1025, 4095, 4096, 4097, 5000, 70001, (1 << 19) - 1,
      (1 << 19) + 1, 600_001]
# (dimensions, grid, log2 tile, W): 11, 36, 4096 - 64 * 3.., 4096+ tiles
GRIDS = [((4096,), 9, 7), ((110, 84), 5, 8), ((1950, 1950), 5, 7),
         ((1954, 1954), 5, 7), ((1984, 1984), 5, 7), ((100, 100, 100), 3, 6)]


@pytest.mark.parametrize("nover,log2tile,W", GRIDS)
def test_order(gpu, nover, log2tile, W):
    from ducc_amd import nufft
    nd = len(nover)
    for M in MS:
        rng = np.random.default_rng(M)
        c = rng.uniform(-np.pi, np.pi, (M, nd))
        if M > 2000:  # a crowded tile and a crowded row of tiles
            c[:1500] = 0.1 + 1e-4 * c[:1500]
            c[1500:2000, 0] = 1.0
        keys, idx = nufft.sort_points(c, nover, W, log2tile)
        kref = O.tile_keys(c, W, nover, 2 * np.pi, log2tile)
        assert np.array_equal(keys, kref)
        assert np.array_equal(idx, np.argsort(kref, kind="stable")), M


@pytest.mark.parametrize("shape", [(60, 50), (700, 900), (20, 24, 28)])
def test_subproblems(gpu, shape):
    """modes of a type 1 against the direct sum: every point is in exactly
    one subproblem"""
    from ducc_amd import nufft
    rng = np.random.default_rng(3)
    nd = len(shape)
    sel = rng.integers(0, int(np.prod(shape)), 16)
    for M in (1, 1500, 4096, 4097, 70001):
        c = rng.uniform(-np.pi, np.pi, (M, nd))
        c[:M // 2] *= 0.01
        p = rng.standard_normal(M) + 1j * rng.standard_normal(M)
        out = np.empty(shape, np.complex128)
        nufft.nu2u(points=p, coord=c, forward=True, epsilon=1e-8, out=out)
        ref = nufft.nudft_direct(1, c, p, shape, True, sel)
        # modes of uniform size ~ sqrt(M): eps of the transform's norm
        lim = 4e-8 * np.linalg.norm(out) * np.sqrt(len(sel) / out.size)
        assert np.linalg.norm(out.reshape(-1)[sel] - ref) <= 4 * lim
