"""GPU: 3-D FP64 type 2 with wide kernels (a wave per point): every support
from 9 to 16, few and many points per tile, tiles smaller than the default,
planned and unplanned, against the direct sum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("digits", [7, 8, 9, 10, 11, 12, 13])
@pytest.mark.parametrize("sigma", [(1.2, 1.5), (1.5, 2.5)])
def test_wide_3d(gpu, digits, sigma):
    from ducc_amd import nufft
    shape = (18, 20, 23)
    eps = 10.0 ** -digits
    rng = np.random.default_rng(digits)
    g = rng.standard_normal(shape) + 1j * rng.standard_normal(shape)
    for M in (1, 70, 3000):
        c = rng.uniform(-np.pi, np.pi, (M, 3))
        c[M // 2:] = 0.3 + 0.01 * c[M // 2:]  # more than one subproblem
        try:
            v = nufft.u2nu(grid=g, coord=c, forward=False, epsilon=eps,
                           sigma_min=sigma[0], sigma_max=sigma[1])
        except RuntimeError as e:
            assert "kernel" in str(e)
            return  # no tabulated kernel in this range
        r = nufft.nudft_direct(2, c, g, shape, False, np.arange(M))
        lim = 4 * eps * np.linalg.norm(g) * np.sqrt(M)
        assert np.linalg.norm(v - r) <= lim + 1e-12 * np.linalg.norm(r)
