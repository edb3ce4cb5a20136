"""ducc0.wgridder (vis2dirty / dirty2vis, ms2dirty / dirty2ms) on the GPU
against the direct sums of oracle/wgridder.py (the sums of the reference's
test_wgridder.py:34-91, pinned there to a 2-D NUDFT and to ducc0 itself),
the reference's accuracy bound (l2error within epsilon,
test_wgridder.py:262-290) and adjointness test (test_wgridder.py:197-235),
and ducc0's own gridder (oracle/_ref) at a larger size."""
import itertools

import numpy as np
import pytest
import torch

from oracle import core as O
from oracle import wgridder as G

pytestmark = pytest.mark.gpu
C = G.SPEED_OF_LIGHT


def _problem(seed, nx, ny, nrow, nchan, fov, single=False):
    rng = np.random.default_rng(seed)
    px = fov * np.pi / 180 / nx
    py = fov * np.pi / 180 / ny * 1.1
    f0 = 1e9
    freq = f0 + np.arange(nchan) * (f0 / nchan)
    uvw = (rng.random((nrow, 3)) - 0.5) / (px * f0 / C)
    ms = rng.random((nrow, nchan)) - 0.5 + 1j * (rng.random((nrow, nchan)) - 0.5)
    wgt = rng.uniform(0.9, 1.1, (nrow, nchan))
    mask = (rng.uniform(0, 1, (nrow, nchan)) > 0.5).astype(np.uint8)
    dirty = rng.random((nx, ny)) - 0.5
    if single:
        ms, wgt, dirty = ms.astype(np.complex64), wgt.astype(np.float32), \
            dirty.astype(np.float32)
    return px, py, freq, uvw, ms, wgt, mask, dirty


# test_wgridder.py:249-261 parameters, a spread of the combinations
CASES = [c for c in itertools.product(
    [(2, 2), (6, 64), (66, 2), (18, 64)],   # (nx, ny)
    [1, 27],                                 # nrow
    [1, 5],                                  # nchan
    [1e-2, 1e-4, 1e-7],                      # epsilon
    [False, True],                           # w-gridding
    [0.001, 0.1, 20.])]                      # fov (degrees)
CASES = CASES[::7]


@pytest.mark.parametrize("nxy,nrow,nchan,eps,wg,fov", CASES)
def test_vis2dirty_against_direct_sum(gpu, nxy, nrow, nchan, eps, wg, fov):
    from ducc_amd import wgridder as W
    nx, ny = nxy
    print(f"vis2dirty {nx}x{ny} nrow={nrow} nchan={nchan} eps={eps} wg={wg} "
          f"fov={fov}", flush=True)
    px, py, freq, uvw, ms, wgt, mask, _ = _problem(42, nx, ny, nrow, nchan,
                                                   fov)
    d = W.ms2dirty(uvw, freq, ms, wgt, nx, ny, px, py, 0, 0, eps, wg, 1, 0,
                   mask)
    ref = G.vis2dirty(uvw, freq, ms, wgt, nx, ny, px, py, wg, mask)
    assert O.l2error(d.astype(complex), ref.astype(complex)) <= eps
    v = W.dirty2ms(uvw, freq, ref, wgt, px, py, 0, 0, eps, wg, 1, 0, mask)
    vref = G.dirty2vis(uvw, freq, ref, wgt, px, py, wg, mask)
    assert O.l2error(v, vref) <= eps


@pytest.mark.parametrize("single,eps", [(False, 2e-13), (False, 3e-5),
                                        (True, 3e-5)])
@pytest.mark.parametrize("wg", [False, True])
@pytest.mark.parametrize("use_wgt,use_mask", [(False, False), (True, True)])
def test_adjointness(gpu, single, eps, wg, use_wgt, use_mask):
    """test_wgridder.py:197-235 (rtol 3 * tol)"""
    from ducc_amd import wgridder as W
    nx, ny = 64, 32
    px = np.pi / 180 / 60 / nx * 0.2398
    py = np.pi / 180 / 60 / nx
    rng = np.random.default_rng(43)
    f0 = 1e9
    nrow, nchan = 100, 5
    freq = f0 + np.arange(nchan) * (f0 / nchan)
    uvw = (rng.random((nrow, 3)) - 0.5) / (py * f0 / C)
    ms = rng.random((nrow, nchan)) - 0.5 + 1j * (rng.random((nrow, nchan)) - 0.5)
    wgt = rng.uniform(0.9, 1.1, (nrow, nchan)) if use_wgt else None
    mask = (rng.uniform(0, 1, (nrow, nchan)) > 0.5).astype(np.uint8) \
        if use_mask else None
    dirty = rng.random((nx, ny)) - 0.5
    if single:
        ms, dirty = ms.astype(np.complex64), dirty.astype(np.float32)
        if wgt is not None:
            wgt = wgt.astype(np.float32)
    d2 = W.ms2dirty(uvw, freq, ms, wgt, nx, ny, px, py, 0, 0, eps, wg, 1, 0,
                    mask).astype(np.float64)
    m2 = W.dirty2ms(uvw, freq, dirty, wgt, px, py, 0, 0, eps, wg, 1, 0,
                    mask).astype(np.complex128)
    ref = max(np.vdot(ms, ms).real, np.vdot(m2, m2).real,
              np.vdot(dirty, dirty).real, np.vdot(d2, d2).real)
    tol = 3e-5 * ref if single else 2e-13 * ref
    lhs = np.vdot(ms.astype(np.complex128), m2).real
    rhs = float(np.sum(d2 * dirty))
    assert abs(lhs - rhs) <= 3 * tol


@pytest.mark.parametrize("kw", [dict(flip_u=True), dict(flip_v=True,
                                                        flip_w=True),
                                dict(center_x=0.002, center_y=-0.003),
                                dict(divide_by_n=False),
                                dict(allow_nshift=False)])
def test_options_against_direct_sum(gpu, kw):
    from ducc_amd import wgridder as W
    nx, ny, eps = 40, 36, 1e-7
    px, py, freq, uvw, ms, wgt, mask, dirty = _problem(5, nx, ny, 30, 3, 5.0)
    okw = {k: v for k, v in kw.items() if k != "allow_nshift"}
    for wg in (False, True):
        d = W.vis2dirty(uvw=uvw, freq=freq, vis=ms, wgt=wgt, npix_x=nx,
                        npix_y=ny, pixsize_x=px, pixsize_y=py, epsilon=eps,
                        do_wgridding=wg, mask=mask, **kw)
        ref = G.vis2dirty(uvw, freq, ms, wgt, nx, ny, px, py, wg, mask, **okw)
        assert O.l2error(d.astype(complex), ref.astype(complex)) <= eps
        v = W.dirty2vis(uvw=uvw, freq=freq, dirty=dirty, wgt=wgt,
                        pixsize_x=px, pixsize_y=py, epsilon=eps,
                        do_wgridding=wg, mask=mask, **kw)
        vref = G.dirty2vis(uvw, freq, dirty, wgt, px, py, wg, mask, **okw)
        assert O.l2error(v, vref) <= eps


@pytest.mark.parametrize("single,eps", [(False, 1e-6), (True, 1e-4)])
@pytest.mark.parametrize("wg", [False, True])
def test_matches_ducc0(gpu, single, eps, wg):
    """1000 rows x 8 channels onto 256 x 256 pixels of 20 degrees: within
    2 eps of ducc0's own ms2dirty / dirty2ms (oracle/_ref, all host cores)"""
    import os
    from oracle import ref as R
    from ducc_amd import wgridder as W
    if not R.available():
        pytest.skip("reference library not built")
    nx = ny = 256
    px, py, freq, uvw, ms, wgt, mask, dirty = _problem(7, nx, ny, 1000, 8,
                                                       20.0, single)
    nth = os.cpu_count() or 1
    d = W.vis2dirty(uvw=uvw, freq=freq, vis=ms, wgt=wgt, npix_x=nx,
                    npix_y=ny, pixsize_x=px, pixsize_y=py, epsilon=eps,
                    do_wgridding=wg, mask=mask)
    r = R.wgridder(False, uvw, freq, ms, wgt, mask, nx, ny, px, py, eps, wg,
                   nthreads=nth)
    assert O.l2error(d.astype(complex), r.astype(complex)) <= 2 * eps
    v = W.dirty2vis(uvw=uvw, freq=freq, dirty=dirty, wgt=wgt, pixsize_x=px,
                    pixsize_y=py, epsilon=eps, do_wgridding=wg, mask=mask)
    rv = R.wgridder(True, uvw, freq, dirty, wgt, mask, nx, ny, px, py, eps,
                    wg, nthreads=nth)
    assert O.l2error(v.astype(np.complex128),
                     rv.astype(np.complex128)) <= 2 * eps


def test_torch_arrays_and_all_masked(gpu):
    from ducc_amd import wgridder as W
    nx, ny, eps = 32, 32, 1e-6
    px, py, freq, uvw, ms, wgt, mask, dirty = _problem(9, nx, ny, 20, 2, 2.0)
    d_np = W.vis2dirty(uvw=uvw, freq=freq, vis=ms, wgt=wgt, npix_x=nx,
                       npix_y=ny, pixsize_x=px, pixsize_y=py, epsilon=eps,
                       do_wgridding=True, mask=mask)
    t = lambda x: torch.from_numpy(x).cuda()
    out = torch.empty((nx, ny), dtype=torch.float64, device="cuda")
    res = W.vis2dirty(uvw=t(uvw), freq=t(freq), vis=t(ms), wgt=t(wgt),
                      pixsize_x=px, pixsize_y=py, epsilon=eps,
                      do_wgridding=True, mask=t(mask), dirty=out)
    assert res is out
    np.testing.assert_allclose(out.cpu().numpy(), d_np, rtol=0, atol=1e-12)
    zero = np.zeros_like(mask)
    d0 = W.vis2dirty(uvw=uvw, freq=freq, vis=ms, wgt=wgt, npix_x=nx,
                     npix_y=ny, pixsize_x=px, pixsize_y=py, epsilon=eps,
                     do_wgridding=True, mask=zero)
    assert np.all(d0 == 0)
    v0 = W.dirty2vis(uvw=uvw, freq=freq, dirty=dirty, wgt=wgt, pixsize_x=px,
                     pixsize_y=py, epsilon=eps, do_wgridding=True, mask=zero)
    assert np.all(v0 == 0)


def _both(uvw, vis, wgt, mask, dirty, px, eps, lim, **kw):
    """vis2dirty and dirty2vis (frequency c: uvw in wavelengths) against the
    direct sums"""
    from ducc_amd import wgridder as W
    nx, ny = dirty.shape
    freq = np.array([C])
    d = W.vis2dirty(uvw=uvw, freq=freq, vis=vis, wgt=wgt, npix_x=nx,
                    npix_y=ny, pixsize_x=px, pixsize_y=px, epsilon=eps,
                    do_wgridding=True, mask=mask, **kw)
    r = G.vis2dirty(uvw, freq, vis, wgt, nx, ny, px, px, True, mask)
    assert O.l2error(d.astype(complex), r.astype(complex)) <= lim
    v = W.dirty2vis(uvw=uvw, freq=freq, dirty=dirty, wgt=wgt, pixsize_x=px,
                    pixsize_y=px, epsilon=eps, do_wgridding=True, mask=mask,
                    **kw)
    r = G.dirty2vis(uvw, freq, dirty, wgt, px, px, True, mask)
    assert O.l2error(v.astype(np.complex128), r) <= lim
    assert np.all(v[mask == 0] == 0)


@pytest.mark.parametrize("single,eps", [(False, 1e-9), (False, 1e-4),
                                        (True, 1e-4)])
def test_plane_order(gpu, single, eps):
    """visibilities by (tile, first plane): a tile with more of a plane's
    visibilities than one subproblem holds, over a hundred planes (several
    batches of lists), a gap of planes without any, masked ones"""
    rng = np.random.default_rng(11)
    nx, ny, n = 100, 60, 4000
    px = np.radians(10.) / nx  # dw is about 100 wavelengths
    uvw = (rng.random((n, 3)) - 0.5) / px
    w = np.where(rng.random(n) < 0.5, rng.uniform(-2000, 0, n),
                 rng.uniform(6000, 9000, n))
    uvw[:, 2] = w
    uvw[:2500] = [0.1 / px, -0.2 / px, 7000.] + rng.random((2500, 3)) * [
        0.01 / px, 0.01 / px, 200.]
    vis = rng.random((n, 1)) - 0.5 + 1j * (rng.random((n, 1)) - 0.5)
    wgt = rng.uniform(0.9, 1.1, (n, 1))
    mask = (rng.random((n, 1)) > 0.2).astype(np.uint8)
    dirty = rng.random((nx, ny)) - 0.5
    if single:
        vis, wgt, dirty = (vis.astype(np.complex64), wgt.astype(np.float32),
                           dirty.astype(np.float32))
    _both(uvw, vis, wgt, mask, dirty, px, eps, eps)


def test_planes_sharing_a_key(gpu):
    """few visibilities, many tiles and planes: more than 2^24 (tile, plane)
    pairs, so that neighbouring planes share a sort key (and more planes than
    are counted in LDS)"""
    rng = np.random.default_rng(12)
    nx, n, eps, sigma = 320, 40, 1e-6, 2.0
    px = np.radians(20.) / nx
    uvw = (rng.random((n, 3)) - 0.5) / px
    # n - 1 runs from 0 to that of the corner, centred by the shift
    nm1 = 1 - np.sqrt(1 - 2 * (nx / 2 * px) ** 2)
    dw = 0.5 / sigma / (0.5 * nm1)
    # clusters over 60000 planes, some a fraction of a plane wide
    uvw[:, 2] = np.repeat(rng.uniform(-3e4, 3e4, 8), 5) * dw + \
        rng.uniform(0, 1, n) * np.repeat([0.1, 1, 2, 3, 4, 9, 20, 40], 5) * dw
    uvw[0, 2], uvw[1, 2] = -3e4 * dw, 3e4 * dw
    tiles = (2 * nx // 32) ** 2  # 32 x 32 cells each
    assert tiles * 6e4 > 1 << 24
    vis = rng.random((n, 1)) - 0.5 + 1j * (rng.random((n, 1)) - 0.5)
    mask = np.ones((n, 1), np.uint8)
    mask[7] = 0
    dirty = rng.random((nx, nx)) - 0.5
    # rounding of phases of w (n - 1) turns: 2 pi 4e3 * 1.1e-16
    _both(uvw, vis, np.ones((n, 1)), mask, dirty, px, eps, eps + 1e-11,
          sigma_min=sigma, sigma_max=sigma)


def test_key_table_is_bounded(gpu):
    """device memory of a call goes with its image and visibilities, not
    with tiles times planes (1.8 GB of table here at one entry each)"""
    from ducc_amd import wgridder as W
    nx, n, sigma = 1400, 16, 2.0
    px = np.radians(20.) / nx
    nm1 = 1 - np.sqrt(1 - 2 * (nx / 2 * px) ** 2)
    dw = 0.5 / sigma / (0.5 * nm1)
    uvw = np.zeros((n, 3))
    uvw[: n // 2, 2], uvw[n // 2:, 2] = -3e4 * dw, 3e4 * dw
    assert (2 * nx // 32) ** 2 * 6e4 * 4 > 1.7e9
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    W.vis2dirty(uvw=uvw, freq=np.array([C]), vis=np.ones((n, 1), complex),
                npix_x=nx, npix_y=nx, pixsize_x=px, pixsize_y=px,
                epsilon=1e-6, do_wgridding=True, sigma_min=sigma,
                sigma_max=sigma)
    assert free - torch.cuda.mem_get_info()[0] < 1 << 30


def test_errors(gpu):
    from ducc_amd import wgridder as W
    px, py, freq, uvw, ms, wgt, mask, dirty = _problem(1, 8, 8, 4, 2, 1.0)
    with pytest.raises(RuntimeError, match="even"):
        W.vis2dirty(uvw=uvw, freq=freq, vis=ms, npix_x=7, npix_y=8,
                    pixsize_x=px, pixsize_y=py, epsilon=1e-5)
    with pytest.raises(RuntimeError, match="ascending"):
        W.vis2dirty(uvw=uvw, freq=freq[::-1].copy(), vis=ms, npix_x=8,
                    npix_y=8, pixsize_x=px, pixsize_y=py, epsilon=1e-5)
    with pytest.raises(RuntimeError, match="epsilon"):
        W.vis2dirty(uvw=uvw, freq=freq, vis=ms, npix_x=8, npix_y=8,
                    pixsize_x=px, pixsize_y=py, epsilon=0.0)
