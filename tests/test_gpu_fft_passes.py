"""GPU: the FFT passes at their edges - every radix alone and combined, line
counts that leave a workgroup partly filled, lines that take two passes over
L1 x L2, out-of-place input with a factor - against a 64-bit FFT."""
import ctypes as ct

import numpy as np
import pytest
import torch

from conftest import kernel_rows
from ducc_amd import _lib, fft, nufft

pytestmark = pytest.mark.gpu

# one length per radix, composite pairs, the longest lines in LDS, and lines
# beyond it (two passes; 16381 is prime: Bluestein over a long line)
LENGTHS = [2, 3, 5, 6, 7, 9, 10, 11, 12, 14, 15, 16, 84, 110, 210, 432, 462,
           1078, 1210, 1440, 3388, 3750, 3840, 4096, 7168, 8192, 8232, 11025,
           16381, 185220]


def tol(dtype, n):
    """Relative error in rms of log2(n) butterfly levels that each round once
    or twice by up to u, half a unit, independently: about u sqrt(log2 n).
    Measured over all lengths here: 0.5 to 0.92 of that in single precision,
    0.5 to 1.5 in double, where the comparison's own error adds.  Bluestein
    (a prime factor above 11): three transforms of twice the length."""
    u = 6e-8 if dtype == torch.complex64 else 1.11e-16
    t = u * np.sqrt(max(np.log2(n), 1.0))
    for p in (2, 3, 5, 7, 11):
        while n % p == 0:
            n //= p
    return t * (1.3 if dtype == torch.complex64 else 2.0) * (
        1.0 if n == 1 else 2.0)


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("n", LENGTHS)
def test_lines(n, dtype):
    g = torch.Generator(device="cuda").manual_seed(n)
    for shape, ax in (((1, n), 1), ((7, n), 1), ((n, 1), 0), ((n, 37), 0),
                      ((2, n, 5), 1)):
        if n > 20000 and shape[0] * shape[-1] > 7 * n:
            continue
        a = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
        keep = a.clone()
        for fwd in (True, False):
            r = fft.c2c(a, axes=[ax], forward=fwd, inorm=0 if fwd else 2)
            f = torch.fft.fft if fwd else torch.fft.ifft
            e = f(a.to(torch.complex128), dim=ax)
            err = ((r - e).norm() / e.norm()).item()
            assert err < tol(dtype, n), (shape, err)
            assert torch.equal(a, keep)


@pytest.mark.parametrize("n,eps,dtype,coord", [
    (700, 1e-5, torch.complex64, torch.float32),
    (5000, 1e-9, torch.complex128, torch.float64),
    (9001, 1e-5, torch.complex64, torch.float64),
    (100003, 1e-4, torch.complex64, torch.float64),
    (60000, 1e-9, torch.complex128, torch.float64)])
def test_long_rows_nufft(n, eps, dtype, coord):
    """1-D transforms whose grid is one long line, both types and orders"""
    rng = np.random.default_rng(n)
    M = 300
    x = rng.uniform(-np.pi, np.pi, M)
    x = x.astype(np.float32 if coord == torch.float32 else np.float64)
    k = np.arange(n) - n // 2
    E = np.exp(1j * np.outer(x.astype(np.float64), k))
    p = rng.standard_normal(M) + 1j * rng.standard_normal(M)
    c = rng.standard_normal(n) + 1j * rng.standard_normal(n)
    xt = torch.from_numpy(x).cuda()[:, None]
    pt = torch.from_numpy(p).cuda().to(dtype)
    ct = torch.from_numpy(c).cuda().to(dtype)
    # float32 coordinates are folded in double: no error beyond eps
    lim = 4 * eps + (2e-6 if dtype == torch.complex64 else 1e-13)
    for fo in (False, True):
        sh = (lambda a: np.fft.ifftshift(a)) if fo else (lambda a: a)
        out = torch.empty(n, dtype=dtype, device="cuda")
        nufft.nu2u(points=pt, coord=xt, forward=True, epsilon=eps, out=out,
                   fft_order=fo)
        e = sh(E.conj().T @ p)
        assert np.linalg.norm(out.cpu().numpy() - e) <= lim * np.linalg.norm(e)
        g = torch.from_numpy(sh(ct.cpu().numpy()).copy()).cuda()
        v = nufft.u2nu(grid=g, coord=xt, forward=False, epsilon=eps,
                       fft_order=fo)
        e = E @ c
        assert np.linalg.norm(v.cpu().numpy() - e) <= lim * np.linalg.norm(e)


def c2c_factor(a, out, axes, forward, fct):
    """dmx_c2c with any factor (the Python call has 1, 1/N and 1/sqrt N)"""
    da, ka = _lib.describe(a)
    do, ko = _lib.describe(out)
    ax = np.asarray(axes, dtype=np.int64)
    opt = _lib.options(stream=torch.cuda.current_stream().cuda_stream)
    _lib.check(_lib.lib().dmx_c2c(ct.byref(da), ct.byref(do), ax.ctypes.data,
                                  len(axes), int(forward), float(fct), 1,
                                  ct.byref(opt)))


# (shape, axes): lines in LDS; strided lines; the two column passes; two
# passes over long lines; global passes; Bluestein first and last; an axis of
# length 1 alone
@pytest.mark.parametrize("shape,axes", [
    ((5, 64), [1]), ((64, 5), [0]), ((1024, 24), [0, 1]), ((2, 16384), [1]),
    ((20000, 3), [0]), ((3, 1009), [1]), ((12, 101), [0, 1]), ((1, 7), [0])])
@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
def test_factor(shape, axes, dtype):
    """out = fct * DFT(in) for every factor, zero among them, whichever step
    applies it: contiguous, strided and real input, out of place and in
    place"""
    g = torch.Generator(device="cuda").manual_seed(7)
    n = int(np.prod([shape[a] for a in axes]))
    a = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
    wide = torch.zeros((shape[0], 2 * shape[1]), dtype=dtype, device="cuda")
    wide[:, ::2] = a
    for x in (a, wide[:, ::2], a.real.contiguous()):
        e = torch.fft.fftn(x.to(torch.complex128), dim=axes)
        for fct in (0.0, 0.3, -2.0, 1.0):
            # (not a zero-filled array: every element has to be written)
            out = torch.full(shape, 3.0, dtype=dtype, device="cuda")
            c2c_factor(x, out, axes, True, fct)
            d = (out - fct * e).norm().item()
            # (the factor rounds once more)
            assert d <= abs(fct) * 2 * tol(dtype, n) * e.norm().item(), fct
            if x is a:
                y = x.clone()
                c2c_factor(y, y, axes, True, fct)
                assert torch.equal(y, out)


@pytest.mark.parametrize("dtype", [torch.complex64, torch.complex128])
@pytest.mark.parametrize("shape,ax", [
    ((512, 8203), 0), ((256, 9001), 0), ((630, 517), 0), ((1021, 84), 1),
    ((4001, 110), 1), ((9, 1 << 18), 1), ((3, 1 << 20), 1)])
def test_full_workgroups(shape, ax, dtype):
    """as many lines as a workgroup takes, the last one partly filled:
    strided and contiguous lines, and both passes of long ones (their
    padded lines take more than 64 KiB of LDS)"""
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn(shape, dtype=dtype, device="cuda", generator=g)
    r = fft.c2c(a, axes=[ax])
    e = torch.fft.fft(a.to(torch.complex128), dim=ax)
    assert ((r - e).norm() / e.norm()).item() < tol(dtype, shape[ax])


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n0,rest", [
    (255, (100, 120)), (511, (8, 9)), (1023, (8, 9)), (2047, (8, 9))])
def test_full_workgroups_3d(gpu, n0, rest, dtype):
    """3-D grids whose strided axis is 512, 1024, 2048 or 4096 long: full
    workgroups with padded lines, both types"""
    single = dtype == np.complex64
    idx = kernel_rows(2.0, 3, single)[6 if single else 9][0]
    shape = (n0,) + rest
    rng = np.random.default_rng(n0)
    M = 2000
    c = rng.uniform(-np.pi, np.pi, (M, 3))
    p = (rng.standard_normal(M) + 1j * rng.standard_normal(M)).astype(dtype)
    q = (rng.standard_normal(shape) +
         1j * rng.standard_normal(shape)).astype(dtype)
    out = np.empty(shape, dtype)
    info = {}
    nufft.nu2u(points=p, coord=c, forward=True, epsilon=1e-3, out=out,
               kernel_idx=idx, info=info)
    assert info["nover"][0] == 2 * (n0 + 1)
    # the row's error (2e-5 and 3e-8 of the result's norm) over 64 entries
    lim = 2 * info["eps_tab"] + (2e-6 if single else 0)
    sel = rng.integers(0, out.size, 64)
    ref = nufft.nudft_direct(1, c, p, shape, True, sel)
    rms = np.linalg.norm(out) / np.sqrt(out.size)
    assert np.linalg.norm(out.reshape(-1)[sel] - ref) <= lim * 8 * rms
    v = nufft.u2nu(grid=q, coord=c, forward=False, epsilon=1e-3,
                   kernel_idx=idx)
    sel = np.arange(64)
    ref = nufft.nudft_direct(2, c, q, shape, False, sel)
    rms = np.linalg.norm(v) / np.sqrt(M)
    assert np.linalg.norm(v[sel] - ref) <= lim * 8 * rms


def test_many_long_lines(gpu):
    """more than 65535 lines beyond LDS (4096 elements in double precision),
    by themselves and as the rows of a 2-D grid"""
    n, L = 65536 + 70, 4116
    g = torch.Generator(device="cuda").manual_seed(3)
    a = torch.randn((n, L), dtype=torch.complex128, device="cuda",
                    generator=g)
    rows = [0, 1, 65534, 65535, 65536, n - 1]
    e = torch.fft.fft(a[rows], dim=1)
    r = fft.c2c(a, axes=[1], out=a)
    for i, q in enumerate(rows):
        d = ((r[q] - e[i]).norm() / e[i].norm()).item()
        assert d < tol(torch.complex128, L), q
    del a, r
    shape = (33000, 2048)
    idx = kernel_rows(2.0, 2, False)[5][0]
    rng = np.random.default_rng(1)
    M = 50
    c = torch.from_numpy(rng.uniform(-np.pi, np.pi, (M, 2))).cuda()
    E = [torch.polar(torch.ones((), dtype=torch.float64, device="cuda"),
                     torch.outer(c[:, d], torch.arange(
                         s, dtype=torch.float64, device="cuda") - s // 2))
         for d, s in enumerate(shape)]
    p = torch.randn(M, dtype=torch.complex128, device="cuda", generator=g)
    info = {}
    out = torch.empty(shape, dtype=torch.complex128, device="cuda")
    nufft.nu2u(points=p, coord=c, forward=False, epsilon=1e-3, out=out,
               kernel_idx=idx, info=info)
    assert info["nover"][0] > 65535 and info["nover"][1] == L
    lim = 2 * info["eps_tab"]
    ref = (E[0] * p[:, None]).T.contiguous() @ E[1]
    assert (out - ref).norm().item() <= lim * ref.norm().item()
    q = torch.randn(shape, dtype=torch.complex128, device="cuda",
                    generator=g)
    v = nufft.u2nu(grid=q, coord=c, forward=False, epsilon=1e-3,
                   kernel_idx=idx)
    ref = ((E[0] @ q) * E[1]).sum(1)
    assert (v - ref).norm().item() <= lim * ref.norm().item()


@pytest.mark.parametrize("shape,ax,most", [
    ((512, 4096), 1, 1.19e-7), ((2048, 2048), 1, 1.124e-7),
    ((81, 4096), 0, 1.01e-7), ((4096, 729), 1, 1.285e-7)])
def test_wide_radices_round_no_more(shape, ax, most):
    """single precision: lines of radices 16 and 9 are no further from the
    64-bit transform than with radices 8 and 3 (`most`)"""
    s = q = 0.0
    for seed in range(3):
        g = torch.Generator(device="cuda").manual_seed(seed)
        a = torch.randn(shape, dtype=torch.complex64, device="cuda",
                        generator=g)
        r = fft.c2c(a, axes=[ax])
        e = torch.fft.fft(a.to(torch.complex128), dim=ax)
        s += (r - e).norm().item() ** 2
        q += e.norm().item() ** 2
    assert np.sqrt(s / q) <= most
