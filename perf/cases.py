"""The work that users of ducc_amd have it do, as measurable cases.

A case is a dict of plain values.  Its "op" is the entry point:

  nu2u / u2nu   ducc_amd.nufft.nu2u / u2nu on device tensors (points sorted
                in the call), 1-D to 3-D
  plan          ducc_amd.nufft.plan, executed: u2nu and then nu2u with the
                other sign, the normal operator of an iterative solver
  grad          ducc_amd.torch_nufft.u2nu, forward and backward (gradients of
                the grid and of the coordinates)
  c2c           ducc_amd.fft.c2c
  sht           ducc_amd.sht.synthesis_general and adjoint_synthesis_general
  wgrid         ducc_amd.wgridder.vis2dirty and dirty2vis

and the rest are its sizes and options.  `exact` restates every operation as
direct sums in 64 bits (torch matrix products), without the package's code.
"""
import math

import numpy as np
import torch

DEV = "cuda"
C = 299792458.0  # m/s


# --------------------------------------------------------------- the cases
def listed():
    return [
        # the smallest call: a handful of points on a small grid, as in an
        # inner loop over many little problems; launches and host work
        dict(name="nu2u_2d_small", op="nu2u", shape="64x48", M=2000,
             eps=1e-6, dtype="c128", coord="f64", points="uniform",
             forward=True, fft_order=False),
        # an accurate 2-D type 1 of moderate size in double precision (the
        # configuration c1 of ducc_amd/configs_bench.py)
        dict(name="nu2u_2d_f64", op="nu2u", shape="256x256", M=100_000,
             eps=1e-9, dtype="c128", coord="f64", points="uniform",
             forward=True, fft_order=False),
        # spectra of long, unevenly sampled series: 1-D, an odd length far
        # beyond what fits a workgroup, single-precision coordinates
        dict(name="u2nu_1d_odd", op="u2nu", shape="100003", M=1_000_000,
             eps=1e-4, dtype="c64", coord="f32", points="uniform",
             forward=False, fft_order=True),
        # the benchmark's workload, one direction each: 1e7 clustered points,
        # 2048 x 2048 modes, eps 1e-5, single precision
        dict(name="nu2u_2d_large", op="nu2u", shape="2048x2048",
             M=10_000_000, eps=1e-5, dtype="c64", coord="f64",
             points="clustered", forward=True, fft_order=False),
        dict(name="u2nu_2d_large", op="u2nu", shape="2048x2048",
             M=10_000_000, eps=1e-5, dtype="c64", coord="f64",
             points="clustered", forward=True, fft_order=False),
        # 3-D imaging, type 1 (c3 of ducc_amd/configs_bench.py)
        dict(name="nu2u_3d_large", op="nu2u", shape="256x256x256",
             M=50_000_000, eps=1e-4, dtype="c64", coord="f64",
             points="uniform", forward=True, fft_order=False),
        # 3-D type 2 in double precision on a box of unequal sides
        dict(name="u2nu_3d_f64", op="u2nu", shape="96x100x108", M=1_000_000,
             eps=1e-9, dtype="c128", coord="f64", points="clustered",
             forward=True, fft_order=False),
        # one iteration of a solver that keeps its plan: the normal operator
        # on an image of unequal, odd sides, all in single precision
        dict(name="plan_2d_normal", op="plan", shape="1023x768",
             M=1_500_000, eps=1e-4, dtype="c64", coord="f32",
             points="uniform", forward=True, fft_order=False),
        # a differentiable transform inside a model (c4 of
        # ducc_amd/configs_bench.py): forward and both gradients
        dict(name="grad_2d", op="grad", shape="512x512", M=2_000_000,
             eps=1e-6, dtype="c64", coord="f64", points="uniform",
             forward=True, fft_order=False),
        # the FFT by itself (bench.py --workload c2c)
        dict(name="c2c_2d_large", op="c2c", shape="4096x4096", dtype="c64",
             axes="all", forward=True),
        # spin-2 fields on the sphere at arbitrary points, both directions
        # (bench.py --workload sht --spin 2, the CMB lensing geometry)
        dict(name="sht_spin2", op="sht", lmax=1187, spin=2, npt=2_000_000,
             eps=1e-7, dtype="c128"),
        # radio imaging with w-gridding, both directions (bench.py
        # --workload wgridder)
        dict(name="wgrid_large", op="wgrid", nrow=20_000, nchan=64,
             npix=2472, fov=5.0, eps=1e-4, dtype="c64", wgridding=True),
    ]


def _log(rng, lo, hi):
    """an integer spread over the logarithm of [lo, hi]"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """Another case of the same ranges.  Taps (points times kernel support
    to the dimension) stay at half of the largest listed case's, sides at
    the listed ones."""
    op = rng.choice(["nu2u", "u2nu", "nu2u", "u2nu", "plan", "grad", "c2c",
                     "sht", "wgrid"])
    dtype = rng.choice(["c64", "c128"])
    fwd = rng.random() < 0.5
    if op == "c2c":
        nd = rng.choice([1, 2, 2, 3])
        top = {1: 1_000_000, 2: 4096, 3: 256}[nd]
        # lines that are smooth, odd or prime alike
        shape = [_log(rng, 8, top) for _ in range(nd)]
        axes = rng.choice(["all", "all", "first", "last"])
        return dict(op=op, shape="x".join(map(str, shape)), dtype=dtype,
                    axes=axes, forward=fwd)
    if op == "sht":
        return dict(op=op, lmax=_log(rng, 32, 1187),
                    spin=rng.choice([0, 0, 1, 2]),
                    npt=_log(rng, 2000, 2_000_000),
                    eps=10.0 ** -rng.randint(4, 5 if dtype == "c64" else 9),
                    dtype=dtype)
    if op == "wgrid":
        return dict(op=op, nrow=_log(rng, 300, 20_000),
                    nchan=_log(rng, 1, 64), npix=2 * _log(rng, 60, 1236),
                    fov=round(rng.uniform(1.0, 5.0), 2),
                    eps=10.0 ** -rng.randint(2, 4 if dtype == "c64" else 7),
                    dtype=dtype, wgridding=rng.random() < 0.7)
    nd = rng.choice([2] if op == "grad" else [1, 2, 2, 3])
    top = {1: 1_000_000, 2: 2048, 3: 256}[nd]
    shape = [_log(rng, 24, top) for _ in range(nd)]
    digits = rng.randint(2, 6 if dtype == "c64" else 11)
    coord = rng.choice(["f32", "f64"])
    if op == "plan":  # a plan's values have its coordinates' precision
        coord = "f32" if dtype == "c64" else "f64"
    if coord == "f32":  # coordinates that carry no more digits
        digits = min(digits, 6)
    most = min(10_000_000, 5e9 / (digits + 2.0) ** nd)
    return dict(op=op, shape="x".join(map(str, shape)),
                M=_log(rng, 1000, most), eps=10.0 ** -digits, dtype=dtype,
                coord=coord, points=rng.choice(["uniform", "clustered"]),
                forward=fwd, fft_order=rng.random() < 0.3)


# -------------------------------------------------------------- the inputs
def _shape(case):
    return tuple(int(s) for s in case["shape"].split("x"))


def _types(case):
    return ((torch.complex64, torch.float32) if case["dtype"] == "c64"
            else (torch.complex128, torch.float64))


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(1000003 * seed + 17)


def _normal(shape, dtype, g):
    return torch.randn(shape, dtype=dtype, device=DEV, generator=g)


def _unit(shape, dtype, g):
    """uniform in [0, 1)"""
    return torch.rand(shape, dtype=dtype, device=DEV, generator=g)


def _coords(case, g):
    """(M, ndim) in [-pi, pi): uniform, or eight Gaussian clusters of
    0.3 rad as in the benchmark"""
    M, nd = case["M"], len(_shape(case))
    if case["points"] == "uniform":
        c = (_unit((M, nd), torch.float64, g) - 0.5) * (2 * math.pi)
    else:
        cen = (_unit((8, nd), torch.float64, g) - 0.5) * (2 * math.pi)
        lab = torch.randint(0, 8, (M,), device=DEV, generator=g)
        c = cen[lab] + 0.3 * _normal((M, nd), torch.float64, g)
        c = torch.remainder(c + math.pi, 2 * math.pi) - math.pi
    return c.to(torch.float32 if case["coord"] == "f32" else torch.float64)


def _alm_start(lmax):
    """start[m] with a_lm at start[m] + l (mmax = lmax)"""
    m = np.arange(lmax + 1)
    return m * (2 * lmax + 1 - m) // 2


def _inputs(case, seed):
    g = _gen(seed)
    op = case["op"]
    cdt, rdt = _types(case)
    if op == "c2c":
        return dict(a=_normal(_shape(case), cdt, g))
    if op == "sht":
        lmax, spin, npt = case["lmax"], case["spin"], case["npt"]
        nc = 1 if spin == 0 else 2
        n = (lmax + 1) * (lmax + 2) // 2
        alm = 2 * torch.complex(_unit((nc, n), torch.float64, g),
                                _unit((nc, n), torch.float64, g)) - (1 + 1j)
        alm[:, :lmax + 1].imag = 0.0  # m = 0: real fields
        for m in range(min(spin, lmax + 1)):  # l < spin: none
            s = int(_alm_start(lmax)[m])
            alm[:, s + m:s + spin] = 0.0
        # a Fibonacci lattice, turned by the seed
        i = torch.arange(npt, dtype=torch.float64, device=DEV)
        turn = _unit((1,), torch.float64, g)
        theta = torch.arccos(1.0 - (2.0 * i + 1.0) / npt)
        phi = torch.remainder(i * (2.0 / (1.0 + math.sqrt(5.0))) + turn, 1.0)
        loc = torch.stack([theta, phi * (2 * math.pi)], dim=1).contiguous()
        mp = 2 * _unit((nc, npt), torch.float64, g) - 1
        return dict(alm=alm.to(cdt), loc=loc, map=mp.to(rdt))
    if op == "wgrid":
        nrow, nchan, npix = case["nrow"], case["nchan"], case["npix"]
        freq = 1e9 + torch.arange(nchan, dtype=torch.float64,
                                  device=DEV) * (1e9 / nchan)
        # baselines that this image samples at half its Nyquist rate and up
        fov = case["fov"] * math.pi / 180
        longest = npix / (2 * fov) * C / 2e9
        uvw = (_unit((nrow, 3), torch.float64, g) - 0.5) * torch.tensor(
            [1.38, 1.38, 0.46], dtype=torch.float64, device=DEV) * longest
        vis = torch.complex(_unit((nrow, nchan), rdt, g),
                            _unit((nrow, nchan), rdt, g)) - (0.5 + 0.5j)
        wgt = _unit((nrow, nchan), rdt, g) + 0.5
        dirty = _unit((npix, npix), rdt, g) - 0.5
        return dict(uvw=uvw, freq=freq, vis=vis, wgt=wgt, dirty=dirty,
                    pix=fov / npix)
    d = dict(coord=_coords(case, g))
    if op in ("nu2u", "grad"):
        d["points"] = _normal((case["M"],), cdt, g)
    if op in ("u2nu", "plan", "grad"):
        d["grid"] = _normal(_shape(case), cdt, g)
    return d


def prepare(case, seed):
    d = dict(_inputs(case, seed), case=case)
    op = case["op"]
    cdt, rdt = _types(case)
    if op == "nu2u":
        d["out"] = torch.empty(_shape(case), dtype=cdt, device=DEV)
    elif op == "plan":
        from ducc_amd import nufft
        d["plan"] = nufft.plan(nu2u=False, coord=d["coord"],
                               grid_shape=_shape(case), epsilon=case["eps"],
                               fft_order=case["fft_order"])
    elif op == "grad":
        d["grid"].requires_grad_(True)
        d["coord"].requires_grad_(True)
    elif op == "sht":
        d["alm_out"] = torch.zeros_like(d["alm"])
    return d


# ----------------------------------------------------------------- one pass
def _axes(case):
    nd = len(_shape(case))
    return {"all": list(range(nd)), "first": [0], "last": [nd - 1]}[
        case["axes"]]


def run(st):
    case = st["case"]
    op = case["op"]
    if op in ("nu2u", "u2nu"):
        from ducc_amd import nufft
        kw = dict(coord=st["coord"], forward=case["forward"],
                  epsilon=case["eps"], fft_order=case["fft_order"])
        if op == "nu2u":
            return nufft.nu2u(points=st["points"], out=st["out"], **kw)
        return nufft.u2nu(grid=st["grid"], **kw)
    if op == "plan":
        v = st["plan"].u2nu(grid=st["grid"], forward=case["forward"])
        h = st["plan"].nu2u(points=v, forward=not case["forward"])
        return {"values": v, "normal": h}
    if op == "grad":
        from ducc_amd import torch_nufft
        v = torch_nufft.u2nu(st["grid"], st["coord"], case["forward"],
                             eps=case["eps"], fft_order=case["fft_order"])
        gg, gc = torch.autograd.grad(v, (st["grid"], st["coord"]),
                                     st["points"])
        return {"values": v.detach(), "grid_grad": gg, "coord_grad": gc}
    if op == "c2c":
        from ducc_amd import fft
        return fft.c2c(st["a"], axes=_axes(case), forward=case["forward"])
    if op == "sht":
        from ducc_amd import sht
        kw = dict(spin=case["spin"], lmax=case["lmax"], loc=st["loc"],
                  epsilon=case["eps"])
        m = sht.synthesis_general(alm=st["alm"], **kw)
        a = sht.adjoint_synthesis_general(map=st["map"], alm=st["alm_out"],
                                          **kw)
        return {"map": m, "alm": a}
    from ducc_amd import wgridder
    kw = dict(uvw=st["uvw"], freq=st["freq"], wgt=st["wgt"],
              pixsize_x=st["pix"], pixsize_y=st["pix"], epsilon=case["eps"],
              do_wgridding=case["wgridding"])
    dirty = wgridder.vis2dirty(vis=st["vis"], npix_x=case["npix"],
                               npix_y=case["npix"], **kw)
    vis = wgridder.dirty2vis(dirty=st["dirty"], **kw)
    return {"dirty": dirty, "vis": vis}


# ----------------------------------------------------- the work of one pass
def work(case):
    """Inputs read once and outputs written once; the operations of the FFT
    of the modes alone (5 N log2 N, without oversampling) and of one tap per
    digit of eps and axis."""
    op = case["op"]
    sv = 8 if case["dtype"] == "c64" else 16
    if op == "c2c":
        s = _shape(case)
        N = math.prod(s)
        return dict(bytes=2 * N * sv, flops=sum(
            5 * N * math.log2(max(s[a], 2)) for a in _axes(case)))
    if op == "sht":
        nc = 1 if case["spin"] == 0 else 2
        L, npt = case["lmax"] + 1, case["npt"]
        taps = max(2, round(-math.log10(case["eps"]))) ** 2
        # two operations per (l, m, ring pair) and component of a_lm, each
        # of two real parts, both ways, and the recursion's three
        return dict(bytes=2 * npt * (16 + nc * sv // 2) + nc * L * L * sv,
                    flops=2 * (L * L / 2 * L / 2 * (3 + 4 * nc) * nc +
                               4 * npt * taps +
                               10 * L * L * math.log2(4 * L * L)))
    if op == "wgrid":
        nvis, N = case["nrow"] * case["nchan"], case["npix"] ** 2
        taps = max(2, round(-math.log10(case["eps"]))) ** (
            3 if case["wgridding"] else 2)
        return dict(bytes=2 * (24 * case["nrow"] + nvis * (sv + sv // 2) +
                               N * sv // 2),
                    flops=2 * (4 * nvis * taps + 5 * N * math.log2(N)))
    s = _shape(case)
    M, N, nd = case["M"], math.prod(s), len(s)
    sc = 4 if case["coord"] == "f32" else 8
    taps = max(2, round(-math.log10(case["eps"]))) ** nd
    b = M * (nd * sc + sv) + N * sv
    f = 4 * M * taps + 5 * N * math.log2(max(N, 2))
    if op == "plan":
        b, f = 2 * b - M * nd * sc, 2 * f
    elif op == "grad":
        b, f = 2 * b + M * nd * sc, (2 + nd) * f
    return dict(bytes=b, flops=f)


def tolerance(case):
    """Four times the error measured against `exact`: the transforms answer
    to eps (0.3 eps in 2-D and 3-D and on the sphere, 0.6 eps in 1-D, 3 eps
    for coordinate gradients), on top of the sums' rounding (2.5e-7 in
    single precision between two runs, whose atomics add in another
    order)."""
    op = case["op"]
    single = case["dtype"] == "c64"
    if op == "c2c":
        return {"rel": 1e-6 if single else 4e-15}
    times = 10.0 if op == "grad" else 1.0
    if "shape" in case and len(_shape(case)) == 1:
        times = 2.0
    return {"rel": times * case["eps"] + (1e-6 if single else 1e-14)}


# ------------------------------------------------ the same in 64-bit sums
def _modes(n, fft_order):
    k = torch.arange(n, dtype=torch.float64, device=DEV) - n // 2
    return torch.roll(k, -(n // 2)) if fft_order else k


def _wave(x, k, s):
    """exp(i s x k), (len(x), len(k))"""
    a = torch.outer(s * x, k)
    return torch.polar(torch.ones_like(a), a)


def _split(case, grid=None):
    """1-D lengths as an array of two axes, k = k0 + B a + b, so that the
    sums are matrix products: (mode lists, array on them or None)"""
    s = _shape(case)
    if len(s) > 1:
        ks = [_modes(n, case["fft_order"]) for n in s]
        return ks, grid
    n = s[0]
    B = max(1, int(math.sqrt(n)))
    A = -(-n // B)
    ks = [torch.arange(A, dtype=torch.float64, device=DEV) * B - n // 2,
          torch.arange(B, dtype=torch.float64, device=DEV)]
    if grid is not None:
        g = torch.roll(grid, n // 2) if case["fft_order"] else grid
        full = torch.zeros(A * B, dtype=torch.complex128, device=DEV)
        full[:n] = g
        grid = full.reshape(A, B)
    return ks, grid


def _chunks(M, ks):
    rows = math.prod(len(k) for k in ks[:-1]) + len(ks[-1]) + len(ks[0])
    step = max(256, min(M, (1 << 27) // rows))
    return [(i, min(M, i + step)) for i in range(0, M, step)]


def _type2(case, grid, coord, sign, deriv=False):
    """values at the points (and, with deriv, the derivative along every
    axis, (M, ndim))"""
    ks, G = _split(case, grid.to(torch.complex128))
    x = coord.to(torch.float64)
    nd, M = len(_shape(case)), x.shape[0]
    out = torch.empty(M, dtype=torch.complex128, device=DEV)
    der = torch.zeros((M, nd), dtype=torch.complex128, device=DEV)
    G2 = G.reshape(-1, G.shape[-1]).T.contiguous()
    for i, j in _chunks(M, ks):
        xs = [x[i:j, 0]] * 2 if nd == 1 else [x[i:j, d] for d in range(nd)]
        E = [_wave(c, k, sign) for c, k in zip(xs, ks)]

        def total(F):
            t = (F[-1] @ G2).reshape((j - i,) + G.shape[:-1])
            for e in F[:-1]:
                t = (t * e.reshape(e.shape + (1,) * (t.dim() - 2))).sum(1)
            return t
        out[i:j] = total(E)
        if deriv:
            for q, k in enumerate(ks):
                F = list(E)
                F[q] = E[q] * (1j * sign * k)
                der[i:j, min(q, nd - 1)] += total(F)
    return (out, der) if deriv else out


def _type1(case, points, coord, sign):
    ks, _ = _split(case)
    p, x = points.to(torch.complex128), coord.to(torch.float64)
    s = _shape(case)
    nd, M = len(s), x.shape[0]
    G = torch.zeros((math.prod(len(k) for k in ks[:-1]), len(ks[-1])),
                    dtype=torch.complex128, device=DEV)
    for i, j in _chunks(M, ks):
        xs = [x[i:j, 0]] * 2 if nd == 1 else [x[i:j, d] for d in range(nd)]
        E = [_wave(c, k, sign) for c, k in zip(xs, ks)]
        t = E[0] * p[i:j, None]
        for e in E[1:-1]:
            t = (t[:, :, None] * e[:, None, :]).reshape(j - i, -1)
        G += t.T.contiguous() @ E[-1]
    if nd > 1:
        return G.reshape(s)
    g = G.reshape(-1)[:s[0]]
    return torch.roll(g, -(s[0] // 2)) if case["fft_order"] else g


def _wigner_rings(lmax, spin, theta):
    """yields l and sqrt((2l+1)/4pi) times the Wigner functions
    d^l_{m,-spin}(theta) and d^l_{m,spin}(theta) as (lmax + 1, len(theta))
    arrays over m: the three-term recursion in l from the closed form at
    l = max(m, spin)"""
    m = torch.arange(lmax + 1, dtype=torch.float64, device=DEV)[:, None]
    ct = torch.cos(theta)[None, :]
    lc = torch.log(torch.cos(theta / 2).abs())[None, :]
    ls = torch.log(torch.sin(theta / 2).abs())[None, :]
    l0 = torch.maximum(m, torch.full_like(m, float(spin)))
    lo = torch.minimum(m, torch.full_like(m, float(spin)))
    # d^{l0}: sqrt(binomial(2 l0, l0 - lo)) cos^a sin^b, a + b = 2 l0
    lb = 0.5 * (torch.lgamma(2 * l0 + 1) - torch.lgamma(l0 - lo + 1) -
                torch.lgamma(l0 + lo + 1))
    starts = []
    for s in (-spin, spin):
        a, b = (m + s).abs(), (m - s).abs()
        # (-1)^(m - s) where m > s: d^l_{m s} starts with (-sin)^(m - s)
        sg = torch.where((m > s) & ((m - s) % 2 == 1), -1.0, 1.0)
        starts.append(sg * torch.exp(
            lb + torch.where(a > 0, a * lc, torch.zeros_like(lc)) +
            torch.where(b > 0, b * ls, torch.zeros_like(ls))))
    cur = [torch.zeros((lmax + 1, theta.numel()), dtype=torch.float64,
                       device=DEV) for _ in range(2)]
    old = [torch.zeros_like(c) for c in cur]
    for l in range(lmax + 1):
        begin = l0 == l
        for q, s in enumerate((-spin, spin)):
            if l > 0:
                n = l - 1.0  # d^{n+1} from d^n and d^{n-1}
                den = n * torch.sqrt(torch.clamp(
                    (l * l - m * m) * (l * l - s * s), min=0.0))
                if n == 0:  # Legendre's first step (m = s = 0)
                    new = ct * cur[q]
                else:
                    new = ((2 * n + 1) * (n * l * ct - m * s) * cur[q] -
                           l * torch.sqrt(torch.clamp(
                               (n * n - m * m) * (n * n - s * s), min=0.0)) *
                           old[q]) / den
                new = torch.where(l0 < l, new, torch.zeros_like(new))
            else:
                new = torch.zeros_like(cur[q])
            new = torch.where(begin, starts[q], new)
            old[q], cur[q] = cur[q], new
        f = math.sqrt((2 * l + 1) / (4 * math.pi))
        yield l, f * cur[0], f * cur[1]


def _sphere(case, d):
    """Both directions through the trigonometric polynomial of the field:
    rings at N + 1 equidistant theta, an FFT in theta over the doubled
    sphere, direct sums at the points."""
    lmax, spin, npt = case["lmax"], case["spin"], case["npt"]
    nc, L1 = d["alm"].shape[0], lmax + 1
    N = 2 * ((lmax + 3) // 2) + 2
    theta = torch.arange(N + 1, dtype=torch.float64, device=DEV) * (
        math.pi / N)
    start = torch.from_numpy(_alm_start(lmax)).to(DEV)
    alm = d["alm"].to(torch.complex128)
    # rows theta_j, j = 0 .. 2N-1; columns m = -lmax .. lmax
    X = torch.zeros((2 * N, 2 * lmax + 1), dtype=torch.complex128,
                    device=DEV)
    case2 = dict(case, shape="%dx%d" % (2 * N, 2 * lmax + 1),
                 fft_order=False)
    E = torch.zeros((L1, N + 1), dtype=torch.complex128, device=DEV)
    F = torch.zeros_like(E)
    # the adjoint's spectrum: sums over the points against exp(-i k x)
    mp = d["map"].to(torch.complex128)
    pts = mp[0] if nc == 1 else torch.complex(d["map"][0].double(),
                                              d["map"][1].double())
    A = _type1(case2, pts, d["loc"], -1)
    A = torch.fft.ifft(torch.fft.ifftshift(A, dim=0), dim=0)
    par = torch.where((torch.arange(-lmax, L1, device=DEV) + spin) % 2 == 0,
                      1.0, -1.0).to(torch.float64)
    # fold the doubled rows (theta > pi) back onto 0 .. pi
    R = A[:N + 1].clone()
    R[1:N] += torch.flip(A[N + 1:], dims=[0]) * par[None, :]
    Rp, Rm = R[:, lmax:].T, torch.flip(R[:, :L1], dims=[1]).T  # (m, ring)
    out = torch.zeros_like(alm)
    odd = -1.0 if spin % 2 else 1.0
    for l, dn, dp in _wigner_rings(lmax, spin, theta):
        if l < spin:
            continue
        k = l + 1
        # order m: (-1)^s d_{m,-s}; order -m, with the symmetry of the a_lm:
        # d_{m,s}
        yp, ym = odd * dn[:k], dp[:k]
        at = start[:k] + l
        hp = (Rp[:k] * yp).sum(1)
        if nc == 1:
            E[:k] += alm[0, at][:, None] * yp
            out[0, at] = hp
            continue
        e, b = alm[0, at][:, None], alm[1, at][:, None]
        E[:k] -= (e + 1j * b) * yp
        F[:k] -= (e.conj() + 1j * b.conj()) * ym
        hm = (Rm[:k] * ym).sum(1).conj()
        out[0, at] = -(hp + hm) / 2
        out[1, at] = 1j * (hp - hm) / 2
    if nc == 1:
        F = E.conj()
    X[:N + 1, lmax:] = E.T
    X[:N + 1, :lmax] = torch.flip(F[1:].T, dims=[1])
    X[N + 1:] = torch.flip(X[1:N], dims=[0]) * par[None, :]
    Y = torch.fft.fftshift(torch.fft.fft(X, dim=0), dim=0) / (2 * N)
    v = _type2(case2, Y, d["loc"], 1)
    return {"map": torch.stack([v.real] if nc == 1 else [v.real, v.imag]),
            "alm": out}


def _radio(case, d):
    """direct sums over pixels and visibilities"""
    npix, pix = case["npix"], d["pix"]
    x = (torch.arange(npix, dtype=torch.float64, device=DEV) -
         npix // 2) * pix
    X, Y = [t.reshape(-1) for t in torch.meshgrid(x, x, indexing="ij")]
    r2 = X * X + Y * Y
    nm1 = -r2 / (torch.sqrt(1 - r2) + 1)
    n = nm1 + 1
    if not case["wgridding"]:
        nm1, n = torch.zeros_like(nm1), torch.ones_like(n)
    uvw = (d["uvw"][:, None, :] * (d["freq"] / C)[None, :, None]).reshape(
        -1, 3) * (2 * math.pi)
    v = (d["vis"].to(torch.complex128) * d["wgt"]).reshape(-1)
    D = (d["dirty"].double().reshape(-1) / n).to(torch.complex128)
    B = torch.stack([X, Y, -nm1])
    dirty = torch.zeros(npix * npix, dtype=torch.float64, device=DEV)
    vis = torch.empty_like(v)
    step = max(1, (1 << 26) // (npix * npix))
    for i in range(0, v.numel(), step):
        a = uvw[i:i + step] @ B
        w = torch.polar(torch.ones_like(a), a)
        dirty += (v[None, i:i + step] @ w)[0].real
        vis[i:i + step] = w.conj() @ D
    vis = vis.reshape(d["vis"].shape) * d["wgt"].double()
    return {"dirty": (dirty / n).reshape(npix, npix), "vis": vis}


def exact(case, seed):
    op = case["op"]
    if op == "wgrid" and case["nrow"] * case["nchan"] * case["npix"] ** 2 \
            > 1.5e11:
        return None
    if op not in ("c2c", "sht", "wgrid") and \
            case["M"] * math.prod(_shape(case)) > 5e13:
        return None
    d = _inputs(case, seed)
    if op == "c2c":
        f = torch.fft.fftn if case["forward"] else torch.fft.ifftn
        return f(d["a"].to(torch.complex128), dim=_axes(case),
                 norm="backward" if case["forward"] else "forward")
    if op == "sht":
        return _sphere(case, d)
    if op == "wgrid":
        return _radio(case, d)
    s = -1 if case["forward"] else 1
    if op == "nu2u":
        return _type1(case, d["points"], d["coord"], s)
    if op == "u2nu":
        return _type2(case, d["grid"], d["coord"], s)
    if op == "plan":
        v = _type2(case, d["grid"], d["coord"], s)
        return {"values": v, "normal": _type1(case, v, d["coord"], -s)}
    v, der = _type2(case, d["grid"], d["coord"], s, deriv=True)
    p = d["points"].to(torch.complex128)
    return {"values": v, "grid_grad": _type1(case, p, d["coord"], -s),
            "coord_grad": (p[:, None] * der.conj()).real}
