"""The work a user has this library do, as cases that can be timed and checked.

A case is a dict of plain values; its "kind" names the entry point:

  rhs      FullRHS.eval: the incompressible right-hand side of a triply
           periodic n^3 grid (nine cd06 gradients, nine cf90 filters, the
           divergence, the FFT Poisson solve and the projection)
  grad     operators%gradient on a derivatives object (cd10 or cd06)
  filter   one cf90 pass along x, y and z on a filters object
  cgrid    getRHS of the compressible solver, viscous, with the artificial
           diffusivities
  igrid    a velocity set into the incompressible solver and one step of it
  closure  the learned subgrid stress of a velocity-gradient field

Fields lie x fastest, so a field (nx, ny, nz) is a torch tensor (nz, ny, nx).
exact() restates each path in FP64 torch: the line operators as dense
matrices A^-1 B built from the schemes' coefficients, the transforms as
torch.fft.
"""
import functools
import math

import numpy as np
import torch

import padeops_amd as P

PI2 = 2 * math.pi
DT = {"f64": torch.float64, "f32_refine": torch.float32}


def listed():
    return [
        # a right-hand side of a small box, as test and tuning runs call it: launches and their latency
        dict(name="rhs_32_f64", kind="rhs", n=32, prec="f64"),
        # an ordinary resolution in the reference's own precision
        dict(name="rhs_256_f64", kind="rhs", n=256, prec="f64"),
        # the benchmark's workload in its benchmark precision
        dict(name="rhs_512_f32r", kind="rhs", n=512, prec="f32_refine"),
        # post-processing of a wall-bounded field on a grid of odd sizes: one-sided ends in y, symmetric in x
        dict(name="grad_walls_201x129x151_f64", kind="grad", nx=201, ny=129, nz=151, method="cd10", prec="f64",
             px=False, py=False, pz=True, xb=1, xn=-1, yb=0, yn=0, zb=0, zn=0),
        # gradients of a large periodic field whose sizes are no powers of two (one above 512)
        dict(name="grad_384x320x640_f32r", kind="grad", nx=384, ny=320, nz=640, method="cd06", prec="f32_refine",
             px=True, py=True, pz=True, xb=0, xn=0, yb=0, yn=0, zb=0, zn=0),
        # de-aliasing filter of a channel field: periodic x and z, walls in y, ragged sizes
        dict(name="filter_300x161x200_f64", kind="filter", nx=300, ny=161, nz=200, prec="f64",
             px=True, py=False, pz=True, xb=0, xn=0, yb=0, yn=0, zb=0, zn=0),
        # the compressible right-hand side at the benchmark's size
        dict(name="cgrid_256_f64", kind="cgrid", nx=256, ny=256, nz=256, prec="f64",
             px=True, py=True, pz=True, xb=0, xn=0, yb=0, yn=0, zb=0, zn=0),
        # a compressible box between a symmetry plane and open ends in x, on a ragged grid, in the fast precision
        dict(name="cgrid_walls_180x96x100_f32r", kind="cgrid", nx=180, ny=96, nz=100, prec="f32_refine",
             px=False, py=True, pz=True, xb=1, xn=0, yb=0, yn=0, zb=0, zn=0),
        # one step of a small isotropic LES (the closure study's coarse grid): a few hundred short launches
        dict(name="igrid_les_64_f32r", kind="igrid", nx=64, ny=64, nz=64, walls=False, Re=600.0, sgs="smagorinsky",
             prec="f32_refine"),
        # one step of the isotropic DNS that the closure study takes its data from
        dict(name="igrid_dns_256_f64", kind="igrid", nx=256, ny=256, nz=256, walls=False, Re=600.0, sgs="none",
             prec="f64"),
        # one step of the wall-modelled LES at the benchmark's size
        dict(name="igrid_wall_les_512x512x256_f32r", kind="igrid", nx=512, ny=512, nz=256, walls=True, Re=0.0,
             sgs="smagorinsky", prec="f32_refine"),
        # the learned stress of a 256^3 field of gradients, as a solver asks for it at every stage
        dict(name="closure_256_f32", kind="closure", npts=256 ** 3, prec="f32_refine"),
    ]


def draw(rng):
    kind = rng.choice(["rhs", "grad", "grad", "filter", "cgrid", "cgrid", "igrid", "igrid", "closure"])
    prec = rng.choice(["f64", "f32_refine"])

    def size(lo, hi):
        n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
        # grids are as often round numbers as odd ones
        return max(lo, min(hi, rng.choice([n, n, n | 1, 8 * ((n + 4) // 8), 32 * ((n + 16) // 32)])))

    def sizes(lo, hi, most):
        while True:
            s = [size(lo, hi) for _ in range(3)]
            if s[0] * s[1] * s[2] <= most:
                return dict(zip(("nx", "ny", "nz"), s))

    def ends(kinds):
        c = {}
        for d in "xyz":
            per = rng.random() < 0.6
            c["p" + d] = per
            c[d + "b"] = 0 if per else rng.choice(kinds)
            c[d + "n"] = 0 if per else rng.choice(kinds)
        return c

    if kind == "rhs":
        return dict(kind=kind, n=2 ** rng.randint(5, 9 if prec == "f32_refine" else 8), prec=prec)
    if kind == "grad":
        method = rng.choice(["cd10", "cd10", "cd06"])
        return dict(kind=kind, method=method, prec=prec, **sizes(16, 640, 40_000_000),
                    **ends([0, 0, 1, -1] if method == "cd10" else [0]))
    if kind == "filter":
        return dict(kind=kind, prec=prec, **sizes(16, 640, 40_000_000), **ends([0, 0, 1]))
    if kind == "cgrid":
        return dict(kind=kind, prec=prec, **sizes(24, 320, 8_000_000), **ends([0, 1]))
    if kind == "igrid":
        walls = rng.random() < 0.4
        n = [2 ** rng.randint(5, 8) for _ in range(3)]
        if walls:
            n[2] = min(n[2], 128)
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], walls=walls, Re=0.0 if walls else rng.choice([150.0, 600.0]),
                    sgs="smagorinsky" if walls else rng.choice(["none", "smagorinsky", "amd"]), prec=prec)
    return dict(kind=kind, npts=int(math.exp(rng.uniform(math.log(30_000), math.log(20_000_000)))), prec=prec)


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _fields(count, nx, ny, nz, seed, k0=None):
    """`count` random fields (nz, ny, nx) of zero mean and unit rms with a
    turbulence spectrum: E ~ k^4 exp(-2 (k/k0)^2), or, without k0, a plateau
    up to k = 4 followed by a k^-5/3 range (density ~ k^-11/3)."""
    dev = _dev()
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    f = lambda n: torch.fft.fftfreq(n, d=1.0 / n, device=dev, dtype=torch.float64)  # noqa: E731
    k = torch.sqrt(f(nz).view(-1, 1, 1) ** 2 + f(ny).view(1, -1, 1) ** 2
                   + torch.arange(nx // 2 + 1, device=dev, dtype=torch.float64).view(1, 1, -1) ** 2)
    amp = (16.0 + k * k) ** (-11.0 / 12.0) if k0 is None else k * torch.exp(-(k / k0) ** 2)
    amp[0, 0, 0] = 0.0
    out = []
    for _ in range(count):
        h = torch.fft.rfftn(torch.randn((nz, ny, nx), generator=g, device=dev, dtype=torch.float64)) * amp
        u = torch.fft.irfftn(h, s=(nz, ny, nx))
        out.append(u / u.square().mean().sqrt())
    return out


def _net(seed):
    """padded parameters of a 10-64-64-64-6 network, He-initialised as for training"""
    r = np.random.default_rng(seed)
    sizes = (10, 64, 64, 64, 6)
    return [(r.normal(0, math.sqrt(2.0 / a), (b, a)).astype(np.float32), r.normal(0, 0.05, b).astype(np.float32))
            for a, b in zip(sizes[:-1], sizes[1:])]


def _inputs(case, seed):
    """the input tensors of a case in its storage type, shape (nz, ny, nx) each"""
    dt = DT[case["prec"]]
    kind = case["kind"]
    if kind == "closure":
        return [_gradients(case["npts"], seed).to(dt)]
    nx, ny, nz = (case["n"],) * 3 if kind == "rhs" else (case["nx"], case["ny"], case["nz"])
    if kind == "rhs":
        v = _fields(3, nx, ny, nz, seed, 8.0)
    elif kind in ("grad", "filter"):
        v = _fields(1, nx, ny, nz, seed)
    elif kind == "cgrid":
        f = _fields(5, nx, ny, nz, seed, 4.0)
        rho, p = 1.0 + 0.05 * f[0], 1.0 + 0.05 * f[4]
        u = [0.2 * q for q in f[1:4]]
        e = p / (0.4 * rho) + 0.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
        v = [rho, rho * u[0], rho * u[1], rho * u[2], rho * e]
    else:
        v = _fields(3, nx, ny, nz, seed, 6.0)
        w = v[2]
        if case["walls"]:
            # the log-law mean flow over a rough wall, w vanishing on both walls
            z = (torch.arange(nz, device=w.device, dtype=torch.float64) + 0.5) * _dims(case)[2] / nz
            v[0] = v[0] + (torch.log(z / 1e-4) / 0.4).view(-1, 1, 1)
            w = torch.cat([w, w[:1]])
            w[0], w[nz] = 0.0, 0.0
        else:
            w = torch.cat([w, w[:1]])
        v[2] = w
    return [q.to(dt).contiguous() for q in v]


def _gradients(npts, seed):
    """velocity gradients (9, npts): trace-free, more rotation than strain, with intermittent magnitude"""
    dev = _dev()
    g = torch.Generator(device=dev)
    g.manual_seed(seed)
    a = torch.randn((9, npts), generator=g, device=dev, dtype=torch.float32)
    a *= torch.exp(0.5 * torch.randn((1, npts), generator=g, device=dev, dtype=torch.float32))
    t = (a[0] + a[4] + a[8]) / 3
    for c in (0, 4, 8):
        a[c] -= t
    return a


def _dims(case):
    """box lengths: cubic cells of a 2 pi wide box"""
    return tuple(PI2 * case[n] / case["nx"] for n in ("nx", "ny", "nz"))


def _bcs(case):
    return tuple((case[d + "b"], case[d + "n"]) for d in "xyz")


def _per(case):
    return case["px"], case["py"], case["pz"]


def _sgs(case):
    if case["sgs"] == "none":
        return None
    L = _dims(case)
    d = (L[0] / case["nx"] * L[1] / case["ny"] * L[2] / case["nz"]) ** (1.0 / 3.0)
    if case["sgs"] == "amd":
        c = tuple(l / case[n] for l, n in zip(L, ("nx", "ny", "nz")))
        return dict(model="amd", camd=c, cglobal=1.0 / 3.0)
    s = dict(model="smagorinsky", cglobal=(0.17 * d) ** 2)
    if case["walls"]:
        s.update(wall_model="moeng", z0=1e-4)
    return s


WALLS = dict(botWall=3, topWall=2, dpFdx=1.0)
CFL = 0.8
GAS = dict(mu_ref=0.01, T_ref=1.0, visc_n=0.75, Pr=0.72)


def prepare(case, seed):
    kind, prec = case["kind"], case["prec"]
    v = _inputs(case, seed)
    s = dict(case=case, v=v)
    e = torch.empty_like
    if kind == "rhs":
        s["op"] = P.FullRHS(case["n"], PI2, prec)
        s["grad"] = torch.empty(9 * case["n"] ** 3, dtype=v[0].dtype, device=v[0].device)
        s["out"] = [e(v[0]) for _ in range(3)]
    elif kind == "grad":
        L = _dims(case)
        s["op"] = P.derivatives()
        s["op"].init(case["nx"], case["ny"], case["nz"], *[l / case[n] for l, n in zip(L, ("nx", "ny", "nz"))],
                     *_per(case), *(case["method"],) * 3)
        s["out"] = [e(v[0]) for _ in range(3)]
    elif kind == "filter":
        s["op"] = P.filters()
        s["op"].init(case["nx"], case["ny"], case["nz"], *_per(case), "cf90", "cf90", "cf90")
        s["out"] = [e(v[0]) for _ in range(3)]
    elif kind == "cgrid":
        L = _dims(case)
        s["op"] = P.cgrid()
        s["op"].init((case["nx"], case["ny"], case["nz"]), [l / case[n] for l, n in zip(L, ("nx", "ny", "nz"))],
                     periodic=_per(case), bc=_bcs(case), inviscid=False, prec=prec, **GAS)
        s["v"] = [torch.stack(v)]
        s["out"] = [e(s["v"][0])]
    elif kind == "igrid":
        s["op"] = P.igrid()
        s["op"].init(case["nx"], case["ny"], case["nz"], *_dims(case), Re=case["Re"], scheme=2, CFL=CFL,
                     sgs=_sgs(case), walls=WALLS if case["walls"] else None, prec=prec)
    else:
        net = P.SGSNet(64)
        net.set_params(P.SGSNet.pack(_net(seed)))
        s["op"] = P.Closure(net, case["npts"])
        s["out"] = [torch.empty((6, case["npts"]), dtype=v[0].dtype, device=v[0].device)]
    return s


def run(s):
    case, op, v = s["case"], s["op"], s["v"]
    kind, prec = case["kind"], case["prec"]
    if kind == "rhs":
        op.eval(*v, s["grad"], *s["out"])
        return [s["grad"]] + s["out"]
    if kind == "grad":
        P.gradient(op, v[0], *s["out"], *_bcs(case), prec=prec)
        return s["out"]
    if kind == "filter":
        (x, y, z), (xb, yb, zb) = s["out"], _bcs(case)
        op.filterx(v[0], x, *xb, prec=prec)
        op.filtery(x, y, *yb, prec=prec)
        op.filterz(y, z, *zb, prec=prec)
        return z
    if kind == "cgrid":
        op.getRHS(v[0], s["out"][0])
        return s["out"][0]
    if kind == "igrid":
        op.set_velocity(*v)
        op.step()
        out = [op.field("u"), op.field("v"), op.field("w")]
        for t in out:
            t.owner = op  # the views lie in the solver's memory: it lives as long as they do
        return out
    op.stress(v[0], case["npts"], 0.05, 1.0, s["out"][0], which=2, prec=prec)
    return s["out"][0]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how far two correct ones may be apart
# ---------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    W = 8 if case["prec"] == "f64" else 4
    if kind == "closure":
        # 9 gradients in, 6 stresses out; the network's products and the tensor algebra
        return dict(bytes=15 * case["npts"] * W, flops=case["npts"] * (2 * (10 * 64 + 2 * 64 * 64 + 64 * 6) + 900))
    N = case["n"] ** 3 if kind == "rhs" else case["nx"] * case["ny"] * case["nz"]
    lg = math.log2(N)
    if kind == "rhs":
        # 3 fields in; 9 gradients and 3 fields out; 14 tridiagonal and 9 pentadiagonal line solves, 2 transforms
        return dict(bytes=15 * N * W, flops=N * (14 * 9 + 9 * 19 + 2 * 2.5 * lg))
    if kind == "grad":
        return dict(bytes=4 * N * W, flops=N * 3 * (15 if case["method"] == "cd10" else 9))
    if kind == "filter":
        return dict(bytes=2 * N * W, flops=N * 3 * 19)
    if kind == "cgrid":
        # 5 fields in, 5 out; 33 first, 18 second derivatives, 18 Gaussian passes, about 300 pointwise operations
        return dict(bytes=10 * N * W, flops=N * (33 * 15 + 18 * 16 + 18 * 13 + 300))
    # the velocity in and out, and the three fields read and written by each of the six projections (a global
    # solve each); about 33 two-dimensional transforms and 20 line solves a stage
    return dict(bytes=(6 + 6 * 6) * N * W, flops=6 * N * (33 * 2.5 * lg * 2 / 3 + 20 * 9 + 150))


def tolerance(case):
    kind, f64 = case["kind"], case["prec"] == "f64"
    if kind == "closure":
        # BF16 weights and activations: 0.7 to 1% from the FP64 network
        return dict(rel=2e-2)
    if kind == "igrid":
        # one step from the same velocity: 5e-7 (FP32), 2e-15 (FP64) from exact()
        return dict(rel=1e-12 if f64 else 4e-6)
    if kind == "cgrid":
        # quotients and moduli of differentiated FP32 fields: 8e-7 on the listed grid, 1e-5 on the largest drawn ones
        return dict(rel=1e-11 if f64 else 2e-5)
    if kind == "rhs":
        # the filter's left-hand side nearly vanishes at the grid scale (1e-13 in FP64); the pressure's FP32
        # gradient at 512^3: 3e-6
        return dict(rel=1e-12 if f64 else 1e-5)
    return dict(rel=1e-12 if f64 else 1e-6)


# ---------------------------------------------------------------------------
# FP64 restatement
# ---------------------------------------------------------------------------
def _matrix(nout, nin, coef, wrap=None, mirror=None):
    """rows i of sum_o coef[o] x[i + o]; columns outside wrap (period) or are
    mirrored: mirror = (left(j), right(j)) give (column, sign)"""
    M = np.zeros((nout, nin))
    for i in range(nout):
        for o, c in coef.items():
            j, s = i + o, 1.0
            if wrap:
                j %= wrap
            elif j < 0:
                j, s = mirror[0](j)
            elif j >= nin:
                j, s = mirror[1](j)
            M[i, j] += s * c
    return M


def _collocated(scheme):
    """(LHS offsets, RHS offsets, parity flip) of the interior rows at unit spacing"""
    if scheme == "cd06":
        al, be, c, anti = 1 / 3, 0.0, [0, 7 / 9, 1 / 36], True
    elif scheme == "cd10":
        al, be, c, anti = 0.5, 0.05, [0, 17 / 24, 101 / 600, 1 / 600], True
    elif scheme == "cd10_d2":
        al, be = 334 / 899, 43 / 1798
        c, anti = [0, 1065 / 1798, (1038 / 899) / 4, (79 / 1798) / 9], False
        c[0] = -2 * sum(c)
    elif scheme == "cf90":
        al, be, c, anti = 6.6624e-1, 1.6688e-1, [9.9965e-1, 6.6652e-1, 1.6674e-1, 4.0e-5, -5.0e-6], False
    else:  # gaussian
        al, be, anti = 0.0, 0.0, False
        c = [3565 / 10368, 3091 / 12960, 1997 / 25920, 149 / 12960, 107 / 103680]
    R = {0: c[0]}
    for q in range(1, len(c)):
        R[q], R[-q] = c[q], (-c[q] if anti else c[q])
    return {-2: be, -1: al, 0: 1.0, 1: al, 2: be}, R, anti


def _end_rows(scheme):
    """one-sided rows of the first points: (LHS offsets, RHS offsets) per row"""
    p, q, r, s = -17 / 6, 1.5, 1.5, -1 / 6
    if scheme == "cd06":
        ah = 1 / 3
        app = ((40 * ah - 1) * q + 7 * (4 * ah - 1) * s) / (16 * (ah + 2) * q + 8 * (1 - 4 * ah) * s)
        w1 = (2 * ah + 1) / (2 * (q + s))
        w2 = ((8 * ah + 7) * q - 6 * (2 * ah + 1) * r + (8 * ah + 7) * s) / (9 * (q + s))
        w3 = (4 * (ah + 2) * q + 2 * (1 - 4 * ah) * s) / (9 * (q + s))
        qpp, rpp = (app + 2) / 3, (4 * app - 1) / 12
        rows = [(w1, {0: 1, 1: 3}, {0: p, 1: q, 2: r, 3: s}), (w2, {-1: .25, 0: 1, 1: .25}, {-1: -.75, 1: .75}),
                (w3, {-1: app, 0: 1, 1: app}, {-2: -rpp, -1: -qpp, 1: qpp, 2: rpp})]
    elif scheme == "cd10":
        qh, rh, sh = 17 / 24, 101 / 600, 1 / 600
        a3 = (8 * rh - 175 * sh) / (18 * rh - 550 * sh)
        b3, q3, r3, s3 = (-3 + 8 * a3) / 20, (12 - 7 * a3) / 12, (568 * a3 - 183) / 600, (9 * a3 - 4) / 300
        t, u = qh + rh - sh * (q3 / s3 - 1), s * (rh + 2 * sh) - q * (qh + rh + sh)
        a2 = ((17 * u) / (72 * (q + s) * t) - 8 / 9) / ((19 * u) / (24 * (q + s) * t) - 1 / 3)
        b2, q2, r2 = (-1 + 3 * a2) / 12, (8 - 3 * a2) / 9, (-17 + 57 * a2) / 72
        w1 = (qh + 2 * rh + 3 * sh) / (q + s)
        w2 = (rh + sh * (1 + q3 / s3) - r * w1) / 0.75
        w3, w4 = (qh + rh + sh * (1 - q3 / s3)) / r2, sh / s3
        rows = [(w1, {0: 1, 1: 3}, {0: p, 1: q, 2: r, 3: s}), (w2, {-1: .25, 0: 1, 1: .25}, {-1: -.75, 1: .75}),
                (w3, {-2: b2, -1: a2, 0: 1, 1: a2, 2: b2}, {-2: -r2, -1: -q2, 1: q2, 2: r2}),
                (w4, {-2: b3, -1: a3, 0: 1, 1: a3, 2: b3}, {-3: -s3, -2: -r3, -1: -q3, 1: q3, 2: r3, 3: s3})]
    elif scheme == "cd10_d2":
        a = 11.0
        b = 344 / 1179
        A3, B3, be = (696 - 1191 * b) / 428, (2454 * b - 294) / 2140, (38 * b - 9) / 214
        rows = [(1, {0: 1, 1: a}, {0: (11 * a + 35) / 12, 1: -(5 * a + 26) / 3, 2: (a + 19) / 2, 3: (a - 14) / 3,
                                   4: (11 - a) / 12}),
                (1, {-1: .1, 0: 1, 1: .1}, {-1: 1.2, 0: -2.4, 1: 1.2}),
                (1, {-2: be, -1: b, 0: 1, 1: b, 2: be}, {-2: B3, -1: A3, 0: -2 * (A3 + B3), 1: A3, 2: B3})]
    elif scheme == "cf90":
        al, be = 6.6624e-1, 1.6688e-1
        lhs = {-2: be, -1: al, 0: 1, 1: al, 2: be}
        rows = [(1, {0: 1}, {0: 1}),
                (1, {-1: .4997, 0: 1, 1: .4997}, {-1: .49985, 0: .9997, 1: .49985}),
                (1, lhs, {-2: .1668, -1: .66656, 0: .99952, 1: .66656, 2: .1668}),
                (1, lhs, {-3: 4e-5, -2: .16672, -1: .66652, 0: .99968, 1: .66652, 2: .16672, 3: 4e-5})]
    else:
        rows = []
        for j, w in enumerate([[5 / 6, 1 / 6], [2 / 3, 1 / 6], [31 / 64, 7 / 32, 5 / 128],
                               [17 / 48, 15 / 64, 7 / 96, 1 / 64]]):
            rows.append((1, {0: 1}, {o: w[abs(o)] for o in range(1 - len(w), len(w)) if j + o >= 0}))
    return [({o: w * x for o, x in lh.items()}, {o: w * x for o, x in rh.items()}) for w, lh, rh in rows]


@functools.lru_cache(maxsize=64)
def _line(scheme, n, h, periodic, b1, bn):
    """dense n x n matrix of a collocated operator"""
    lh, rh, anti = _collocated(scheme)
    order = {"cd06": 1, "cd10": 1, "cd10_d2": 2}.get(scheme, 0)
    if periodic:
        A, B = _matrix(n, n, lh, wrap=n), _matrix(n, n, rh, wrap=n)
    else:
        def ends(sg):
            return [lambda j: (-j, sg * (b1 or 1)), lambda j: (2 * (n - 1) - j, sg * (bn or 1))]
        A, B = _matrix(n, n, lh, mirror=ends(-1 if anti else 1)), _matrix(n, n, rh, mirror=ends(1))
        for k, (l, r) in enumerate(_end_rows(scheme)):
            for side, b in ((0, b1), (1, bn)):
                if b:
                    continue
                i, d = (k, 1) if side == 0 else (n - 1 - k, -1)
                A[i], B[i] = 0, 0
                for o, x in l.items():
                    A[i, i + d * o] = x
                for o, x in r.items():
                    B[i, i + d * o] = x * (d if anti else 1)
    return np.linalg.solve(A, B) / h ** order


def _along(M, f, axis):
    """M along an axis of a (z, y, x) field; axis 0, 1, 2 = x, y, z"""
    M = torch.as_tensor(M, device=f.device).to(f.dtype)
    if axis == 0:
        return f @ M.T
    if axis == 1:
        return torch.stack([M @ p for p in f])
    return (M @ f.reshape(f.shape[0], -1)).reshape((M.shape[0],) + f.shape[1:])


def exact(case, seed):
    v = [q.double() for q in _inputs(case, seed)]
    return dict(rhs=_exact_rhs, grad=_exact_grad, filter=_exact_filter, cgrid=_exact_cgrid, igrid=_exact_igrid,
                closure=_exact_closure)[case["kind"]](case, seed, v)


def _exact_rhs(case, seed, u):
    n = case["n"]
    h = PI2 / n
    D, F = _line("cd06", n, h, True, 0, 0), _line("cf90", n, 1.0, True, 0, 0)
    dt = DT[case["prec"]]
    grad = torch.empty((9,) + tuple(u[0].shape), dtype=dt, device=u[0].device)
    for i in range(3):
        for j in range(3):
            grad[3 * i + j] = _along(D, u[i], j)
    for i in range(3):
        for j in range(3):
            u[i] = _along(F, u[i], j)
    div = _along(D, u[0], 0)
    for j in (1, 2):
        div += _along(D, u[j], j)
    k = torch.fft.fftfreq(n, d=1.0 / n, device=div.device, dtype=torch.float64) * PI2 / n
    kp2 = ((14 / 9 * torch.sin(k) + 1 / 18 * torch.sin(2 * k)) / (1 + 2 / 3 * torch.cos(k)) / h) ** 2
    kp2[n // 2] = 0.0
    ks = kp2.view(n, 1, 1) + kp2.view(1, n, 1) + kp2[:n // 2 + 1].view(1, 1, -1)
    ks = torch.where(ks <= 1e-14, torch.inf, ks)
    p = torch.fft.irfftn(torch.fft.rfftn(div) / -ks, s=(n, n, n))
    del ks, div
    return [grad] + [(u[j] - _along(D, p, j)).to(dt) for j in range(3)]


def _exact_grad(case, seed, v):
    L = _dims(case)
    return [_along(_line(case["method"], case[n], L[i] / case[n], _per(case)[i], *_bcs(case)[i]), v[0], i)
            for i, n in enumerate(("nx", "ny", "nz"))]


def _exact_filter(case, seed, v):
    f = v[0]
    for i, n in enumerate(("nx", "ny", "nz")):
        f = _along(_line("cf90", case[n], 1.0, _per(case)[i], *_bcs(case)[i]), f, i)
    return f


def _exact_cgrid(case, seed, W):
    n = [case[q] for q in ("nx", "ny", "nz")]
    h = [l / m for l, m in zip(_dims(case), n)]
    per, bc = _per(case), _bcs(case)

    def op(scheme, f, i, sg=1):
        return _along(_line(scheme, n[i], h[i], per[i], sg * bc[i][0], sg * bc[i][1]), f, i)

    def smooth(f):
        for i in (1, 0, 2):
            for _ in range(2):
                f = op("gauss", f, i)
        return f

    def d4(f, i):
        return op("cd10_d2", op("cd10_d2", f, i), i)

    gam, Cmu, Cbeta, Ckap = 1.4, 0.002, 1.75, 0.01
    rho, E = W[0], W[4]
    u = [q / rho for q in W[1:4]]
    e = E / rho - 0.5 * (u[0] ** 2 + u[1] ** 2 + u[2] ** 2)
    p, T = (gam - 1) * rho * e, (gam - 1) * e
    g = [[op("cd10", u[i], j, -1 if i == j else 1) for j in range(3)] for i in range(3)]
    mu = GAS["mu_ref"] * (T / GAS["T_ref"]) ** GAS["visc_n"]
    kap = gam / (gam - 1) * mu / GAS["Pr"]
    f = torch.sqrt(g[0][0] ** 2 + g[1][1] ** 2 + g[2][2] ** 2 + 0.5 * (g[1][0] + g[0][1]) ** 2
                   + 0.5 * (g[2][0] + g[0][2]) ** 2 + 0.5 * (g[2][1] + g[1][2]) ** 2)
    mu = mu + smooth(Cmu * rho * sum(d4(f, i) * h[i] ** 6 for i in range(3)).abs())
    f = g[0][0] + g[1][1] + g[2][2]
    r = [op("cd10", rho, i) ** 2 for i in range(3)]
    s = r[0] + r[1] + r[2] + 1e-32
    b = sum(d4(f, i) * h[i] ** 4 * (h[i] * r[i] / s) ** 2 for i in range(3))
    curl2 = (g[2][1] - g[1][2]) ** 2 + (g[0][2] - g[2][0]) ** 2 + (g[1][0] - g[0][1]) ** 2
    bulk = smooth(Cbeta * rho * torch.where(f >= 0, 0.0, f * f / (f * f + curl2 + 1e-32)) * b.abs())
    r = [op("cd10", e, i) ** 2 for i in range(3)]
    s = r[0] + r[1] + r[2] + 1e-32
    b = sum(d4(e, i) * h[i] ** 4 * (h[i] * r[i] / s) for i in range(3))
    kap = kap + smooth(Ckap * rho * torch.sqrt(gam * p / rho) * b.abs() / T)
    lam = bulk - 2 / 3 * mu
    dil = g[0][0] + g[1][1] + g[2][2]
    tau = [[mu * (g[i][j] + g[j][i]) + (lam * dil if i == j else 0) for j in range(3)] for i in range(3)]
    out = [torch.zeros_like(rho) for _ in range(5)]
    for d in range(3):
        q = -kap * op("cd10", T, d)
        F = [W[1 + d]] + [W[1 + d] * u[i] + (p if i == d else 0) - tau[i][d] for i in range(3)]
        F.append((E + p) * u[d] - sum(u[i] * tau[i][d] for i in range(3)) + q)
        for c in range(5):
            out[c] -= op("cd10", F[c], d, 1 if c == 1 + d else -1)
    return torch.stack(out)


def _exact_closure(case, seed, v):
    W = [(torch.as_tensor(w, device=v[0].device).double(), torch.as_tensor(b, device=v[0].device).double())
         for w, b in _net(seed)]
    A = v[0].T.reshape(-1, 3, 3)
    scale = torch.sqrt((A * A).sum(dim=(1, 2)).mean())
    out = torch.empty((6, A.shape[0]), dtype=DT[case["prec"]], device=A.device)
    step = 1 << 21
    for o in range(0, A.shape[0], step):
        a = A[o:o + step] / scale
        eye = torch.eye(3, dtype=a.dtype, device=a.device)
        tr = lambda m: m.diagonal(dim1=1, dim2=2).sum(-1)  # noqa: E731

        def mm(x, y):
            return (x[:, :, :, None] * y[:, None, :, :]).sum(2)
        s = 0.5 * (a + a.mT) - (tr(a) / 3).view(-1, 1, 1) * eye
        r = 0.5 * (a - a.mT)
        s2, r2, sr = mm(s, s), mm(r, r), mm(s, r)
        rs, rs2, r2s = mm(r, s), mm(r, s2), mm(r2, s)
        i1, i2, i3, i4, i5 = tr(s2), -tr(r2), tr(mm(s2, s)), tr(r2s), tr(mm(r2, s2))
        i6 = tr(mm(r2s, rs2))

        def root(x, k):
            return torch.sign(x) * x.abs() ** (1.0 / k)
        pq = 0.5 * i1
        c = (0.5 * i3 / pq * torch.sqrt(3 / pq)).clamp(-1, 1)
        ph, m = torch.acos(c) / 3, 2 * torch.sqrt(pq / 3)
        x = [torch.sqrt(i1), torch.sqrt(i2), root(i3, 3), root(i4, 3), (-i5).clamp(min=0) ** 0.25, root(i6, 6)]
        x += [m * torch.cos(ph - k * PI2 / 3) for k in range(3)] + [torch.ones_like(ph)]
        y = torch.stack(x, 1)
        for k, (w, b) in enumerate(W):
            y = y @ w.T + b
            if k < 3:
                y = torch.nn.functional.gelu(y, approximate="tanh")
        sr2 = mm(s, r2)
        Tn = [s, sr - rs, s2 - (i1 / 3).view(-1, 1, 1) * eye, r2 + (i2 / 3).view(-1, 1, 1) * eye, rs2 - mm(s2, r),
              r2s + sr2 - (2 / 3 * tr(sr2)).view(-1, 1, 1) * eye]
        t = sum(y[:, k].view(-1, 1, 1) * Tn[k] for k in range(6)) * (0.05 * scale) ** 2
        for k, (i, j) in enumerate(((0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2))):
            out[k, o:o + step] = 0.5 * (t[:, i, j] + t[:, j, i])
    return out


def _staggered(op, n, h, periodic, bot, top):
    """dense matrix of a cd06stagg operator between n cells and n + 1 edges:
    "dEC", "dCE" first derivatives, "iEC", "iCE" interpolations, "ddC", "ddE"
    second derivatives; bot, top 1 even, -1 odd, 0 one-sided"""
    ein, eout = op in ("dEC", "iEC", "ddE"), op in ("dCE", "iCE", "ddE")
    order = {"d": 1, "i": 0}[op[0]] if op[1] != "d" else 2
    if order == 1:
        al, c, anti = 9 / 62, (63 / 62, 17 / 186), -1
    elif order == 0:
        al, c, anti = 0.3, (0.75, 0.05), 1
    else:
        al, c, anti = 2 / 11, (12 / 11, 3 / 44), 1
    if order == 2:
        rh = {0: -2 * (c[0] + c[1]), -1: c[0], 1: c[0], -2: c[1], 2: c[1]}
    else:
        rh = {1: c[0], 0: anti * c[0], 2: c[1], -1: anti * c[1]}
        if eout:
            rh = {o - 1: x for o, x in rh.items()}
    lh = {-1: al, 0: 1.0, 1: al}
    if periodic:
        M = np.linalg.solve(_matrix(n, n, lh, wrap=n), _matrix(n, n, rh, wrap=n)) / h ** order
        if ein:
            M = np.hstack([M, np.zeros((n, 1))])
        return np.vstack([M, M[:1]]) if eout else M
    nin, nout = n + int(ein), n + int(eout)

    def ends(edge, sg):
        b, t = bot or 1, top or 1
        return [lambda j: (-j if edge else -1 - j, sg * b), lambda j: (2 * n - j - (0 if edge else 1), sg * t)]
    A, B = _matrix(nout, nout, lh, mirror=ends(eout, -1 if order == 1 else 1)), _matrix(nout, nin, rh, mirror=ends(ein, 1))
    w0, w1 = 223 / 186, 61 / 62
    a1 = 37 / 183
    b1 = (-1 + 22 * a1) / 24
    sided = {"dEC": [({0: w0, 1: -w0}, [-w0, 2 * w0, -w0, 0]),
                     ({-1: w1 * a1, 0: w1, 1: w1 * a1},
                      [-w1 * b1, -w1 * 3 / 8 * (3 - 2 * a1), w1 * 3 / 8 * (3 - 2 * a1), w1 * b1])],
             "dCE": [({0: 1}, [-71 / 24, 47 / 8, -31 / 8, 23 / 24]), ({-1: 1 / 22, 0: 1, 1: 1 / 22}, [-12 / 11, 12 / 11])],
             "iEC": [({0: 1, 1: 1}, [1 / 4, 3 / 2, 1 / 4, 0])],
             "iCE": [({0: 1}, [15 / 8, -5 / 4, 3 / 8]), ({-1: 1 / 6, 0: 1, 1: 1 / 6}, [2 / 3, 2 / 3])]}.get(op, [])
    for k, (l, r) in enumerate(sided):
        for b, i, d, j0 in ((bot, k, 1, 0), (top, nout - 1 - k, -1, nin - 1)):
            if b:
                continue
            A[i], B[i] = 0, 0
            for o, x in l.items():
                A[i, i + d * o] = x
            for o, x in enumerate(r):
                B[i, j0 + d * o] = x * (d if order == 1 else 1)
    return np.linalg.solve(A, B) / h ** order


def _exact_igrid(case, seed, vel):
    """one SSP-RK45 step of the rotational-form solver from the projected velocity"""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    Lx, Ly, Lz = _dims(case)
    dx, dy, dz = Lx / nx, Ly / ny, Lz / nz
    walls, Re, sgs = case["walls"], case["Re"], _sgs(case)
    dev = vel[0].device
    ar = lambda n: torch.fft.fftfreq(n, d=1.0 / n, device=dev, dtype=torch.float64)  # noqa: E731
    # the highest mode carries a plus sign in the derivatives, a minus sign in the pressure's k^2 and potential
    k1 = torch.arange(nx // 2 + 1, device=dev, dtype=torch.float64) * PI2 / Lx
    k2m = ar(ny) * PI2 / Ly
    k2 = k2m.clone()
    k2[ny // 2] *= -1
    k1m = k1.clone()
    k1m[nx // 2] *= -1
    g2 = ((k1.abs() < 2 / 3 * math.pi / dx).view(1, 1, -1) & (k2.abs() < 2 / 3 * math.pi / dy).view(1, -1, 1)).double()
    K1, K2 = k1.view(1, 1, -1), k2.view(1, -1, 1)

    def fft(f):
        return torch.fft.fft(torch.fft.rfft(f, dim=2), dim=1)

    def ifft(f):
        return torch.fft.irfft(torch.fft.ifft(f, dim=1), n=nx, dim=2)

    @functools.lru_cache(maxsize=32)
    def zmat(op, b, t):
        return torch.as_tensor(_staggered(op, nz, dz, not walls, b, t), device=dev)

    def z(op, f, b=0, t=0):
        M = zmat(op, b, t)
        flat = f.reshape(f.shape[0], -1)
        if f.is_complex():
            r = torch.view_as_complex((M @ torch.view_as_real(flat).reshape(f.shape[0], -1)).reshape(M.shape[0], -1, 2))
        else:
            r = M @ flat
        return r.reshape((M.shape[0],) + f.shape[1:])

    nk = 2 * nz if walls else nz
    k3 = ar(nk) * PI2 / (nk * dz)
    kd = k3 * dz
    k3p = (2 * (63 / 62) * torch.sin(kd / 2) + 2 * (17 / 186) * torch.sin(3 * kd / 2)) / (1 + 18 / 62 * torch.cos(kd)) / dz
    ks = k1m.view(1, 1, -1) ** 2 + k2m.view(1, -1, 1) ** 2 + (k3p ** 2).view(-1, 1, 1)
    kinv = torch.where(ks <= 1e-14, 0.0, 1 / torch.where(ks <= 1e-14, 1.0, ks))
    del ks
    if walls:
        uB, uT, wB, wT, dUB, dUT, dWB, dWT = 0, 1, -1, -1, 0, -1, 0, 0
        shift = torch.polar(torch.ones_like(k3), 0.5 * kd).view(-1, 1, 1)
        lam = torch.sqrt(k1m.view(1, -1) ** 2 + k2m.view(-1, 1) ** 2)
        t = lam * Lz
        den = torch.where(t < 500, 1 / (lam * torch.sinh(t.clamp(max=500)) + 1e-13), 0.0)
        den = torch.where(den < 1e-16, 0.0, den)
        den[0, 0] = 0.0
        ze = torch.arange(nz + 1, device=dev, dtype=torch.float64) * dz
        zc = 0.5 * (ze[1:] + ze[:-1])

        def hyp(f, z_, cap, scale):
            t = lam * z_
            return torch.where(t < 32, scale * f(t.clamp(max=32)), cap)
    else:
        uB, uT, wB, wT, dUB, dUT, dWB, dWT = 1, 1, -1, -1, -1, -1, 0, 0
        g3 = (k3.abs() < 2 / 3 * math.pi / dz).double().view(-1, 1, 1)

    def dealias(f):
        if walls:
            return f * g2
        c = torch.fft.ifft(torch.fft.fft(f[:nz], dim=0) * (g2 * g3), dim=0)
        return c if f.shape[0] == nz else torch.cat([c, c[:1]])

    def project(u, v, w):
        a, b = K1, K2
        if walls:
            a, b = k1m.view(1, 1, -1), k2m.view(1, -1, 1)
            w = w.clone()
            cb = -w[0] * den
            ct = (w[nz] - cb * hyp(torch.sinh, Lz - ze[nz], -4e13, -lam)) * den
            u, v = u.clone(), v.clone()
            for k in range(nz):
                ph = 1j * (cb * hyp(torch.cosh, Lz - zc[k], 4e13, 1.0) + ct * hyp(torch.cosh, zc[k], 1e13, 1.0))
                u[k] -= a[0] * ph
                v[k] -= b[0] * ph
            for k in range(1, nz):
                w[k] -= cb * hyp(torch.sinh, Lz - ze[k], -4e13, -lam) + ct * hyp(torch.sinh, ze[k], 4e13, lam)
            w[0], w[nz] = 0, 0
            f = 1j * (a * u + b * v)
            F = torch.fft.fft(torch.cat([f.flip(0), f]), dim=0)
            Wt = torch.fft.fft(torch.cat([-w[1:nz].flip(0), w]), dim=0)
            F = -(F + 1j * (k3p.view(-1, 1, 1) * shift.conj()) * Wt) * kinv
            p = torch.fft.ifft(F, dim=0)[nz:]
            Wt = Wt - 1j * (k3p.view(-1, 1, 1) * shift) * F
            w = torch.fft.ifft(Wt, dim=0)[nz - 1:].clone()
            w[0], w[nz] = 0, 0
        else:
            p = torch.fft.ifft(-kinv * torch.fft.fft(z("dEC", w) + 1j * (K1 * u + K2 * v), dim=0), dim=0)
            w = w - z("dCE", p)
        return u - 1j * a * p, v - 1j * b * p, w

    def prep(S):
        S = project(*[dealias(q) for q in S])
        return S

    def rhs(S):
        u, v, w = S
        uE, vE, wC = z("iCE", u, uB, uT), z("iCE", v, uB, uT), z("iEC", w, wB, wT)
        dzu, dzv, dzw = z("dCE", u, uB, uT), z("dCE", v, uB, uT), z("dEC", w, wB, wT)
        pu, pv, pw, puE, pvE = ifft(u), ifft(v), ifft(w), ifft(uE), ifft(vE)
        oz = ifft(1j * K1 * v - 1j * K2 * u)
        ox, oy = ifft(1j * K1 * w - dzu), ifft(1j * K2 * w - dzv)
        ru = z("iEC", fft(ox * pw)) + fft(oz * pv)
        rv = z("iEC", fft(oy * pw)) - fft(oz * pu)
        rw = -fft(ox * puE + oy * pvE)
        del oz, ox, oy, puE, pvE
        if Re > 0:
            kk = -(K1 * K1 + K2 * K2)
            ru = ru + (kk * u + z("ddC", u, uB, uT)) / Re
            rv = rv + (kk * v + z("ddC", v, uB, uT)) / Re
            rw = rw + (kk * w + z("ddE", w, wB, wT)) / Re
        if sgs:
            gC = [ifft(1j * K1 * u), ifft(1j * K2 * u), ifft(z("iEC", dzu, dUB, dUT)),
                  ifft(1j * K1 * v), ifft(1j * K2 * v), ifft(z("iEC", dzv, dUB, dUT)),
                  ifft(1j * K1 * wC), ifft(1j * K2 * wC), ifft(dzw)]
            s = [gC[0], 0.5 * (gC[1] + gC[3]), 0.5 * (gC[2] + gC[6]), gC[4], 0.5 * (gC[5] + gC[7]), gC[8]]
            if sgs["model"] == "amd":
                c = sgs["camd"]

                def row(i, j):
                    return sum(c[q] ** 2 * gC[3 * i + q] * gC[3 * j + q] for q in range(3))
                num = (row(0, 0) * s[0] + row(1, 1) * s[3] + row(2, 2) * s[5]
                       + 2 * (row(0, 1) * s[1] + row(0, 2) * s[2] + row(1, 2) * s[4]))
                nu = (-num / (sum(q * q for q in gC) + 1e-32)).clamp(min=0)
            else:
                nu = torch.sqrt(2 * (s[0] ** 2 + s[3] ** 2 + s[5] ** 2 + 2 * (s[1] ** 2 + s[2] ** 2 + s[4] ** 2)))
            nu = nu * sgs["cglobal"]
            nuE = z("iCE", nu).clamp(min=0)
            t13 = -nuE * ifft(dzu + 1j * K1 * w)
            t23 = -nuE * ifft(dzv + 1j * K2 * w)
            if walls:
                sp = torch.sqrt(pu[0] ** 2 + pv[0] ** 2).mean()
                us = sp * 0.4 / math.log(dz / 2 / sgs["z0"])
                m = -us * us / (sp + 1e-13)
                t13[0], t23[0] = m * pu[0], m * pv[0]
            t11, t12, t22, t33 = [fft(-2 * nu * s[q]) for q in (0, 1, 3, 5)]
            t13, t23 = fft(t13), fft(t23)
            ru = ru - 1j * K1 * t11 - 1j * K2 * t12 - z("dEC", t13)
            rv = rv - 1j * K1 * t12 - 1j * K2 * t22 - z("dEC", t23)
            rw = rw - 1j * K1 * t13 - 1j * K2 * t23 - z("dCE", t33)
        if walls:
            ru[:, 0, 0] += WALLS["dpFdx"] * nx * ny
        return ru, rv, rw

    def mix(*terms):
        return prep([sum(c * S[q] for c, S in terms) for q in range(3)])

    S0 = prep([fft(q) for q in vel])
    m = (ifft(S0[0]).abs() / dx + ifft(S0[1]).abs() / dy + ifft(z("iEC", S0[2], wB, wT)).abs() / dz).max().item()
    dt = CFL / m
    if Re > 0:
        dt = min(dt, CFL * Re * min(dx, dy, dz) ** 2)
    S1 = mix((1.0, S0), (0.39175222657189 * dt, rhs(S0)))
    S2 = mix((0.444370493651235, S0), (0.555629506348765, S1), (0.368410593050371 * dt, rhs(S1)))
    S3 = mix((0.620101851488403, S0), (0.379898148511597, S2), (0.25189177427169 * dt, rhs(S2)))
    R3 = rhs(S3)
    S4 = mix((0.17807995439313, S0), (0.821920045606868, S3), (0.54497475022852 * dt, R3))
    S = mix((0.517231671970585, S2), (0.096059710526147, S3), (0.06369246866629 * dt, R3),
            (0.386708617503269, S4), (0.22600748323690 * dt, rhs(S4)))
    return [ifft(q).reshape(-1) for q in S]
