"""Overlapping segments: pencils of lengths that are no multiple of 32, all
ends of the x direction, and more than 512 rows.

On the CPU the exported tables drive a numpy model of the kernels' solve,
compared with the dense systems over every scheme, boundary pair and a range
of lengths.  On the GPU the kernels are compared with the oracle."""
import ctypes

import numpy as np
import pytest

import oracle as O
import padeops_amd as P
from padeops_amd import _lib

BCS = [(a, b) for a in (-1, 0, 1) for b in (-1, 0, 1)]


def _tables(op, kind, bc1, bcn):
    L = _lib.lib()
    meta = (ctypes.c_int * 9)()
    assert L.pdo_op_overlap_tables(op._handle(), kind, bc1, bcn, meta, None, None, None, None) == 0
    m, p, K, nbl, nbr, q0, nd, d0, guni = list(meta)
    if p == 0:
        return None
    fac, spk = np.zeros((4, m, 5)), np.zeros((4, m, 4))
    G, sp = np.zeros((p, nd, 2 * K, 2 * K)), np.zeros((2, 4, 8))
    dp = ctypes.POINTER(ctypes.c_double)
    assert L.pdo_op_overlap_tables(op._handle(), kind, bc1, bcn, meta,
                                   *[a.ctypes.data_as(dp) for a in (fac, spk, G, sp)]) == 0
    return dict(m=m, P=p, K=K, nbl=nbl, nbr=nbr, q0=q0, nd=nd, d0=d0, guni=guni, fac=fac, spk=spk, G=G, sp=sp)


def _solve(t, d, periodic):
    """y = A^-1 d as the kernels compute it"""
    m, p, K, n = t["m"], t["P"], t["K"], len(d)
    start = [s * n // p if periodic else (s * (n - m) // (p - 1) if p > 1 else 0) for s in range(p)]
    own = [(start[s + 1] if s < p - 1 else (n if periodic else start[s] + m)) - start[s] for s in range(p)]
    assert all(o in (t["q0"], t["q0"] + 1) for o in (own if periodic else own[:-1] or [t["q0"]]))
    z = np.zeros((p, m))
    types = [1 if periodic else (3 if p == 1 else (0 if s == 0 else (2 if s == p - 1 else 1))) for s in range(p)]
    for s in range(p):
        F, v = t["fac"][types[s]], d[(start[s] + np.arange(m)) % n].copy()
        for j in range(1, m):
            v[j] -= F[j, 0] * v[j - 1] + (F[j, 1] * v[j - 2] if j > 1 else 0)
        for j in range(m - 1, -1, -1):
            v[j] = v[j] * F[j, 2] - (F[j, 3] * v[j + 1] if j + 1 < m else 0) - (F[j, 4] * v[j + 2] if j + 2 < m else 0)
        z[s] = v
    ends = np.zeros((p, 2 * K))
    for s in range(p):
        if periodic or s > 0:
            ends[s, :K] = z[s, m - own[s - 1]:m - own[s - 1] + K]
        if periodic or s < p - 1:
            ends[s, K:] = z[s, own[s] - K:own[s]]
    y = np.full(n, np.nan)
    for s in range(p):
        g = sum(t["G"][s, i] @ ends[(s + t["d0"] + i) % p] for i in range(t["nd"]))
        S = t["spk"][types[s]]
        v = z[s] - S[:, :K] @ g[:K] - S[:, 2:2 + K] @ g[K:]
        y[start[s]:start[s] + own[s]] = v[:own[s]]
    if t["guni"]:
        assert np.allclose(t["G"], t["G"][:1], rtol=0, atol=1e-13 * np.abs(t["G"]).max())
    return y


def _ops():
    for per in (True, False):
        yield "cd06", lambda n, per=per: (P.cd06(), lambda o: o.init(n, 0.1, per, 0, 0)), [0], [(0, 0)], per
        yield "cd06b", lambda n, per=per: (P.cd06(), lambda o: o.init(n, 0.1, per, 1, -1)), [0], [(0, 0)], per
        yield "cd10", lambda n, per=per: (P.cd10(), lambda o: o.init(n, 0.1, per)), [0, 1], BCS, per
        yield "cf90", lambda n, per=per: (P.cf90(), lambda o: o.init(n, per)), [2], BCS, per
    yield "cd06stagg", lambda n: (P.cd06stagg(), lambda o: o.init(n, 0.1)), [10, 11, 12, 13, 14, 15], [(0, 0)], True
    for fl in range(16):
        a = [bool(fl & b) for b in (1, 2, 4, 8)]
        yield ("cd06stagg%d" % fl, lambda n, a=a: (P.cd06stagg(), lambda o: o.init(n, 0.1, *a)),
               [10, 11, 12, 13, 14, 15, 16, 17], [(0, 0)], False)


@pytest.mark.parametrize("case", list(_ops()), ids=lambda c: c[0] + ("_per" if c[4] else ""))
def test_tables_solve_the_dense_system(case):
    _, make, kinds, bcs, per = case
    rng = np.random.default_rng(1)
    taken = 0
    for n in (16, 17, 20, 24, 31, 32, 33, 36, 37, 48, 63, 64, 65, 96, 100, 129, 151, 200, 201, 300, 384, 511, 513,
              600, 640, 1000, 1024):
        op, init = make(n)
        assert init(op) == 0
        for kind in kinds:
            for bc in bcs if not per else bcs[:1]:
                t = _tables(op, kind, *bc)
                if t is None:
                    continue
                taken += 1
                A, _ = op.dense(kind, *bc)
                d = rng.standard_normal(A.shape[0])
                y = _solve(t, d, per)
                # a backward stable solve: residual at rounding, against |A| |y|
                res = np.abs(A @ y - d) / (np.abs(A) @ np.abs(y) + np.abs(d))
                assert res.max() < 1e-13, (n, kind, bc, res.max())
                if not per:
                    B = op.dense(kind, *bc)[1]
                    for j in range(t["nbl"]):
                        assert np.allclose(B[j, :8], t["sp"][0, j], rtol=0, atol=1e-12 * np.abs(B).max())
                        assert not B[j, 8:].any()
                    for j in range(t["nbr"]):
                        r = A.shape[0] - t["nbr"] + j
                        assert np.allclose(B[r, -8:], t["sp"][1, j], rtol=0, atol=1e-12 * np.abs(B).max())
                        assert not B[r, :-8].any()
    assert taken > 15


def _fields(n, dir, seed):
    """a field (na, nb pencils of n points along dir) with ragged pencil counts"""
    shape = {1: (n, 7, 11), 2: (37, n, 5), 3: (9, 13, n)}[dir]
    r = np.random.default_rng(seed)
    return np.asfortranarray(r.standard_normal(shape))


# lengths at the edges of the segment counts: one 16- or 32-row segment, one
# row more, the last and first of a count, primes, above 512
LENGTHS = [16, 17, 23, 32, 33, 36, 47, 63, 64, 65, 97, 101, 151, 200, 257, 300, 509, 513, 640, 1021]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["f64", "f32_refine"])
@pytest.mark.parametrize("dir", [1, 2, 3])
@pytest.mark.parametrize("n", LENGTHS)
def test_against_oracle(cuda, n, dir, prec):
    import torch

    from fields import from_dev, rel_l2, to_dev
    dt = torch.float64 if prec == "f64" else torch.float32
    f = _fields(n, dir, n + dir)
    if prec != "f64":
        f = np.asfortranarray(f.astype(np.float32).astype(np.float64))
    F = to_dev(f, dt, cuda)
    na, nb = {1: f.shape[1:], 2: (f.shape[0], f.shape[2]), 3: f.shape[:2]}[dir]
    h = 2 * np.pi / n
    cases = []
    for per in (True, False):
        d6, d10, fl = P.cd06(), P.cd10(), P.cf90()
        assert d6.init(n, h, per) == 0 and d10.init(n, h, per) == 0 and fl.init(n, per) == 0
        for bc in [(0, 0)] if per else [(0, 0), (1, -1), (-1, 1)]:
            cases.append(((d10.dd1, d10.dd2, d10.dd3), O.CD10_D1, h, per, bc, bc))
            cases.append(((d10.d2d1, d10.d2d2, d10.d2d3), O.CD10_D2, h, per, bc, bc))
            cases.append(((fl.filter1, fl.filter2, fl.filter3), O.CF90, 1.0, per, bc, bc))
        cases.append(((d6.dd1, d6.dd2, d6.dd3), O.CD06_D1, h, per, (0, 0), ()))
    # FP64 rounding of a solve whose condition grows to 1e3 near the grid
    # scale (cf90); FP32 storage rounds the output alone
    tol = 1e-12 if prec == "f64" else 1e-7
    for fns, op, dx, per, bc, args in cases:
        ref = O.apply(op, f, dir, dx, per, *bc)
        out = torch.full_like(F, float("nan"))
        fns[dir - 1](F, out, na, nb, *args, prec=prec)
        torch.cuda.synchronize()
        assert rel_l2(from_dev(out, f.shape), ref) < tol, (op, per, bc)


@pytest.mark.gpu
@pytest.mark.parametrize("n,prec", [(n, "f64") for n in (16, 24, 40, 48, 65, 100)]
                         + [(n, "f32_refine") for n in (32, 64, 96, 100, 511, 512, 513)])
def test_staggered_against_oracle(cuda, n, prec):
    import torch

    from fields import from_dev, rel_l2, to_dev
    dt = torch.float64 if prec == "f64" else torch.float32
    tol = 1e-13 if prec == "f64" else 1e-7  # FP32 storage rounds the output alone
    r = np.random.default_rng(n)
    n1, n2 = 11, 6
    for per in (True, False):
        s = P.cd06stagg()
        assert s.init(n, 0.1, *([] if per else [True, False, False, True])) == 0
        for name, op, ein, eout in (("ddz_E2C", O.STG_D1_E2C, 1, 0), ("ddz_C2E", O.STG_D1_C2E, 0, 1),
                                    ("d2dz2_C2C", O.STG_D2_C2C, 0, 0), ("d2dz2_E2E", O.STG_D2_E2E, 1, 1),
                                    ("InterpZ_E2C", O.STG_IN_E2C, 1, 0), ("InterpZ_C2E", O.STG_IN_C2E, 0, 1)):
            # the last edge of a periodic field need not repeat the first
            f = np.asfortranarray(r.standard_normal((n1, n2, n + ein)))
            if prec != "f64":
                f = np.asfortranarray(f.astype(np.float32).astype(np.float64))
            ref = (O.apply(op, f, 3, 0.1, True, n=n) if per
                   else O.stagg_np(op, f, 0.1, O.TOP_EVEN | O.BOT_SIDED, n))
            out = torch.full((n1 * n2 * (n + eout),), float("nan"), dtype=dt, device=cuda)
            getattr(s, name)(to_dev(f, dt, cuda), out, n1, n2, prec=prec)
            torch.cuda.synchronize()
            assert rel_l2(from_dev(out, (n1, n2, n + eout)), ref) < tol, (name, per)


@pytest.mark.gpu
@pytest.mark.parametrize("dir,prec,per", [(1, "f32_refine", False), (2, "f32_refine", False), (2, "f32_refine", True),
                                          (2, "f64", False), (3, "f32_refine", False), (3, "f64", True)])
def test_fields_of_4_gib(cuda, dir, prec, per):
    """fields whose byte offsets pass 32 bits: planes (y) or rows (z) of their
    own 64-bit offsets, and whole lines along x, against the same passes over
    parts of the field, which are addressed within 32 bits"""
    import torch
    n, dt = 400, torch.float64 if prec == "f64" else torch.float32
    pencils = (2 ** 32 // dt.itemsize + (1 << 22)) // n
    na = 1 << 12
    nb = pencils // na + 1
    f = torch.empty(n * na * nb, dtype=dt, device=cuda)
    assert f.numel() * f.element_size() > 2 ** 32
    g = torch.Generator(device=cuda).manual_seed(dir)
    for part in f.chunk(64):
        part.normal_(generator=g)
    out = torch.full_like(f, float("nan"))
    op = P.cd10()
    assert op.init(n, 0.1, per) == 0
    fn = (op.dd1, op.dd2, op.dd3)[dir - 1]
    fn(f, out, na, nb, prec=prec)
    # x, y: whole planes (nb the slowest index); z: pencils of one plane index
    axis = 0 if dir < 3 else 1
    shape = (nb, n * na) if dir < 3 else (n, nb, na)
    F, G = f.view(shape), out.view(shape)
    for b in (0, 1, nb // 2, nb - 2):
        part = F.narrow(axis, b, 2).contiguous().flatten()
        ref = torch.full_like(part, float("nan"))
        fn(part, ref, na, 2, prec=prec)
        got = G.narrow(axis, b, 2).contiguous().flatten()
        torch.cuda.synchronize()
        assert torch.equal(got, ref), (b, (got - ref).abs().max().item())
    assert all(bool(torch.isfinite(part).all()) for part in out.chunk(16))
    del f, out, F, G
    torch.cuda.empty_cache()
