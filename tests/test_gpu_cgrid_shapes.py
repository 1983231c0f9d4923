"""GPU: cgrid at the sizes where its kernels change over, against the oracle.

Filters: the strided kernel gives a lane 16 rows of a pencil and shares the
rows out evenly, the x kernel holds whole lines, and either applies the
filter once or twice in a pass; other sizes take the general kernel, once per
pass.  Right-hand side: flux derivatives are summed in the passes of the
register, the overlapping-segment and the general kernels."""
import numpy as np
import pytest

import oracle.explicit as X
import padeops_amd as P
from fields import from_dev, random_field, rel_l2, to_dev
from oracle.cgrid import Cgrid

pytestmark = pytest.mark.gpu

D = (0.1, 0.13, 0.17)


@pytest.mark.parametrize("periodic,bc", [(True, (0, 0)), (False, (0, 0)), (False, (1, -1)), (False, (-1, 1))])
@pytest.mark.parametrize("n", [8, 9, 15, 16, 17, 23, 24, 25, 32, 33, 49, 100])
@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("prec", ["f64", "f32_refine"])
def test_filter_once_and_twice(cuda, axis, n, periodic, bc, prec):
    import torch
    dt = torch.float64 if prec == "f64" else torch.float32
    shape = [11, 9, 10]
    shape[axis] = n
    shape = tuple(shape)
    per, bcs = [True] * 3, [(0, 0)] * 3
    per[axis], bcs[axis] = periodic, bc
    f = from_dev(to_dev(random_field(shape, seed=n + axis), dt, cuda), shape)
    for kind in ("gaussian", "lstsq"):
        cg = P.cgrid()
        assert cg.init(shape, D, prec=prec, periodic=tuple(per), bc=tuple(bcs), filter=(kind,) * 3) == 0
        for times in (1, 2, 3, 4):
            ref = f
            for ax in (1, 0, 2):
                for _ in range(times):
                    ref = X.filter_axis(ref, ax, kind, per[ax], *bcs[ax])
            fd = to_dev(f, dt, cuda)
            assert cg.filter(fd, numtimes=times, gaussian=kind == "gaussian") == 0
            torch.cuda.synchronize()
            # 9-point sums with weights of at most 1 in magnitude, FP64; FP32
            # storage rounds each of at most 3 times fields by 2^-24, which
            # the filters that follow damp like the field
            tol = 1e-14 if prec == "f64" else 2.0 ** -24
            assert rel_l2(from_dev(fd, shape), ref) <= tol * 3 * times, (kind, times)


@pytest.mark.parametrize("axis,n,other", [(a, n, (128, 129)) for a in (1, 2) for n in (16, 17, 24, 25, 33, 100)]
                         + [(0, n, (23, 23)) for n in (255, 256, 257, 300)] + [(0, 512, (16, 32)), (0, 4096, (16, 32)),
                                                                             (0, 16, (64, 129))])
@pytest.mark.parametrize("prec", ["f64", "f32_refine"])
def test_filter_large_fields(cuda, axis, n, other, prec):
    """one application in chunks along y and z and in lines along x: more than
    2^18 points, and 512 lines or more of above 256 points (smaller fields
    take a thread per point)"""
    import torch
    dt = torch.float64 if prec == "f64" else torch.float32
    shape = list(other)
    shape.insert(axis, n)
    f = random_field(shape, seed=n + axis)
    ft = to_dev(f, dt, cuda)
    f = from_dev(ft, tuple(shape))
    for periodic, bc in ((True, (0, 0)), (False, (0, 0)), (False, (1, -1))):
        o = P.gaussian()
        o.init(n, periodic)
        out = torch.full_like(ft, float("nan"))
        (o.filter1, o.filter2, o.filter3)[axis](ft, out, *other, *bc, prec=prec)
        torch.cuda.synchronize()
        ref = X.filter_axis(f, axis, "gaussian", periodic, *bc)
        # a 9-point sum in FP64; FP32 storage rounds the output alone
        assert rel_l2(from_dev(out, tuple(shape)), ref) <= (1e-14 if prec == "f64" else 2.0 ** -24), (periodic, bc)


@pytest.mark.parametrize("n", [257, 300, 1023, 1025, 4096, 4097])
@pytest.mark.parametrize("periodic,bc", [(True, (0, 0)), (False, (1, -1))])
@pytest.mark.parametrize("prec", ["f64", "f32_refine"])
def test_filter_long_lines_twice(cuda, n, periodic, bc, prec):
    """few long lines: two applications with up to 1024 threads and 64 KiB of
    LDS up to 4096 points, one after the other beyond"""
    import torch
    dt = torch.float64 if prec == "f64" else torch.float32
    shape = (n, 10, 1)
    ft = to_dev(random_field(shape, seed=n), dt, cuda)
    ref = from_dev(ft, shape)
    cg = P.cgrid()
    assert cg.init(shape, D, prec=prec, periodic=(periodic, True, True), bc=(bc, (0, 0), (0, 0))) == 0
    for ax in (1, 0):  # one point along z: no filter
        for _ in range(2):
            ref = X.filter_axis(ref, ax, "gaussian", periodic if ax == 0 else True, *(bc if ax == 0 else (0, 0)))
    assert cg.filter(ft, numtimes=2, gaussian=True) == 0
    torch.cuda.synchronize()
    # as above, four applications
    assert rel_l2(from_dev(ft, shape), ref) <= 4 * (1e-14 if prec == "f64" else 2.0 ** -24)


@pytest.mark.parametrize("n", [4095, 4096, 4097, 6000])
@pytest.mark.parametrize("prec", ["f64", "f32_refine"])
def test_filter_long_lines(cuda, n, prec):
    import torch
    dt = torch.float64 if prec == "f64" else torch.float32
    shape = (n, 3, 2)
    for periodic in (True, False):
        o = P.gaussian()
        o.init(n, periodic)
        ft = to_dev(random_field(shape, seed=n), dt, cuda)
        out = torch.full_like(ft, float("nan"))
        o.filter1(ft, out, 3, 2, *((0, 0) if periodic else (1, -1)), prec=prec)
        torch.cuda.synchronize()
        ref = X.filter_axis(from_dev(ft, shape), 0, "gaussian", periodic, *((0, 0) if periodic else (1, -1)))
        assert rel_l2(from_dev(out, shape), ref) <= (1e-14 if prec == "f64" else 1e-7)


def _state(shape):
    """phases of no symmetry: no point has a zero density gradient, whose
    direction the artificial bulk viscosity takes"""
    x = list(np.meshgrid(*[2 * np.pi * (np.arange(s) + 0.37) / s for s in shape], indexing="ij"))
    x[0] = x[0] + 0.3 * np.sin(x[1] + 0.7)
    rho = 1.0 + 0.1 * np.sin(x[0] + 0.2) * np.cos(x[1] + 0.9) + 0.05 * np.cos(x[2] + 2 * x[1])
    u, v, w = 0.3 * np.cos(x[1] + x[2] + 0.4), 0.2 * np.sin(x[0] - x[2]), 0.25 * np.sin(x[0] + 1) * np.cos(x[1])
    p = 1.0 + 0.1 * np.cos(x[0] + x[1] + 0.6)
    e = p / (0.4 * rho)
    return np.stack([rho, rho * u, rho * v, rho * w, rho * (e + 0.5 * (u * u + v * v + w * w))], axis=-1)


@pytest.mark.parametrize("periodic", [(True, True, True), (False, True, False), (False, False, False)])
@pytest.mark.parametrize("shape", [(32, 64, 32), (33, 17, 20), (16, 40, 49), (12, 10, 14), (32, 36, 1),
                                   # above 512 rows: two segments per wave, in several passes per launch and
                                   # with the flux sums
                                   (20, 544, 12), (12, 10, 600), (600, 10, 12), (10, 12, 1023)])
def test_rhs(cuda, shape, periodic):
    import torch
    bc = tuple((0, 0) if q else (1, -1) for q in periodic)
    kw = dict(periodic=periodic, bc=bc, inviscid=False, mu_ref=0.02, T_ref=0.9, visc_n=0.7, Pr=0.72)
    W = _state(shape).astype(np.float32).astype(np.float64)
    ref, parts = Cgrid(shape, D, **kw).rhs(W, parts=True)
    for prec in ("f64", "f32_refine"):
        dt = torch.float64 if prec == "f64" else torch.float32
        cg = P.cgrid()
        assert cg.init(shape, D, prec=prec, **kw) == 0
        wd = to_dev(W, dt, cuda)
        rhs = torch.full_like(wd, float("nan"))
        for _ in range(2):  # the second call starts from the first one's sums
            assert cg.getRHS(wd, rhs) == 0
        torch.cuda.synchronize()
        got = from_dev(rhs, shape + (5,))
        for c in range(5):
            err = np.sqrt(np.mean((got[..., c] - ref[..., c]) ** 2))
            if prec == "f64":
                assert err <= 1e-12 * np.sqrt(np.mean(ref[..., c] ** 2)), c
            else:
                # the fluxes, at most 1.5 and the stresses (large where a wall
                # cuts the state), are stored to 2^-24 and a derivative lifts
                # what is rounded by at most 2.6 / dx inside, up to 4 / dx in
                # one-sided closure rows
                top = 1.5 + np.abs(parts["tau"]).max() + np.abs(parts["q"]).max()
                assert err <= 2.0 ** -24 * top * np.sqrt(sum((4.0 / d) ** 2 for d in D)), c


def test_rhs_beyond_shared_launches(cuda):
    """FP32 fields above 16 MiB take one pass per launch, the FP64 ones of the
    same grid (below 64 MiB) several: the two agree to FP32 rounding"""
    import torch
    shape = (170, 160, 160)
    W = _state(shape).astype(np.float32).astype(np.float64)
    out = {}
    for prec, dt in (("f64", torch.float64), ("f32_refine", torch.float32)):
        cg = P.cgrid()
        assert cg.init(shape, D, prec=prec, inviscid=False, mu_ref=0.02, T_ref=0.9, visc_n=0.7, Pr=0.72) == 0
        wd = to_dev(W, dt, cuda)
        rhs = torch.empty_like(wd)
        assert cg.getRHS(wd, rhs) == 0
        torch.cuda.synchronize()
        out[prec] = rhs.double().reshape(5, -1)
    err = (out["f32_refine"] - out["f64"]).square().mean(dim=1).sqrt()
    # the bound of test_rhs inside the domain, 2.6 / dx, fluxes of at most 1.5
    assert err.max().item() <= 2.0 ** -24 * 1.5 * np.sqrt(sum((2.6 / d) ** 2 for d in D))


@pytest.mark.parametrize("prec,n", [("f64", 208), ("f32_refine", 164)])
def test_work_memory_of_large_fields(cuda, prec, n):
    """fields beyond the shared launches (64 MiB, 16 MiB) form one artificial
    coefficient at a time and hold work for one: 46 fields"""
    import gc

    import torch
    gc.collect()  # no earlier object's memory comes back in between
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    cg = P.cgrid()
    assert cg.init((n, n, n), D, prec=prec) == 0
    used = free - torch.cuda.mem_get_info()[0]
    field = n ** 3 * (8 if prec == "f64" else 4)
    assert used <= 47 * field, used / field
