"""igrid steps on boxes at the edges of the line transforms' ranges: the
shortest and longest lines of x and y, several fields to a launch and one,
plane counts of cells and edges that end inside a group of lines."""
import numpy as np
import pytest

import padeops_amd as P
from oracle.igrid import Igrid

pytestmark = pytest.mark.gpu

# (nx, ny, nz): nx from 16 to 1024, ny from 8 to 1024
SHAPES = [(16, 8, 16), (32, 128, 16), (128, 16, 32), (1024, 8, 16), (16, 1024, 16), (512, 64, 32)]


def _velocity(nx, ny, nz, walls):
    x = np.arange(nx)[:, None, None] * 2 * np.pi / nx
    y = np.arange(ny)[None, :, None] * 2 * np.pi / ny
    zc = (np.arange(nz) + 0.5)[None, None, :] * 2 * np.pi / nz
    ze = np.arange(nz + 1)[None, None, :] * 2 * np.pi / nz
    u = np.sin(x) * np.cos(2 * y) * np.cos(zc) + 0.3 * np.cos(3 * x + y) + (2.0 if walls else 0.0)
    v = -np.cos(x) * np.sin(y) + 0.2 * np.sin(2 * y + zc)
    w = 0.3 * np.sin(x + y) * np.sin(ze)
    return u, v, w


@pytest.mark.parametrize("prec", ["f64", "f32_refine"])
@pytest.mark.parametrize("walls", [False, True])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_step_matches_oracle(cuda, shape, walls, prec):
    import torch

    from fields import from_dev, rel_l2, to_dev
    nx, ny, nz = shape
    W = dict(botWall=1, topWall=2, dpFdx=0.5) if walls else None
    L = (2 * np.pi,) * 3
    ref = Igrid(nx, ny, nz, *L, Re=200.0, scheme=1, dt=2e-3, sgs=dict(model=0, cglobal=1e-3), walls=W)
    dt = torch.float64 if prec == "f64" else torch.float32
    vel = [q.astype(np.float32).astype(np.float64) for q in _velocity(nx, ny, nz, walls)]
    ref.set_velocity(*vel)
    ref.step()
    g = P.igrid()
    assert g.init(nx, ny, nz, *L, Re=200.0, scheme=1, dt=2e-3, sgs=dict(model="smagorinsky", cglobal=1e-3), walls=W,
                  prec=prec) == 0
    g.set_velocity(*[to_dev(np.asfortranarray(q), dt, cuda) for q in vel])
    g.step()
    torch.cuda.synchronize()
    # one step of rounding errors: a few hundred ulp of the storage type in
    # the velocity, a factor k_max dz (at most 500 here) more in its gradients
    tol = 1e-13 if prec == "f64" else 3e-6
    for name, nzz in (("u", nz), ("v", nz), ("w", nz + 1), ("wC", nz), ("uE", nz + 1), ("vE", nz + 1)):
        assert rel_l2(from_dev(g.field(name), (nx, ny, nzz)), ref.f[name]) < tol, name
    for name, nzz in (("duidxjC", nz), ("duidxjE", nz + 1)):
        assert rel_l2(from_dev(g.field(name), (nx, ny, nzz, 9)), ref.f[name]) < 500 * tol, name
