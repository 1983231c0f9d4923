"""igrid.field: a view keeps the solver whose memory it shows."""
import ctypes
import gc
import types
import weakref

import numpy as np
import pytest

import padeops_amd as P


def test_view_keeps_its_solver(monkeypatch):
    """a library whose solver is a host buffer, and as_tensor over it through
    numpy, which like the device form holds the object it wraps"""
    import torch
    buf = (ctypes.c_double * (4 * 4 * 4))(*range(64))
    freed = []

    def field(h, which, out):
        ctypes.cast(out, ctypes.POINTER(ctypes.c_void_p))[0] = ctypes.addressof(buf)
        return 0

    def as_tensor(holder, device):
        holder.__array_interface__ = holder.__cuda_array_interface__
        return torch.from_numpy(np.asarray(holder))

    fake = types.SimpleNamespace(pdo_igrid_field=field, pdo_igrid_destroy=lambda h: freed.append(1))
    monkeypatch.setattr(P, "lib", lambda: fake)
    monkeypatch.setattr(torch, "as_tensor", as_tensor)
    g = P.igrid()
    g._h, g.shape, g.prec = ctypes.c_void_p(1), (4, 4, 4), "f64"
    view, alive = g.field("u"), weakref.ref(g)
    del g
    gc.collect()
    assert alive() is not None and not freed
    part = view.view(4, 4, 4)[1:]
    del view
    gc.collect()
    assert not freed and torch.equal(part.flatten(), torch.arange(16.0, 64.0, dtype=torch.float64))
    del part
    gc.collect()
    assert freed and alive() is None


@pytest.mark.gpu
def test_views_after_the_solver_goes(cuda):
    import torch
    n = 16
    r = np.random.default_rng(0)

    def views():
        g = P.igrid()
        assert g.init(n, n, n, 1.0, 1.0, 1.0, dt=1e-3, prec="f64") == 0
        u = [torch.as_tensor(r.standard_normal(m), device=cuda) for m in (n ** 3, n ** 3, n * n * (n + 1))]
        u[2][-n * n:] = u[2][:n * n]
        assert g.set_velocity(*u) == 0
        return g, {k: g.field(k) for k in g.FIELDS}

    g, v = views()
    torch.cuda.synchronize()
    kept = {k: t.clone() for k, t in v.items()}
    alive = weakref.ref(g)
    del g
    gc.collect()
    assert alive() is not None
    fill = [torch.zeros(9 * n * n * (n + 1), dtype=torch.float64, device=cuda) for _ in range(8)]
    assert all(torch.equal(v[k], kept[k]) for k in v) and len(fill) == 8
    del v
    gc.collect()
    assert alive() is None
