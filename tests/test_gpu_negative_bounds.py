"""Tolerances and step bounds below zero through the device entry points, which
take them as they are (the builders refuse them): no step's error meets a
negative tolerance, and with a negative step the signed error of the
predictor-corrector is below every positive one.  The kernels decide from
squares, whose comparison loses the signs; the outcome has to be the oracle's.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from bacon_amd import _lib as L
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _solve(w, method, cap):
    import torch
    n, dim = w["y0"].shape[1], w["dim"]

    def T(a, dt=torch.float64):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda:0")

    b = dict(y0=T(w["y0"]), params=T(w["params"]), t_end=T(w["t_end"]), tol=T(w["tol"]),
             t=T(np.zeros(n)), y=T(np.zeros((dim, n))), st=T(np.full(n, -7), torch.int32),
             cnt=T(np.zeros((n, 2)), torch.int32))
    d = L.EnsembleDesc(n=n, dim=dim, n_params=w["params"].shape[0], y0=b["y0"].data_ptr(),
                       params=b["params"].data_ptr(), t0_s=0.0, t_end=b["t_end"].data_ptr(),
                       tol=b["tol"].data_ptr(), dt_min_s=w["dt_min"], dt_max_s=w["dt_max"],
                       max_attempts=cap, t_out=b["t"].data_ptr(), y_out=b["y"].data_ptr(),
                       status=b["st"].data_ptr(), counts=b["cnt"].data_ptr())
    if method in (L.ADAMS5, L.ADAMS3):
        rc = L.lib().bg_adams_solve_device(method, L.RHS[w["rhs"]], L.INTENDED, C.byref(d), None)
    else:
        rc = L.lib().bg_bdf_solve_device(method, L.RHS[w["rhs"]], L.INTENDED, 64, C.byref(d),
                                         None)
    assert rc == 0
    torch.cuda.synchronize()
    cnt = b["cnt"].cpu().numpy()
    return dict(t=b["t"].cpu().numpy(), y=b["y"].cpu().numpy(), status=b["st"].cpu().numpy(),
                n_accepted=cnt[:, 0], n_rejected=cnt[:, 1])


def _oracle(w, method, cap):
    return O.solve_ensemble(method, w["rhs"], w["y0"], w["params"], w["t_end"], w["tol"],
                            t0=0.0, dt_min=w["dt_min"], dt_max=w["dt_max"],
                            semantics=O.INTENDED, profile=O.PROFILE_DEVICE, threads=0,
                            max_attempts=cap)


def _lv(n, tol):
    w = W.lotka_volterra(n)
    w.update(t_end=np.full(n, 2.0), tol=np.asarray(tol), dt_min=1e-9)
    return w


@pytest.mark.parametrize("method", ["ADAMS5", "ADAMS3"])
@pytest.mark.parametrize("case", ["tol", "mixed tol", "dt", "dt and tol"])
def test_adams(gpu, orc, method, case):
    n = 130
    mag = np.geomspace(1e-9, 1e-2, n)
    w = _lv(n, mag)
    if "tol" in case:
        w["tol"] = np.where(np.arange(n) % 2 == 0, mag, -mag) if case == "mixed tol" else -mag
    if "dt" in case:
        w.update(dt_min=-0.02, dt_max=-0.01)
    g = _solve(w, getattr(L, method), 150)
    o = _oracle(w, getattr(O, method), 150)
    for k in ("status", "n_accepted", "n_rejected"):
        assert np.array_equal(g[k], o[k]), k
    for k in ("t", "y"):
        assert np.array_equal(g[k], o[k], equal_nan=True), k


@pytest.mark.parametrize("method", ["BDF6", "BDF2"])
@pytest.mark.parametrize("rhs", ["exp", "lotka_volterra", "robertson", "b2", "b4", "b8", "b16"])
def test_bdf(gpu, orc, rhs, method):
    n = 40
    if rhs == "exp":
        w = dict(rhs="exp", dim=1, y0=np.linspace(0.5, 2.0, n)[None], params=np.zeros((0, n)),
                 dt_min=1e-9, dt_max=0.1, t_end=np.full(n, 1.0))
    elif rhs == "lotka_volterra":
        w = _lv(n, np.zeros(n))
    elif rhs == "robertson":
        w = W.robertson(n)
        w["t_end"] = np.full(n, 0.02)
    else:
        w = W.brusselator(n, cells=int(rhs[1:]))
        w["t_end"] = np.full(n, 0.3)
    w["tol"] = -np.geomspace(1e-9, 1e-2, n)
    g = _solve(w, getattr(L, method), 60)
    o = _oracle(w, getattr(O, method), 60)
    for k in ("status", "n_accepted", "n_rejected"):
        assert np.array_equal(g[k], o[k]), k
