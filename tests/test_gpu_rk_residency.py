"""The RK launch's default residency: where the counter kernel chooses between
two and three waves per SIMD (per-instance bounds, 131,073 to 262,144 instances
on 256 CUs), next to it on both sides, and in every block size, each instance has
the bits of the solve with one wave per CU, whatever the bounds are: alike,
different, given for the end, the tolerance or the start alone, scheduled or not,
infinite or already reached.
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from bacon_amd import _lib as L
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _run(w, fields, order, launch):
    import torch
    n = w["y0"].shape[1]

    def T(a, dt=torch.float64):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda:0")

    keep = dict(y0=T(w["y0"]), params=T(w["params"]), t=T(np.zeros(n)), y=T(np.zeros((2, n))),
                st=T(np.full(n, -7), torch.int32), cnt=T(np.zeros((n, 2)), torch.int32))
    d = L.EnsembleDesc(n=n, dim=2, n_params=4, y0=keep["y0"].data_ptr(),
                       params=keep["params"].data_ptr(), dt_min_s=1e-12, dt_max_s=0.1,
                       t_out=keep["t"].data_ptr(), y_out=keep["y"].data_ptr(),
                       status=keep["st"].data_ptr(), counts=keep["cnt"].data_ptr())
    for k in ("t0", "t_end", "tol"):
        if k in fields:
            keep[k] = T(w[k])
            setattr(d, k, keep[k].data_ptr())
        else:
            setattr(d, k + "_s", float(w[k][0]))
    if order is not None:
        keep["order"] = T(order, torch.int32)
        d.order = keep["order"].data_ptr()
    assert L.lib().bg_rk_solve_device(L.RK45, L.RHS["lotka_volterra"], L.INTENDED, C.byref(d),
                                      C.byref(launch), None) == 0
    torch.cuda.synchronize()
    return {k: keep[k].cpu().numpy() for k in ("t", "y", "st", "cnt")}


@pytest.mark.parametrize("n", [131072, 131073, 200001, 262144, 262145])
@pytest.mark.parametrize("case", ["alike", "t_end", "tol", "t0", "odd"])
def test_choice_of_residency(gpu, orc, n, case):
    w = W.lotka_volterra(n)
    s = W.Stream(50, n)
    w.update(t0=np.zeros(n), t_end=np.full(n, 0.2), tol=np.full(n, 1e-6))
    fields = ("t_end", "tol")
    if case == "t_end":
        w["t_end"], fields = s.uniform(0.0, 0.4), ("t_end",)
    elif case == "tol":
        w["tol"], fields = s.log_uniform(1e-9, 1e-4), ("tol",)
    elif case == "t0":
        w["t0"], fields = s.uniform(0.0, 0.25), ("t0",)
    elif case == "odd":
        # bounds for which the predicted cost is no number to compare
        w["tol"] = np.where(np.arange(n) % 5 == 0, np.inf, 1e-6)
        w["t0"] = np.where(np.arange(n) % 3 == 0, 0.2, 0.0)
        fields = ("t0", "t_end", "tol")
    ref = _run(w, fields, None, L.Launch(block=64, blocks_per_cu=1))
    order = np.random.default_rng(n).permutation(n)
    for block in (0, 64, 128, 192):
        for o in (None, order):
            g = _run(w, fields, o, L.Launch(block=block))
            for k in ref:
                assert np.array_equal(g[k], ref[k]), (k, block)
    pick = np.arange(0, n, 997)
    for t0 in np.unique(w["t0"][pick])[:2]:  # the oracle takes one start
        p = pick[w["t0"][pick] == t0]
        r = O.solve_ensemble(O.RK45, "lotka_volterra", w["y0"][:, p], w["params"][:, p],
                             w["t_end"][p], w["tol"][p], t0=t0, dt_min=1e-12, dt_max=0.1,
                             profile=O.PROFILE_DEVICE, threads=0)
        assert np.array_equal(ref["y"][:, p], r["y"])
        assert np.array_equal(ref["st"][p], r["status"])
