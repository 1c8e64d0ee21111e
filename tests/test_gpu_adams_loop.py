"""The Adams ensemble kernel's two phases at their edges, bit for bit against
the oracle's DEVICE profile: caps that fall on every kind of call (bootstrap,
first multistep, the yields after it, an ordinary step, the final step),
ensembles of one lane up to more than the resident ones, and tolerances for
which no step is an ordinary one.
"""
import numpy as np
import pytest

import oracle as O
from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _same(w, method, semantics=L.INTENDED, cap=0):
    g = ivp.solve_ensemble(getattr(L, method), w, semantics=semantics, max_attempts=cap)
    o = O.solve_ensemble(getattr(O, method), w["rhs"], w["y0"], w["params"], w["t_end"], w["tol"],
                         t0=w["t0"], dt_min=w["dt_min"], dt_max=w["dt_max"], semantics=semantics,
                         profile=O.PROFILE_DEVICE, threads=0, max_attempts=cap)
    for k in ("status", "n_accepted", "n_rejected", "t", "y"):
        assert np.array_equal(g[k], o[k]), k
    return o


def _lv(n, t_end, tol_lo, tol_hi):
    w = W.lotka_volterra(n)
    s = W.Stream(41, n)
    w["t_end"] = s.uniform(0.01, t_end)
    w["tol"] = s.log_uniform(tol_lo, tol_hi)
    w["dt_min"] = 1e-9
    return w


@pytest.mark.parametrize("semantics", [L.AS_BUILT, L.INTENDED])
@pytest.mark.parametrize("method", ["ADAMS5", "ADAMS3"])
@pytest.mark.parametrize("cap", [1, 2, 3, 4, 5, 6, 7, 8, 9, 13, 40, 150])
def test_caps(gpu, orc, method, semantics, cap):
    o = _same(_lv(400, 6.0, 1e-7, 1e-3), method, semantics, cap)
    assert np.any(o["status"] == 9)


@pytest.mark.parametrize("n", [1, 2, 63, 65, 1000, 340001])
def test_sizes(gpu, orc, n):
    _same(_lv(n, 0.4 if n > 10000 else 5.0, 1e-6, 1e-3), "ADAMS5")


@pytest.mark.parametrize("tol", [1e-145, 1e-30, 1e60, 1e145])
def test_no_ordinary_steps(gpu, orc, tol):
    w = _lv(100, 2.0, 1e-6, 1e-3)
    w["tol"] = np.full(100, tol)
    w["dt_min"] = 1e-4
    _same(w, "ADAMS5", cap=2000)
