"""The BDF ensemble kernels' passes at their edges.

  * Caps that fall on every kind of call (bootstrap, multistep, the yields
    after a bootstrap, the final step): status and accepted calls as the oracle
    counts them.
  * The ensemble's calls, bootstraps and multisteps taken together, yield as
    often as the single-instance iterator's, one by one, and end at the same
    state bit for bit (the same device code), and an instance has the same bits in any company: alone, in a wave
    with others, and behind the queue.
"""
import numpy as np
import pytest

import oracle as O
from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _workload(rhs, n):
    if rhs == "lotka_volterra":
        w = W.lotka_volterra(n)
        w.update(tol=np.full(n, 1e-6), t_end=W.Stream(45, n).uniform(0.05, 1.0), dt_min=1e-9)
    elif rhs == "robertson":
        w = W.robertson(n)
        w["t_end"] = W.Stream(45, n).uniform(0.002, 0.02)
    else:
        w = W.brusselator(n, cells=int(rhs[1:]))
        w.update(tol=np.full(n, 1e-6), t_end=W.Stream(45, n).uniform(0.02, 0.3))
    return w


def _part(w, sel):
    p = dict(w)
    for k in ("y0", "params"):
        p[k] = np.ascontiguousarray(w[k][:, sel])
    for k in ("t_end", "tol"):
        p[k] = w[k][sel]
    return p


@pytest.mark.parametrize("method", ["BDF6", "BDF2"])
@pytest.mark.parametrize("rhs", ["lotka_volterra", "robertson", "b2"])
@pytest.mark.parametrize("cap", [1, 2, 3, 5, 9, 10, 11, 25])
def test_caps(gpu, orc, rhs, method, cap):
    w = _workload(rhs, 70)
    g = ivp.solve_ensemble(getattr(L, method), w, max_attempts=cap)
    o = O.solve_ensemble(getattr(O, method), w["rhs"], w["y0"], w["params"], w["t_end"], w["tol"],
                         dt_min=w["dt_min"], dt_max=w["dt_max"], profile=O.PROFILE_DEVICE,
                         threads=0, max_attempts=cap)
    assert np.array_equal(g["status"], o["status"])
    assert np.array_equal(g["n_accepted"], o["n_accepted"])


@pytest.mark.parametrize("cls,method", [(ivp.BDF6, L.BDF6), (ivp.BDF2, L.BDF2)])
@pytest.mark.parametrize("rhs", ["lotka_volterra", "robertson", "b2", "b4", "b8"])
def test_iterator_and_ensemble_agree(gpu, rhs, cls, method):
    w = _workload(rhs, 40)
    g = ivp.solve_ensemble(method, w)
    assert np.all(g["status"] == 0)
    for i in (0, 7, 39):
        s = (cls.new(w["dim"]).with_minimum_dt(w["dt_min"]).with_maximum_dt(w["dt_max"])
             .with_tolerance(w["tol"][i]).with_initial_time(0.0).with_ending_time(w["t_end"][i])
             .with_initial_conditions(w["y0"][:, i]).with_derivative(w["rhs"], w["params"][:, i]))
        path = s.solve().collect_vec()
        assert len(path) == g["n_accepted"][i]
        # a bootstrap that reaches the end yields none of its values
        # (bdf.rs:519-546): then the path stops before the final state
        if path and path[-1][0] == g["t"][i]:
            assert np.array_equal(path[-1][1], g["y"][:, i])


@pytest.mark.parametrize("rhs,n", [("lotka_volterra", 140001), ("robertson", 50007),
                                   ("b2", 50007), ("b4", 17003), ("b8", 9001), ("b16", 4500)])
def test_same_bits_in_any_company(gpu, rhs, n):
    w = _workload(rhs, n)
    w["t_end"] = w["t_end"] * 0.2
    g = ivp.solve_ensemble(L.BDF6, w)
    assert np.all(g["status"] == 0)
    for sel in (np.arange(0, 200), np.array([3]), np.arange(n - 65, n)):
        p = ivp.solve_ensemble(L.BDF6, _part(w, sel))
        for k in ("t", "n_accepted", "n_rejected", "n_newton", "n_lu"):
            assert np.array_equal(p[k], g[k][sel]), k
        assert np.array_equal(p["y"], g["y"][:, sel])


@pytest.mark.parametrize("n", [1, 768, 3073, 5120, 5121])
def test_inverses_of_the_whole_wave_solver(gpu, n):
    """The 32-component solver around the sizes at which its kernel changes:
    the same bits as in another ensemble, and the FP32 inverse (an error of
    about 1e-7 of the correction) leads to the accepted steps and, within 2 %,
    to the iterations of the FP64 one."""
    w = W.brusselator(n, cells=16)
    w["t_end"] = np.full(n, 0.4)
    g = ivp.solve_ensemble(L.BDF6, w)
    assert (g["status"] == 0).all()
    pick = np.unique(np.linspace(0, n - 1, 7).astype(int))
    p = ivp.solve_ensemble(L.BDF6, _part(w, pick))
    for k in ("t", "status", "n_accepted", "n_rejected", "n_newton", "n_lu"):
        assert np.array_equal(p[k], g[k][pick]), k
    assert np.array_equal(p["y"], g["y"][:, pick])
    f = ivp.solve_ensemble(L.BDF6, w, lu_bits=32)
    assert (f["status"] == 0).all()
    assert np.mean(f["n_accepted"] != g["n_accepted"]) <= 0.01
    assert abs(f["n_newton"].sum() - g["n_newton"].sum()) <= 0.02 * g["n_newton"].sum()
    assert np.abs(f["y"] - g["y"]).max() < 1e-5
