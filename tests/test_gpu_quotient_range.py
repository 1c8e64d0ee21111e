"""Instances whose controller quotients may leave the range of the division
without scaling (no lower step bound, an end or a stop at t = 0, tolerances up
to 1e+-145): every attempt decides by its own numerator, in waves that hold both
kinds.  Compared bit for bit with the oracle's DEVICE profile, whose quotient is
the IEEE division throughout, or with the solve that stays within the range.
"""
import numpy as np
import pytest

import oracle as O
from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W
from test_gpu_rk_loop import _same, _solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("method", ["RK45", "RK23"])
@pytest.mark.parametrize("dt_min", [0.0, 1e-300])
def test_numerators_around_the_range(gpu, orc, method, dt_min):
    """q2 = (tol h)^2 crosses 2^-920 at tol h = 3.4e-139 and 2^900 at 2.9e135."""
    n = 400
    w = W.lotka_volterra(n)
    s = W.Stream(47, n)
    tol = np.where(np.arange(n) % 2 == 0, s.log_uniform(1e-9, 1e-4),
                   np.where(np.arange(n) % 4 == 1, s.log_uniform(1e-145, 1e-125),
                            s.log_uniform(1e128, 1e145)))
    w.update(t_end=s.uniform(0.1, 3.0), tol=tol, dt_min=dt_min)
    g = _solve(w, method=getattr(L, method), max_attempts=400)
    _same(w, g, getattr(O, method), 400)


@pytest.mark.parametrize("N", [32, 64, 128])
def test_linear(gpu, N):
    """No lower bound against 1e-40: the first steps, (dt_max + dt_min) / 2, are
    the same."""
    w = W.linear_shared(90, N=N)
    s = W.Stream(48, 90)
    w.update(t_end=s.uniform(0.1, 2.0), dt_min=1e-40,
             tol=np.where(np.arange(90) % 3 == 0, 1e140, s.log_uniform(1e-8, 1e-2)))
    a, b = (ivp.solve_ensemble(L.RK45, dict(w, dt_min=d)) for d in (1e-40, 1e-300))
    for k in ("t", "status", "n_accepted", "n_rejected", "y"):
        assert np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("method", ["RK45", "RK23"])
@pytest.mark.parametrize("start,end", [(-2.0, 0.0), (0.0, 1e-300), (-1e-300, 1.5), (-1e-70, 0.0),
                                       (1e-250, 2.0), (-3.0, -1e-62), (1e-62, 1.0)])
def test_times_around_zero(gpu, orc, method, start, end):
    n = 130
    w = W.lotka_volterra(n)
    s = W.Stream(49, n)
    w.update(t0=start, t_end=np.full(n, end), tol=s.log_uniform(1e-9, 1e-4))
    g = _solve(w, method=getattr(L, method), max_attempts=400)
    _same(w, g, getattr(O, method), 400)


@pytest.mark.parametrize("near", [0.0, 1e-300, -1e-300, 1e-70, -1e-70, 5e-324])
@pytest.mark.parametrize("n_more", [0, 1100])
def test_stops_around_zero(gpu, near, n_more):
    """A stop at or next to zero, among few stops (in LDS) and among more than
    fit there: every stop is landed on, and the states at the others are those
    of the solve without it (global errors at tol 1e-8 stay far below 1e-5)."""
    n = 70
    w = W.lotka_volterra(n)
    w.update(t0=-1.0, t_end=np.full(n, 1.0), tol=np.full(n, 1e-8))
    more = np.linspace(0.25, 0.75, n_more) if n_more else np.array([0.5])
    stops = np.concatenate([[-0.5, near], more])
    for only in (True, False):
        g = ivp.solve_path(L.RK45, w, 4000, stops=stops, stops_only=only)
        assert np.all(g["status"] == 0)
        times = g["path_t"][:, 0][:g["path_len"][0]]
        assert np.all(np.isin(stops, times)) and times[-1] == 1.0
        if only:
            assert np.array_equal(times, np.append(stops, 1.0))
            r = ivp.solve_path(L.RK45, w, 4000, stops=np.concatenate([[-0.5], more]),
                               stops_only=True)
            assert np.abs(g["path_y"][2:stops.size + 1] - r["path_y"][1:stops.size]).max() < 1e-5
