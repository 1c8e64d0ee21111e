"""Path output through the packed records (ensembles whose buffers exceed the
chip's L2) against the direct stores of a smaller ensemble of the same
instances: every entry, written or not, is the same bit for bit, in both
layouts, for each record size (1 to 4 components), with the ring wrapped and
not, every step and every third one, with stops between.
"""
import numpy as np
import pytest

from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _workload(rhs, n):
    if rhs == "lotka_volterra":
        w = W.lotka_volterra(n)
        w.update(t_end=W.Stream(42, n).uniform(0.5, 6.0), tol=np.full(n, 1e-7))
    elif rhs == "two_level":
        w = W.two_level(n)
        w.update(t_end=W.Stream(42, n).uniform(0.5, 4.0))
    elif rhs == "lorenz":
        w = W.lorenz_plain(n)
        w.update(t_end=W.Stream(42, n).uniform(0.05, 0.5))
    else:
        w = dict(rhs="neg", dim=1, y0=W.Stream(43, n).uniform(0.5, 2.0)[None], t0=0.0,
                 params=np.zeros((0, n)), t_end=W.Stream(42, n).uniform(0.5, 6.0),
                 tol=np.full(n, 1e-9), dt_min=1e-12, dt_max=0.1)
    return w


def _part(w, m):
    p = dict(w)
    for k in ("y0", "params"):
        p[k] = np.ascontiguousarray(w[k][:, :m])
    for k in ("t_end", "tol"):
        p[k] = w[k][:m]
    return p


@pytest.mark.parametrize("inst_major", [False, True])
@pytest.mark.parametrize("rhs,n,capacity", [("lotka_volterra", 20011, 61),
                                            ("two_level", 17001, 67), ("lorenz", 40003, 33),
                                            ("neg", 65601, 45), ("neg", 300001, 9)])
def test_packed_equals_direct(gpu, rhs, n, capacity, inst_major):
    w = _workload(rhs, n)
    m = 777
    for every, stops in ((1, None), (3, np.array([0.02, 0.3, 0.9, 2.5]))):
        a = ivp.solve_path(L.RK45, w, capacity, every=every, stops=stops,
                           instance_major=inst_major)
        b = ivp.solve_path(L.RK45, _part(w, m), capacity, every=every, stops=stops,
                           instance_major=inst_major)
        for k in ("t", "status", "n_accepted", "n_rejected", "path_len"):
            assert np.array_equal(a[k][:m], b[k]), k
        assert np.array_equal(a["y"][:, :m], b["y"])
        assert np.array_equal(a["path_t"][:, :m], b["path_t"])
        assert np.array_equal(a["path_y"][:, :, :m], b["path_y"])
        # the whole ensemble: no entry beyond its instance's records is written
        assert np.all(a["status"] == 0)
        kept = np.minimum(a["path_len"], capacity)
        written = np.arange(capacity)[:, None] < kept[None]
        assert np.array_equal(a["path_t"] != 0.0, written)
