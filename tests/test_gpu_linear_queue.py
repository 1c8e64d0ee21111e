"""The shared-matrix kernel's column queue and controller: an ensemble larger
than the resident columns gives every instance the bits it has in a small one,
at ends and tolerances that differ; the quotient without range scaling (dt_min
1e-40) and the scaled IEEE division (dt_min 1e-300) give the same bits, also where
dt sits at dt_max.
"""
import numpy as np
import pytest

from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _workload(N, n, t_end=0.4):
    w = W.linear_shared(n, N=N)
    s = W.Stream(44, n)
    w["t_end"] = s.uniform(0.0, t_end)
    w["tol"] = s.log_uniform(1e-9, 1e-2)
    return w


def _equal(a, b, m):
    for k in ("t", "status", "n_accepted", "n_rejected"):
        assert np.array_equal(a[k][:m], b[k][:m]), k
    assert np.array_equal(a["y"][:, :m], b["y"][:, :m])


@pytest.mark.parametrize("N,n", [(32, 33001), (64, 16499), (128, 8209)])
def test_more_instances_than_columns(gpu, N, n):
    w = _workload(N, n)
    a = ivp.solve_ensemble(L.RK45, w)
    m = 203
    part = dict(w, y0=np.ascontiguousarray(w["y0"][:, :m]), params=np.zeros((0, m)),
                t_end=w["t_end"][:m], tol=w["tol"][:m])
    _equal(a, ivp.solve_ensemble(L.RK45, part), m)
    assert np.all(a["status"] == 0)


@pytest.mark.parametrize("N", [32, 64, 128])
def test_division_forms_agree(gpu, N):
    # both lower bounds leave the first step, (dt_max + dt_min) / 2, the same
    w = dict(_workload(N, 150, t_end=3.0), dt_min=1e-40)
    a = ivp.solve_ensemble(L.RK45, w)
    tiny = dict(w, dt_min=1e-300)  # outside the range of the short division
    _equal(a, ivp.solve_ensemble(L.RK45, tiny), 150)
