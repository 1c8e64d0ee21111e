"""The RK ensemble kernel's attempt loop and work queue at their edges.

Each case is compared with the oracle's DEVICE profile bit for bit (status,
counts, final time and state), as the operations are the same:
  * ensembles around the resident lanes' number (queue or not), with a schedule
    and without, in several launch shapes;
  * attempt caps that instances reach at different times;
  * step-size factors outside the root's range: quotients of 65536 and more
    (loose tolerance, dt at dt_max), of 1e-8 and less (first step far too
    long), NaN (overflowing state), and bounds for which the quotient has to be
    the scaled IEEE division (dt_min 0, an end time at 0).
"""
import ctypes as C

import numpy as np
import pytest

import oracle as O
from bacon_amd import _lib as L
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _solve(w, method=L.RK45, order=None, max_attempts=0, launch=None, semantics=L.INTENDED):
    import torch
    n, dim = w["y0"].shape[1], w["dim"]

    def T(a, dt=torch.float64):
        return torch.as_tensor(np.ascontiguousarray(a), dtype=dt, device="cuda:0")

    b = dict(y0=T(w["y0"]), params=T(w["params"]), t_end=T(w["t_end"]), tol=T(w["tol"]),
             t=T(np.zeros(n)), y=T(np.zeros((dim, n))), st=T(np.full(n, -7), torch.int32),
             cnt=T(np.zeros((n, 2)), torch.int32),
             order=None if order is None else T(order, torch.int32))
    d = L.EnsembleDesc(n=n, dim=dim, n_params=w["params"].shape[0], y0=b["y0"].data_ptr(),
                       params=b["params"].data_ptr(), t0_s=w.get("t0", 0.0),
                       t_end=b["t_end"].data_ptr(), tol=b["tol"].data_ptr(),
                       dt_min_s=w["dt_min"], dt_max_s=w["dt_max"],
                       order=b["order"].data_ptr() if order is not None else None,
                       max_attempts=max_attempts, t_out=b["t"].data_ptr(),
                       y_out=b["y"].data_ptr(), status=b["st"].data_ptr(),
                       counts=b["cnt"].data_ptr())
    rc = L.lib().bg_rk_solve_device(method, L.RHS[w["rhs"]], semantics, C.byref(d),
                                    C.byref(launch) if launch is not None else None, None)
    assert rc == 0
    torch.cuda.synchronize()
    cnt = b["cnt"].cpu().numpy()
    return dict(t=b["t"].cpu().numpy(), y=b["y"].cpu().numpy(), status=b["st"].cpu().numpy(),
                n_accepted=cnt[:, 0], n_rejected=cnt[:, 1])


def _same(w, g, method=O.RK45, max_attempts=0, semantics=O.INTENDED):
    o = O.solve_ensemble(method, w["rhs"], w["y0"], w["params"], w["t_end"], w["tol"],
                         t0=w.get("t0", 0.0), dt_min=w["dt_min"], dt_max=w["dt_max"],
                         semantics=semantics, profile=O.PROFILE_DEVICE, threads=0,
                         max_attempts=max_attempts)
    if max_attempts:
        # the oracle meets the cap before it looks whether the instance is
        # done; the kernels report one that ends with its last attempt as done
        o["status"] = np.where((o["status"] == 9) & (o["t"] >= w["t_end"]), 0, o["status"])
    for k in ("status", "n_accepted", "n_rejected"):
        assert np.array_equal(g[k], o[k]), k
    for k in ("t", "y"):
        assert np.array_equal(g[k], o[k], equal_nan=True), k
    return o


def _lv(n, t_end=0.75, tol=1e-6):
    w = W.lotka_volterra(n)
    s = W.Stream(40, n)
    w["t_end"] = s.uniform(0.0, t_end)
    w["tol"] = s.log_uniform(tol * 1e-3, tol * 1e3)
    return w


@pytest.mark.parametrize("ordered", [False, True])
@pytest.mark.parametrize("n", [1, 63, 64, 65, 16383, 16384, 16385, 16384 + 97, 40001])
def test_sizes_around_the_resident_lanes(gpu, orc, n, ordered):
    """One wave per CU (256 CUs): 16,384 lanes; beyond them the queue hands out
    positions."""
    w = _lv(n)
    order = np.random.default_rng(n).permutation(n) if ordered else None
    for refill in (0, 7, 64):
        lc = L.Launch(block=64, blocks_per_cu=1, refill_min=refill, prio_cutoff=n // 3)
        _same(w, _solve(w, order=order, launch=lc))
    _same(w, _solve(w, order=order))


@pytest.mark.parametrize("cap", [1, 2, 7, 40])
def test_attempt_caps(gpu, orc, cap):
    w = _lv(20000, t_end=6.0)
    lc = L.Launch(block=64, blocks_per_cu=1)
    for launch in (lc, None):
        o = _same(w, _solve(w, max_attempts=cap, launch=launch), max_attempts=cap)
    assert np.any(o["status"] == 9)


@pytest.mark.parametrize("method", ["RK45", "RK23"])
@pytest.mark.parametrize("semantics", [0, 1])
@pytest.mark.parametrize("case", ["at dt_max", "first step too long", "overflow", "dt_min 0",
                                  "end at 0", "huge tol"])
def test_quotients_outside_the_root(gpu, orc, case, method, semantics):
    w = _lv(300, t_end=4.0)
    cap = 3000
    if case == "at dt_max":
        w.update(dt_max=1e-3, tol=np.full(300, 1e-3))
    elif case == "first step too long":
        w.update(dt_max=50.0, tol=np.full(300, 1e-9))
    elif case == "overflow":
        w.update(y0=w["y0"] * 1e160)
    elif case == "dt_min 0":
        w.update(dt_min=0.0)
    elif case == "end at 0":
        w.update(t0=-1.0, t_end=np.zeros(300))
    else:
        w.update(tol=np.geomspace(1e60, 1e140, 300))
    g = _solve(w, method=getattr(L, method), max_attempts=cap, semantics=semantics)
    _same(w, g, getattr(O, method), cap, semantics)


@pytest.mark.parametrize("fields", ["equal", "tol", "t_end", "all"])
@pytest.mark.parametrize("n", [1, 2, 257, 4099])
def test_builder_schedules(gpu, orc, n, fields):
    """The builder's arrays: of one value, or of several (scheduled on the
    device, with an infinite tolerance among them)."""
    from bacon_amd import ivp
    w = _lv(n)
    rng = np.random.default_rng(n)
    w["t_end"], w["tol"], w["t0"] = np.full(n, 0.75), np.full(n, 1e-6), 0.125
    if fields in ("tol", "all"):
        w["tol"] = 10.0 ** rng.uniform(-8, -4, n)
        w["tol"][n // 2] = np.inf
    if fields in ("t_end", "all"):
        w["t_end"] = rng.uniform(0.5, 1.5, n)
    _same(w, ivp.solve_ensemble(L.RK45, dict(w, t0=np.full(n, 0.125))))
