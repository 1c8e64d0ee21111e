"""Packed path output with a capacity far above the records, and with more
entries than a grid's y dimension has blocks for: the same entries, written or
not, as the direct stores of a smaller ensemble of the same instances (sizes
below 32 MiB of records are not packed).
"""
import numpy as np
import pytest

from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu


def _part(w, m):
    p = dict(w)
    for k in ("y0", "params"):
        p[k] = np.ascontiguousarray(w[k][:, :m])
    for k in ("t_end", "tol"):
        p[k] = w[k][:m]
    return p


def _same(w, m, capacity, **kw):
    a = ivp.solve_path(L.RK45, w, capacity, **kw)
    b = ivp.solve_path(L.RK45, _part(w, m), capacity, **kw)
    for k in ("t", "status", "n_accepted", "n_rejected", "path_len"):
        assert np.array_equal(a[k][:m], b[k]), k
    assert np.array_equal(a["path_t"][:, :m], b["path_t"])
    assert np.array_equal(a["path_y"][:, :, :m], b["path_y"])
    assert np.all(a["status"] == 0)
    kept = np.minimum(a["path_len"], capacity)
    assert np.array_equal(a["path_t"] != 0.0, np.arange(capacity)[:, None] < kept[None])
    return a


@pytest.mark.parametrize("stops", [None, np.array([0.1, 0.4])])
@pytest.mark.parametrize("n,capacity", [(20011, 301), (135001, 41)])
def test_capacity_above_the_records(gpu, n, capacity, stops):
    """Some instances of each 64 record nothing, some a few entries of one tile
    of eight, some several tiles."""
    w = W.lotka_volterra(n)
    s = W.Stream(46, n)
    w.update(t_end=s.uniform(-0.3, 0.9), tol=np.full(n, 1e-6))
    for inst_major in (False, True):
        a = _same(w, 500, capacity, stops=stops, instance_major=inst_major)
        assert a["path_len"].min() == 0 and 8 < a["path_len"].max() < capacity


@pytest.mark.parametrize("inst_major", [False, True])
def test_few_instances_with_a_large_capacity(gpu, inst_major):
    """Six instances, 530,000 entries of one component: 66,250 tiles of eight,
    the last of them written before the ring wraps."""
    n, capacity = 6, 530000
    w = dict(rhs="neg", dim=1, y0=np.linspace(0.5, 2.0, n)[None], params=np.zeros((0, n)), t0=0.0,
             t_end=np.linspace(0.05, 0.54, n), tol=np.full(n, 1e-6), dt_min=1e-12, dt_max=1e-6)
    a = _same(w, 1, capacity, instance_major=inst_major)
    assert a["path_len"][0] < 60000 and a["path_len"][-1] > capacity
    assert np.all(np.abs(a["path_y"][:1000, 0] / (w["y0"][0] * np.exp(-a["path_t"][:1000])) - 1)
                  < 1e-6)


def test_packed_on_two_streams(gpu):
    """Calls on two streams, from two threads, without a synchronisation between
    them: the packed records' workspaces, which come from one pool and go back
    while the other stream's kernels run, keep the calls apart."""
    import ctypes as C
    import threading

    import torch
    n, capacity = 20011, 61
    sizes = [capacity, capacity - 3, capacity + 7]

    def inputs(index):
        s = W.Stream(52 + index, n)
        w = W.lotka_volterra(n, first=index * n)
        y0, p, end = (torch.as_tensor(a, device="cuda:0")
                      for a in (w["y0"], w["params"], s.uniform(0.5, 4.0)))
        return y0.contiguous(), p.contiguous(), end

    def call(inp, cap, stream):
        y0, p, end = inp
        out = dict(pt=torch.zeros((cap, n), dtype=torch.float64, device="cuda:0"),
                   py=torch.zeros((cap, 2, n), dtype=torch.float64, device="cuda:0"),
                   pl=torch.zeros(n, dtype=torch.int32, device="cuda:0"))
        torch.cuda.current_stream().synchronize()
        d = L.EnsembleDesc(n=n, dim=2, n_params=4, y0=y0.data_ptr(), params=p.data_ptr(),
                           t_end=end.data_ptr(), tol_s=1e-7, dt_min_s=1e-12, dt_max_s=0.1)
        pd = L.PathDesc(capacity=cap, every=1, n_stops=0, flags=0, stops=None,
                        path_t=out["pt"].data_ptr(), path_y=out["py"].data_ptr(),
                        path_len=out["pl"].data_ptr())
        rc = L.lib().bg_rk_solve_path_device(L.RK45, L.RHS["lotka_volterra"], L.INTENDED,
                                             C.byref(d), C.byref(pd),
                                             C.c_void_p(stream.cuda_stream))
        assert rc == 0
        return out

    ins = [inputs(0), inputs(1)]
    want = []
    for inp in ins:
        want.append([call(inp, cap, torch.cuda.current_stream()) for cap in sizes])
        torch.cuda.synchronize()
    got = [[], []]

    def work(index):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for k in range(12):
                got[index].append(call(ins[index], sizes[k % 3], stream))
        stream.synchronize()

    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for index in (0, 1):
        assert len(got[index]) == 12
        for k, g in enumerate(got[index]):
            for key, v in g.items():
                assert torch.equal(v, want[index][k % 3][key]), (index, k, key)
