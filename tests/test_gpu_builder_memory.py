"""The batched builder where the stream-ordered allocator has no room for the
schedule's workspace: the solve takes the instances in input order, with the
results of the scheduled one."""
import ctypes as C

import numpy as np
import pytest

from bacon_amd import _lib as L
from bacon_amd import ivp
from bacon_amd import workloads as W

pytestmark = pytest.mark.gpu

VP = C.c_void_p


class _Location(C.Structure):
    _fields_ = [("type", C.c_int), ("id", C.c_int)]


class _PoolProps(C.Structure):
    _fields_ = [("alloc_type", C.c_int), ("handle_types", C.c_int), ("location", _Location),
                ("security", VP), ("max_size", C.c_size_t), ("reserved", C.c_ubyte * 56)]


def _runtime():
    """The HIP runtime that the process has loaded."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    return C.CDLL(path)


def test_no_room_for_the_schedule(gpu):
    n = 400000
    w = W.lotka_volterra(n)
    s = W.Stream(51, n)
    w.update(t_end=s.uniform(0.1, 0.5), tol=s.log_uniform(1e-8, 1e-5))
    want = ivp.solve_ensemble(L.RK45, w)
    hip = _runtime()
    # a pool of 4 MiB: enough for a launch's counter, not for the sort (three
    # words per instance)
    props = _PoolProps(alloc_type=1, location=_Location(1, 0), max_size=4 << 20)
    small, default, p = VP(), VP(), VP()
    assert hip.hipMemPoolCreate(C.byref(small), C.byref(props)) == 0
    assert hip.hipDeviceGetMemPool(C.byref(default), 0) == 0
    assert hip.hipDeviceSetMemPool(0, small) == 0
    try:
        hip.hipMallocAsync.argtypes = [C.POINTER(VP), C.c_size_t, VP]
        assert hip.hipMallocAsync(C.byref(p), 12 * n, None) != 0
        hip.hipGetLastError()
        got = ivp.solve_ensemble(L.RK45, w)
    finally:
        assert hip.hipDeviceSetMemPool(0, default) == 0
        hip.hipDeviceSynchronize()
        hip.hipMemPoolDestroy(small)
    for k in want:
        assert np.array_equal(got[k], want[k]), k
