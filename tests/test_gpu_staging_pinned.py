"""State arrays in pinned memory, which long copies leave to the runtime, next to
pageable ones: every value comes back as it went, also where one array is pinned
and the other is not, and while an adaptive run works in another thread."""
import ctypes as C
import threading

import numpy as np
import pytest

import rhydro
from rhydro import RH_UNEW, RH_UOLD

pytestmark = pytest.mark.gpu

hip = C.CDLL("libamdhip64.so")
hip.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
hip.hipHostFree.argtypes = [C.c_void_p]


def _round_trip(s, m):
    want = m.uold.copy(), m.unew.copy()
    s.sync_to_device()
    m.uold[:] = -1.0
    m.unew[:] = -2.0
    s.sync_to_host(RH_UOLD)
    assert (m.unew == -2.0).all()
    s.sync_to_host(RH_UNEW)
    np.testing.assert_array_equal(m.uold, want[0])
    np.testing.assert_array_equal(m.unew, want[1])


@pytest.mark.parametrize("pinned", [("uold",), ("unew",), ("uold", "unew")])
@pytest.mark.parametrize("ngridmax", [100, 33001, 150001])  # 0.03, 10.6 and 48 MB
def test_pinned(ngridmax, pinned):
    print(f"case staging pinned {pinned} ngridmax {ngridmax}", flush=True)
    m = rhydro.uniform_mesh(2, ngridmax=ngridmax)
    held = []
    for k in pinned:
        p = C.c_void_p()
        assert hip.hipHostMalloc(C.byref(p), m.arrays[k].nbytes, 0) == 0
        held.append(p)
        m.arrays[k] = np.ctypeslib.as_array((C.c_double * m.arrays[k].size).from_address(p.value))
    rng = np.random.default_rng(ngridmax)
    for k in ("uold", "unew"):
        m.arrays[k][:] = rng.random(m.arrays[k].size)
    s = rhydro.Solver()
    s.bind(m)
    _round_trip(s, m)
    s.close()
    m.arrays.clear()
    for p in held:
        hip.hipHostFree(p)


def test_beside_an_adaptive_run():
    print("case staging beside an adaptive run", flush=True)
    kw = dict(levelmin=4, levelmax=6, ngridmax=40000, err_grad_d=0.1, err_grad_p=0.1, riemann="hllc",
              regions=rhydro.sedov_regions(4))
    runs, errs = [], []

    def work():
        try:
            a = rhydro.AmrRun(**kw)
            a.step(6)
            runs.append(a.state()["uold"].copy())
            a.close()
        except BaseException as e:
            errs.append(e)

    work()
    t = threading.Thread(target=work)
    t.start()
    for r in range(4):
        m = rhydro.uniform_mesh(2, ngridmax=60000 + r)
        m.uold[:] = np.random.default_rng(r).random(m.uold.size)
        m.unew[:] = 2.0 * m.uold
        s = rhydro.Solver()
        s.bind(m)
        _round_trip(s, m)
        s.close()
    t.join()
    assert not errs, errs
    np.testing.assert_array_equal(runs[0], runs[1])
