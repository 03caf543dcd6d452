"""rh_interpol_hydro with operands and results in one buffer, within one batch
of its pinned buffer (8,192 octs) and beyond: the octs are those of separate
arrays, and the columns beyond the hydro variables stay as passed."""
import ctypes as C

import numpy as np
import pytest

import rhydro

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [3, 8192, 8193, 20000])
@pytest.mark.parametrize("shift", [0, 64])
def test_shared_buffer(n, shift):
    print(f"case interpol overlap n {n} shift {shift}", flush=True)
    rng = np.random.default_rng(n)
    buf = rng.normal(size=n * 512 + 64)
    u1 = buf[shift:shift + n * 448].reshape(n, 7, 64)
    u1[:, :, 0] = rng.uniform(0.1, 2.0, (n, 7))
    u1[:, :, 4] = rng.uniform(2.0, 4.0, (n, 7))
    s = rhydro.Solver(gamma=1.4, interpol_type=1, interpol_var=0)
    want = s.interpol(u1.copy())[:, :, :5].copy()
    before = buf[:n * 512].reshape(n, 8, 64)[:, :, 5:].copy()
    dp = C.POINTER(C.c_double)
    st = rhydro.lib().rh_interpol_hydro(s._ctx, n, buf[shift:].ctypes.data_as(dp), buf.ctypes.data_as(dp))
    s.close()
    assert st == rhydro.RH_OK
    got = buf[:n * 512].reshape(n, 8, 64)
    np.testing.assert_array_equal(got[:, :, :5], want)
    np.testing.assert_array_equal(got[:, :, 5:], before)
