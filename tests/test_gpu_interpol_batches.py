"""rh_interpol_hydro at the edges of its blocks (64 octs), of its pinned buffer
and of its batches (8,192 octs): every oct must equal the oracle's, and the
columns beyond the hydro variables must be returned as they were passed."""
import numpy as np
import pytest

import oracle
import rhydro

pytestmark = pytest.mark.gpu


def _rows(n, seed):
    rng = np.random.default_rng(seed)
    u1 = rng.normal(size=(n, 7, 64))
    u1[:, :, 0] = rng.uniform(0.1, 2.0, (n, 7))
    u1[:, :, 4] = rng.uniform(2.0, 4.0, (n, 7))
    return u1


def _check(got, u1, po, octs):
    for o in octs:
        np.testing.assert_array_equal(got[o][:, :5], oracle.interpol(po, u1[o])[:, :5])


@pytest.mark.parametrize("n", [1, 63, 65, 8191, 8192, 8193])
def test_batches(n):
    print(f"case interpol batches n {n}", flush=True)
    u1 = _rows(n, n)
    s = rhydro.Solver(gamma=1.4, interpol_type=1, interpol_var=0)
    got = s.interpol(u1)
    again = s.interpol(u1[: max(1, n // 3)])
    s.close()
    po = oracle.params(gamma=1.4, interpol_type=1, interpol_var=0)
    octs = sorted({0, n // 2, n - 1, min(n - 1, 64), min(n - 1, 8191)})
    _check(got, u1, po, octs)
    np.testing.assert_array_equal(again[:, :, :5], got[: max(1, n // 3), :, :5])


def test_other_columns_stay():
    print("case interpol other columns", flush=True)
    n = 65
    u1 = _rows(n, 7)
    u2 = np.random.default_rng(8).normal(size=(n, 8, 64))
    before = u2.copy()
    s = rhydro.Solver(gamma=1.4, interpol_type=3, interpol_var=2)
    s.interpol(u1, u2)
    s.close()
    _check(u2, u1, oracle.params(gamma=1.4, interpol_type=3, interpol_var=2), [0, 63, 64])
    np.testing.assert_array_equal(u2[:, :, 5:], before[:, :, 5:])
