"""State copies between the caller's arrays and the device at the edges of the
staged form: arrays just below and above the length from which it is used,
lengths that end inside a piece, many short runs (ensembles), and several
contexts copying at once.  Every value must come back as it went."""
import threading

import numpy as np
import pytest

import rhydro
from rhydro import RH_UNEW, RH_UOLD

pytestmark = pytest.mark.gpu


def _mesh(ngridmax, seed):
    m = rhydro.uniform_mesh(2, ngridmax=ngridmax)
    rng = np.random.default_rng(seed)
    m.uold[:] = rng.random(m.uold.shape)
    m.unew[:] = rng.random(m.unew.shape)
    return m


def _round_trip(s, meshes):
    want = [(m.uold.copy(), m.unew.copy()) for m in meshes]
    s.sync_to_device()
    for m in meshes:
        m.uold[:] = -1.0
        m.unew[:] = -2.0
    s.sync_to_host(RH_UOLD)
    assert all((m.unew == -2.0).all() for m in meshes)
    s.sync_to_host(RH_UNEW)
    for m, (uold, unew) in zip(meshes, want):
        np.testing.assert_array_equal(m.uold, uold)
        np.testing.assert_array_equal(m.unew, unew)


# 40 bytes per cell, 8 * ngridmax + 1 cells: 2^25/10 octs are 10 MB.
@pytest.mark.parametrize("ngridmax", [9, 32767, 32768, 52428, 150001])
def test_round_trip(ngridmax):
    print(f"case staging ngridmax {ngridmax}", flush=True)
    m = _mesh(ngridmax, ngridmax)
    s = rhydro.Solver()
    s.bind(m)
    _round_trip(s, [m])
    s.close()


@pytest.mark.parametrize("sizes", [[9], [9, 10, 11, 12, 13], [3001, 9, 8000, 257, 9, 30011], [9] * 40 + [40000, 50021]])
def test_ensemble_round_trip(sizes):
    print(f"case staging ensemble {len(sizes)} boxes", flush=True)
    ms = [_mesh(n, 100 + k) for k, n in enumerate(sizes)]
    s = rhydro.Solver()
    s.bind_ensemble(ms)
    _round_trip(s, ms)
    s.close()


def test_contexts_copy_at_once():
    print("case staging threads", flush=True)
    errs = []

    def work(k):
        try:
            for r in range(3):
                m = _mesh(33000 + 7001 * k, 10 * k + r)
                s = rhydro.Solver()
                s.bind(m)
                _round_trip(s, [m])
                s.close()
        except BaseException as e:
            errs.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errs, errs
