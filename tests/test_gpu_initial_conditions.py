"""Initial conditions of adaptive runs computed on the device: regions of both
kinds that overlap (the last one counts), that lie off the cells' centres or
hold none, boxes of several coarse cells, and the shear layer.  The tree and
the state must equal the oracle's."""
import numpy as np
import pytest

import oracle
import rhydro
from helpers import assert_same

pytestmark = pytest.mark.gpu


def _region(kind, centre, lengths, d, v, p):
    r = dict(type=kind, d=d, p=p)
    r.update(zip(("x_center", "y_center", "z_center"), centre))
    r.update(zip(("length_x", "length_y", "length_z"), lengths))
    r.update(zip("uvw", v))
    return r


BASE = _region("square", (0.5, 0.5, 0.5), (10.0, 10.0, 10.0), 1.0, (0.0, 0.1, 0.0), 0.1)
CASES = {
    # Each later region covers a part of the one before.
    "overlap": [BASE, _region("sphere", (0.45, 0.5, 0.55), (0.3, 0.0, 0.0), 2.0, (0.3, 0.0, -0.2), 1.0),
                _region("square", (0.5, 0.5, 0.5), (0.25, 0.5, 0.125), 0.5, (0.0, 0.0, 0.7), 2.0),
                _region("sphere", (0.5, 0.53125, 0.5), (0.0625, 0.0, 0.0), 4.0, (-1.0, 0.0, 0.0), 5.0)],
    # A region that holds no cell centre, then one whose faces run through
    # cell centres (strictly inside counts).
    "edges": [BASE, _region("sphere", (0.5, 0.5, 0.5), (1e-6, 0.0, 0.0), 9.0, (0.0, 0.0, 0.0), 9.0),
              _region("square", (0.5, 0.5, 0.5), (0.5625, 0.5625, 0.5625), 3.0, (0.0, 0.2, 0.0), 3.0)],
    # No region covers the corners: they keep their state.
    "uncovered": [_region("sphere", (0.5, 0.5, 0.5), (0.8, 0.0, 0.0), 1.0, (0.0, 0.0, 0.1), 1.0),
                  _region("sphere", (0.5, 0.5, 0.5), (0.2, 0.0, 0.0), 3.0, (0.0, 0.0, 0.0), 2.0)],
}


def _compare(kw):
    g = rhydro.AmrRun(**kw)
    o = oracle.OracleAmr(**{k: (rhydro.resolve_riemann(v) if k == "riemann" else v) for k, v in kw.items()})
    a, b = g.state(), o.state()
    for k in ("numbl", "headl", "next", "father", "son", "nbor"):
        np.testing.assert_array_equal(a[k], b[k], err_msg=k)
    for k in ("xg", "uold", "unew"):
        assert_same(a[k], b[k], k)
    g.close()
    o.close()
    return a


@pytest.mark.parametrize("nx", [1, 3])
@pytest.mark.parametrize("name", sorted(CASES))
def test_regions(name, nx):
    print(f"case initial conditions {name} nx {nx}", flush=True)
    a = _compare(dict(levelmin=3 if nx == 3 else 4, levelmax=6, ngridmax=40000, nx=nx, err_grad_d=0.1,
                      err_grad_p=0.2, riemann="hllc", regions=CASES[name]))
    assert a["numbl"][5] > 0


@pytest.mark.parametrize("nx", [1, 2])
def test_layer(nx):
    print(f"case initial conditions layer nx {nx}", flush=True)
    a = _compare(dict(levelmin=4, levelmax=6, ngridmax=60000, nx=nx, err_grad_d=0.2, ic="kh",
                      kh_amp=0.01, riemann="hllc"))
    assert a["numbl"][6] > 0
