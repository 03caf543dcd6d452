"""The mixed form where states are in the step kernels' range and the products
of the Riemann solvers overflow FP32: dense, hot and fast cells together, alone
on the mesh and among ordinary ones, and long time steps.  Equal to the
per-cell kernel (variant 0), which knows no range."""
import numpy as np
import pytest

import rhydro
from helpers import assert_same, clone

pytestmark = pytest.mark.gpu

LEVEL = 4


def _mesh(kind):
    m = rhydro.uniform_mesh(LEVEL)
    rng = np.random.default_rng(5)
    cells = m.cells_of_level(LEVEL)
    n = cells.size
    u = m.state("uold")
    if kind == "uniform":  # supersonic, sound speed 5e5
        d, v, t = np.full(n, 2.0 ** 36), np.full((3, n), 0.0), np.full(n, 5e5 ** 2 / (1.4 * 0.4))
        v[0] = 9e5
    else:
        d = 2.0 ** rng.uniform(20, 48, n)
        v = rng.choice([-1.0, 1.0], (3, n)) * 2.0 ** rng.uniform(0, 23, (3, n))
        t = 2.0 ** rng.uniform(10, 48, n)
        if kind == "mixed":
            o = rng.random(n) < 0.5
            d[o], t[o] = rng.uniform(0.5, 2.0, o.sum()), rng.uniform(1.0, 3.0, o.sum())
            v[:, o] = rng.uniform(-1.0, 1.0, (3, o.sum()))
    u[0, cells] = d
    u[1:4, cells] = d * v
    u[4, cells] = d * (t + 0.5 * (v ** 2).sum(0))
    m.unew[:] = m.uold
    return m


@pytest.mark.parametrize("kind", ["uniform", "dense", "mixed"])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc", "acoustic"])
@pytest.mark.parametrize("dt", [1e-12, 1e-3, 1e3])
def test_products_beyond_fp32(riemann, kind, dt):
    print(f"case mixed overflow {riemann} {kind} dt {dt}", flush=True)
    m0 = _mesh(kind)
    dx = 1.0 / 2 ** LEVEL
    want = None
    for variant in (0, 2, 6):
        s = rhydro.Solver(gamma=1.4, riemann=riemann, variant=variant, precision=rhydro.RH_PREC_MIXED)
        m = clone(m0)
        s.bind(m)
        s.set_unew(LEVEL)
        s.godunov_fine(LEVEL, dt, dx)
        s.sync_to_host()
        s.close()
        if want is None:
            want = m.unew.copy()
        assert_same(m.unew, want, f"unew variant {variant}")
