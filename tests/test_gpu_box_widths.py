"""Ensembles whose waves of eight octs hold cells of boxes with different cell
widths: every box's time steps and states equal those of its own run.  The
fastest cells lie in a box's first and last octs, where a wave begins or ends
inside the neighbouring box, so another box's width shows in the time step."""
import numpy as np
import pytest

import rhydro
from helpers import assert_same, clone

pytestmark = pytest.mark.gpu


def _box(nx, seed):
    m = rhydro.uniform_mesh(2, nx=nx, ny=nx, nz=nx)
    rhydro.init_lognormal(m, 2, seed, 1.4, 0.2, 0.2)
    cells = m.cells_of_level(2)
    u = m.state("uold")
    u[4, np.r_[cells[:8], cells[-8:]]] *= 20.0
    m.unew[:] = m.uold
    return m, 1.0 / (nx * 4)


# Octs per box: nx^3 -- 343, 27, 125, 729, 1.
@pytest.mark.parametrize("sides", [(7, 3), (3, 5), (9, 7, 3), (3, 1, 1, 5, 9)])
@pytest.mark.parametrize("variant", [-1, 2, 6])
@pytest.mark.parametrize("precision", [rhydro.RH_PREC_FP64, rhydro.RH_PREC_MIXED])
def test_boxes_of_different_widths(sides, variant, precision):
    print(f"case box widths {sides} variant {variant} precision {precision}", flush=True)
    boxes = [_box(nx, 60 + k) for k, nx in enumerate(sides)]
    kw = dict(gamma=1.4, riemann="hllc", variant=variant, precision=precision)
    alone = []
    for m0, dx in boxes:
        m = clone(m0)
        s = rhydro.Solver(**kw)
        s.bind(m)
        dts = s.run_uniform(2, dx, 0.8, 4)
        s.sync_to_host()
        s.close()
        alone.append((dts, m.uold.copy()))
    ms = [clone(m) for m, _ in boxes]
    s = rhydro.Solver(**kw)
    s.bind_ensemble(ms)
    dts = s.run_ensemble([2] * len(ms), [dx for _, dx in boxes], 0.8, 4)
    s.sync_to_host()
    s.close()
    for b, (dt, u) in enumerate(alone):
        assert_same(dts[:, b], dt, f"dt of box {b}")
        assert_same(ms[b].uold, u, f"uold of box {b}")
