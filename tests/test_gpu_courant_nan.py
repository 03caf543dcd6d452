"""The Courant minimum that a multi-step run takes along with its update, in
waves where some lanes' cells are NaN: those are skipped, wherever they sit in
the wave, and the fastest of the others counts, as in the Courant step by
itself and in the oracle."""
import numpy as np
import pytest

import oracle
import rhydro
from helpers import assert_same, clone, oracle_params

pytestmark = pytest.mark.gpu

LEVEL = 4  # 8^3 cells: 64 octs, eight waves, each a block of 4^3 cells


# (lanes of the wave that hold a NaN, lane of the fastest cell)
@pytest.mark.parametrize("nan,fast", [((0,), 63), ((0, 16), 59), ((1, 32), 62), ((48,), 7)])
@pytest.mark.parametrize("slope_type,gravity", [(1, False), (1, True), (4, False)])
@pytest.mark.parametrize("variant", [1, 2, 3, 4, 5, 6])
def test_nan_lanes(variant, slope_type, gravity, nan, fast):
    print(f"case courant nan {nan} fast {fast} slope {slope_type} gravity {gravity} variant {variant}", flush=True)
    m0 = rhydro.uniform_mesh(LEVEL)
    rhydro.init_lognormal(m0, LEVEL, 9, 1.4, 0.1, 0.1)
    cells = m0.cells_of_level(LEVEL)
    u = m0.state("uold")
    wave = cells[64 * 3: 64 * 4]
    u[4, wave[fast]] *= 1e4
    u[4, wave[list(nan)]] = np.nan
    m0.unew[:] = m0.uold
    f = np.random.default_rng(2).normal(0.0, 0.1, 3 * m0.ncell) if gravity else None
    dx = 1.0 / 2 ** LEVEL
    for precision in (rhydro.RH_PREC_FP64, rhydro.RH_PREC_MIXED):
        s = rhydro.Solver(gamma=1.4, slope_type=slope_type, riemann="hllc", variant=variant, precision=precision)
        m = clone(m0)
        s.bind(m, f=f)
        dts = s.run_uniform(LEVEL, dx, 0.8, 2)
        m1 = clone(m0)
        s.bind(m1, f=f)
        s.run_uniform(LEVEL, dx, 0.8, 1)
        assert s.courant(LEVEL, dx, 1.4, 0.8) == dts[1]
        if precision == rhydro.RH_PREC_FP64:
            mo = clone(m0)
            want = oracle.OracleMesh(mo, f=f).run_uniform(oracle_params(s), LEVEL, dx, 0.8, 2)
            assert_same(dts, want, "dt")
        s.close()
