"""Runs of one level whose Courant minimum is handed from step to step through
slots: run lengths around the rotation of the three sets, levels of fewer octs
than a launch has slots and of more, runs one after another, and the time step
of a state that the general path updates.  Equal to the oracle value for value."""
import numpy as np
import pytest

import oracle
import rhydro
from helpers import assert_same, clone, oracle_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("variant", [2, 6])
@pytest.mark.parametrize("level,nx", [(2, 1), (2, 3), (4, 1), (4, 3)])
def test_run_lengths(level, nx, variant):
    print(f"case slots level {level} nx {nx} variant {variant}", flush=True)
    m0 = rhydro.uniform_mesh(level, nx=nx, ny=nx, nz=nx)
    rhydro.init_lognormal(m0, level, 3, 1.4, 0.4, 0.4)
    dx = 1.0 / (nx * 2 ** level)
    s = rhydro.Solver(gamma=1.4, slope_type=1, riemann="hllc", variant=variant)
    m, mo = clone(m0), clone(m0)
    s.bind(m)
    p = oracle_params(s)
    om = oracle.OracleMesh(mo)
    for n in (1, 2, 3, 4, 5, 7, 1):
        dt = s.run_uniform(level, dx, 0.8, n)
        assert_same(dt, om.run_uniform(p, level, dx, 0.8, n), f"dt of {n} steps")
    s.sync_to_host()
    s.close()
    assert_same(m.uold, mo.uold, "uold")
    assert_same(m.unew, mo.unew, "unew")


@pytest.mark.parametrize("variant", [2, 6])
def test_general_path_takes_the_same_step(variant):
    """A quarter of the cells lies outside the range of the fast form."""
    print(f"case slots general path variant {variant}", flush=True)
    level = 4
    m0 = rhydro.uniform_mesh(level)
    rhydro.init_lognormal(m0, level, 5, 1.4, 0.3, 0.3)
    cells = m0.cells_of_level(level, leaf_only=True)
    c = np.random.default_rng(1).choice(cells, cells.size // 4, replace=False)
    u = m0.state("uold")
    u[1:4, c] = 1e-310
    u[4, c] = 0.3 * u[0, c]
    m0.unew[:] = m0.uold
    dx = 1.0 / 2 ** level
    s = rhydro.Solver(gamma=1.4, slope_type=1, riemann="hllc", variant=variant)
    m, mo = clone(m0), clone(m0)
    s.bind(m)
    p = oracle_params(s)
    dt = s.run_uniform(level, dx, 0.8, 5)
    s.sync_to_host()
    s.close()
    assert_same(dt, oracle.OracleMesh(mo).run_uniform(p, level, dx, 0.8, 5), "dt")
    assert_same(m.uold, mo.uold, "uold")
