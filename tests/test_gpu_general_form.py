"""Waves of the step kernels that leave the ordinary form: a few cells out of
range among ordinary ones, so that of a wave all, two, one or none of the
dimensions meet them, for every slope and interpolation type, whole and partial
last waves.  The FP64 form must equal the oracle value for value, the mixed form
the per-cell kernel (variant 0)."""
import numpy as np
import pytest

import oracle
import rhydro
from amr_meshes import refined_mesh
from helpers import assert_same, clone, oracle_params

pytestmark = pytest.mark.gpu


def _sprinkle(m, level, seed):
    """Tiny and denormal velocities, cold, thin, dense and NaN cells, one in 150."""
    rng = np.random.default_rng(seed)
    cells = m.cells_of_level(level, leaf_only=True)
    c = rng.choice(cells, max(4, cells.size // 150), replace=False)
    u = m.state("uold")
    for k, i in enumerate(c):
        kind = k % 6
        if kind == 0:
            u[1:4, i] = rng.choice([2.0 ** -500, 2.0 ** -900, 1e-310], 3)
        elif kind == 1:
            u[1:4, i], u[4, i] = 0.0, u[0, i] * 1e-11
        elif kind == 2:
            u[:, i] *= 1e-11
        elif kind == 3:
            u[0, i] *= 2.0 ** 52
        elif kind == 4:
            u[4, i] = np.nan
        else:
            u[1, i] = 2.0 ** 30 * u[0, i]
    m.unew[:] = m.uold


def _call(m0, level, dx, f=None, **kw):
    m = clone(m0)
    s = rhydro.Solver(gamma=1.4, **kw)
    s.bind(m, f=f)
    s.set_unew(level)
    s.godunov_fine(level, 2e-3, dx)
    s.sync_to_host()
    p = oracle_params(s)
    s.close()
    return m.unew, p


@pytest.mark.parametrize("slope_type,interpol_type", [(0, 0), (1, 1), (1, 2), (2, 1), (3, 3), (6, 2), (7, 1), (8, 3)])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc", "acoustic"])
def test_few_cells(riemann, slope_type, interpol_type):
    kw = dict(riemann=riemann, slope_type=slope_type, interpol_type=interpol_type)
    for nx, level in ((1, 5), (5, 3)):  # 512 octs; 1,000 octs and a cell width that is no power of two
        m0 = rhydro.uniform_mesh(level, nx=nx, ny=nx, nz=nx)
        rhydro.init_lognormal(m0, level, 61, 1.4, 0.3, 0.3)
        _sprinkle(m0, level, 62)
        dx = 1.0 / (nx * 2 ** level)
        want = None
        mixed = _call(m0, level, dx, variant=0, precision=rhydro.RH_PREC_MIXED, **kw)[0]
        for variant in (2, 6):
            print(f"case general {riemann} {slope_type} {interpol_type} nx={nx} v{variant}", flush=True)
            got, p = _call(m0, level, dx, variant=variant, **kw)
            if want is None:
                want = clone(m0)
                om = oracle.OracleMesh(want)
                om.set_unew(level)
                om.godunov_fine(p, level, 2e-3, dx)
            assert_same(got, want.unew, f"fp64 nx {nx} variant {variant}")
            got = _call(m0, level, dx, variant=variant, precision=rhydro.RH_PREC_MIXED, **kw)[0]
            assert_same(got, mixed, f"mixed nx {nx} variant {variant}")


@pytest.mark.parametrize("level", [4, 5, 6])
@pytest.mark.parametrize("riemann", ["llf", "hllc"])
def test_few_cells_at_refined_neighbours(riemann, level):
    m0 = refined_mesh(4, ((0.4, 0.5, 0.6, 0.3), (0.45, 0.5, 0.55, 0.17)), seed=13)
    _sprinkle(m0, level, 63)
    for slope_type, interpol_type in ((1, 1), (2, 3)):
        kw = dict(riemann=riemann, slope_type=slope_type, interpol_type=interpol_type)
        mixed = _call(m0, level, 1.0 / 2 ** level, variant=0, precision=rhydro.RH_PREC_MIXED, **kw)[0]
        for variant in (2, 6):
            print(f"case general amr {riemann} level {level} v{variant}", flush=True)
            got, p = _call(m0, level, 1.0 / 2 ** level, variant=variant, **kw)
            mo = clone(m0)
            om = oracle.OracleMesh(mo)
            om.set_unew(level)
            om.godunov_fine(p, level, 2e-3, 1.0 / 2 ** level)
            assert_same(got, mo.unew, f"fp64 level {level} variant {variant}")
            got = _call(m0, level, 1.0 / 2 ** level, variant=variant, precision=rhydro.RH_PREC_MIXED, **kw)[0]
            assert_same(got, mixed, f"mixed level {level} variant {variant}")
