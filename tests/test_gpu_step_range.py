"""The step kernels at the edges of their range: states, time steps and
cell widths on both sides of the bounds within which they skip the scaling of
divisions and the NaN cases of minima, and waves that mix both.  The FP64 form
must equal the oracle value for value, the mixed form the per-cell kernel
(variant 0), which knows no range."""
import numpy as np
import pytest

import oracle
import rhydro
from amr_meshes import refined_mesh
from helpers import assert_same, clone, oracle_params

pytestmark = pytest.mark.gpu

RIEMANNS = ["llf", "hll", "hllc", "acoustic"]


def _spoil(m, level, kind, seed):
    """Puts states of the kind into an eighth of the level's octs."""
    rng = np.random.default_rng(seed)
    cells = m.cells_of_level(level, leaf_only=True)
    c = rng.choice(cells, max(1, cells.size // 40), replace=False)
    u = m.state("uold")
    sign = rng.choice([-1.0, 1.0], (3, c.size))
    if kind == "slow":  # velocities around the smallest in range, and denormal ones
        u[1:4, c] = sign * rng.choice([0.0, 2.0 ** -199, 2.0 ** -200, 2.0 ** -201, 2.0 ** -60, 1e-310], (3, c.size))
    elif kind == "fast":  # kinetic and total energies around the largest
        e = rng.choice([2.0 ** 49, 2.0 ** 50, 2.0 ** 51, 2.0 ** 20], c.size)
        u[0, c] = 1.0
        u[1:4, c] = sign * np.sqrt(e / 4)
        u[4, c] = e
    elif kind == "dense":
        u[0, c] = rng.choice([2.0 ** 49, 2.0 ** 50, 2.0 ** 51, 2.0 ** 30], c.size)
    elif kind == "thin":  # density and pressure around their floors
        u[0, c] = rng.choice([1e-10, 1e-9, 2.0 ** -45, 2.0 ** -44], c.size)
        u[1:4, c] = sign * u[0, c] * 0.1
        u[4, c] = u[0, c] * rng.choice([1e-12, 1e-3, 1.0], c.size)
    m.unew[:] = m.uold


SPHERES = ((0.4, 0.5, 0.6, 0.3), (0.45, 0.5, 0.55, 0.17))
KINDS = ["slow", "fast", "dense", "thin"]
# Time steps: ordinary, none, below and above the bounds.
DTS = [1e-3, 0.0, 2.0 ** -101, 2.0 ** -51, 2.0 ** 17]


def _one_call(m0, level, dx, dt, f=None, **kw):
    s = rhydro.Solver(**kw)
    m = clone(m0)
    s.bind(m)
    s.set_unew(level)
    s.godunov_fine(level, dt, dx)
    s.sync_to_host()
    p = oracle_params(s)
    s.close()
    return m, p


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("riemann", RIEMANNS)
def test_range_edges_fp64(riemann, kind):
    for nx, level in ((1, 4), (3, 3)):
        m0 = rhydro.uniform_mesh(level, nx=nx, ny=nx, nz=nx)
        rhydro.init_lognormal(m0, level, 31, 1.4)
        _spoil(m0, level, kind, 17)
        dx = 1.0 / (nx * 2 ** level)
        for slope in (1, 2):
            for dt in DTS:
                mo = clone(m0)
                om = oracle.OracleMesh(mo)
                om.set_unew(level)
                om.godunov_fine(oracle.params(1.4, slope, rhydro.resolve_riemann(riemann)), level, dt, dx)
                for variant in (2, 6):
                    print(f"case range fp64 {riemann} {kind} nx={nx} slope={slope} dt={dt} v{variant}", flush=True)
                    mg, _ = _one_call(m0, level, dx, dt, gamma=1.4, slope_type=slope, riemann=riemann, variant=variant)
                    assert_same(mg.unew, mo.unew, f"unew dt={dt} variant {variant}")


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("riemann", RIEMANNS)
def test_range_edges_mixed(riemann, kind):
    for nx, level in ((1, 4), (3, 3)):
        m0 = rhydro.uniform_mesh(level, nx=nx, ny=nx, nz=nx)
        rhydro.init_lognormal(m0, level, 32, 1.4)
        _spoil(m0, level, kind, 18)
        dx = 1.0 / (nx * 2 ** level)
        for dt in (1e-3, 0.0, 2.0 ** -51):
            want = None
            for variant in (0, 2, 6):
                print(f"case range mixed {riemann} {kind} nx={nx} dt={dt} v{variant}", flush=True)
                mg, _ = _one_call(m0, level, dx, dt, gamma=1.4, riemann=riemann, variant=variant,
                                  precision=rhydro.RH_PREC_MIXED)
                if want is None:
                    want = mg.unew.copy()
                assert_same(mg.unew, want, f"unew dt={dt} variant {variant}")


@pytest.mark.parametrize("kind", KINDS)
def test_range_edges_at_refined_neighbours(kind):
    """Out-of-range states next to coarser and refined cells: the general form's
    records, refined siblings and coarse reflux."""
    m0 = refined_mesh(4, SPHERES, seed=13)
    for L in (4, 5, 6):
        m = clone(m0)
        _spoil(m, L, kind, 19)
        mo = clone(m)
        om = oracle.OracleMesh(mo)
        om.set_unew(L)
        om.godunov_fine(oracle.params(1.4, 1, 2), L, 1e-3, 1.0 / 2 ** L)
        for variant in (2, 6):
            print(f"case range amr {kind} level {L} v{variant}", flush=True)
            mg, _ = _one_call(m, L, 1.0 / 2 ** L, 1e-3, gamma=1.4, riemann="hllc", variant=variant)
            assert_same(mg.unew, mo.unew, f"unew level {L} variant {variant}")


@pytest.mark.parametrize("gamma", [1.0 + 2.0 ** -11, 1.0 + 2.0 ** -10, 65.0, 66.0])
def test_gamma_bounds(gamma):
    """gamma at the bounds of the step kernels' rule; beyond them the launch
    takes the kernels without a range."""
    m0 = rhydro.uniform_mesh(4)
    rhydro.init_lognormal(m0, 4, 33, gamma)
    mo = clone(m0)
    om = oracle.OracleMesh(mo)
    om.set_unew(4)
    om.godunov_fine(oracle.params(gamma, 1, 2), 4, 1e-4, 1.0 / 16)
    for variant in (2, 6):
        print(f"case range gamma={gamma} v{variant}", flush=True)
        mg, _ = _one_call(m0, 4, 1.0 / 16, 1e-4, gamma=gamma, riemann="hllc", variant=variant)
        assert_same(mg.unew, mo.unew, f"unew gamma={gamma}")


def test_waves_across_boxes():
    """Boxes of 27 octs: waves of eight octs hold two boxes with different time
    steps and cell widths.  Each box equals its own run."""
    boxes = []
    for b in range(3):
        m = rhydro.uniform_mesh(2, nx=3, ny=3, nz=3)
        rhydro.init_lognormal(m, 2, 40 + b, 1.4, 0.3 * (b + 1))
        boxes.append(m)
    levels, dxs = [2] * 3, [1.0 / 12, 1.0 / 12, 1.0 / 12]
    for variant in (2, 6):
        alone = []
        for m0 in boxes:
            m = clone(m0)
            s = rhydro.Solver(gamma=1.4, riemann="hllc", variant=variant)
            s.bind(m)
            dts = s.run_uniform(2, dxs[0], 0.8, 3)
            s.sync_to_host()
            s.close()
            alone.append((dts, m.uold.copy()))
        print(f"case range boxes of 27 octs v{variant}", flush=True)
        ms = [clone(m) for m in boxes]
        s = rhydro.Solver(gamma=1.4, riemann="hllc", variant=variant)
        s.bind_ensemble(ms)
        dts = s.run_ensemble(levels, dxs, 0.8, 3)
        s.sync_to_host()
        s.close()
        for b in range(3):
            assert_same(dts[:, b], alone[b][0], f"dt box {b}")
            assert_same(ms[b].uold, alone[b][1], f"uold box {b}")


def test_courant_of_long_minima_arrays():
    """2^18 octs: the step kernels leave 32,768 block minima, which are folded
    before the last reduction.  The next time step of a run equals the Courant
    step of its state, with the fastest cell, a second one and NaN cells (which
    are skipped) at the ends and in the middle of the list."""
    level = 8
    m = rhydro.uniform_mesh(level)
    rhydro.init_lognormal(m, level, 51, 1.4)
    cells = m.cells_of_level(level)
    dx = 1.0 / 2 ** level
    for where in (0, cells.size // 2 + 5, cells.size - 1):
        mg = clone(m)
        u = mg.state("uold")
        u[4, cells[where]] *= 50.0
        u[0, cells[(where + 9999) % cells.size]] = np.nan
        mg.unew[:] = mg.uold
        print(f"case long courant at {where}", flush=True)
        for variant in (2, 6):
            s = rhydro.Solver(gamma=1.4, riemann="hllc", variant=variant)
            s.bind(mg)
            dts = s.run_uniform(level, dx, 0.8, 3)
            s.bind(mg)
            assert s.courant(level, dx, 1.4, 0.8) == dts[0]
            for k in range(1, 3):
                s.bind(mg)
                s.run_uniform(level, dx, 0.8, k)
                assert s.courant(level, dx, 1.4, 0.8) == dts[k], f"step {k} variant {variant}"
            s.close()


@pytest.mark.parametrize("prec,low", [("mixed", 30), ("mixed", 90), ("mixed", 160), ("fp64", 380), ("fp64", 700)])
@pytest.mark.parametrize("variant", [2, 6])
@pytest.mark.parametrize("slope_type,interpol_type", [(1, 1), (2, 1), (8, 3), (7, 2), (6, 1)])
def test_front_velocities(slope_type, interpol_type, variant, prec, low):
    """Gas nearly at rest, its velocities falling off by orders of magnitude
    from cell to cell down to 2^-low, as ahead of a front: products of two
    differences, and in FP32 differences too, vanish."""
    print(f"case front {prec} low {low} variant {variant} slopes {slope_type} {interpol_type}", flush=True)
    level = 4
    m0 = rhydro.uniform_mesh(level)
    u = m0.state("uold")
    cells = m0.cells_of_level(level, leaf_only=True)
    rng = np.random.default_rng(low)
    x = np.arange(cells.size) // 8 / (cells.size // 8)
    for i in range(1, 4):
        e = low * x * rng.uniform(0.7, 1.0, cells.size)
        u[i, cells] = rng.choice([-1.0, 0.0, 1.0, 1.0, 1.0], cells.size) * rng.uniform(0.5, 1.0, cells.size) * np.exp2(-e)
    u[0, cells] = np.where(rng.random(cells.size) < 0.3, rng.uniform(0.5, 1.0, cells.size), 1.0)
    u[4, cells] = 2.5 + 0.5 * (u[1:4, cells] ** 2).sum(0) / u[0, cells]
    m0.unew[:] = m0.uold
    kw = dict(gamma=1.4, slope_type=slope_type, interpol_type=interpol_type, riemann="hllc")
    for dx, dt in ((1.0 / 2 ** level, 1e-2), (1.0 / (3 * 2 ** level), 5e-3)):
        if prec == "mixed":
            got, _ = _one_call(m0, level, dx, dt, variant=variant, precision=rhydro.RH_PREC_MIXED, **kw)
            want, _ = _one_call(m0, level, dx, dt, variant=0, precision=rhydro.RH_PREC_MIXED, **kw)
        else:
            got, p = _one_call(m0, level, dx, dt, variant=variant, **kw)
            want = clone(m0)
            oracle.OracleMesh(want).godunov_fine(p, level, dt, dx)
        assert_same(got.unew, want.unew, f"dx {dx}")
