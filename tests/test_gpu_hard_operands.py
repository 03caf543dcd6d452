"""Operands on which the step kernels' reciprocals, quotients and square roots
round hardest: densities whose significand is all ones, pressures over densities
and squared sound speeds whose quotient or root lies next to a midpoint of two
doubles.  The FP64 form must equal the oracle value for value."""
import random

import numpy as np
import pytest

import oracle
import rhydro
from helpers import assert_same, clone, oracle_params

pytestmark = pytest.mark.gpu

LEVEL = 5  # 16^3 cells


def _roots():
    """Doubles in [1, 4) next to the square of a midpoint: M*M = X + r with M of 54
    bits, X a multiple of 2^54 or 2^55, r small (r = 1 mod 8 has roots)."""
    out = []
    for r in range(-799, 800):
        if r % 8 != 1:
            continue
        for e in (54, 55):
            m = 1
            for j in range(3, e):
                if (m * m - r) % (1 << (j + 1)):
                    m += 1 << (j - 1)
            for s in {m, -m % (1 << e), (m + (1 << (e - 1))) % (1 << e), (-m + (1 << (e - 1))) % (1 << e)}:
                for mm in (s, s + (1 << e)):
                    if (1 << 53) <= mm < (1 << 54):
                        x = (mm * mm - r) >> e
                        if (1 << 52) <= x < (1 << 53):
                            out.append(float(x) * 2.0 ** (e - 106))
    return np.array(out + [np.nextafter(4.0, 0.0), np.nextafter(1.0, 2.0), np.nextafter(2.0, 0.0)])


def _quotients(n, seed):
    """(2p, d): d odd, 2^54 * 2p = (odd 54-bit number) * d + r with r small, kept
    where the cell's energy can be chosen so that its pressure is exactly p."""
    rng = random.Random(seed)
    out = []
    while len(out) < n:
        d = rng.getrandbits(52) | (1 << 52) | 1
        if len(out) < n // 4:
            d = (1 << 53) - 1 - 2 * rng.randrange(1 << 12)
        inv = pow(d, -1, 1 << 54)
        for r in (1, -1, 3, -3):
            q = r * inv % (1 << 54)
            a = (q * d - r) >> 54
            if q < 1 << 53 or not (1 << 52) <= a < (1 << 53):
                continue
            dd, p = float(d) * 2.0 ** -52, float(a) * 2.0 ** -53
            o = 1.0 / dd
            e = p
            for _ in range(-20, 20):
                e = np.nextafter(e, 0.0)
            for _ in range(40):
                if dd * (e * o) == p:
                    out.append((dd, float(e)))
                    break
                e = np.nextafter(e, 10.0)
    return np.array(out[:n])


def _states(kind):
    rng = np.random.default_rng(8)
    n = 16 ** 3
    d, v, e = np.ones(n), np.zeros((3, n)), np.ones(n)
    if kind == "roots":  # gamma = 2: c^2 = 2p/d = x
        e = 0.5 * rng.choice(_roots(), n)
    elif kind == "quotients":
        q = _quotients(1500, 9)
        i = rng.integers(0, len(q), n)
        d, e = q[i, 0], q[i, 1]
    else:  # densities just below powers of two, and their neighbours
        d = 2.0 ** rng.integers(-20, 15, n)
        for _ in range(3):
            d = np.where(rng.random(n) < 0.7, np.nextafter(d, 0.0), d)
        v = rng.uniform(-1.0, 1.0, (3, n))
        e = d * (rng.uniform(1.0, 2.0, n) + 0.5 * (v ** 2).sum(0))
    return d, v, e


@pytest.mark.parametrize("kind", ["roots", "quotients", "ones"])
@pytest.mark.parametrize("riemann", ["llf", "hll", "hllc", "acoustic"])
def test_hard_operands(riemann, kind):
    m0 = rhydro.uniform_mesh(LEVEL)
    cells = m0.cells_of_level(LEVEL)
    d, v, e = _states(kind)
    u = m0.state("uold")
    u[0, cells], u[1:4, cells], u[4, cells] = d, d * v, e
    m0.unew[:] = m0.uold
    dx = 1.0 / 2 ** LEVEL
    # Without slopes the face states are the cells' own.
    for slope_type, interpol_type in ((0, 0), (1, 1)):
        for variant in (2, 6):
            print(f"case hard operands {kind} {riemann} slopes {slope_type} v{variant}", flush=True)
            s = rhydro.Solver(gamma=2.0, riemann=riemann, slope_type=slope_type, interpol_type=interpol_type,
                              variant=variant)
            m, mo = clone(m0), clone(m0)
            s.bind(m)
            dts = s.run_uniform(LEVEL, dx, 0.8, 2)
            s.sync_to_host()
            want = oracle.OracleMesh(mo).run_uniform(oracle_params(s), LEVEL, dx, 0.8, 2)
            s.close()
            assert_same(dts, want, "dt")
            assert_same(m.uold, mo.uold, f"{kind} slopes {slope_type} variant {variant}")
