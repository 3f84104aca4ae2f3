"""The quotients and square roots with shared parts that the step kernels form,
against IEEE division and square root on the host: the same bits.  The
reciprocals alone: their formulas end in one rounding of a value that is off by
at most half an ulp (1 / sqrt(b), from the rounding of b y; half the reciprocal
of the rounded root, from its estimate) or far less (1 / b), so 1.01 and 0.51
ulp; measured in 64-bit mantissas.
"""
import numpy as np
import pytest

from hgswe import capi

pytestmark = pytest.mark.gpu

N = 1 << 22


def operands(kind, seed):
    rng = np.random.default_rng(seed)
    sign = rng.choice([-1.0, 1.0], N)
    if kind == "wide":
        return sign * 10.0 ** rng.uniform(-100, 100, N), 10.0 ** rng.uniform(-100, 100, N)
    if kind == "solver":  # discharges over depths, fluxes over areas
        return sign * 10.0 ** rng.uniform(-16, 8, N), 10.0 ** rng.uniform(-3, 6, N)
    if kind == "roots":  # eps under a square root, and up
        return sign * rng.uniform(0.0, 10.0, N), 2.0 ** -52 + 10.0 ** rng.uniform(-17, 6, N)
    near = rng.integers(0, 64, N) - 32  # mantissas within 32 ulp of a power of two, over each other
    a = np.ldexp(1.0 + near * 2.0 ** -52, rng.integers(-40, 40, N))
    b = np.ldexp(1.0 + rng.permutation(near) * 2.0 ** -52, rng.integers(-40, 40, N))
    return sign * a, b


def ulps(x, exact):
    return np.max(np.abs((x.astype(np.longdouble) - exact) / np.spacing(np.abs(x)).astype(np.longdouble)))


@pytest.mark.parametrize("kind", ["wide", "solver", "roots", "near_powers_of_two"])
def test_against_ieee(kind):
    assert np.finfo(np.longdouble).nmant >= 63
    a, b = operands(kind, 5)
    a[:4], b[:4] = [0.0, -0.0, np.inf, np.nan], 3.0
    q, s, o, r, y = capi.rounding_probe(a, b)
    assert np.array_equal(q.view(np.int64)[np.isfinite(q)], (a / b).view(np.int64)[np.isfinite(a)])
    assert q[2] == np.inf and np.isnan(q[3]) and np.signbit(q[1])
    assert np.array_equal(s, np.sqrt(b))
    root = np.sqrt(b.astype(np.longdouble))
    assert ulps(o, 0.5 / s.astype(np.longdouble)) <= 1.01 and ulps(r, 1.0 / root) <= 1.01
    assert ulps(y, 1.0 / b.astype(np.longdouble)) <= 0.51
