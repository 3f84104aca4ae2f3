"""The FP64 tanh of the device networks, its operations emulated on the host:
fused multiply-adds through an extended type (64-bit significand: the product
and sum are rounded once more, by at most 2^-64), the reciprocal correctly
rounded (the device's is within an ulp, and only scales residuals and a
first quotient that is corrected).  Bound: 0.75 ulp, from the last rounding
(half an ulp) and a carried-error tail of at most a quarter."""
import math

import numpy as np
import pytest

L = np.longdouble


def fma(a, b, c):
    return (L(a) * L(b) + L(c)).astype(np.float64)


def tanh64(x):
    y = 2 * np.abs(x)
    y = np.where(y > 80.0, 80.0, y)
    k = np.rint(y * 1.4426950408889634)
    lo = float.fromhex("0x1.a39ef35793c76p-33")
    r0 = fma(-k, float.fromhex("0x1.62e42feep-1"), y)
    r = fma(-k, lo, r0)
    rl = fma(-k, lo, r0 - r)
    p = np.full_like(r, 1 / math.factorial(14))
    for n in range(13, 1, -1):
        p = fma(p, r, 1 / math.factorial(n))
    c = p * r * r
    ph = r + c
    pl = ((r - ph) + c) + fma(rl, ph, rl)
    s = np.ldexp(1.0, k.astype(int))
    a, b = s * ph, s - 1
    e = b + a
    el = fma(s, pl, (b - e) + a)
    d = e + 2
    t = d - e
    dl = (e - (d - t)) + (2 - t) + el
    yd = 1 / d
    q = e * yd
    return np.copysign(fma(fma(-q, dl, fma(-d, q, e)) + el, yd, q), x)


@pytest.mark.parametrize("lo,hi", [(1e-300, 1e-200), (1e-12, 1e-6), (1e-6, 1e-2), (1e-2, 0.2), (0.2, 0.5), (0.5, 2),
                                   (2, 20), (20, 700)])
def test_error_bound(lo, hi):
    if np.finfo(L).nmant < 63:
        pytest.skip("no extended type here")
    x = np.exp(np.random.default_rng(1).uniform(math.log(lo), math.log(hi), 200_000))
    x *= np.where(np.arange(x.size) % 2, 1, -1)
    ref = np.tanh(L(x))
    ulp = np.spacing(np.abs(ref.astype(np.float64)))
    assert np.max(np.abs(tanh64(x).astype(L) - ref) / ulp) <= 0.75


def test_special_values():
    x = np.array([0.0, -0.0, np.inf, -np.inf, 5e-324])
    y = tanh64(x)
    assert np.array_equal(y, np.tanh(x)) and np.array_equal(np.signbit(y), np.signbit(x))
