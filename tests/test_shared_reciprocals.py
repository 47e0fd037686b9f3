"""Quotients that share a denominator are formed on the device from its
correctly rounded reciprocal (divBy in acts_amd/csrc/kf_common.hpp): the
sixths and thirds of a step length, the components of a direction over its
norm, d(time)/d(q/p) over its momentum denominator.  In exact rational
arithmetic (every operation rounded once) the sequence gives the correctly
rounded quotient of the division it replaces, over the magnitudes those
operands have."""
from fractions import Fraction

import numpy as np
import pytest

from test_recip_division import div_recip, quotient, rn64


@pytest.mark.parametrize("den", [3.0, 6.0])
def test_constant_denominators(den):
    rng = np.random.default_rng(31)
    y = rn64(1 / Fraction(den))
    for e in rng.integers(-400, 80, size=1500):
        a = float(rng.uniform(-2.0, 2.0) * 2.0 ** int(e))
        assert div_recip(a, den, y, rn64) == quotient(a, den, rn64), a


def test_norm_of_a_direction():
    rng = np.random.default_rng(32)
    for _ in range(500):
        v = rng.normal(size=3) * 10.0 ** rng.uniform(-12, 0, size=3)
        v = v / np.linalg.norm(v) * (1 + 1e-3 * rng.normal())
        n = float(np.sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]))
        y = rn64(1 / Fraction(n))
        for c in v:
            assert div_recip(float(c), n, y, rn64) == quotient(float(c), n, rn64), (c, n)


def test_momentum_denominator():
    """h m^2 / (p^2 q/p dt/ds), p from 10 MeV to 10 TeV, h from 1 nm to 10 m."""
    rng = np.random.default_rng(33)
    m = float(np.float32(0.1056583755))
    for _ in range(1500):
        p = 10.0 ** rng.uniform(-2, 4)
        qop = float(rng.choice([-1.0, 1.0]) / p)
        dtds = float(np.sqrt(1 + (m / p) * (m / p)))
        den = p * p * qop * dtds
        y = rn64(1 / Fraction(den))
        a = float(10.0 ** rng.uniform(-6, 4)) * m * m
        assert div_recip(a, den, y, rn64) == quotient(a, den, rn64), (a, den)
