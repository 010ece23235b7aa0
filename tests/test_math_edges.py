"""The edges of ctsm_math.h's straight-line log, exp and pow: the arguments that
are settled by clamping and selecting (zeros, infinities, NaN, overflow,
underflow, subnormal results) against the host's C library, and the error of
exp and pow against 40-digit values.

The bounds: a result's last rounding is half an ulp; rounding the reduced
argument (half of 2^-54 for |r| <= 0.35, results from 0.7 up) adds a quarter and
the polynomial's own roundings a few hundredths: 0.8 for exp.  pow rounds the
reduced argument once more when it folds the low word in: 1.05.
"""
import math
from decimal import Decimal

import numpy as np
import pytest

from test_math import _rng, _ulp_err, _vec

INF, NAN = math.inf, math.nan


def _same(got, want):
    return (got == want) | (np.isnan(got) & np.isnan(want))


def test_log_exp_special_values():
    x = np.array([0.0, -0.0, INF, -INF, NAN, -1.0, -5e-324, 1.0])
    with np.errstate(all="ignore"):
        assert np.all(_same(_vec("log", x), np.log(x)))
        assert np.all(_same(_vec("exp", np.array([INF, -INF, NAN, 0.0, -0.0, 1e300, -1e300, 710.0, 712.5, -746.0])),
                            np.array([INF, 0.0, NAN, 1.0, 1.0, INF, 0.0, INF, INF, 0.0])))


@pytest.mark.parametrize("lo,hi", [(709.7, 709.8), (-745.4, -744.0), (-709.0, -708.0)])
def test_exp_at_overflow_and_underflow(lo, hi):
    x = np.linspace(lo, hi, 401)
    want = np.array([Decimal(v).exp() for v in x])
    got = _vec("exp", x)
    for g, w in zip(got, want):
        if w > Decimal(1.7976931348623157e308):
            assert g == INF
        elif w < Decimal(2.2250738585072014e-308):
            assert abs(Decimal(g) - w) <= Decimal(5e-324)
        else:
            assert _ulp_err(g, w) < 0.8


def test_pow_special_values():
    x = np.array([0.0, -0.0, INF, -INF, NAN, -1.0, -2.0, 1.0, 2.0, 0.5, 1e-310])
    y = np.array([0.0, -0.0, 1.0, 2.0, 3.0, -1.0, -3.0, 0.5, -0.5, INF, -INF, NAN, 1e300, -1e300, 1e-300])
    X, Y = (a.ravel() for a in np.meshgrid(x, y))
    with np.errstate(all="ignore"):
        want = np.power(X, Y)
    ulp = np.array([math.ulp(w) if math.isfinite(w) else 0.0 for w in want])
    got = _vec("pow", X, Y)
    with np.errstate(invalid="ignore"):
        assert np.all(_same(got, want) | (np.abs(got - want) <= ulp))


@pytest.mark.parametrize("lo,hi,ylo,yhi", [(0.01, 1.0, -13.0, -2.5), (0.01, 1.0, 8.0, 30.0), (1e-3, 3e3, -3.0, 3.0)])
def test_pow_error(lo, hi, ylo, yhi):
    r = _rng(31)
    x, y = np.exp(r.uniform(math.log(lo), math.log(hi), 1500)), r.uniform(ylo, yhi, 1500)
    got = _vec("pow", x, y)
    assert max(_ulp_err(g, (Decimal(b) * Decimal(a).ln()).exp()) for a, b, g in zip(x, y, got)) < 1.05


def test_exp_error():
    x = _rng(32).uniform(-50.0, 50.0, 3000)
    assert max(_ulp_err(g, Decimal(v).exp()) for v, g in zip(x, _vec("exp", x))) < 0.8
