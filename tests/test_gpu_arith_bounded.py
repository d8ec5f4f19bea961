"""The device quotient and square root sequences of the bounded-state fluxes
(pip_riemann.h quob, sqrtb, sqrt_rcp) against IEEE division and square root on
the host, over the operands that bounded states can give them: divisors and
radicands from 2^-404 to 2^404 (four factors in (2^-100, 2^100) and a few small
ones), numerators from 0 over 2^-500 to 2^404.

The quotient n / sqrt(x) takes the reciprocal that the root's own iteration
gives.  Its bits decide only whether an exact residual is rounded back the right
way, so the operands close to midpoints of two doubles matter most."""
import ctypes

import numpy as np
import pytest

from pip_amd import _lib

pytestmark = pytest.mark.gpu


def _p(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


def _check(n, d):
    n, d = (np.ascontiguousarray(x, dtype=np.float64) for x in (n, d))
    q, r, s = (np.empty_like(n) for _ in range(3))
    _lib.check(_lib.lib().pip_check_arith_bounded(_p(n), _p(d), _p(q), _p(r), _p(s), n.size))
    root = np.sqrt(d)
    for name, got, want in (("n / d", q, n / d), ("sqrt(d)", r, root), ("n / sqrt(d)", s, n / root)):
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, f"{bad.size} of {name} differ, first n={n[bad[0]]!r} d={d[bad[0]]!r}"


def _positive(rng, size, emin, emax):
    return np.ldexp(rng.uniform(1.0, 2.0, size), rng.integers(emin, emax, size))


SIZE = 1 << 22


@pytest.mark.parametrize("seed", range(3))
def test_random_operands(seed):
    rng = np.random.default_rng(seed)
    n = rng.choice([-1.0, 1.0], SIZE) * _positive(rng, SIZE, -500, 404)
    n[::1000] = 0.0
    _check(n, _positive(rng, SIZE, -404, 404))


@pytest.mark.parametrize("seed", range(3))
def test_quotients_close_to_rounding_ties(seed):
    """Numerators a last place or less from (q + half a last place) times the
    divisor, for the divisor d and for its root."""
    rng = np.random.default_rng(100 + seed)
    d = _positive(rng, SIZE, -60, 60)
    q = _positive(rng, SIZE, -60, 60)
    for root in (False, True):
        g = np.sqrt(d) if root else d
        with np.errstate(all="ignore"):
            n = (q.astype(np.longdouble) + np.spacing(q).astype(np.longdouble) / 2) * g.astype(np.longdouble)
        n = n.astype(np.float64)
        for m in (n, np.nextafter(n, np.inf), np.nextafter(n, 0.0), g * q, np.nextafter(g, np.inf)):
            _check(m, d)


def test_roots_of_squares_and_their_neighbours():
    rng = np.random.default_rng(9)
    g = _positive(rng, SIZE, -200, 200)
    x = g * g
    for d in (x, np.nextafter(x, np.inf), np.nextafter(x, 0.0), np.ldexp(1.0, rng.integers(-404, 404, SIZE))):
        _check(g, d)
