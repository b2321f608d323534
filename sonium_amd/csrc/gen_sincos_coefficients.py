"""Coefficients of the device sin/cos polynomials.

Two pairs, both near-minimax: for |r| <= pi/2 (P and Q of degree 7, used after
a reduction by pi and for moderate phase differences) and for |r| <= 0.32 (P of
degree 4, Q of degree 3, for the phase differences inside one panel).

sin r = r + r^3 P(r^2),   cos r = 1 - r^2/2 + r^4 Q(r^2),

with P and Q interpolating (sin r - r)/r^3 and
(cos r - 1 + r^2/2)/r^4 as functions of u = r^2 at the Chebyshev nodes
of [0, r_max^2] (Chebyshev interpolation, near-minimax for these entire
functions), computed in 50-digit arithmetic with mpmath and rounded to double.
After the reduction by pi one sign flip finishes both values.
``python gen_sincos_coefficients.py`` prints the constants and the maximum
error of the polynomials with the rounded coefficients, measured against
mpmath on 2001 points of [0, r_max].
"""

from __future__ import annotations

import mpmath as mp

# r_max (evaluated at the working precision), degree of P, degree of Q
RANGES = {"half period": (lambda: mp.pi / 2, 7, 7), "panel": (lambda: mp.mpf("0.32"), 4, 3)}


def _g(u):
    if u == 0:
        return mp.mpf(-1) / 6
    r = mp.sqrt(u)
    return (mp.sin(r) - r) / r ** 3


def _h(u):
    if u == 0:
        return mp.mpf(1) / 24
    r = mp.sqrt(u)
    return (mp.cos(r) - 1 + u / 2) / u ** 2


def _interpolate(f, degree, r_max):
    upper = r_max ** 2
    n = degree + 1
    nodes = [upper / 2 * (1 - mp.cos((2 * i + 1) * mp.pi / (2 * n))) for i in range(n)]
    vander = mp.matrix([[x ** j for j in range(n)] for x in nodes])
    values = mp.matrix([f(x) for x in nodes])
    return [float(c) for c in mp.lu_solve(vander, values)]


def coefficients(name="half period"):
    """(P, Q) as lists of doubles, lowest degree first."""
    with mp.workdps(50):
        r_max, dp, dq = RANGES[name]
        return _interpolate(_g, dp, r_max()), _interpolate(_h, dq, r_max())


def max_errors(P, Q, name="half period", samples=2001):
    """Maximum |poly - exact| of sin and cos over [0, r_max] with the given coefficients."""
    es = ec = mp.mpf(0)
    with mp.workdps(50):
        r_max = RANGES[name][0]()
        for i in range(samples):
            r = r_max * i / (samples - 1)
            u = r * r
            p = sum(mp.mpf(c) * u ** j for j, c in enumerate(P))
            q = sum(mp.mpf(c) * u ** j for j, c in enumerate(Q))
            es = max(es, abs(r + r ** 3 * p - mp.sin(r)))
            ec = max(ec, abs(1 - u / 2 + u * u * q - mp.cos(r)))
    return float(es), float(ec)


if __name__ == "__main__":
    for name in RANGES:
        P, Q = coefficients(name)
        print(name)
        print("P =", ", ".join(repr(c) for c in P))
        print("Q =", ", ".join(repr(c) for c in Q))
        print("max error sin %.3e cos %.3e" % max_errors(P, Q, name))
