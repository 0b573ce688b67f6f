"""Print the constants of fastmath.h: Chebyshev interpolants computed with mpmath at 40 digits and rounded once to
double, and the parts of ln(2)/2 and pi/2.

  atanh(s) = s + s^3 p(s^2),              |s| <= (sqrt(2) - 1) / (sqrt(2) + 1), p of degree 6
  sin r = r + r^3 p(r^2), cos r = 1 - r^2/2 + r^4 p(r^2), |r| <= pi/4, p of degree 5

The intervals of s^2 and r^2 are 2e-4 longer, for arguments that rounding leaves beyond their ends.

Usage: python gen_fastmath.py
"""
import mpmath as mp

from gen_hank64 import cheb_interp_monomial

mp.mp.dps = 40


def interpolant(f, top, deg):
    """Monomial coefficients, low order first, of the interpolant of f on (0, top]."""
    top = mp.mpf(top)
    return [float(mp.re(c) / top ** k) for k, c in enumerate(cheb_interp_monomial(lambda v: f(v * top), deg))]


def split(x, bits):
    """x to `bits` fractional bits, rounded down, and the double nearest to the rest."""
    head = mp.floor(x * 2 ** bits) / 2 ** bits
    return float(head), float(x - head)


def constants():
    q, more = mp.sqrt, 1 + mp.mpf(2) / 10 ** 4
    smax = (q(2) - 1) / (q(2) + 1)
    half_pi = float(mp.pi / 2)
    return {
        "atanh": interpolant(lambda z: (mp.atanh(q(z)) / q(z) - 1) / z, more * smax ** 2, 6),
        "sin": interpolant(lambda z: (mp.sin(q(z)) / q(z) - 1) / z, more * (mp.pi / 4) ** 2, 5),
        "cos": interpolant(lambda z: (mp.cos(q(z)) - 1 + z / 2) / z ** 2, more * (mp.pi / 4) ** 2, 5),
        "ln2/2": split(mp.log(2) / 2, 32),
        "pi/2": (half_pi, float(mp.pi / 2 - half_pi)),
    }


if __name__ == "__main__":
    for name, values in constants().items():
        print(name, *map(repr, values))
