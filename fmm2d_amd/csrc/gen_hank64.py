"""Generate hank64_tables.h: the FP64 coefficient tables of the real-argument
Hankel pair (hankel.h, hank01_real).

For x < X1: the sums of the ascending series (Abramowitz & Stegun 9.1.10, 9.1.11,
9.1.13) in q = x^2/4 as their Chebyshev interpolants on [0, X1^2/4], NSER
coefficients each (interpolation error below 1e-19; the series itself needs 17
terms), computed with mpmath and rounded once to double:
  J0 = sum a_k q^k,            a_k = (-1)^k / (k!)^2
  J1 = (x/2) sum b_k q^k,      b_k = (-1)^k / (k! (k+1)!)
  Y0 = (2/pi) [(ln(x/2) + gamma) J0 + sum c_k q^k],  c_k = -H_k a_k
  Y1 = (2/pi) (ln(x/2) + gamma) J1 - 2/(pi x) - (x/(2 pi)) sum d_k q^k,
                               d_k = (2 H_k + 1/(k+1)) b_k
(H_k the harmonic numbers).

For x >= X1:  H_nu(x) = sqrt(2/(pi x)) e^{i (x - nu pi/2 - pi/4)} (P_nu + i Q_nu)(s),
s = X1/x in (0, 1].  The amplitude M_nu = P_nu + i Q_nu is smooth in s (it tends
to 1 as s -> 0 along Hankel's asymptotic expansion, A&S 9.2.5-9.2.10); P_nu and
Q_nu are its Chebyshev interpolants of degree NFIT on [0, 1] (nodes at the
Chebyshev points of the first kind), computed with mpmath at 40 digits, converted
to monomial coefficients in s at that precision and rounded once to double.
The maximum error of the rounded polynomials evaluated by Horner's rule in
double, against mpmath's hankel1 on x in [X1, 1e6], is printed to stderr
(about one unit in the last place of |M| ~ 1).
Run:  python fmm2d_amd/csrc/gen_hank64.py > fmm2d_amd/csrc/hank64_tables.h
"""
import sys
from fractions import Fraction

import mpmath as mp
import numpy as np

X1 = 4
NFIT = 18
NSER = 15
mp.mp.dps = 40


def series():
    """Rows (a_k, b_k, c_k, d_k), k = 0..NSER-1, as doubles."""
    rows = []
    fk, H = Fraction(1), Fraction(0)
    for k in range(45):
        if k > 0:
            fk *= k
            H += Fraction(1, k)
        ak = Fraction((-1) ** k) / (fk * fk)
        bk = Fraction((-1) ** k) / (fk * fk * (k + 1))
        rows.append([mp.mpf(v.numerator) / v.denominator
                     for v in (ak, bk, -H * ak, (2 * H + Fraction(1, k + 1)) * bk)])
    qmax = mp.mpf(X1) ** 2 / 4
    cols = []
    for j in range(4):
        # in v = q / qmax on [0, 1]
        c = cheb_interp_monomial(
            lambda v: sum(r[j] * (v * qmax) ** k for k, r in enumerate(rows)), NSER - 1)
        cols.append([float(p.real / qmax ** k) for k, p in enumerate(c)])
    return [[cols[j][k] for j in range(4)] for k in range(NSER)]


def amplitude(nu, x):
    x = mp.mpf(x)
    return mp.hankel1(nu, x) * mp.sqrt(mp.pi * x / 2) * mp.expj(-(x - nu * mp.pi / 2 - mp.pi / 4))


def cheb_interp_monomial(f, deg):
    """Monomial coefficients (in s, low order first) of the degree-deg Chebyshev
    interpolant of f on s in [0, 1]."""
    n = deg + 1
    half = mp.mpf(1) / 2
    fv = [f((mp.cos(mp.pi * (k + half) / n) + 1) / 2) for k in range(n)]
    c = [sum(fv[k] * mp.cos(mp.pi * j * (k + half) / n) for k in range(n)) * (2 if j else 1) / n
         for j in range(n)]
    T = [[mp.mpf(1)], [mp.mpf(0), mp.mpf(1)]]  # T_j(u) in powers of u
    for j in range(2, n):
        a = [mp.mpf(0)] + [2 * v for v in T[-1]]
        b = T[-2] + [mp.mpf(0)] * (len(a) - len(T[-2]))
        T.append([p - q for p, q in zip(a, b)])
    pu = [mp.mpc(0)] * n
    for j in range(n):
        for i, v in enumerate(T[j]):
            pu[i] += c[j] * v
    ps = [mp.mpc(0)] * n  # u = 2 s - 1
    for i in range(n):
        for k in range(i + 1):
            ps[k] += pu[i] * mp.binomial(i, k) * 2 ** k * (-1) ** (i - k)
    return ps


def main():
    print("// Generated by gen_hank64.py -- FP64 coefficients of H0, H1 for real")
    print("// arguments.  FMM2D_H64_SER: rows (a_k, b_k, c_k, d_k) of the ascending")
    print("// series' interpolants in q = x^2/4, k = 0..NSER-1 (x < X1).  FMM2D_H64_AMP: rows")
    print("// (P0, Q0, P1, Q1)_k of the amplitude polynomials in s = X1 / x, k = 0..NFIT")
    print("// (x >= X1).  Low order first.")
    print("#pragma once")
    print(f"#define FMM2D_H64_X1 {X1}.0")
    print(f"#define FMM2D_H64_NFIT {NFIT}")
    print(f"#define FMM2D_H64_NSER {NSER}")
    print("#define FMM2D_H64_SER \\")
    print(", \\\n".join("  " + ", ".join(repr(v) for v in row) for row in series()))
    amp = []
    for nu in (0, 1):
        ps = cheb_interp_monomial(
            lambda s: amplitude(nu, X1 / s) if s > 0 else mp.mpc(1), NFIT)
        cr = [float(p.real) for p in ps]
        ci = [float(p.imag) for p in ps]
        amp += [cr, ci]
        err = 0.0
        for x in np.concatenate([np.linspace(X1, 8 * X1, 400), np.geomspace(8 * X1, 1e6, 60)]):
            s = X1 / x
            pr = pi = 0.0
            for k in range(NFIT, -1, -1):
                pr = pr * s + cr[k]
                pi = pi * s + ci[k]
            err = max(err, abs(complex(pr, pi) - complex(amplitude(nu, x))))
        print(f"nu={nu}: max |M - poly| = {err:.2e}", file=sys.stderr)
    print("#define FMM2D_H64_AMP \\")
    print(", \\\n".join("  " + ", ".join(repr(amp[j][k]) for j in range(4))
                         for k in range(NFIT + 1)))


if __name__ == "__main__":
    main()
