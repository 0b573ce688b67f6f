"""The pair kernels' own logarithm, reciprocals, square root and sine/cosine (csrc/fastmath.h) and the real-argument
Hankel pair (csrc/hankel.h) at the edges of their ranges, through single-source direct sums against numpy and scipy.

Tolerances: 8 units in the last place for the logarithm and 1/r; for H0, H1 relative to |H|, 1e-14 (the documented
accuracy 5e-15, and scipy's own) plus the phase error of two units in the last place of k r."""
import numpy as np
import pytest
from scipy.special import hankel1

pytestmark = pytest.mark.gpu

ULP = np.finfo(float).eps


def single_source(kind, x, zk=None, dip=False):
    """pot and d pot / dx at the targets (x, 0) of one unit charge or x-dipole at the origin."""
    from fmm2d_amd import fmm2d as F
    src = np.zeros((2, 1))
    trg = np.array([x, np.zeros_like(x)])
    one, vec = np.ones(1, dtype=complex), np.array([[1.0], [0.0]])
    (p, g, _), _ = F._direct(kind, zk, src, trg, None if dip else one, one if dip else None,
                             vec if dip else None, 2, 1, 1e-300)
    return p[0], np.asarray(g).reshape(2, -1)[0]


def edges():
    r = np.sqrt(0.5)
    base = [1.0, r, np.nextafter(r, 0), np.nextafter(r, 2), np.sqrt(r), 2 ** 0.25, np.nextafter(1, 0),
            np.nextafter(1, 2), 1 + 1e-9, 1 - 1e-5, 1.1, 0.9]
    return np.array([b * s for b in base for s in (1.0, 2.0, 0.5, 1e-8, 1e8, 1e-100, 1e100)])


def test_log_and_reciprocal():
    x = edges()
    p, g = single_source("l", x)
    lg = np.log(x)
    # log(r) from log(r^2) / 2: the rounding of r^2 is half a unit of 1
    assert np.all(np.abs(p.real - lg) <= 8 * ULP * np.abs(lg) + ULP), np.max(np.abs(p.real - lg))
    assert np.all(np.abs(g.real * x - 1) <= 8 * ULP)


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_nan_and_infinite_targets(bad):
    p, _ = single_source("l", np.array([1.0, bad, 2.0]))
    assert not np.isfinite(p[1].real)
    assert np.all(np.isfinite(p[[0, 2]]))
    p, _ = single_source("h", np.array([1.0, bad, 2.0]), zk=2.0)
    assert not np.isfinite(p[1])
    assert np.all(np.isfinite(p[[0, 2]]))


@pytest.mark.parametrize("dip", [False, True])
@pytest.mark.parametrize("zk", [1.0, 37.5])
def test_hankel_edges(zk, dip):
    kr = np.concatenate([[1e-8, 1e-3, 0.5, 2.4, np.nextafter(4, 0), 4.0, np.nextafter(4, 5)],
                         np.arange(1, 40) * np.pi / 4, np.geomspace(4, 1e6, 60), np.linspace(0.1, 9, 50)])
    x = kr / zk
    z = zk * x
    p, g = single_source("h", x, zk=complex(zk), dip=dip)
    h0, h1 = hankel1(0, z), hankel1(1, z)
    tol = 1e-14 + 4 * ULP * z
    if not dip:
        want, scale = 0.25j * h0, 0.25 * np.abs(h0)
        wantg, scaleg = -0.25j * zk * h1, 0.25 * zk * np.abs(h1)
    else:
        want, scale = 0.25j * zk * h1, 0.25 * zk * np.abs(h1)
        wantg = 0.25j * zk * zk * (h0 - h1 / z)  # d/dx of (i k / 4) H1(k x)
        # (x = the sum's own terms: H2 = 2 H1 / z - H0 cancels for small z)
        scaleg = 0.25 * zk * zk * (np.abs(h0) + 2 * np.abs(h1) / z)
    assert np.all(np.abs(p - want) <= tol * scale), np.max(np.abs(p - want) / scale / tol)
    assert np.all(np.abs(g - wantg) <= 2 * tol * scaleg), np.max(np.abs(g - wantg) / scaleg / tol)


@pytest.mark.parametrize("zk", [1e155, 1e155 + 1e154j])
def test_subnormal_squares(zk):
    """Distances whose square is subnormal (r < 1.5e-154).  The square's own rounding, half of 4.9e-324, is an error of
    k r times half of that over r^2 in the argument, more for the singular part of small arguments."""
    z = np.array([0.3, 1.0, 3.0, 7.0])
    x = z * 1e-155
    p, _ = single_source("h", x, zk=zk)
    h0 = hankel1(0, zk * x)
    tol = 1e-14 + 4 * ULP * z + 2 * (1 + z) * 4.9406564584124654e-324 / (x * x)
    assert np.all(np.abs(p - 0.25j * h0) <= tol * 0.25 * np.abs(h0)), np.abs(p / (0.25j * h0) - 1) / tol


def test_large_arguments():
    x = np.array([1e7, 2.0 ** 40, 2.0 ** 49, 2.0 ** 50, 2.0 ** 55, 1e30])  # exact squares or far beyond phase accuracy
    p, _ = single_source("h", x, zk=1.0)
    amp = 0.25 * np.sqrt(2 / np.pi / x)
    assert np.all(np.isfinite(p)) and np.all(np.abs(np.abs(p) / amp - 1) < 1e-7)
    want = 0.25j * np.sqrt(2 / np.pi / x) * np.exp(1j * x) * np.exp(-0.25j * np.pi)
    # 1/x terms of the amplitude, and one unit of x in the phase
    assert abs(p[0] - want[0]) < (1 / x[0] + 4 * ULP * x[0]) * amp[0]
