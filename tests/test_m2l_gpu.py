"""The M2L of four rotated sources per operator (csrc/m2l.h) at every padding of its tiles, up to and beyond
the length where the one-source operators take over: FMM potentials with a given expansion order against
the oracle's direct sums.

The truncation error of order p is bounded by C (sqrt(2)/2 / 1.5)^(p+1) (the rule of l2dterms, and of
h2dterms at low frequency); a misplaced coefficient, phase or slot would leave errors of the size of the
potential itself."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def points(n, rng):
    return np.concatenate([rng.random((2, n // 2)), 0.3 + 0.02 * rng.standard_normal((2, n - n // 2))], axis=1)


def bound(p, floor):
    return (np.sqrt(0.5) / 1.5) ** (p + 1) + floor


@pytest.mark.parametrize("nd,prec", [(1, "fp64"), (3, "fp64"), (1, "mixed"), (2, "mixed")])
@pytest.mark.parametrize("p", [2, 7, 8, 14, 15, 16, 18, 23, 24, 31, 32, 39, 40, 48, 56, 63, 64])
def test_laplace_orders(p, nd, prec):
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(100 * p + nd)
    n, m = 2000, 60
    src, trg = points(n, rng), points(301, rng)
    ch = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n))
    opts = {"nterms": [p], "ndiv": 12, "precision": prec}
    res, ier = _fmm("l", 1e-6, None, src, ch[0] if nd == 1 else ch, None, None, trg, 2, 2, nd, opts)
    assert ier == 0
    floor = 1e-12 if prec == "fp64" else 2e-6
    for pts, end in ((src[:, :m], ""), (trg[:, :m], "targ")):
        ex = O.direct("l", nd, src, pts, ch, None, None, 2, 1e-16)
        for what in ("pot", "grad"):
            a = np.reshape(res[what + end], np.shape(ex[what + "targ"])[:-1] + (-1,))[..., :m]
            e = np.linalg.norm(a - ex[what + "targ"]) / np.linalg.norm(ex[what + "targ"])
            assert e < (1 if what == "pot" else 4) * bound(p, floor), (what + end, e)


@pytest.mark.parametrize("nd,prec", [(1, "fp64"), (2, "fp64"), (1, "mixed")])
@pytest.mark.parametrize("p", [4, 7, 8, 11, 12, 15, 16, 19, 20, 24, 27, 28, 31, 32])
def test_helmholtz_orders(p, nd, prec):
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(100 * p + nd)
    n, m, zk = 2000, 60, 1.5
    src = points(n, rng)
    ch = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n))
    opts = {"nterms": [p], "ndiv": 12, "precision": prec}
    res, ier = _fmm("h", 1e-6, zk, src, ch[0] if nd == 1 else ch, None, None, None, 1, 0, nd, opts)
    assert ier == 0
    ex = O.direct("h", nd, src, src[:, :m], ch, None, None, 1, 1e-16, zk=zk)["pottarg"]
    a = np.reshape(res["pot"], (nd, n))[:, :m]
    e = np.linalg.norm(a - ex) / np.linalg.norm(ex)
    assert e < bound(p, 1e-11 if prec == "fp64" else 4e-6), e


@pytest.mark.parametrize("kind,p,prec", [(k, p, prec) for k, ps in (("l", (71, 79, 87, 95)), ("h", (36, 40, 44, 47)))
                                         for p in ps for prec in (("fp64", "mixed") if k == "l" else ("fp64",))])
def test_last_row_tiles_of_long_operators(kind, p, prec):
    """Operators of 65 coefficients and more (csrc/translate.h) with one to four row tiles in their last chunk (9 to
    12 tiles in all), in one wavefront or split over slots and k steps, one density or two.  (Helmholtz operators of
    these orders at this wavenumber are beyond FP32's range: 71! (1/2 pi)^72 > 3.4e38.)"""
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(p)
    n, m, zk = 2000, 60, 1.5
    src = points(n, rng)
    for nd in (1, 2):
        ch = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n))
        opts = {"nterms": [p], "ndiv": 12, "precision": prec}
        res, ier = _fmm(kind, 1e-6, zk if kind == "h" else None, src, ch[0] if nd == 1 else ch, None, None, None, 1, 0,
                        nd, opts)
        assert ier == 0
        ex = O.direct(kind, nd, src, src[:, :m], ch, None, None, 1, 1e-16, **({"zk": zk} if kind == "h" else {}))
        a = np.reshape(res["pot"], (nd, n))[:, :m]
        e = np.linalg.norm(a - ex["pottarg"]) / np.linalg.norm(ex["pottarg"])
        assert e < bound(p, {"fp64": 1e-11, "mixed": 4e-6}[prec]), e


@pytest.mark.parametrize("prec", ["fp64", "mixed"])
@pytest.mark.parametrize("unit", [1.0, 1j])
def test_log_term_of_either_part(prec, unit):
    """Charges of one sign, all real or all imaginary: the M2L's log(boxsize) M_0 is most of that part of L_0, and
    an update of it that gets lost (its row has the translation's own sum to add as well) leaves an error of order one."""
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(7)
    n, m, p = 3000, 80, 16
    src = points(n, rng)
    ch = unit * (1.0 + rng.random((2, n))) + 0j
    opts = {"nterms": [p], "ndiv": 12, "precision": prec}
    for nd in (1, 2):
        c = (ch[0] if nd == 1 else ch) * (1.0 if nd == 1 else np.array([[1.0], [1j]]))
        res, ier = _fmm("l", 1e-6, None, src, c, None, None, None, 1, 0, nd, opts)
        assert ier == 0
        ex = O.direct("l", nd, src, src[:, :m], np.reshape(c, (nd, n)), None, None, 1, 1e-16)["pottarg"]
        a = np.reshape(res["pot"], (nd, n))[:, :m]
        e = np.linalg.norm(a - ex) / np.linalg.norm(ex)
        assert e < bound(p, 1e-12 if prec == "fp64" else 2e-6), e
