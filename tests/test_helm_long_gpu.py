"""Helmholtz P2M and list 4 (csrc/helm_fmm.hip, accumulate_rows) where an expansion no longer fits two coefficients a
lane (orders from 64 on) and goes in tiles of 60 orders: around 64, at and beside the tiles' edges, and several
tiles, with charges, dipoles and both, one density and two, against the oracle's direct sums.

Orders are set level by level, at least what the rule of h2dterms asks for at eps; the result is then within a few
eps (10, as for the M2M and L2L), and a misplaced order or phase leaves an error of the size of the potential."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

EPS, ZK, NDIV = 1e-9, 300.0, 150


def rule(size):
    from fmm2d_amd import _native as nat
    v = ctypes.c_int(0)
    assert nat.lib().fmm2d_h2dterms(size, ZK, 0.0, EPS, ctypes.byref(v)) == 0
    return v.value


@pytest.mark.parametrize("what", ["c", "d", "cd"])
@pytest.mark.parametrize("p", [62, 63, 64, 65, 119, 120, 121, 180, 241])
def test_long_rows(p, what):
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(p)
    n, m = 4001, 60
    src = np.concatenate([rng.random((2, n // 2)), 0.3 + 0.02 * rng.standard_normal((2, n - n // 2))], axis=1)
    size = np.ptp(src, axis=1).max()
    # (from level 3 on, k times the box size 37 and less, M2L operators of orders beyond 121 pass the range of a double:
    # H_2p(k r) grows like (4 p / e k r)^2p)
    nterms = [rule(size / 2 ** l) if l > 2 and p > 121 else max(p, rule(size / 2 ** l)) for l in range(12)]
    assert all(t >= rule(size / 2 ** l) for l, t in enumerate(nterms))
    for nd in (1, 2):
        ch = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n)) if "c" in what else None
        ds = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n)) if "d" in what else None
        dv = rng.standard_normal((nd, 2, n)) if "d" in what else None
        one = [None if a is None else a[0] if nd == 1 else a for a in (ch, ds, dv)]
        res, ier = _fmm("h", EPS, ZK, src, *one, None, 1, 0, nd, {"nterms": nterms, "ndiv": NDIV})
        assert ier == 0
        ex = O.direct("h", nd, src, src[:, :m], ch, ds, dv, 1, 1e-16, zk=ZK)["pottarg"]
        a = np.reshape(res["pot"], (nd, n))[:, :m]
        e = np.linalg.norm(a - ex) / np.linalg.norm(ex)
        assert e < 10 * EPS, e
