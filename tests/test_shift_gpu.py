"""M2M and L2L by the 4-point DFT over a parent's children (csrc/shift.h) where its shapes change: a small tree
(one column a thread, rows split over threads) and a large one (two columns a thread), several row tiles, expansions
that pass through LDS in chunks, orders that differ from level to level, several densities.

Tolerances as in the M2L test: the truncation error of the smallest order p is bounded by
(sqrt(2)/2 / 1.5)^(p+1) of the potential, and a misplaced coefficient or phase leaves errors of its size."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def points(n, rng):
    return np.concatenate([rng.random((2, n // 2)), 0.3 + 0.02 * rng.standard_normal((2, n - n // 2))], axis=1)


def bound(p, floor):
    return (np.sqrt(0.5) / 1.5) ** (p + 1) + floor


@pytest.mark.parametrize("n,ndiv,nd", [(3000, 6, 1), (3000, 6, 5), (150000, 5, 1), (60000, 5, 3)])
@pytest.mark.parametrize("p", [2, 3, 20, 33, 63, 64, 65, 100, [30, 26, 22, 21, 20, 17, 16, 15, 14, 13, 12, 11, 10, 9, 8]])
def test_laplace(p, n, ndiv, nd):
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(n + nd)
    m = 40
    src = points(n, rng)
    ch = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n))
    opts = {"nterms": p if isinstance(p, list) else [p], "ndiv": ndiv}
    res, ier = _fmm("l", 1e-6, None, src, ch[0] if nd == 1 else ch, None, None, None, 1, 0, nd, opts)
    assert ier == 0
    ex = O.direct("l", nd, src, src[:, :m], ch, None, None, 1, 1e-16)["pottarg"]
    a = np.reshape(res["pot"], (nd, n))[:, :m]
    e = np.linalg.norm(a - ex) / np.linalg.norm(ex)
    assert e < bound(min(p) if isinstance(p, list) else p, 1e-11), e


@pytest.mark.parametrize("zk", [30.0, 160.0, 400.0, 60.0 + 3.0j])
@pytest.mark.parametrize("n,ndiv,nd", [(4000, 8, 1), (4000, 8, 2), (80000, 6, 1)])
def test_helmholtz_orders_change(zk, n, ndiv, nd):
    from fmm2d_amd.fmm2d import _fmm
    rng = np.random.default_rng(n + nd)
    m, eps = 40, 1e-9
    src = points(n, rng)
    ch = rng.standard_normal((nd, n)) + 1j * rng.standard_normal((nd, n))
    res, ier = _fmm("h", eps, zk, src, ch[0] if nd == 1 else ch, None, None, None, 1, 0, nd, {"ndiv": ndiv})
    assert ier == 0
    ex = O.direct("h", nd, src, src[:, :m], ch, None, None, 1, 1e-16, zk=zk)["pottarg"]
    a = np.reshape(res["pot"], (nd, n))[:, :m]
    e = np.linalg.norm(a - ex) / np.linalg.norm(ex)
    assert e < 10 * eps, e
