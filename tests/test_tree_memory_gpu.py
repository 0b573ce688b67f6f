"""Device memory of the tree build (csrc/tree.hip): calls fit a workspace limit that their arrays can live in (bytes
measured of a build that doubled its box arrays when they were full and reorganised into a second set as large), and
where the reserved boxes are too few -- the one-workgroup restriction run again, room for the flagged boxes made
after they are counted, the whole build again for the last sweep -- the tree is the C oracle's, array for array."""
import numpy as np
import pytest

from oracle import oracle as O
from test_tree_sizes_gpu import KEYS, points

pytestmark = pytest.mark.gpu


def limited(nbytes, call):
    from fmm2d_amd import _native as nat
    L = nat.lib()
    L.fmm2d_release_workspace()
    assert L.fmm2d_set_workspace_limit(nbytes) == 0
    try:
        return call()
    finally:
        assert L.fmm2d_set_workspace_limit(0) == 0
        L.fmm2d_release_workspace()


@pytest.mark.parametrize("kind,n,nt,ndiv,idivflag,nbytes", [
    ("uniform", 1000, 0, 15, 0, 344064), ("curve", 30000, 0, 15, 0, 16220160), ("curve", 200000, 0, 20, 0, 80871424),
    ("clusters", 100000, 50000, 10, 2, 82575360), ("uniform", 300000, 0, 200, 0, 15892480),
])
def test_tree_fits(kind, n, nt, ndiv, idivflag, nbytes):
    from fmm2d_amd.tree import build_tree
    rng = np.random.default_rng(n + nt)
    src = points(kind, n, rng)
    trg = points(kind, nt, rng) if nt else None
    t = limited(nbytes, lambda: build_tree(src, trg, ndiv=ndiv, idivflag=idivflag))
    assert t["nboxes"] == O.tree(src, trg, ndiv, idivflag)["nboxes"]


@pytest.mark.parametrize("kind,n,nbytes", [("l", 2000, 851968), ("c", 10000, 3780608), ("h", 3000, 17039360)])
def test_call_fits(kind, n, nbytes):
    from fmm2d_amd import fmm2d as F
    rng = np.random.default_rng(n)
    src = points("uniform", n, rng)
    ch = rng.standard_normal(n) + 0j
    _, ier = limited(nbytes, lambda: F._fmm(kind, 1e-6, 10.0 if kind == "h" else None, src, ch, None, None, None, 2, 0,
                                            1))
    assert ier == 0


@pytest.mark.parametrize("kind,n,ndiv", [("tight", 1000, 1), ("tight", 1000, 5), ("tight", 10000, 5),
                                         ("tight", 20000, 1), ("curve", 1000, 1), ("curve", 10000, 1)])
def test_too_few_reserved(kind, n, ndiv):
    from fmm2d_amd.tree import build_tree
    rng = np.random.default_rng(n + ndiv)
    src = points(kind, n, rng)
    t = build_tree(src, ndiv=ndiv)
    o = O.tree(src, None, ndiv)
    assert (t["nlevels"], t["nboxes"]) == (o["nlevels"], o["nboxes"])
    for k in KEYS:
        if not k.startswith("itarg"):
            assert np.array_equal(t[k], o[k]), k
