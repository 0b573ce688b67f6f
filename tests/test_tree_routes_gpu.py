"""The ways of the tree build that refinement on sources at ordinary depth does not take (csrc/tree.hip), against the
C oracle's tree, array for array: refinement on targets and on the larger of both (level by level: one workgroup up to
4096 boxes a level, batches of levels beyond, with too few boxes reserved in either), sets whose boxes are deeper
than the 20 levels of the keys with more than 4096 boxes a level there; and the 64-bit status words of the sort
(csrc/radix_sort.h), which 2^27 points and more take."""
import ctypes

import numpy as np
import pytest

from oracle import oracle as O
from test_refine_keys_gpu import pairs
from test_tree_sizes_gpu import KEYS, points, rows

pytestmark = pytest.mark.gpu


def compare(src, trg, ndiv, idivflag):
    from fmm2d_amd.tree import build_tree
    t = build_tree(src, trg, ndiv=ndiv, idivflag=idivflag, lists=True)
    o = O.tree(src, trg, ndiv, idivflag)
    assert (t["nlevels"], t["nboxes"]) == (o["nlevels"], o["nboxes"])
    for k in KEYS:
        if trg is not None or not k.startswith("itarg"):
            assert np.array_equal(t[k], o[k]), k
    for k in range(1, 5):
        assert np.array_equal(t[f"nlist{k}"], o[f"nlist{k}"]), f"nlist{k}"
        assert np.array_equal(rows(t[f"list{k}"], t[f"nlist{k}"]), rows(o[f"list{k}"], o[f"nlist{k}"])), f"list{k}"


@pytest.mark.parametrize("idivflag", [1, 2])
@pytest.mark.parametrize("kind,ns,nt,ndiv", [
    ("uniform", 5, 1, 1), ("uniform", 300, 700, 15), ("uniform", 700, 300, 15), ("clusters", 1000, 16385, 10),
    ("uniform", 2000, 100000, 5),    # levels of 16384 boxes
    ("clusters", 100, 200000, 5), ("curve", 50000, 60000, 4),
    ("tight", 40, 1000, 5),          # one workgroup runs out of room
    ("tight", 4000, 20000, 5),       # more than 4096 boxes a level, and out of room
])
def test_targets(kind, ns, nt, ndiv, idivflag):
    rng = np.random.default_rng(ns + nt)
    compare(points(kind, ns, rng), points(kind, nt, rng), ndiv, idivflag)


@pytest.mark.parametrize("n,gap,idivflag", [(4000, 1e-8, 0), (4000, 1e-8, 1), (6000, 3e-7, 0), (3000, 2e-9, 2)])
def test_deep_and_wide(n, gap, idivflag):
    rng = np.random.default_rng(n)
    src = pairs(n, gap, rng)
    compare(src, pairs(n, gap, rng) if idivflag else None, 1, idivflag)


@pytest.mark.parametrize("kind", ["l", "h"])
@pytest.mark.parametrize("idivflag", [1, 2])
def test_calls_refined_on_targets(kind, idivflag):
    """Potentials within eps of the direct sum (the library's own bar).  (cfmm2d's potential is analytic, not the direct
    sum's log|z|, where the far field is; lfmm2d runs on the same driver.)"""
    from fmm2d_amd import fmm2d as F
    rng = np.random.default_rng(idivflag)
    ns, nt, m, eps = 3000, 20000, 200, 1e-9
    src, trg = points("clusters", ns, rng), points("curve", nt, rng)
    ch = rng.standard_normal(ns) + 1j * rng.standard_normal(ns)
    zk = 12.0 if kind == "h" else None
    res, ier = F._fmm(kind, eps, zk, src, ch, None, None, trg, 1, 1, 1, {"ndiv": 12, "idivflag": idivflag})
    assert ier == 0
    for pts, out in ((src[:, :m], res["pot"]), (trg[:, :m], res["pottarg"])):
        ex = O.direct(kind, 1, src, pts, ch, None, None, 1, 1e-16, **({"zk": zk} if zk else {}))["pottarg"][0]
        assert np.linalg.norm(out[:m] - ex) < eps * np.linalg.norm(ex)


def test_status_words_of_64_bits():
    """2^27 + 3 uniform points in the unit square (its corners among them), leaves of 8192 at level 7: the order is a
    permutation, leaves follow each other in path order, and a leaf keeps the input order."""
    import torch

    from fmm2d_amd import _native as nat
    L, n, ndiv, lev = nat.lib(), 2 ** 27 + 3, 20000, 7
    g = torch.Generator(device="cuda")
    g.manual_seed(1)
    p = torch.rand(n, 2, dtype=torch.float64, device="cuda", generator=g)
    p[0], p[1] = 0.0, 1.0
    nl, nb, h = ctypes.c_int(0), ctypes.c_int(0), ctypes.c_void_p()
    assert L.fmm2d_tree_build(nat.ptr(p), n, None, 0, 0, ndiv, 51, ctypes.byref(nl), ctypes.byref(nb), ctypes.byref(h),
                              nat.stream_ptr()) == 0
    try:
        isrc = np.zeros(n, np.int32)
        args = [None] * 21
        args[9] = isrc.ctypes.data_as(ctypes.c_void_p)
        assert L.fmm2d_tree_get(h, *args) == 0
    finally:
        L.fmm2d_tree_free(h)
        L.fmm2d_release_workspace()
    assert nl.value == lev and nb.value == sum(4 ** k for k in range(lev + 1))
    order = torch.from_numpy(isrc).cuda().long() - 1
    assert int(order.min()) == 0 and int(order.max()) == n - 1
    assert int(torch.bincount(order, minlength=n).max()) == 1
    path = torch.zeros_like(order)
    for axis in range(2):  # (a column at a time: torch's p[order] of this many rows has come back wrong)
        cell = torch.clamp((p[:, axis].contiguous()[order] * 2 ** lev).long(), max=2 ** lev - 1)
        for k in range(lev):
            path |= ((cell >> k) & 1) << (2 * k + axis)
    assert bool((path[1:] >= path[:-1]).all())
    assert bool(((path[1:] > path[:-1]) | (order[1:] > order[:-1])).all())
