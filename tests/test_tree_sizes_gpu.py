"""The GPU quadtree against the C oracle's (oracle/oracle.c), array for array, at the sizes where the
build changes its ways: the sort's tiles (512, 1024, 4096 keys, by size), one workgroup's scan (16384
boxes) and scan tiles of 4096, room for the level restriction (the last case builds again with more), and
trees from a single leaf to more than a million boxes."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

KEYS = ("laddr", "ilevel", "iparent", "nchild", "ichild", "ncoll", "coll", "centers", "boxsize", "isrc", "isrcse",
        "itarg", "itargse")


def points(kind, n, rng):
    if kind == "uniform":
        return rng.random((2, n))
    if kind == "clusters":
        c = rng.random((2, 9))
        lab = rng.integers(0, 9, n)
        return c[:, lab] + np.exp(rng.uniform(np.log(1e-4), np.log(1e-2), 9))[lab] * rng.standard_normal((2, n))
    if kind == "tight":  # 20 points each: the level restriction adds five times the boxes
        return np.repeat(rng.random((2, n // 20)), 20, axis=1) + 1e-6 * rng.standard_normal((2, n))
    t = rng.uniform(0, 2 * np.pi, n)
    r = 1 + 0.3 * np.cos(5 * t)
    return np.stack([r * np.cos(t), r * np.sin(t)]) + 1e-4 * rng.standard_normal((2, n))


def rows(lists, count):
    """A list's rows as sorted sets."""
    used = np.arange(lists.shape[0])[:, None] < count
    return np.sort(np.where(used, lists, np.iinfo(np.int32).max), axis=0)


@pytest.mark.parametrize("kind,n,nt,ndiv", [
    ("uniform", 1, 0, 15), ("uniform", 15, 0, 15), ("uniform", 16, 3, 15), ("uniform", 300, 1, 1),
    ("clusters", 1000, 0, 15), ("clusters", 4095, 4097, 15), ("curve", 8192, 1000, 20), ("clusters", 8193, 70, 3),
    ("uniform", 16384, 513, 15), ("clusters", 16385, 512, 15), ("curve", 30011, 20003, 20), ("clusters", 262145, 1, 60), ("clusters", 131072, 0, 40), ("uniform", 131073, 0, 15), ("clusters", 135169, 5, 8),
    ("tight", 1000, 0, 15), ("tight", 14000, 0, 15), ("tight", 160000, 0, 15),
])
def test_tree_sizes(kind, n, nt, ndiv):
    from fmm2d_amd.tree import build_tree
    rng = np.random.default_rng(n + nt)
    src = points(kind, n, rng)
    trg = points(kind, nt, rng) if nt else None
    t = build_tree(src, trg, ndiv=ndiv, lists=True)
    o = O.tree(src, trg, ndiv)
    assert (t["nlevels"], t["nboxes"]) == (o["nlevels"], o["nboxes"])
    for k in KEYS:
        if nt or not k.startswith("itarg"):
            assert np.array_equal(t[k], o[k]), k
    for k in range(1, 5):
        assert np.array_equal(t[f"nlist{k}"], o[f"nlist{k}"]), f"nlist{k}"
        assert np.array_equal(rows(t[f"list{k}"], t[f"nlist{k}"]), rows(o[f"list{k}"], o[f"nlist{k}"])), f"list{k}"
