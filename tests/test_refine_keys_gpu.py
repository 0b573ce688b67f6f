"""The refinement from the sorted keys (csrc/tree.hip, k_ref_keys) against the C oracle's tree, array for array, where
it changes its ways: tiles of 256 and 1024 keys, boxes around the depth of the keys (20 levels) and beyond it
(level by level then), more boxes than expected (made again with more room), leaves of one point, targets."""
import numpy as np
import pytest

from oracle import oracle as O
from test_tree_sizes_gpu import KEYS, points

pytestmark = pytest.mark.gpu


def pairs(n, gap, rng):
    """n points in pairs gap apart, in the unit square (whose corners are points)."""
    p = rng.random((2, n // 2))
    p[:, 0], p[:, 1] = 0.0, 1.0
    q = p + gap * np.sign(0.5 - p)
    return np.concatenate([p, q], axis=1)


CASES = [
    ("uniform", 1, 0, 1), ("uniform", 2, 0, 1), ("uniform", 255, 0, 3), ("uniform", 256, 0, 3), ("uniform", 257, 9, 3),
    ("uniform", 1023, 1025, 7), ("uniform", 1025, 0, 1), ("uniform", 3, 5000, 1), ("curve", 65537, 65, 20),
    ("pairs1e-5", 1200, 0, 1), ("pairs1e-5", 1200, 300, 1), ("pairs2e-6", 512, 0, 1), ("pairs9e-7", 64, 0, 1),
    ("pairs4e-7", 64, 10, 1), ("pairs1e-8", 64, 0, 1), ("pairs0.0", 64, 0, 2), ("clusters", 1048577, 0, 200),
    ("uniform", 1048576, 1000, 90),
]


@pytest.mark.parametrize("kind,n,nt,ndiv", CASES)
def test_refinement(kind, n, nt, ndiv):
    from fmm2d_amd.tree import build_tree
    rng = np.random.default_rng(n + nt)
    src = pairs(n, float(kind[5:]), rng) if kind.startswith("pairs") else points(kind, n, rng)
    trg = points("uniform", nt, rng) if nt else None
    t = build_tree(src, trg, ndiv=ndiv)
    o = O.tree(src, trg, ndiv)
    assert (t["nlevels"], t["nboxes"]) == (o["nlevels"], o["nboxes"])
    for k in KEYS:
        if nt or not k.startswith("itarg"):
            assert np.array_equal(t[k], o[k]), k
