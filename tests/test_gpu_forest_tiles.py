"""Regression trees on the device against a NumPy walk, bit for bit: batches
of 16 trees and tiles of 128 rows with remainders, the largest trees and
feature counts that the tiles take and the smallest beyond them, thresholds
met exactly, NaN and infinite features."""

import ctypes

import numpy as np
import numpy.testing as npt
import pytest

pytestmark = pytest.mark.gpu


def _tree(rng, leaves, nfeat):
    left, right, feat, thr = [0], [0], [0], [0.0]
    ends = [0]
    while len(ends) < leaves:
        p = ends.pop(int(rng.integers(len(ends))))
        left[p], right[p] = len(left), len(left) + 1
        feat[p], thr[p] = int(rng.integers(nfeat)), float(rng.integers(-3, 4)) / 2
        for _ in range(2):
            ends.append(len(left))
            left.append(0), right.append(0), feat.append(0), thr.append(0.0)
    leaf = np.zeros(len(left), np.uint8)
    leaf[ends] = 1
    return [np.array(a) for a in (feat, thr, left, right)] + [leaf, rng.standard_normal(len(left))]


def _walk(trees, base, X):
    out = np.full(len(X), base)
    for feat, thr, left, right, leaf, value in trees:
        at = np.zeros(len(X), int)
        while not leaf[at].all():
            go = X[np.arange(len(X)), feat[at]] <= thr[at]
            at = np.where(leaf[at] == 1, at, np.where(go, left[at], right[at]))
        out = out + value[at]
    return out


@pytest.mark.parametrize("ntrees, leaves, nfeat", [(1, 1, 1), (1, 64, 16), (15, 9, 3), (16, 63, 10),
                                                   (17, 64, 16), (33, 40, 13), (5, 65, 16),
                                                   (5, 30, 17)])
def test_forest_matches_numpy_walk(gpu, ntrees, leaves, nfeat):
    from fd_adi_amd import _lib
    from fd_adi_amd.SizedArrayPtr import SizedArrayPtr
    rng = np.random.default_rng(ntrees * 100 + leaves)
    trees = [_tree(rng, leaves if k == 0 else int(rng.integers(1, leaves + 1)), nfeat)
             for k in range(ntrees)]
    start = np.zeros(ntrees + 1, np.int64)
    start[1:] = np.cumsum([len(t[0]) for t in trees])
    cat = [np.ascontiguousarray(np.concatenate(a), dtype=d) for a, d in
           zip(zip(*trees), (np.int32, float, np.int32, np.int32, np.uint8, float))]
    h = ctypes.c_void_p()
    _lib.call("fdadi_forest_create", ntrees, _lib.ptr(start), nfeat, *[_lib.ptr(a) for a in cat],
              0.25, ctypes.byref(h))
    try:
        for n in (1, 64, 127, 128, 129, 1000):
            X = rng.integers(-5, 6, (n, nfeat)) / 2.0
            X[rng.random(X.shape) < 0.05] = np.nan
            X[rng.random(X.shape) < 0.02] = np.inf
            dX, out = SizedArrayPtr(X), SizedArrayPtr().alloc(n)
            _lib.call("fdadi_forest_predict", h, dX.p, n, out.p, _lib.default_stream())
            npt.assert_array_equal(out.to_numpy(), _walk(trees, 0.25, X))
    finally:
        _lib.lib.fdadi_forest_destroy(h)
