"""Prediction with rows and runs of trees in LDS (fbhip_predict.hip) at the edges
of its tiles, runs and feature counts: margins bit for bit the float32 additions
of the walked leaves in tree order, leaf ids equal."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

from test_gpu_shap_paths import _ensemble, lib  # noqa: F401

pytestmark = pytest.mark.gpu


def _walk(offs, a, words, x):
    """Margins from 0.25 and leaf ids, tree by tree, in float32."""
    n = x.shape[0]
    m = np.full(n, np.float32(0.25))
    ids = np.zeros((n, offs.size - 1), np.float32)
    rows = np.arange(n)
    for t in range(offs.size - 1):
        at = np.full(n, offs[t], np.int64)
        while True:
            split = a["leaf"][at] == 0
            if not split.any():
                break
            v = x[rows, a["feat"][at]]
            left = v < a["cond"][at]
            cat = a["clen"][at] > 0
            code = np.where(cat & (v >= 0) & (v < 2**24), v, 0).astype(np.int64)
            word = code // 32
            listed = cat & (v >= 0) & (v < 2**24) & (word < a["clen"][at])
            w = words[np.where(listed, a["coff"][at] + word, 0)]
            left = np.where(cat, ~(listed & ((w >> (code % 32)) & 1 == 1)), left)
            left = np.where(np.isnan(v), a["dl"][at] == 1, left)
            nxt = offs[t] + np.where(left, a["left"][at], a["right"][at])
            at = np.where(split, nxt, at)
        ids[:, t] = at - offs[t]
        m = (m + a["val"][at]).astype(np.float32)
    return m, ids


@pytest.mark.parametrize("rows,n_trees,depth,nf,n_cat,full", [
    (1, 1, 3, 4, 0, True),          # one row, a single-leaf tree
    (64, 33, 6, 28, 0, True),       # several runs, split over workgroups
    (65, 40, 8, 200, 40, True),     # runs ended by their nodes, categories, a row past a tile
    (300, 20, 4, 500, 0, False),    # the widest rows
    (300, 20, 4, 501, 3, False),    # wider: rows from memory
    (100, 3, 13, 9, 2, True),       # 16,383 nodes: larger than a run
    (33_000, 18, 5, 130, 4, False),  # several tiles a workgroup, one group of rows, one run
    (33_001, 60, 6, 100, 4, False),  # two groups, several runs
    (131_100, 30, 5, 28, 4, False),  # four groups, the last tile one group and a bit
])
def test_margins_and_leaf_ids(lib, rows, n_trees, depth, nf, n_cat, full):  # noqa: F811
    N = lib
    rng = np.random.default_rng(rows + nf)
    offs, a, words = _ensemble(rng, n_trees, depth, nf, n_cat, full)
    x = rng.normal(size=(rows, nf)).astype(np.float32)
    if n_cat:
        x[:, nf - n_cat:] = rng.integers(-2, 80, (rows, n_cat))
    x[rng.random(x.shape) < 0.1] = np.nan
    h = C.c_void_p()
    N.check_hip(N.hip().fbh_shap_model_create(
        0, n_trees, N.ptr(offs), N.ptr(a["feat"]), N.ptr(a["cond"]), N.ptr(a["left"]),
        N.ptr(a["right"]), N.ptr(a["dl"]), N.ptr(a["leaf"]), N.ptr(a["val"]), N.ptr(a["hess"]),
        N.ptr(a["coff"]), N.ptr(a["clen"]), N.ptr(words), words.size, nf, 0.25, C.byref(h)))
    try:
        want, ids = _walk(offs, a, words, x)
        got = np.full(rows, np.nan, np.float32)
        N.check_hip(N.hip().fbh_predict(h, N.ptr(x), rows, None, 0, N.ptr(got)))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        leaf = np.full((rows, n_trees), np.nan, np.float32)
        N.check_hip(N.hip().fbh_predict(h, N.ptr(x), rows, None, 2, N.ptr(leaf)))
        assert np.array_equal(leaf, ids)
    finally:
        N.hip().fbh_shap_model_destroy(h)


@pytest.mark.parametrize("rows,n_trees,depth,nf,n_cat,full", [
    (20_000, 3, 12, 28, 3, True),    # a tree a run: walked from memory, rows in LDS
    (20_000, 6, 11, 40, 0, True),    # three trees a run: likewise
    (1_000, 3, 12, 28, 3, True),     # few rows: the runs split over workgroups
    (40_000, 1, 2, 28, 0, True),     # one small tree
    (33_000, 2, 5, 400, 5, True),    # two small trees of wide rows: read in place
    (500, 2, 13, 240, 3, True),      # trees larger than a run, rows past 64 KiB of LDS
    (130, 2, 13, 255, 0, True),      # the widest of those
    (130, 2, 13, 256, 3, True),      # wider: read in place
])
def test_large_and_few_trees(lib, rows, n_trees, depth, nf, n_cat, full):  # noqa: F811
    """Both sides of predict_tiles_pay, and of the row widths of the walk it leaves
    the others to."""
    test_margins_and_leaf_ids(lib, rows, n_trees, depth, nf, n_cat, full)


@pytest.mark.parametrize("rows,n_trees,depth,nf,n_cat", [
    (300, 40, 6, 28, 4),       # rows and trees in LDS
    (20_000, 3, 12, 28, 4),    # nodes from memory, rows in LDS
    (33_000, 2, 5, 400, 5),    # both from memory
])
def test_values_at_the_ends_of_the_order(lib, rows, n_trees, depth, nf, n_cat):  # noqa: F811
    """Cells and thresholds among both zeros, infinities, denormals, the largest and
    smallest numbers and NaN, equal ones among them: the walk's float comparisons."""
    N = lib
    rng = np.random.default_rng(nf + depth)
    offs, a, words = _ensemble(rng, n_trees, depth, nf, n_cat, True)
    tiny, big = np.float32(1.4e-45), np.finfo(np.float32).max
    ends = np.array([0.0, -0.0, np.inf, -np.inf, tiny, -tiny, 3 * tiny, 1.17e-38, -1.17e-38, big,
                     -big, 1.0, -1.0, np.nan], np.float32)
    a["cond"] = rng.choice(ends, a["cond"].size).astype(np.float32)
    x = rng.choice(ends, (rows, nf)).astype(np.float32)
    h = C.c_void_p()
    N.check_hip(N.hip().fbh_shap_model_create(
        0, n_trees, N.ptr(offs), N.ptr(a["feat"]), N.ptr(a["cond"]), N.ptr(a["left"]),
        N.ptr(a["right"]), N.ptr(a["dl"]), N.ptr(a["leaf"]), N.ptr(a["val"]), N.ptr(a["hess"]),
        N.ptr(a["coff"]), N.ptr(a["clen"]), N.ptr(words), words.size, nf, 0.25, C.byref(h)))
    try:
        want, ids = _walk(offs, a, words, x)
        got = np.full(rows, np.nan, np.float32)
        N.check_hip(N.hip().fbh_predict(h, N.ptr(x), rows, None, 0, N.ptr(got)))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        leaf = np.full((rows, n_trees), np.nan, np.float32)
        N.check_hip(N.hip().fbh_predict(h, N.ptr(x), rows, None, 2, N.ptr(leaf)))
        assert np.array_equal(leaf, ids)
    finally:
        N.hip().fbh_shap_model_destroy(h)
