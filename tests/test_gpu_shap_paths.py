"""TreeSHAP by the closed sums (fbhip_shap_paths.hip) against the host engine's
operation order (fbh_shap_set_host_order, which the other suites pin to the
oracle), at the edges of its tiles, depths, path shapes and feature counts.

Tolerance: both sides round every product and sum of a path of at most 8 splits
at 4 or 8 quadrature points, at most 16 roundings of one leaf's terms a level,
each relative to terms of at most the leaf's size (a path's weights sum to 1 over
the leaves of a tree): 8 * 16 * 2^-24 of the sum over trees of the largest leaf."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from ferrisboost_amd import _native as N

    if not N.device_available(0):
        pytest.fail("no gfx950 device: the GPU suite needs an MI355X")
    return N


def _ensemble(rng, n_trees, depth, nf, n_cat, full):
    """Flattened trees: nodes split with probability 1 (full) or 0.75; the last
    n_cat features categorical with 40 codes; the first tree a single leaf."""
    cols = {k: [] for k in ("feat", "cond", "left", "right", "dl", "leaf", "val", "hess", "coff",
                            "clen")}
    words, offs = [], [0]
    for t in range(n_trees):
        level, n, nodes = [(0, 1000.0)], 1, {}
        for d in range(depth + 1):
            nxt = []
            for i, cover in level:
                if d == depth or t == 0 or (not full and rng.random() > 0.75):
                    nodes[i] = (0, 0.0, -1, -1, 0, 1, rng.normal(), cover, 0, 0)
                    continue
                f = int(rng.integers(nf))
                share = rng.uniform(0.05, 0.95)
                coff = clen = 0
                if f >= nf - n_cat:
                    coff, clen = len(words), 2
                    words.extend(rng.integers(0, 2**32, 2, dtype=np.uint32).tolist())
                nodes[i] = (f, rng.normal(), n, n + 1, int(rng.integers(2)), 0, 0.0, cover, coff,
                            clen)
                nxt += [(n, cover * share), (n + 1, cover * (1.0 - share))]
                n += 2
            level = nxt
        for i in range(n):
            for k, v in zip(cols, nodes[i]):
                cols[k].append(v)
        offs.append(offs[-1] + n)
    kinds = {"feat": np.uint32, "cond": np.float32, "left": np.int32, "right": np.int32,
             "dl": np.uint8, "leaf": np.uint8, "val": np.float32, "hess": np.float32,
             "coff": np.uint32, "clen": np.uint32}
    a = {k: np.array(v, kinds[k]) for k, v in cols.items()}
    return np.array(offs, np.uint32), a, np.array(words + [0], np.uint32)


@pytest.mark.parametrize("rows,n_trees,depth,nf,n_cat,full", [
    (1, 1, 3, 4, 0, True),        # one row, nothing but a single-leaf tree
    (63, 2, 1, 1, 0, True),       # one split, one feature, a tile less a row
    (64, 9, 8, 3, 1, False),      # every path repeats features, one full tile
    (65, 17, 8, 40, 5, True),     # full depth, a row past a tile, a run past 8 x 2 trees
    (1000, 40, 7, 600, 100, False),  # the widest sums LDS holds
    (130, 5, 6, 601, 0, True),    # wider: the general kernel
    (130, 5, 9, 12, 0, True),     # deeper: the general kernel
])
def test_paths_match_the_host_order(lib, rows, n_trees, depth, nf, n_cat, full):
    N = lib
    rng = np.random.default_rng(rows + depth)
    offs, a, words = _ensemble(rng, n_trees, depth, nf, n_cat, full)
    x = rng.normal(size=(rows, nf)).astype(np.float32)
    if n_cat:  # codes, some past the sets, some negative
        x[:, nf - n_cat:] = rng.integers(-2, 80, (rows, n_cat))
    x[rng.random(x.shape) < 0.1] = np.nan
    margin = rng.normal(size=rows).astype(np.float32)
    h = C.c_void_p()
    N.check_hip(N.hip().fbh_shap_model_create(
        0, n_trees, N.ptr(offs), N.ptr(a["feat"]), N.ptr(a["cond"]), N.ptr(a["left"]),
        N.ptr(a["right"]), N.ptr(a["dl"]), N.ptr(a["leaf"]), N.ptr(a["val"]), N.ptr(a["hess"]),
        N.ptr(a["coff"]), N.ptr(a["clen"]), N.ptr(words), words.size, nf, 0.25, C.byref(h)))
    most = sum(float(np.abs(a["val"][b:e]).max()) for b, e in zip(offs[:-1], offs[1:]))
    tol = 8 * 16 * 2.0 ** -24 * most
    kinds = [("fbh_shap_contribs", (rows, nf + 1))]
    if nf <= 40:
        kinds.append(("fbh_shap_interactions", (rows, nf + 1, nf + 1)))
    try:
        for name, shape in kinds:
            for mg in (None, margin):
                got, want = np.full(shape, np.nan, np.float32), np.zeros(shape, np.float32)
                N.check_hip(N.hip().fbh_shap_set_host_order(h, 0))
                N.check_hip(getattr(N.hip(), name)(h, N.ptr(x), rows, N.ptr(mg), N.ptr(got)))
                N.check_hip(N.hip().fbh_shap_set_host_order(h, 1))
                N.check_hip(getattr(N.hip(), name)(h, N.ptr(x), rows, N.ptr(mg), N.ptr(want)))
                # an interaction line sums nf cells, the diagonal with them
                t = tol * (1 if len(shape) == 2 else nf)
                assert np.max(np.abs(got - want)) <= t, (name, np.max(np.abs(got - want)), t)
    finally:
        N.hip().fbh_shap_model_destroy(h)


@pytest.mark.parametrize("nan_threshold", [False, True])
def test_decisions_at_the_ends_of_the_order(lib, nan_threshold):
    """Cells and thresholds among zeros, infinities, denormals and NaN: the lane masks'
    decisions are the engine's (a NaN threshold takes its order whole). Tolerance as
    above."""
    N = lib
    rng = np.random.default_rng(3)
    rows, n_trees, nf = 200, 12, 9
    offs, a, words = _ensemble(rng, n_trees, 6, nf, 2, True)
    tiny, big = np.float32(1.4e-45), np.finfo(np.float32).max
    ends = np.array([0.0, -0.0, np.inf, -np.inf, tiny, -tiny, 1.17e-38, big, -big, 1.0, np.nan],
                    np.float32)
    a["cond"] = rng.choice(ends[:-1], a["cond"].size).astype(np.float32)
    if nan_threshold:
        a["cond"][np.flatnonzero((a["leaf"] == 0) & (a["clen"] == 0))[0]] = np.nan
    x = rng.choice(ends, (rows, nf)).astype(np.float32)
    h = C.c_void_p()
    N.check_hip(N.hip().fbh_shap_model_create(
        0, n_trees, N.ptr(offs), N.ptr(a["feat"]), N.ptr(a["cond"]), N.ptr(a["left"]),
        N.ptr(a["right"]), N.ptr(a["dl"]), N.ptr(a["leaf"]), N.ptr(a["val"]), N.ptr(a["hess"]),
        N.ptr(a["coff"]), N.ptr(a["clen"]), N.ptr(words), words.size, nf, 0.25, C.byref(h)))
    tol = 8 * 16 * 2.0 ** -24 * sum(float(np.abs(a["val"][b:e]).max())
                                    for b, e in zip(offs[:-1], offs[1:]))
    try:
        out = {}
        for order in (0, 1):
            out[order] = np.full((rows, nf + 1), np.nan, np.float32)
            N.check_hip(N.hip().fbh_shap_set_host_order(h, order))
            N.check_hip(N.hip().fbh_shap_contribs(h, N.ptr(x), rows, None, N.ptr(out[order])))
        assert np.max(np.abs(out[0] - out[1])) <= (0.0 if nan_threshold else tol)
    finally:
        N.hip().fbh_shap_model_destroy(h)


@pytest.mark.parametrize("share,fits", [(1e-3, True), (1e-5, True), (1e-6, False)])
def test_weights_near_the_range_of_a_float(lib, share, fits):
    """A path of eight splits on as many features that each pass `share` of the cover
    on, to leaves of value 0. The factors above its last split grow to 1e21, 1e35 and
    1e42; the last is beyond a float, and the model takes the engine's order, whose
    values it then has. The others stay finite and add up."""
    N = lib
    D = 8
    n = 2 * D + 1
    a = {"feat": np.zeros(n, np.uint32), "cond": np.zeros(n, np.float32),
         "left": np.full(n, -1, np.int32), "right": np.full(n, -1, np.int32),
         "dl": np.zeros(n, np.uint8), "leaf": np.ones(n, np.uint8),
         "val": np.full(n, 0.5, np.float32), "hess": np.zeros(n, np.float32)}
    at, a["hess"][0] = 0, 1e10
    for d in range(D):
        a["feat"][at], a["leaf"][at], a["val"][at] = d, 0, 0
        a["left"][at], a["right"][at] = 2 * d + 1, 2 * d + 2
        a["hess"][2 * d + 1] = a["hess"][at] * np.float32(share)
        a["hess"][2 * d + 2] = a["hess"][at]
        at = 2 * d + 1
    a["val"][2 * (D - 2) + 1:] = 0.0  # every leaf below the sixth split
    offs = np.array([0, n], np.uint32)
    h = C.c_void_p()
    N.check_hip(N.hip().fbh_shap_model_create(0, 1, N.ptr(offs), *(N.ptr(v) for v in a.values()),
                                              None, None, None, 0, D, 0.0, C.byref(h)))
    x = np.ones((65, D), np.float32)
    x[0] = -1.0        # down the whole path
    x[1, :7] = -1.0    # to its last right leaf
    x[2, ::2] = -1.0
    try:
        out = {}
        for order in (0, 1):
            out[order] = np.full((65, D + 1), np.nan, np.float32)
            N.check_hip(N.hip().fbh_shap_set_host_order(h, order))
            N.check_hip(N.hip().fbh_shap_contribs(h, N.ptr(x), 65, None, N.ptr(out[order])))
        if not fits:
            assert np.array_equal(out[0], out[1], equal_nan=True)
            return
        margin = np.zeros(65, np.float32)
        N.check_hip(N.hip().fbh_predict(h, N.ptr(x), 65, None, 0, N.ptr(margin)))
        # (the weights sum to 1 + share at each node, not to 1: rows add up to within
        # the covers' own error)
        assert np.isfinite(out[0]).all()
        assert np.max(np.abs(out[0].sum(1) - margin)) <= 16 * share + 8 * 16 * 2.0 ** -24
    finally:
        N.hip().fbh_shap_model_destroy(h)
