"""Calls of one model that share its kept device models and buffers: sizes on both
sides of the page-locked, staged and threaded paths, tree ranges, threads at once,
and the reserved value in a large input. Every result equals the host's scoring bit
for bit."""

from __future__ import annotations

import os
import sys
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(__file__))
from helpers import product_params  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def trained():
    import ferrisboost_amd as fb

    if not fb.device_available(0):
        pytest.fail("no gfx950 device: the GPU suite needs an MI355X")
    rng = np.random.default_rng(5)
    x = rng.normal(size=(9_000, 31)).astype(np.float32)
    x[rng.random(x.shape) < 0.05] = np.nan
    y = (np.nan_to_num(x[:, 0]) + np.nan_to_num(x[:, 1]) > 0).astype(np.float32)
    return fb.train(product_params({"max_depth": 5, "eta": 0.3}), x, y, num_boost_round=12), x


@pytest.mark.parametrize("rows", [1, 2_000, 2_048, 2_200, 9_000, 40_000])
def test_sizes_and_tree_ranges(trained, rows):
    m, x = trained
    x = np.ascontiguousarray(np.resize(x, (rows, x.shape[1])))
    for r in (None, (0, 5), (3, 12), (7, 7)):
        kw = {} if r is None else {"iteration_range": r}
        for _ in range(2):  # a new device model, then the kept one
            got = m.predict(x, **kw)
            assert np.array_equal(got.view(np.uint32),
                                  m.predict(x, use_gpu=False, **kw).view(np.uint32)), r


def test_threads_at_once(trained):
    m, x = trained
    want = {n: m.predict(x[:n], use_gpu=False, output_margin=True) for n in (7, 500, 9_000)}
    phi = {n: m.predict(x[:n], pred_contribs=True) for n in want}

    def call(i):
        n = (7, 500, 9_000)[i % 3]
        if i % 2:
            return np.array_equal(m.predict(x[:n], output_margin=True), want[n])
        return np.array_equal(m.predict(x[:n], pred_contribs=True), phi[n])

    with ThreadPoolExecutor(6) as ex:
        assert all(ex.map(call, range(48)))


@pytest.mark.parametrize("rows", [10, 9_000, 40_000])
def test_a_reserved_value_is_an_error(trained, rows):
    m, x = trained
    x = np.resize(x, (rows, x.shape[1])).copy()
    x[-1, -1] = np.finfo(np.float32).max
    with pytest.raises(ValueError, match="largest float32"):
        m.predict(x)
