"""Rows uploaded once and kept on the device for the binning against rows uploaded
twice (a memory budget keeps none) and against host sketch and binning: the same
models, at sizes on both sides of the piped upload and of the row packing's blocks."""

from __future__ import annotations

import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(__file__))
from helpers import product_params  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fb():
    import ferrisboost_amd as fb

    if not fb.device_available(0):
        pytest.fail("no gfx950 device: the GPU suite needs an MI355X")
    return fb


@pytest.mark.parametrize("rows,nf,n_cat,max_bin", [
    (1, 3, 0, 16),            # one row
    (255, 28, 0, 255),        # a packing block less a row, one bundle of two tiles
    (257, 41, 2, 300),        # a row past a block, planar 16-bit and interleaved tiles
    (1000, 5, 1, 64),         # one planar tile without a bundle
    (1_060_000, 64, 0, 256),  # 271 MB: the piped upload, its last piece short
])
def test_kept_rows_give_the_same_model(fb, rows, nf, n_cat, max_bin):
    rng = np.random.default_rng(rows + nf)
    x = rng.normal(size=(rows, nf)).astype(np.float32)
    if n_cat:
        x[:, nf - n_cat:] = rng.integers(0, 9, (rows, n_cat))
    if max_bin != 256:
        x[rng.random(x.shape) < 0.05] = np.nan
    y = (np.nan_to_num(x[:, 0]) > 0).astype(np.float32)
    p = product_params({"max_depth": 3, "max_bin": max_bin, "eta": 0.3})
    if n_cat:
        p["feature_types"] = ["q"] * (nf - n_cat) + ["c"] * n_cat
    want = fb.train(dict(p, gpu_memory_budget=64 << 30), x, y, num_boost_round=2)
    others = [{}]
    if rows <= 1000:
        others.append({"hip_host_sketch": True, "hip_host_binning": True})
    for extra in others:
        got = fb.train(dict(p, **extra), x, y, num_boost_round=2)
        assert got.to_json() == want.to_json(), extra
        assert np.array_equal(got.train_margins(rows), want.train_margins(rows))
