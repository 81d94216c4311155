"""Jobs on memory and streams that earlier jobs have left against jobs on fresh
ones: the same models and predictions, from one thread and from two at once; what is
kept is bounded, goes back on request and is not held beside a memory budget."""

from __future__ import annotations

import os
import sys
import threading

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.dirname(__file__))
from helpers import product_params  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def fb():
    import ferrisboost_amd as fb

    if not fb.device_available(0):
        pytest.fail("no gfx950 device: the GPU suite needs an MI355X")
    return fb


def release():
    from ferrisboost_amd import _native as N

    N.check_hip(N.hip().fbh_release_cached(0))


def free_bytes():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def job(fb, seed, rows, nf, n_cat=0, **params):
    rng = np.random.default_rng(seed)
    x = rng.normal(size=(rows, nf)).astype(np.float32)
    x[rng.random(x.shape) < 0.05] = np.nan
    if n_cat:
        x[:, nf - n_cat:] = rng.integers(0, 40, (rows, n_cat))
    y = np.nan_to_num(x[:, 0] * x[:, 1 % nf])
    y = np.digitize(y, [-0.3, 0.3]).astype(np.float32) if "num_class" in params else \
        (y > 0).astype(np.float32)
    p = product_params({"max_depth": 5, "eta": 0.3, **params})
    if n_cat:
        p["feature_types"] = ["q"] * (nf - n_cat) + ["c"] * n_cat
    m = fb.train(p, x, y, num_boost_round=4)
    return m.to_json(), m.train_margins(rows).tobytes(), m.predict(x).tobytes(), \
        m.predict(x[:50], pred_contribs=True).tobytes()


CASES = [
    dict(rows=1, nf=3),
    dict(rows=4099, nf=28, max_bin=255),
    dict(rows=30_011, nf=60, max_bin=256, colsample_bytree=0.4, subsample=0.7),
    dict(rows=20_003, nf=24, n_cat=6, max_bin=600, grow_policy="lossguide", max_leaves=20),
    dict(rows=9_001, nf=17, objective="multi:softprob", num_class=3),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c['rows']}x{c['nf']}")
def test_job_on_kept_memory_equals_job_on_fresh_memory(fb, case):
    release()
    want = job(fb, 5, **case)
    for other in (6, 7):  # leave their contents in the blocks that the next job takes
        job(fb, other, **case)
        assert job(fb, 5, **case) == want


def test_two_threads(fb):
    want = {s: job(fb, s, **CASES[1]) for s in (1, 2)}
    got, errors = {}, []

    def work(s):
        try:
            got[s] = [job(fb, s, **CASES[1]) for _ in range(5)]
        except Exception as e:  # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors
    for s in (1, 2):
        assert all(g == want[s] for g in got[s])


def test_kept_memory_is_bounded_and_goes_back(fb):
    big = dict(rows=400_000, nf=40)
    release()
    job(fb, 1, **big)
    release()
    before = free_bytes()
    job(fb, 1, **big)
    total = torch.cuda.mem_get_info()[1]
    assert 0 < before - free_bytes() <= total // 16 + (64 << 20)
    release()
    assert abs(before - free_bytes()) <= 64 << 20
    # a job under a memory budget keeps nothing and clears what others kept
    job(fb, 1, **big)
    assert before - free_bytes() > 64 << 20
    rng = np.random.default_rng(0)
    x = rng.normal(size=(400_000, 40)).astype(np.float32)
    y = (x[:, 0] > 0).astype(np.float32)
    fb.train(product_params({"max_depth": 3, "gpu_memory_budget": 8 << 30}), x, y, num_boost_round=1)
    assert abs(before - free_bytes()) <= 64 << 20
