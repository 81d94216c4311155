"""Device models between calls: what models that are alive leave on the device goes
back on request and before a job with a memory budget; models of many outputs find
theirs again; calls give the same values throughout."""

from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

SLACK = 64 << 20  # the driver's own bookkeeping


@pytest.fixture(scope="module")
def fb():
    import ferrisboost_amd as fb

    if not fb.device_available(0):
        pytest.fail("no gfx950 device: the GPU suite needs an MI355X")
    return fb


def _free():
    torch.cuda.synchronize()
    return torch.cuda.mem_get_info()[0]


def _model(fb, n_class=1, rows=20_000, nf=30):
    rng = np.random.default_rng(n_class)
    x = rng.normal(size=(rows, nf)).astype(np.float32)
    y = x[:, 0] + 0.3 * rng.normal(size=rows)
    p = {"max_depth": 5, "objective": "reg:squarederror"}
    if n_class > 1:
        y = np.digitize(y, np.quantile(y, np.linspace(0, 1, n_class + 1)[1:-1]))
        p.update(objective="multi:softprob", num_class=n_class)
    return fb.train(p, x, y.astype(np.float32), num_boost_round=3), x


def test_memory_goes_back_with_models_alive(fb):
    single, x = _model(fb)
    classes, _ = _model(fb, 4)
    wide = np.tile(x, (8, 1))
    fb.release_cached()
    before = _free()
    want = None
    for _ in range(2):
        got = [single.predict(wide), single.predict(wide, pred_contribs=True),
               classes.predict(wide),
               classes.predict(x, pred_contribs=True, engine_order=False)]
        got += [single.predict(wide, iteration_range=(b, e)) for b in range(3)
                for e in range(b + 1, 4)]
        if want is not None:  # on models made again
            assert all(np.array_equal(a, b) for a, b in zip(want, got))
        want = got
        assert before - _free() > 32 << 20  # staging and workspaces wait for the next call
        fb.release_cached()
        assert before - _free() <= SLACK
    # a job with a memory budget finds nothing beside it
    single.predict(wide, pred_contribs=True)
    assert before - _free() > 32 << 20
    fb.train({"max_depth": 2, "gpu_memory_budget": 4 << 30, "objective": "reg:squarederror"}, x,
             x[:, 0], num_boost_round=1)
    assert before - _free() <= SLACK
    assert np.array_equal(single.predict(wide), want[0])


def test_ten_classes(fb):
    m, x = _model(fb, 10)
    for n in (5, 3_000):
        want = m.predict(x[:n], use_gpu=False, output_margin=True)
        first = m.predict(x[:n], pred_contribs=True)
        for _ in range(3):
            got = m.predict(x[:n], output_margin=True)
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
            assert np.array_equal(m.predict(x[:n], pred_contribs=True), first)


def _tiny(N, value):
    """A device model of one leaf."""
    h = C.c_void_p()
    a = {k: np.array([v], t) for k, v, t in (
        ("feat", 0, np.uint32), ("cond", 0, np.float32), ("left", -1, np.int32),
        ("right", -1, np.int32), ("dl", 0, np.uint8), ("leaf", 1, np.uint8),
        ("val", value, np.float32), ("hess", 1, np.float32))}
    offs = np.array([0, 1], np.uint32)
    N.check_hip(N.hip().fbh_shap_model_create(
        0, 1, N.ptr(offs), *(N.ptr(v) for v in a.values()), None, None, None, 0, 3, 0.0,
        C.byref(h)))
    return h


def test_parked_models_are_found_by_owner_and_name(fb):
    from ferrisboost_amd import _native as N

    L = N.hip()
    mine, other = 1 << 63, (1 << 63) + 1  # no model's own numbers

    def take(owner, trees, output):
        h = C.c_void_p()
        N.check_hip(L.fbh_shap_model_unpark(0, owner, trees, output, C.byref(h)))
        return h

    for k in range(40):
        N.check_hip(L.fbh_shap_model_park(_tiny(N, float(k)), mine, 7, k))
    assert not take(mine, 8, 3) and not take(other, 7, 3) and not take(mine, 7, 40)
    x = np.zeros((2, 3), np.float32)
    for _ in range(2):  # in turn, as a model of 40 outputs is scored
        for k in range(40):
            h = take(mine, 7, k)
            out = np.zeros(2, np.float32)
            N.check_hip(L.fbh_predict(h, N.ptr(x), 2, None, 0, N.ptr(out)))
            assert out.tolist() == [k, k]
            N.check_hip(L.fbh_shap_model_park(h, mine, 7, k))
    N.check_hip(L.fbh_shap_models_drop(mine))
    assert not take(mine, 7, 0)
