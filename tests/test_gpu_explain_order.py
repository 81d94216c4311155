"""TreeSHAP of one model takes one arithmetic, whatever the call's row count: the
engine's order (bit for bit the oracle's values; the default of several outputs, and
engine_order=True) or the closed sums (engine_order=False), for single-output, class
and quantile models on both sides of a 64-row tile and above 512 rows.

Tolerance of the sums: 8 * 16 * 2^-24 of the trees' largest leaves, as in
test_gpu_shap_paths.py; an interaction's diagonal sums its line."""

from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ROWS = 700


@pytest.fixture(scope="module")
def models(oracle):
    import ferrisboost_amd as fb
    from ferrisboost_amd import _native as N

    if not N.device_available(0):
        pytest.fail("no gfx950 device: the GPU suite needs an MI355X")
    rng = np.random.default_rng(17)
    x = rng.normal(size=(3_000, 7)).astype(np.float32)
    x[rng.random(x.shape) < 0.05] = np.nan
    z = np.nan_to_num(x[:, 0]) + np.nan_to_num(x[:, 1] * x[:, 2])
    labels = {"single": (z > 0), "classes": np.digitize(z, [-0.5, 0.5]), "quantiles": z}
    params = {"single": {"objective": "binary:logistic"},
              "classes": {"objective": "multi:softprob", "num_class": 3},
              "quantiles": {"objective": "reg:quantileerror", "quantile_alpha": [0.2, 0.5, 0.8]}}
    out = {}
    for name, p in params.items():
        m = fb.train(dict(p, max_depth=5, eta=0.3), x, labels[name].astype(np.float32),
                     num_boost_round=4)
        k = m.num_class
        trees = m.trees()
        bias = m.class_margins() if k > 1 else [m.base_margin]
        oms = [oracle.model_from_nodes(trees[c::k], np.zeros(0, np.uint32), "reg:squarederror",
                                       float(bias[c])) for c in range(k)]
        most = max(sum(float(np.abs(t["leaf_value"]).max()) for t in trees[c::k])
                   for c in range(k))
        out[name] = (m, oms, 8 * 16 * 2.0 ** -24 * most)
    return x[:ROWS], out


def _call(m, x, kind, order):
    got = m.predict(x, **{"pred_" + kind: True}, engine_order=order)
    return got if m.num_class > 1 else got[:, None]


@pytest.mark.parametrize("name", ["single", "classes", "quantiles"])
@pytest.mark.parametrize("kind", ["contribs", "interactions"])
def test_values_of_each_order(models, name, kind):
    x, all_models = models
    m, oms, tol = all_models[name]
    want = np.stack([om.explain(x, kind) for om in oms], axis=1)
    engine, sums, default = (_call(m, x, kind, o) for o in (True, False, None))
    assert np.array_equal(engine.view(np.uint32), want.view(np.uint32))
    assert np.max(np.abs(sums - want)) <= tol * (1 if kind == "contribs" else x.shape[1])
    assert not np.array_equal(sums, engine)
    chosen = sums if name == "single" else engine
    assert np.array_equal(default.view(np.uint32), chosen.view(np.uint32))


@pytest.mark.parametrize("name", ["single", "classes", "quantiles"])
@pytest.mark.parametrize("kind", ["contribs", "interactions"])
@pytest.mark.parametrize("order", [None, True, False])
def test_a_row_has_one_value_in_any_batch(models, name, kind, order):
    x, all_models = models
    m = all_models[name][0]
    whole = _call(m, x, kind, order)
    for n in (1, 63, 64, 65, 511, 512, 513):
        part = _call(m, x[:n], kind, order)
        assert np.array_equal(part.view(np.uint32), whole[:n].view(np.uint32)), n


def test_the_order_applies_to_treeshap_alone(models):
    x, all_models = models
    m = all_models["single"][0]
    for kw in ({}, {"output_margin": True}, {"pred_leaf": True},
               {"pred_contribs": True, "approx_contribs": True}):
        with pytest.raises(ValueError, match="engine_order"):
            m.predict(x, engine_order=True, **kw)


@pytest.mark.parametrize("nf,rows", [(1, 3), (63, 64), (64, 65), (255, 64), (256, 9), (319, 64),
                                     (320, 64), (500, 40), (500, 41)])
def test_wide_rows_on_both_sides_of_the_copies(nf, rows):
    """Contributions of rows read over the link and of rows copied first (160 KiB of 64
    rows in and out is where they part): the same bits as in a batch of 700."""
    import ferrisboost_amd as fb

    rng = np.random.default_rng(nf)
    x = rng.normal(size=(ROWS, nf)).astype(np.float32)
    m = fb.train({"max_depth": 4, "objective": "reg:squarederror"}, x, x[:, 0] * x[:, -1],
                 num_boost_round=5)
    whole = m.predict(x, pred_contribs=True)
    part = m.predict(x[:rows], pred_contribs=True)
    assert np.array_equal(part.view(np.uint32), whole[:rows].view(np.uint32))
