"""Workloads of the training and scoring paths, through the package's public entry points.

Three kinds of case, which are what a program does with a boosted-tree library:

  train    fb.train on a host matrix: the whole job (sketch, binning, rounds, model and
           training margins back). Timed whole, since a user waits for all of it.
  predict  margins, values or leaf ids of new rows, either Model.predict on host arrays
           (a service or a batch job) or fbh_predict_device on resident buffers (a
           pipeline whose features are already in device memory).
  shap     TreeSHAP contributions or interactions, again on host arrays or in place.

The explained and scored ensembles are synthetic (drawn from the seed, nearly complete
trees with the odd early leaf, skewed feature use, thresholds inside the range that the
path leaves open, covers that fit the data), so the 64-bit results need nothing of this
package.
"""

from __future__ import annotations

import ctypes as C
import json
import math

import numpy as np
import torch

import ferrisboost_amd as fb
from ferrisboost_amd import _native as N

DEV = "cuda:0"
# The most work of exact(): rows x trees x leaves x quadrature points of one SHAP case.
EXACT_SHAP_MOST = 2.5e10


# --------------------------------------------------------------------- cases
def _train(name, **kw):
    c = {"name": name, "kind": "train", "rows": 0, "features": 0, "cats": 0, "codes": 0,
         "nan": 0.0, "max_bin": 255, "objective": "binary:logistic", "classes": 0, "depth": 6,
         "rounds": 10, "grow": "depthwise", "leaves": 0, "subsample": 1.0, "colsample": 1.0,
         "given_cuts": False}
    c.update(kw)
    return c


def _score(name, kind, **kw):
    c = {"name": name, "kind": kind, "rows": 0, "features": 0, "cats": 0, "codes": 0, "nan": 0.0,
         "trees": 100, "depth": 6, "device": False, "output": "value"}
    c.update(kw)
    return c


def listed():
    return [
        # A request to a scoring service: a few rows on a small model. Launches, copies and
        # host work are all there is.
        _score("serve_64", "predict", rows=64, features=28, trees=100, depth=6),
        # A batch job that scores a table with categories and missing values from host memory.
        _score("predict_batch", "predict", rows=200_000, features=50, cats=6, codes=40, nan=0.05,
               trees=300, depth=6),
        # The prediction workload of bench.py (1M x 200, 100 trees of depth 8) with the rows
        # already on the device, as a pipeline has them.
        _score("predict_resident", "predict", rows=1_000_000, features=200, trees=100, depth=8,
               device=True, output="margin"),
        # The explanation workload of bench.py (200 features, 100 trees of depth 8), resident.
        _score("shap_resident", "shap", rows=100_000, features=200, trees=100, depth=8,
               device=True, output="contribs"),
        # A report over a table in host memory: smaller trees, categories, missing values.
        _score("shap_batch", "shap", rows=20_000, features=28, cats=4, codes=30, nan=0.05,
               trees=300, depth=6, output="contribs"),
        # Interactions of a sample of rows, which is how they are used: the output is
        # quadratic in the features.
        _score("interactions", "shap", rows=2_000, features=28, trees=100, depth=6,
               output="interactions"),
        # A small table, as in a search over parameters or a test: rounds are a few launches
        # on nearly nothing.
        _train("train_small", rows=5_000, features=20, rounds=50, nan=0.02),
        # 100k x 28, 100 rounds of depth 6 at max_bin 256: the smallest of the configurations.
        _train("train_100k", rows=100_000, features=28, max_bin=256, rounds=100),
        # The headline configuration: 10.5M x 28 at max_bin 255, depth 8, from raw floats.
        _train("train_narrow", rows=10_500_000, features=28, depth=8, rounds=100),
        # The wide configuration: 400k x 2000, half the columns sampled for each tree.
        _train("train_wide", rows=400_000, features=2000, max_bin=256, depth=8, rounds=40,
               colsample=0.5),
        # The wide-bin configuration: 80 numeric columns with 10 % missing and 20 categorical
        # ones of 500 codes, 1024 bins, best-first trees of 255 leaves, squared error.
        _train("train_widebin", rows=2_000_000, features=100, cats=20, codes=500, nan=0.1,
               max_bin=1024, objective="reg:squarederror", grow="lossguide", leaves=255,
               rounds=40),
        # Several models over one matrix with its cuts kept, with four classes and the
        # customary row and column sampling.
        _train("train_classes", rows=500_000, features=28, objective="multi:softprob", classes=4,
               rounds=25, subsample=0.8, colsample=0.8, given_cuts=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["train", "train", "predict", "shap"])
    if kind == "train":
        objective = rng.choice(["binary:logistic", "reg:squarederror", "multi:softprob"])
        features = _log_int(rng, 5, 400)
        cats = rng.choice([0, 0, min(features // 4, 12)])
        max_bin = rng.choice([64, 255, 256, 512])
        c = dict(rows=_log_int(rng, 1_000, min(3_000_000, 300_000_000 // features)),
                 features=features, cats=cats, codes=rng.randrange(5, 200) if cats else 0,
                 nan=rng.choice([0.0, 0.03, 0.2]), max_bin=max_bin, objective=objective,
                 classes=rng.randrange(3, 6) if objective.startswith("multi") else 0,
                 depth=rng.randrange(3, 9), rounds=rng.randrange(10, 31),
                 subsample=rng.choice([1.0, 1.0, 0.7]), colsample=rng.choice([1.0, 1.0, 0.6]))
        if rng.random() < 0.3:
            c.update(grow="lossguide", leaves=rng.randrange(8, 256))
        c = _train("", **c)
    else:
        features = _log_int(rng, 5, 300)
        cats = rng.choice([0, 0, features // 4])
        c = dict(features=features, cats=cats, codes=rng.randrange(3, 64) if cats else 0,
                 nan=rng.choice([0.0, 0.05, 0.3]), depth=rng.randrange(3, 9),
                 trees=_log_int(rng, 20, 400), device=rng.random() < 0.5)
        if kind == "predict":
            c.update(rows=_log_int(rng, 1, 1_000_000),
                     output=rng.choice(["value", "margin", "leaf"]))
            if c["output"] == "leaf":
                c["rows"] = min(c["rows"], 100_000)
        else:
            c.update(rows=_log_int(rng, 1, 60_000), output="contribs")
            if not c["device"] and features <= 40 and rng.random() < 0.5:
                c.update(rows=min(c["rows"], 3_000), output="interactions")
        c = _score("", kind, **c)
    del c["name"]
    return c


# -------------------------------------------------------------------- inputs
def _rows(case, seed):
    """The feature matrix on the device: standard normals, every third numeric column made
    heavy-tailed, Zipf codes in the last `cats` columns, missing values in the numeric ones."""
    n, nf, nc = case["rows"], case["features"], case["cats"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn((n, nf), generator=g, device=DEV, dtype=torch.float32)
    if case["kind"] == "train":
        x[:, 2:nf - nc:3] = torch.exp(0.5 * x[:, 2:nf - nc:3])
    if case["nan"] > 0.0:
        for f in range(nf - nc):
            x[torch.rand(n, generator=g, device=DEV) < case["nan"], f] = float("nan")
    if nc:
        p = torch.arange(1, case["codes"] + 1, device=DEV, dtype=torch.float64) ** -1.2
        cdf = torch.cumsum(p / p.sum(), 0)
        for f in range(nf - nc, nf):
            u = torch.rand(n, generator=g, device=DEV, dtype=torch.float64)
            x[:, f] = torch.searchsorted(cdf, u).clamp_(max=case["codes"] - 1).float()
    return x


def _labels(case, x, seed):
    """Labels of a nonlinear score of the first columns and of every fourth category code."""
    n, nf, nc = case["rows"], case["features"], case["cats"]
    g = torch.Generator(device=DEV).manual_seed(seed + 7919)
    k = max(1, min(nf - nc, 40))
    w = torch.randn(k, generator=g, device=DEV)
    z = torch.zeros(n, device=DEV)
    for f in range(k):
        z += w[f] * torch.nan_to_num(x[:, f], nan=0.5)
    if k > 3:
        z += 0.8 * torch.nan_to_num(x[:, 0]) * torch.nan_to_num(x[:, 3])
    for f in range(nf - nc, nf):
        z += torch.randn(case["codes"], generator=g, device=DEV)[x[:, f].long()]
    z = (z - z.mean()) / z.std()
    if case["objective"] == "reg:squarederror":
        return z + 0.1 * torch.randn(n, generator=g, device=DEV)
    if case["objective"] == "binary:logistic":
        return (torch.rand(n, generator=g, device=DEV) < torch.sigmoid(1.5 * z)).float()
    z = z + 0.3 * torch.randn(n, generator=g, device=DEV)
    order = torch.argsort(z)
    y = torch.empty(n, device=DEV)
    y[order] = torch.floor(torch.arange(n, device=DEV, dtype=torch.float64)
                           * case["classes"] / n).float()
    return y


def _normal_quantile(u):
    t = torch.from_numpy(np.clip(u, 1e-6, 1.0 - 1e-6))
    return torch.special.ndtri(t).numpy().astype(np.float32)


def _ensemble(case, seed):
    """A list of trees (dicts of node arrays) on normal columns and Zipf codes: level by
    level, each node splits with probability 0.97 (always above level 3), on a feature of
    skewed popularity, at 20 to 80 % of the mass its path leaves open."""
    nt, depth, nf, nc = case["trees"], case["depth"], case["features"], case["cats"]
    r = np.random.default_rng(seed)
    pop = 1.0 / (1.0 + np.arange(nf)) ** 0.5
    pop = r.permutation(pop / pop.sum())
    codes = case["codes"]
    mass = np.arange(1, codes + 1, dtype=np.float64) ** -1.2 if nc else np.zeros(0)
    mass /= max(mass.sum(), 1e-30)
    trees = []
    for _ in range(nt):
        most = 2 ** (depth + 1) - 1
        t = {"feat": np.zeros(most, np.uint32), "cond": np.zeros(most, np.float32),
             "left": np.full(most, -1, np.int32), "right": np.full(most, -1, np.int32),
             "dl": np.zeros(most, np.uint8), "leaf": np.ones(most, np.uint8),
             "value": np.zeros(most, np.float32), "hess": np.zeros(most, np.float32),
             "cats": {}}
        # the open nodes of a level: id, cover, and (feature, low, high) of the path
        ids, cover, paths = [0], [1.0], [{}]
        count = 1
        for d in range(depth):
            k = len(ids)
            split = r.random(k) < (1.0 if d < 3 else 0.97)
            feats = r.choice(nf, size=k, p=pop)
            share = r.uniform(0.2, 0.8, k)
            dl = r.random(k) < 0.5
            nids, ncover, npaths, cut_at, cut_u = [], [], [], [], []
            for i in range(k):
                if not split[i]:
                    continue
                f, u, me = int(feats[i]), float(share[i]), ids[i]
                t["leaf"][me] = 0
                t["feat"][me] = f
                t["dl"][me] = dl[i]
                t["left"][me], t["right"][me] = count, count + 1
                if f >= nf - nc:
                    goes_right = r.random(codes) < u
                    goes_right[int(r.integers(codes))] = True
                    t["cats"][me] = np.flatnonzero(goes_right).astype(np.int64)
                    frac = float(np.clip(1.0 - mass[goes_right].sum(), 0.02, 0.98))
                    lp = rp = paths[i]
                else:
                    lo, hi = paths[i].get(f, (0.0, 1.0))
                    mid = lo + u * (hi - lo)
                    cut_at.append(me)
                    cut_u.append(mid)
                    frac = u
                    lp, rp = dict(paths[i]), dict(paths[i])
                    lp[f], rp[f] = (lo, mid), (mid, hi)
                nids += [count, count + 1]
                ncover += [cover[i] * frac, cover[i] * (1.0 - frac)]
                npaths += [lp, rp]
                count += 2
            if cut_at:
                t["cond"][cut_at] = _normal_quantile(np.array(cut_u))
            for i in range(k):
                t["hess"][ids[i]] = 2.0e5 * cover[i]
            ids, cover, paths = nids, ncover, npaths
        for i in range(len(ids)):
            t["hess"][ids[i]] = 2.0e5 * cover[i]
        t["value"][:] = np.where(t["leaf"] == 1, r.normal(0.0, 0.05, most), 0.0)
        for key, a in t.items():
            if key != "cats":
                t[key] = a[:count]
        trees.append(t)
    return trees


BASE_SCORE = 0.5  # the margin 0 of binary:logistic


def _model_json(case, trees):
    nf, nc = case["features"], case["cats"]
    out = []
    for i, t in enumerate(trees):
        n = t["feat"].size
        leaf = t["leaf"] == 1
        seg, sizes, cats = [], [], []
        for k in sorted(t["cats"]):
            seg.append(len(cats))
            sizes.append(int(t["cats"][k].size))
            cats += t["cats"][k].tolist()
        stype = np.zeros(n, np.int64)
        stype[sorted(t["cats"])] = 1
        out.append({
            "base_weights": [0.0] * n, "categories": cats, "categories_nodes": sorted(t["cats"]),
            "categories_segments": seg, "categories_sizes": sizes,
            "default_left": t["dl"].tolist(), "id": i, "left_children": t["left"].tolist(),
            "loss_changes": [0.0] * n, "parents": [2147483647] * n,
            "right_children": t["right"].tolist(),
            "split_conditions": np.where(leaf, t["value"], t["cond"]).astype(float).tolist(),
            "split_indices": t["feat"].tolist(), "split_type": stype.tolist(),
            "sum_hessian": t["hess"].astype(float).tolist(),
            "tree_param": {"num_deleted": "0", "num_feature": str(nf), "num_nodes": str(n),
                           "size_leaf_vector": "1"}})
    return json.dumps({"version": [2, 0, 0], "learner": {
        "attributes": {}, "feature_names": [],
        "feature_types": ["q"] * (nf - nc) + ["c"] * nc if nc else [],
        "gradient_booster": {"name": "gbtree", "model": {
            "gbtree_model_param": {"num_trees": str(len(out)), "num_parallel_tree": "1"},
            "iteration_indptr": list(range(len(out) + 1)), "tree_info": [0] * len(out),
            "trees": out}},
        "learner_model_param": {"base_score": str(BASE_SCORE), "boost_from_average": "1",
                                "num_class": "0", "num_feature": str(nf), "num_target": "1"},
        "objective": {"name": "binary:logistic",
                      "reg_loss_param": {"scale_pos_weight": "1"}}}})


class _DeviceModel:
    """The C ABI's explanation and prediction model of an ensemble."""

    def __init__(self, case, trees):
        a = {k: np.ascontiguousarray(np.concatenate([t[k] for t in trees]))
             for k in ("feat", "cond", "left", "right", "dl", "leaf", "value", "hess")}
        offs = np.concatenate([[0], np.cumsum([t["feat"].size for t in trees])]).astype(np.uint32)
        coff, clen = np.zeros(offs[-1], np.uint32), np.zeros(offs[-1], np.uint32)
        words = []
        for t, b in zip(trees, offs):
            for k, codes in sorted(t["cats"].items()):
                w = np.zeros(int(codes.max()) // 32 + 1, np.uint32)
                np.bitwise_or.at(w, codes // 32, np.uint32(1) << (codes % 32).astype(np.uint32))
                coff[b + k], clen[b + k] = sum(x.size for x in words), w.size
                words.append(w)
        w = np.concatenate(words) if words else np.zeros(0, np.uint32)
        self.h = C.c_void_p()
        N.check_hip(N.hip().fbh_shap_model_create(
            0, len(trees), N.ptr(offs), N.ptr(a["feat"]), N.ptr(a["cond"]), N.ptr(a["left"]),
            N.ptr(a["right"]), N.ptr(a["dl"]), N.ptr(a["leaf"]), N.ptr(a["value"]),
            N.ptr(a["hess"]), N.ptr(coff), N.ptr(clen), N.ptr(w), int(w.size), case["features"],
            0.0, C.byref(self.h)))

    def __del__(self):
        if self.h:
            N.hip().fbh_shap_model_destroy(self.h)
            self.h = None


def prepare(case, seed):
    x = _rows(case, seed)
    if case["kind"] == "train":
        y = _labels(case, x, seed).cpu().numpy()
        X = x.cpu().numpy()
        params = {"objective": case["objective"], "max_depth": case["depth"], "eta": 0.1,
                  "max_bin": case["max_bin"], "grow_policy": case["grow"], "device": "cuda:0",
                  "max_leaves": case["leaves"], "subsample": case["subsample"],
                  "colsample_bytree": case["colsample"], "seed": 1}
        if case["classes"]:
            params["num_class"] = case["classes"]
        types = None
        if case["cats"]:
            types = ["q"] * (case["features"] - case["cats"]) + ["c"] * case["cats"]
        cuts = fb.sketch(X, case["max_bin"], feature_types=types) if case["given_cuts"] else None
        return {"case": case, "X": X, "y": y, "params": params, "types": types, "cuts": cuts}
    trees = _ensemble(case, seed)
    if case["device"]:
        width = {"leaf": case["trees"], "contribs": case["features"] + 1}.get(case["output"], 0)
        shape = (case["rows"], width) if width else (case["rows"],)
        return {"case": case, "x": x, "model": _DeviceModel(case, trees),
                "out": torch.empty(shape, device=DEV, dtype=torch.float32)}
    return {"case": case, "X": x.cpu().numpy(),
            "model": fb.Model.from_json(_model_json(case, trees), device="cuda:0")}


# --------------------------------------------------------------------- calls
def _filled(a, size):
    out = np.zeros(size, a.dtype)
    out[: a.size] = a
    return out


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        m = fb.train(state["params"], state["X"], state["y"], num_boost_round=case["rounds"],
                     feature_types=state["types"], cuts=state["cuts"])
        nodes = np.concatenate(m.trees())
        values, offsets = m.cuts()
        # filled up with zeros to the most a model of these parameters can hold
        most = 2 ** (case["depth"] + 1) - 1
        if case["leaves"]:
            most = min(most, 2 * case["leaves"] - 1)
        most *= case["rounds"] * max(1, case["classes"])
        return {"nodes": _filled(nodes.view(np.uint8), most * nodes.itemsize),
                "cats": _filled(m.cat_words(), most * (case["codes"] // 32 + 2) if case["cats"]
                                else 0),
                "cuts": _filled(values, case["features"] * max(case["max_bin"], case["codes"])),
                "cut_offsets": offsets, "margins": m.train_margins(case["rows"])}
    if case["device"]:
        x, out, h = state["x"], state["out"], state["model"].h
        if case["kind"] == "shap":
            N.check_hip(N.hip().fbh_shap_contribs_device(h, x.data_ptr(), case["rows"], None,
                                                         out.data_ptr(), 1))
        else:
            kind = {"margin": 0, "value": 1, "leaf": 2}[case["output"]]
            N.check_hip(N.hip().fbh_predict_device(h, x.data_ptr(), case["rows"], None, kind,
                                                   out.data_ptr(), 1))
        return out
    how = {"value": {}, "margin": {"output_margin": True}, "leaf": {"pred_leaf": True},
           "contribs": {"pred_contribs": True}, "interactions": {"pred_interactions": True}}
    return state["model"].predict(state["X"], **how[case["output"]])


# ------------------------------------------------------------ work, tolerance
def work(case):
    n, nf = case["rows"], case["features"]
    if case["kind"] == "train":
        # the matrix, the labels and the margins once; each round every row's cells of the
        # tree's features, its label and its margin (read and written) for each output
        outputs = max(1, case["classes"])
        cell = 1 if case["max_bin"] <= 256 else 2
        per_round = n * case["subsample"] * nf * case["colsample"] * cell + 12.0 * n
        return {"bytes": 4.0 * n * (nf + 2) + case["rounds"] * outputs * per_round,
                # two additions for each cell of a tree, once
                "flops": 2.0 * n * nf * case["subsample"] * case["colsample"] * case["rounds"]
                * outputs}
    nodes = case["trees"] * (2.0 ** (case["depth"] + 1) - 1)
    out = {"leaf": case["trees"], "contribs": nf + 1, "interactions": (nf + 1) ** 2}
    moved = 4.0 * n * (nf + out.get(case["output"], 1)) + 16.0 * nodes
    if case["kind"] == "predict":
        return {"bytes": moved, "flops": 1.0 * n * case["trees"] * case["depth"]}
    # every decision of a tree counts for a row's contributions, not only those on its path
    pairs = case["depth"] if case["output"] == "interactions" else 1
    return {"bytes": moved, "flops": 1.0 * n * nodes / 2 * pairs}


def tolerance(case):
    if case["kind"] == "train" or case["output"] == "leaf":
        return "exact"  # trees are sums of whole numbers; margins follow from them
    if case["kind"] == "predict":
        return {"rel": 8e-7}  # f32 sums of the trees' leaves: 0.6 to 1.8e-7 measured
    return {"rel": 3e-6}  # f32 products and sums along every path: 2.0 to 7.5e-7 measured


# ---------------------------------------------------------------------- exact
def _decisions(t, x):
    """goes-left of every (row, split node) of a tree; the split nodes' ids."""
    at = np.flatnonzero(t["leaf"] == 0)
    f = torch.from_numpy(t["feat"][at].astype(np.int64)).to(x.device)
    v = x[:, f]
    cond = torch.from_numpy(t["cond"][at]).to(x.device)
    dl = torch.from_numpy(t["dl"][at].astype(bool)).to(x.device)
    left = v < cond
    for j, i in enumerate(at):
        if int(i) in t["cats"]:
            right = torch.zeros(1 << 12, dtype=torch.bool, device=x.device)
            right[torch.from_numpy(t["cats"][int(i)]).to(x.device)] = True
            left[:, j] = ~right[torch.nan_to_num(v[:, j]).long()]
    return torch.where(torch.isnan(v), dl[None, :], left), at


def _exact_predict(case, trees, x):
    n = case["rows"]
    m = torch.zeros(n, dtype=torch.float64, device=x.device)
    leaf = torch.zeros((n, len(trees)), dtype=torch.float64, device=x.device)
    for k, t in enumerate(trees):
        for b in range(0, n, 1 << 17):
            e = min(n, b + (1 << 17))
            gl, at = _decisions(t, x[b:e])
            col = np.full(t["feat"].size, 0, np.int64)
            col[at] = np.arange(at.size)
            col = torch.from_numpy(col).to(x.device)
            L = torch.from_numpy(t["left"].astype(np.int64)).to(x.device)
            R = torch.from_numpy(t["right"].astype(np.int64)).to(x.device)
            is_leaf = torch.from_numpy(t["leaf"] == 1).to(x.device)
            node = torch.zeros(e - b, dtype=torch.int64, device=x.device)
            for _ in range(case["depth"]):
                go = torch.gather(gl, 1, col[node][:, None])[:, 0]
                node = torch.where(is_leaf[node], node, torch.where(go, L[node], R[node]))
            leaf[b:e, k] = node.double()
            m[b:e] += torch.from_numpy(t["value"]).to(x.device).double()[node]
    if case["output"] == "leaf":
        return leaf
    return torch.sigmoid(m) if case["output"] == "value" else m


def _paths(t):
    """Each leaf's path as (node, went left) pairs."""
    out, stack = [], [(0, [])]
    while stack:
        i, p = stack.pop()
        if t["leaf"][i]:
            out.append((i, p))
        else:
            stack.append((int(t["left"][i]), p + [(i, True)]))
            stack.append((int(t["right"][i]), p + [(i, False)]))
    return out


def _exact_shap(case, trees, x, pairs):
    n, nf, dev = case["rows"], case["features"], x.device
    nc = nf + 1
    s, w = np.polynomial.legendre.leggauss(8)
    q = torch.from_numpy(0.5 * (s + 1.0)).to(dev)
    w = torch.from_numpy(0.5 * w).to(dev)
    phi = torch.zeros((n, nc), dtype=torch.float64, device=dev)
    inter = torch.zeros((n, nc * nc), dtype=torch.float64, device=dev) if pairs else None
    chunk = 256 if pairs else 2048
    for t in trees:
        col = np.zeros(t["feat"].size, np.int64)
        at = np.flatnonzero(t["leaf"] == 0)
        col[at] = np.arange(at.size)
        paths = _paths(t)
        D, nl = case["depth"], len(paths)
        feat = np.full((nl, D), nf, np.int64)   # unused slots: weight 1, always met
        z = np.ones((nl, D))
        step_col, step_left = np.zeros((nl, D), np.int64), np.zeros((nl, D), bool)
        step_slot, step_on = np.zeros((nl, D), np.int64), np.zeros((nl, D), bool)
        val = np.zeros(nl)
        for i, (node, p) in enumerate(paths):
            val[i] = t["value"][node]
            slots = {}
            for k, (j, went_left) in enumerate(p):
                f = int(t["feat"][j])
                a = slots.setdefault(f, len(slots))
                feat[i, a] = f
                c = int(t["left"][j] if went_left else t["right"][j])
                z[i, a] *= float(t["hess"][c]) / float(t["hess"][j])
                step_col[i, k], step_left[i, k] = col[j], went_left
                step_slot[i, k], step_on[i, k] = a, True
        z, val, featd = (torch.from_numpy(a).to(dev) for a in (z, val, feat))
        step_left, step_on, step_slot, step_col = (torch.from_numpy(a).to(dev) for a in
                                                   (step_left, step_on, step_slot, step_col))
        phi[:, nf] += (val * z.prod(1)).sum()
        for b in range(0, n, chunk):
            e = min(n, b + chunk)
            gl, _ = _decisions(t, x[b:e])
            met = torch.ones((e - b, nl, D), dtype=torch.bool, device=dev)
            for k in range(D):
                ok = (gl[:, step_col[:, k]] == step_left[None, :, k]) | ~step_on[None, :, k]
                idx = step_slot[:, k][None, :, None].expand(e - b, nl, 1)
                met.scatter_(2, idx, met.gather(2, idx) & ok[:, :, None])
            one = met.double()
            prod = torch.ones((e - b, nl, 8), dtype=torch.float64, device=dev)
            for a in range(D):
                prod *= z[None, :, a, None] + (one[:, :, a] - z[None, :, a])[:, :, None] * q
            delta = one - z[None]
            for a in range(D):
                fa = z[None, :, a, None] + delta[:, :, a, None] * q
                rest = prod / fa
                got = val[None] * delta[:, :, a] * (rest * w).sum(2)
                phi[b:e].index_add_(1, featd[:, a], got)
                if not pairs:
                    continue
                for c in range(a + 1, D):
                    fc = z[None, :, c, None] + delta[:, :, c, None] * q
                    both = 0.5 * val[None] * delta[:, :, a] * delta[:, :, c] * (rest / fc * w).sum(2)
                    inter[b:e].index_add_(1, featd[:, a] * nc + featd[:, c], both)
                    inter[b:e].index_add_(1, featd[:, c] * nc + featd[:, a], both)
    if not pairs:
        return phi
    inter = inter.reshape(n, nc, nc)
    d = torch.arange(nf, device=dev)
    inter[:, d, d] = 0.0
    inter[:, nf, :] = 0.0
    inter[:, :, nf] = 0.0
    inter[:, d, d] = phi[:, :nf] - inter.sum(2)[:, :nf]
    inter[:, nf, nf] = phi[:, nf]
    return inter


def exact(case, seed):
    if case["kind"] == "train":
        return None  # trees of fixed-point sums have no 64-bit value to compare with
    x = _rows(case, seed)
    trees = _ensemble(case, seed)
    if case["kind"] == "predict":
        return _exact_predict(case, trees, x)
    pairs = case["output"] == "interactions"
    load = case["rows"] * case["trees"] * 2.0 ** case["depth"] * 8 * (case["depth"] if pairs else 1)
    return None if load > EXACT_SHAP_MOST else _exact_shap(case, trees, x, pairs)
