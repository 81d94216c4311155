"""bench.py's operation counts: the VALU counts are those of the committed counter
summaries of the kernels that run, and the arithmetic of TreeSHAP is counted node by
node."""

from __future__ import annotations

import os
import re
import sys

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def _text(name):
    with open(os.path.join(ROOT, "profiles", name)) as f:
        return f.read()


def test_valu_counts_are_the_profiles():
    shap = _text("shap_kernel.md")
    assert float(re.search(r"\*\*([\d.]+)M\*\*, the\s+figure `bench.py`", shap).group(1)) * 1e6 == \
        bench.SHAP_VALU_OPS_PER_ROW
    row = next(line for line in shap.splitlines() if line.startswith("| VALU instructions |"))
    total = sum(int(c.replace(",", "")) for c in row.split("|")[2:5])
    assert abs(total * 64 / 55_872 / bench.SHAP_VALU_OPS_PER_ROW - 1) < 1e-3
    pred = _text("predict_kernel.md")
    got = re.search(r"\*\*([\d,]+)\*\*, the figure `bench.py`", pred).group(1)
    assert float(got.replace(",", "")) == bench.PREDICT_VALU_OPS_PER_ROW
    n = int(re.search(r"VALU instructions \(wave\) \| ([\d,]+) \|", pred).group(1).replace(",", ""))
    assert abs(n * 64 / 664_576 / bench.PREDICT_VALU_OPS_PER_ROW - 1) < 1e-3


def test_rooflines_stay_below_the_peak():
    # the rates of the committed lines
    import json

    lines = [json.loads(x) for x in re.findall(r"```json\n(\{.*?\})\n```", _text("bench_workloads.md"))]
    fracs = [ln["roofline"].get(k) for ln in lines for k in ("frac", "valu_frac", "hbm_frac")]
    assert len(lines) > 10 and all(0 < f < 1 for f in fracs if f is not None)


def test_shap_flops():
    class Model:
        def __init__(self, *trees):
            self.t = trees

        def trees(self):
            return self.t

    def tree(left, right):
        t = np.zeros(len(left), [("left", np.int32), ("right", np.int32), ("is_leaf", np.uint8)])
        t["left"], t["right"] = left, right
        t["is_leaf"] = np.array(left) < 0
        return t

    stump = tree([1, -1, -1], [2, -1, -1])
    chain = tree([1, 3, -1, -1, -1], [2, 4, -1, -1, -1])
    full = tree([1, 3, 5, -1, -1, -1, -1], [2, 4, 6, -1, -1, -1, -1])
    leaf = tree([-1], [-1])
    two = 3 + 2 * 4 + 4  # a node of two leaves
    assert bench.shap_flops_per_row(Model(leaf)) == 0
    assert bench.shap_flops_per_row(Model(stump)) == two
    assert bench.shap_flops_per_row(Model(chain)) == 24 + 16 + 3 + two
    assert bench.shap_flops_per_row(Model(full, stump)) == 48 + 16 + 3 + 2 * two + two
