"""Device models on both sides of the size from which their records are made on
threads and sent array by array: predictions, contributions and leaf ids agree with
the trees walked on the host, and a model refused by one kernel's records still serves
the others."""

from __future__ import annotations

import pytest

from test_gpu_predict_tiles import test_margins_and_leaf_ids as check_margins
from test_gpu_shap_paths import lib, test_paths_match_the_host_order as check_paths  # noqa: F401

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,n_trees,depth,nf,n_cat", [
    (70, 128, 8, 30, 4),     # 64,897 nodes and a single leaf: one thread
    (70, 130, 8, 30, 4),     # past 65,536: records made beside the copies
    (70, 20, 12, 12, 2),     # deeper than the sums take: prediction's records alone
])
def test_records(lib, rows, n_trees, depth, nf, n_cat):  # noqa: F811
    check_margins(lib, rows, n_trees, depth, nf, n_cat, True)
    check_paths(lib, rows, n_trees, depth, nf, n_cat, True)


def test_two_threads_make_models_at_once(lib):  # noqa: F811
    from concurrent.futures import ThreadPoolExecutor

    with ThreadPoolExecutor(3) as ex:
        for f in [ex.submit(check_margins, lib, 65 + k, 130, 8, 20, 3, True) for k in range(6)]:
            f.result()
