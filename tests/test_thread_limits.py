"""Calls that would use threads where no thread can be made (here: no address space for
another stack) do the work on the caller's."""

from __future__ import annotations

import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_host_scoring_without_threads():
    """Three million cells are looked through for reserved values by threads; without
    them the margins are the same and a reserved value is still an error."""
    script = textwrap.dedent("""
        import resource, sys, threading
        import numpy as np
        sys.path[:0] = [%r, %r]
        import ferrisboost_amd as fb
        from ferrisboost_amd import _native as N
        from test_model_io import XGB_DUMP

        m = fb.Model.from_json(XGB_DUMP)
        nf, n = m.n_features, 3_000_000 // m.n_features
        x = np.random.default_rng(0).normal(size=(n, nf)).astype(np.float32)
        L, out, want = N.train_lib(), np.zeros(n, np.float32), np.zeros(n, np.float32)
        call = lambda o, x=x: L.fbt_predict(m._h, N.ptr(x), len(x), nf, N.OUT_MARGIN, 0,
                                            m.num_trees, None, -1, N.ptr(o))
        step = (1 << 17) // nf  # few enough cells for no thread (whose stack would be kept)
        for b in range(0, n, step):
            N.check_train(call(want[b:b + step], x[b:b + step]))
        now = next(int(s.split()[1]) for s in open("/proc/self/status") if s.startswith("VmSize"))
        resource.setrlimit(resource.RLIMIT_AS, (now * 1024 + (2 << 20), resource.RLIM_INFINITY))
        try:
            threading.Thread(target=int).start()
            print("a thread was made")
        except RuntimeError:
            pass
        N.check_train(call(out))
        assert np.array_equal(out, want)
        x[-1, -1] = np.finfo(np.float32).max
        try:
            N.check_train(call(out))
            raise SystemExit("accepted")
        except ValueError as e:
            assert "largest float32" in str(e)
        print("ok")
    """ % (ROOT, os.path.join(ROOT, "tests")))
    got = subprocess.run([sys.executable, "-c", script], capture_output=True, text=True,
                         timeout=120, env=dict(os.environ, MALLOC_ARENA_MAX="1"))
    assert got.stdout.strip() == "ok", got.stdout + got.stderr
