"""The autotuner keeps a shape per kernel: runs of one shape class that go to
different kernels are each tuned."""
from __future__ import annotations

import time

import numpy as np
import pytest

from immunodbscan_amd import _lib, configs, engine, synth

pytestmark = pytest.mark.gpu


def test_fixed_thresholds_of_two_kernels_are_tuned_apart(gpu_ctx):
    """Thresholds 4 (the general pass) and 3 (the matrix-core pass) on the same
    rows and about as many tiles: the second kernel's first tuned run times its
    own shapes (48 extra count passes), its second one does not."""
    rep = synth.generate(configs.c2_params(200_000, 20_000, 11))
    ctx = _lib.Context(0)
    plain = {}
    for k in (4, 3):  # every buffer is there before the first timed run
        cl = configs.Clustering(eps=0.0, abs_k=k, min_pts=3)
        plain[k] = engine.dbscan(rep, cl, ctx=ctx)
    tiles = [plain[k].stats["tiles"].bit_length() for k in (4, 3)]
    assert tiles[0] == tiles[1]

    def run(k):
        cl = configs.Clustering(eps=0.0, abs_k=k, min_pts=3)
        t0 = time.perf_counter()
        got = engine.dbscan(rep, cl, ctx=ctx, flags=_lib.IDB_FLAG_AUTOTUNE)
        dt = time.perf_counter() - t0
        for f in ("clone_id", "core", "copies", "uniques", "counts"):
            assert np.array_equal(getattr(got, f), getattr(plain[k], f)), (k, f)
        assert got.stats["tuned_trials"] == 24
        return dt

    run(4)
    again4 = run(4)
    first3, again3 = run(3), run(3)
    print(f"threshold 4 again {again4 * 1e3:.2f} ms; threshold 3 first {first3 * 1e3:.2f}, again {again3 * 1e3:.2f}")
    # 48 count passes of at least 60 us each come on top
    assert first3 > again3 + 0.0025
    ctx.close()
