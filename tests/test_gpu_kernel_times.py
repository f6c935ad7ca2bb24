"""The kernel times that a run reports are the kernels' own."""
from __future__ import annotations

import pytest

from immunodbscan_amd import configs, engine, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rep,cl", [(lambda: configs.c2_params(200_000, 20_000, 3), configs.C2),
                                    (lambda: configs.c1_params(200_000, 20_000, 3), configs.C1)])
def test_count_time_does_not_depend_on_where_the_rows_are(gpu_ctx, rep, cl):
    """The same count pass over rows and outputs in host memory and in HBM: host
    outputs are prepared and sent while the run goes on, which is no part of the
    kernel (it added 25 to 30 us)."""
    rep = synth.generate(rep())
    host, dev = engine.HostRun(rep, cl), engine.DeviceRun(rep, cl)
    count, fuse = [], []
    for run in (host, dev):
        st = [run() and (run.stats.count_kernel_ms, run.stats.fuse_kernel_ms, run.stats.stage_ms[3]) for _ in range(20)]
        count.append(min(s[0] for s in st))
        fuse.append(min(s[1] for s in st))
        assert all(0 < s[0] < s[2] and s[1] > 0 for s in st)  # within the core-point stage
    print(f"count {count[0] * 1e3:.0f} / {count[1] * 1e3:.0f} us, growth {fuse[0] * 1e3:.0f} / {fuse[1] * 1e3:.0f}")
    assert abs(count[0] - count[1]) < 0.012
    assert abs(fuse[0] - fuse[1]) < 0.012
