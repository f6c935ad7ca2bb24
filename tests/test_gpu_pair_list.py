"""The neighbour-pair list of a requested capacity: what it holds, and that a
short one costs the count pass nothing."""
from __future__ import annotations

import numpy as np
import pytest

from immunodbscan_amd import configs, engine, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name,rep,cl", [
    ("hamming", lambda: configs.c1_params(150_000, 15_000, 3), configs.C1),
    ("protein", lambda: configs.c2_params(200_000, 20_000, 3), configs.C2),
    ("long", lambda: configs.c5_params(60_000, 300, 3), configs.C5),
])
def test_short_list_leaves_the_count_pass_its_grid(gpu_ctx, name, rep, cl):
    """Past the list's capacity only the growth changes (its second pass): the
    same results, and a count pass that still fills the chip.  On a grid cut to the
    list it took 20 to 300 times as long as with the default list; the claims
    of every wave make it 2 to 4 times."""
    rep = synth.generate(rep())

    def best(cap):
        runs = [engine.dbscan(rep, cl, edge_capacity=cap) for _ in range(5)]
        return runs[0], min(r.stats["count_kernel_ms"] for r in runs)

    full, t_full = best(0)
    assert full.stats["fuse_from_edges"] == 1
    for cap in (64, 256, 2048, 4096, 16384):
        got, t = best(cap)
        print(f"{name} capacity {cap}: {t * 1e3:.0f} us against {t_full * 1e3:.0f}", flush=True)
        for k in ("clone_id", "core", "copies", "uniques", "counts"):
            assert np.array_equal(getattr(got, k), getattr(full, k)), (cap, k)
        assert got.stats["fuse_from_edges"] == 0
        assert t < 8 * t_full, cap


def pairs_of(ctx, rep, cl, capacity):
    import ctypes as C

    from immunodbscan_amd import _lib

    cap = 1 << 20
    out = np.zeros((cap, 2), np.uint32)
    n = C.c_uint64()
    ctx.check(_lib.lib.idb_neighbour_pairs(ctx.handle, engine._dataset(rep),
                                           engine._params(cl, False, 0, edge_capacity=capacity), out.ctypes.data, cap,
                                           C.byref(n)))
    pairs = out[: n.value]
    return pairs[np.lexsort((pairs[:, 1], pairs[:, 0]))]


RELATIVE = configs.Clustering(eps=0.15, abs_k=-1, min_pts=2, use_hamming=False)


@pytest.mark.parametrize("rep,cl,factor", [
    (lambda: configs.c1_params(60, 6, 5), RELATIVE, 2.0),
    (lambda: configs.c1_params(700, 70, 5), RELATIVE, 2.0),
    (lambda: configs.c1_params(6_000, 600, 5), RELATIVE, 2.0),
    (lambda: configs.c1_params(6_000, 600, 5), configs.C1, 2.0),
    (lambda: configs.c2_params(6_000, 600, 5), configs.C2, 2.0),
    (lambda: configs.c5_params(300, 1, 5), configs.C5, 1.25),
])
def test_neighbour_pairs_within_the_capacity(gpu_ctx, rep, cl, factor):
    """A list of some more pairs than there are holds them, however few of them
    each wave finds; a list of fewer is refused."""
    from immunodbscan_amd import _lib

    rep = synth.generate(rep())
    want = pairs_of(gpu_ctx, rep, cl, 0)
    assert len(want) > 64
    assert np.array_equal(pairs_of(gpu_ctx, rep, cl, int(factor * len(want)) + 1), want)
    with pytest.raises(_lib.IdbError, match="raise edge_capacity"):
        pairs_of(gpu_ctx, rep, cl, len(want) // 2)
    with pytest.raises(_lib.IdbError, match="raise edge_capacity"):
        pairs_of(gpu_ctx, rep, cl, 64)
