"""The matrix-core passes with tiles taken whole, in halves and in quarters,
count and fuse: small tables are always taken in parts, so these have the
tiles for each form.  The general passes (the allocation-free entry point runs
them, the other tests hold them to the oracle) give the expected results."""
from __future__ import annotations

import random

import numpy as np
import pytest

from immunodbscan_amd import _lib, configs, engine
from tests.test_gpu_parity import rep_from_rows
from tests.test_mx import AA
from tests.test_zz_no_alloc import noalloc

pytestmark = pytest.mark.gpu


def one_bucket(n, letters, length, seed):
    """n different rows of length - 1 to length + 1 letters under one gene pair,
    in clones of a few and of some hundred rows."""
    rng = random.Random(seed)
    rows = set()
    while len(rows) < n:
        clone = [rng.choice(letters) for _ in range(length)]
        for _ in range(rng.choice([1, 3, 20, 300])):
            s = list(clone)
            for _ in range(rng.randrange(4)):
                s[rng.randrange(len(s))] = rng.choice(letters)
            if rng.random() < 0.2:
                s.pop(rng.randrange(len(s)))
            elif rng.random() < 0.2:
                s.insert(rng.randrange(len(s)), rng.choice(letters))
            rows.add(bytes(s))
    rows = sorted(rows)[:n]
    rng.shuffle(rows)
    return rep_from_rows([(r, [0], [0]) for r in rows])


# of 6,144 resident waves (protein form) half are filled by the parts, of 4,096
# (nucleotide form) twice as many: quarters up to 768 and 2,048 tiles, halves up
# to 1,536 and 4,096
@pytest.mark.parametrize("letters,length,t,n,tiles", [
    (AA, 15, 2, 2_400, (600, 768)), (AA, 15, 2, 3_200, (800, 1_536)), (AA, 15, 2, 4_600, (1_700, 3_000)),
    (AA, 24, 3, 4_601, (1_700, 3_000)),
    (b"ACGT", 80, 3, 3_000, (600, 2_048)), (b"ACGT", 80, 3, 5_000, (2_100, 4_096)), (b"ACGT", 80, 3, 7_003, (4_500, 8_000)),
    (b"ACGT", 30, 2, 7_040, (4_500, 8_000))])
def test_whole_tiles_and_parts(gpu_ctx, letters, length, t, n, tiles):
    rep = one_bucket(n, letters, length, n + t)
    cl = configs.Clustering(eps=0.0, abs_k=t, min_pts=3)
    rc, want, st = noalloc(rep, cl, gpu_ctx)
    assert rc == _lib.IDB_OK, gpu_ctx.last_error()
    assert tiles[0] <= st["tiles"] <= tiles[1]
    print(f"case {len(letters)} letters of {length}, t {t}: {n} rows, {st['tiles']} tiles, {st['neighbour_pairs']} pairs",
          flush=True)
    for cap in (0, 64):
        got = engine.dbscan(rep, cl, edge_capacity=cap)
        # one chunk of 64 pairs: the fuse pass over the same tiles
        assert st["neighbour_pairs"] > 64 and got.stats["fuse_from_edges"] == (cap == 0)
        for k in ("clone_id", "core", "copies", "uniques", "counts"):
            assert np.array_equal(getattr(got, k), want[k]), (cap, k)
        for k in ("n_cores", "n_clusters", "n_noise", "neighbour_pairs", "gated_pairs", "gated_letters"):
            assert got.stats[k] == st[k], (cap, k)
