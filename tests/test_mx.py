"""The matrix-core count and fuse passes of fixed-threshold runs
(idb_mx.hip): their pair decision and features on the CPU against plain
definitions, and whole runs against the oracle at the edges of what they take
(thresholds, alphabets, row lengths around the word edges, buckets around the
tile edges), and just past them, where the general passes run."""
from __future__ import annotations

import os
import random
import subprocess
import tempfile

import numpy as np
import pytest

from immunodbscan_amd import configs, engine
from tests.test_gpu_parity import check, rep_from_rows

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("name", ["test_lvdist", "test_mxfeat"])
def test_host(name):
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "t")
        subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(ROOT, "tests", "cpp", name + ".cpp"), "-o", exe],
                       check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr


def clones(rng, n, letters, lo, hi, edits, genes=3, p_second=0.3, empty=0.01):
    """Rows in clones: copies of a seed with up to `edits` edits, lengths kept
    in [lo, hi]; one or two V genes, so that rows share several buckets."""
    rows = []
    while len(rows) < n:
        L = rng.choice([lo, hi, rng.randrange(lo, hi + 1)])
        seed = [rng.choice(letters) for _ in range(L)]
        v = rng.randrange(genes)
        for _ in range(rng.choice([1, 2, 5, 40])):
            s = list(seed)
            for _ in range(rng.randrange(edits + 1)):
                k = rng.randrange(3)
                if k == 0 and s:
                    s[rng.randrange(len(s))] = rng.choice(letters)
                elif k == 1 and len(s) < hi:
                    s.insert(rng.randrange(len(s) + 1), rng.choice(letters))
                elif len(s) > lo:
                    s.pop(rng.randrange(len(s)))
            vs = {v} | ({rng.randrange(genes)} if rng.random() < p_second else set())
            js = {rng.randrange(2)} if rng.random() < 0.1 else {0}
            rows.append((b"" if rng.random() < empty else bytes(s), sorted(vs), sorted(js)))
    rng.shuffle(rows)
    return rows[:n]


AA = b"ACDEFGHIKLMNPQRSTVWY"
LETTERS30 = bytes(range(65, 95))
CASES = (
    # protein form: 8 to 30 letters, up to 32 letters a row, t 0..3
    [(AA, 8, 25, t, 1500) for t in (0, 1, 2, 3)]
    + [(AA[:8], 1, 32, 2, 1200), (LETTERS30, 28, 32, 3, 1200), (AA, 32, 32, 1, 700), (AA, 1, 3, 2, 900)]
    # past it: 31 letters, t = 4, 33 letters
    + [(LETTERS30 + b"z", 10, 20, 2, 900), (AA, 8, 25, 4, 900), (AA, 20, 33, 2, 900)]
    # nucleotide form: rows of up to 256 letters in 1, 2, 3, 5 and 8 words, t 0..4
    + [(b"ACGT", 24, 150, t, 1500) for t in (0, 1, 2, 3, 4)]
    + [(b"ACGT", 1, 32, 3, 1200), (b"ACGT", 30, 64, 4, 1000), (b"ACGT", 63, 96, 3, 1000), (b"ACG", 127, 160, 2, 800),
       (b"ACGT", 190, 256, 3, 800), (b"ACGT", 255, 256, 4, 500), (b"A", 16, 40, 1, 200), (b"AC", 16, 33, 2, 600)]
    # past it: t = 5, rows under 16 letters
    + [(b"ACGT", 24, 100, 5, 800), (b"ACGT", 1, 15, 1, 800)]
)


@pytest.mark.gpu
@pytest.mark.parametrize("letters,lo,hi,t,n", CASES)
def test_fixed_thresholds(gpu_ctx, letters, lo, hi, t, n):
    rng = random.Random(1000 * t + lo + hi)
    rep = rep_from_rows(clones(rng, n, letters, lo, hi, t + 2))
    cl = configs.Clustering(eps=0.0, abs_k=t, min_pts=rng.choice([1, 2, 3]))
    got, _ = check(rep, cl, tag=f"{len(letters)} letters {lo}-{hi} t{t}")
    # the pair list far too short: the same tiles again, joined row by row
    small, _ = check(rep, cl, tag="fuse", edge_capacity=64)
    if got.stats["neighbour_pairs"] > 8192:
        assert small.stats["fuse_from_edges"] == 0


# buckets of 1, 63, 64, 65, 128 and 129 entries: full and ragged tiles, one row's genes in several buckets
@pytest.mark.gpu
@pytest.mark.parametrize("letters,lo,hi,t", [(AA, 10, 12, 2), (b"ACGT", 40, 42, 3)])
@pytest.mark.parametrize("size", [1, 2, 31, 32, 33, 63, 64, 65, 96, 97, 128, 129])
def test_tile_edges(gpu_ctx, letters, lo, hi, t, size):
    rng = random.Random(size)
    rows = []
    for v in range(3):
        for s, _, _ in clones(rng, size, letters, lo, hi, t + 1, empty=0):
            rows.append((s, [v] if rng.random() < 0.8 else sorted({v, (v + 1) % 3}), [0] if rng.random() < 0.9 else [0, 1]))
    check(rep_from_rows(rows), configs.Clustering(eps=0.0, abs_k=t, min_pts=2), tag=f"buckets of {size}")


@pytest.mark.gpu
def test_one_dense_clone_fills_every_batch(gpu_ctx):
    """Hundreds of rows within the threshold of each other: every pair of a
    tile passes, in tiles taken whole and in parts."""
    for letters, L, t in ((AA, 15, 2), (b"ACGT", 90, 3)):
        rng = random.Random(L)
        seed = [rng.choice(letters) for _ in range(L)]
        rows = []
        for _ in range(700):
            s = list(seed)
            s[rng.randrange(L)] = rng.choice(letters)
            if rng.random() < 0.3:
                s.pop(rng.randrange(len(s)))
            rows.append((bytes(s), [0], [0]))
        got, _ = check(rep_from_rows(rows), configs.Clustering(eps=0.0, abs_k=t, min_pts=4), tag=f"dense t{t}")
        assert got.stats["neighbour_pairs"] > 1000


@pytest.mark.gpu
def test_neighbour_pairs_name_rows(gpu_ctx):
    """The pair list holds entries; callers get rows."""
    from immunodbscan_amd import learned

    rng = random.Random(4)
    rep = rep_from_rows(clones(rng, 600, AA, 8, 20, 3))
    cl = configs.Clustering(eps=0.0, abs_k=2, min_pts=2)
    pairs = learned.neighbour_pairs(rep, cl)
    got = engine.dbscan(rep, cl)
    assert len(pairs) == got.stats["neighbour_pairs"] > 50
    assert (pairs[:, 0] < pairs[:, 1]).all() and len(np.unique(pairs, axis=0)) == len(pairs)
    counts = got.copies.astype(np.int64)
    np.add.at(counts, pairs[:, 0], got.copies[pairs[:, 1]])
    np.add.at(counts, pairs[:, 1], got.copies[pairs[:, 0]])
    assert np.array_equal(np.where(got.copies > 0, counts, 0), got.counts)
