"""The general Myers count pass with tiles taken in parts of their queries
(few tiles), and cluster growth over dense and sparse pair lists: buckets
around the tile and part edges, against the oracle."""
from __future__ import annotations

import random

import numpy as np
import pytest

from immunodbscan_amd import configs, synth
from tests.test_gpu_parity import check, rep_from_rows


def _rows(sizes, letters, L, edits, seed):
    """One bucket per size: mutated copies of one seed row per bucket."""
    rng = random.Random(seed)
    rows = []
    for g, n in enumerate(sizes):
        seed_row = [rng.choice(letters) for _ in range(L)]
        for _ in range(n):
            s = list(seed_row)
            for _ in range(rng.randrange(edits + 1)):
                k = rng.randrange(len(s))
                s[k] = rng.choice(letters)
                if rng.random() < 0.2:
                    s.pop(k)
            rows.append((bytes(s), [g % 30], [g // 30]))
    rng.shuffle(rows)
    return rows


@pytest.mark.gpu
@pytest.mark.parametrize("letters,L", [(b"ACGT", 60), (b"ACGT", 150), (b"ACDEFGHIKLMNPQRSTVWY", 40), (b"ABC", 12)])
@pytest.mark.parametrize("sizes", [(1, 7, 8, 9, 15, 16, 17), (31, 32, 33, 63, 64, 65), (57, 56, 128, 129, 200)])
def test_parts_of_tiles(gpu_ctx, letters, L, sizes):
    rep = rep_from_rows(_rows(sizes, letters, L, max(2, L // 8), 5 + len(sizes)))
    check(rep, configs.Clustering(eps=0.15, abs_k=-1, min_pts=2, use_hamming=False), ctx=gpu_ctx)


@pytest.mark.gpu
@pytest.mark.parametrize("n,eps", [(2400, 0.3), (2400, 0.05)])
def test_growth_over_dense_and_sparse_lists(gpu_ctx, n, eps):
    """One bucket of large clones: hundreds of pairs per row at the larger
    threshold, a few at the smaller one."""
    rep = rep_from_rows(_rows((n // 2, n // 2), b"ACGT", 45, 6, 9))
    check(rep, configs.Clustering(eps=eps, abs_k=-1, min_pts=3, use_hamming=True), ctx=gpu_ctx)
