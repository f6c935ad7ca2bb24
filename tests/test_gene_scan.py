"""The multi-name automaton behind idb_gene_bitsets_gpu: its table on the CPU
against a plain search of every name, and its kernel against the oracle at
both table widths, both output forms and around the long-string cut."""
from __future__ import annotations

import os
import random
import subprocess
import tempfile

import numpy as np
import pytest

from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_gene_table_against_plain_search():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "t")
        subprocess.run(["g++", "-O1", "-fsanitize=address,undefined", "-std=c++17",
                        os.path.join(ROOT, "tests", "cpp", "test_gene_table.cpp"), "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True)
        assert r.returncode == 0, r.stdout + r.stderr


def word(rng, letters, lo, hi):
    return bytes(rng.choice(letters) for _ in range(rng.randrange(lo, hi + 1)))


# names, shortest and longest name, letters: 16-bit tables (bit words in
# registers and in memory), then 32-bit tables (more than 32,768 entries)
@pytest.mark.gpu
@pytest.mark.parametrize("n_names,lo,hi,letters", [(1, 1, 1, b"AB"), (33, 1, 6, b"ABC"), (128, 1, 9, b"ACGT"),
                                                   (129, 2, 9, b"ACGT"), (700, 3, 12, b"ACGT"),
                                                   (128, 20, 40, b"ABCDEFGHIJ"),
                                                   (900, 4, 8, bytes(range(60, 90)))])
def test_gene_scan_forms(gpu_ctx, n_names, lo, hi, letters):
    from immunodbscan_amd.interlink import gene_bitsets_gpu

    rng = random.Random(n_names)
    names = [word(rng, letters, lo, hi) for _ in range(n_names)]
    names[-1] = names[0]
    calls = []
    for i in range(12000):
        L = rng.choice([0, 1, 15, 16, 17, 31, 32, 33, rng.randrange(0, 100)])
        c = bytearray(word(rng, letters, L, L))
        for _ in range(rng.randrange(0, 3)):
            c += rng.choice(names) + b"-"
        calls.append(bytes(c))
    for L in (2047, 2048, 2049, 2050, 4096, 5000):
        c = bytearray(b"~" * L)
        for _ in range(12):
            g = rng.choice(names)
            if len(g) <= L:
                p = rng.randrange(0, L - len(g) + 1)
                c[p:p + len(g)] = g
        calls.insert(rng.randrange(len(calls)), bytes(c))
    got, _ = gene_bitsets_gpu(calls, names)
    assert np.array_equal(got, O.gene_bitsets(calls, names))
