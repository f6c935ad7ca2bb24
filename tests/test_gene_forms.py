"""The gene scan's forms at the edges of what they take, each case checked to
run the form that it is meant for (tests/cpp/gene_form.cpp applies the same
rule to the same names)."""
from __future__ import annotations

import os
import random
import subprocess

import numpy as np
import pytest

from oracle import oracle as O

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def form_of(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("genes") / "gene_form")
    subprocess.run(["g++", "-O1", "-std=c++17", os.path.join(ROOT, "tests", "cpp", "gene_form.cpp"), "-o", exe],
                   check=True)

    def form(n_calls, names):
        r = subprocess.run([exe], input=b"%d %d\n" % (n_calls, len(names)) + b"".join(n + b"\n" for n in names),
                           capture_output=True, check=True)
        kind, entries, lds = r.stdout.split()
        return kind.decode(), int(entries), int(lds)

    return form


def test_reach_of_tables(tmp_path):
    exe = str(tmp_path / "reach")
    subprocess.run(["g++", "-O1", "-fsanitize=address,undefined", "-std=c++17",
                    os.path.join(ROOT, "tests", "cpp", "test_gene_reach.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe, os.path.join(ROOT, "tests", "golden")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr


def names_with(rng, k, letters, states):
    """k names over the letters whose automaton has exactly `states` states."""
    prefixes, names = {b""}, []
    for left in range(k, 0, -1):
        room = states - len(prefixes)
        n = bytes(rng.choice(letters) for _ in range(min(room, room // left + 4)))
        names.append(n or rng.choice(names))  # (no room: a name twice)
        prefixes |= {n[:i] for i in range(1, len(n) + 1)}
    while len(prefixes) < states:  # the first name, letter by letter
        names[0] += rng.choice(letters).to_bytes(1, "little")
        prefixes.add(names[0])
    assert len(prefixes) == states
    return names


def calls_of(rng, n, names, letters):
    calls = []
    for _ in range(n):
        c = bytes(rng.choice(letters) for _ in range(rng.choice([0, 1, 15, 16, 17, 40])))
        for _ in range(rng.randrange(0, 3)):
            c += rng.choice(names) + b"-"
        calls.append(c)
    for L in (2047, 2048, 2049, 5000):
        c = bytearray(b"~" * L)
        for _ in range(12):
            g = rng.choice(names)
            p = rng.randrange(0, L - len(g) + 1)
            c[p:p + len(g)] = g
        calls[rng.randrange(n)] = bytes(c)
    return calls


LETTERS = b"ABCDEFGHIJ"  # table rows of 12 entries
# names, states, calls, form, LDS of a block: the largest 16-bit tables (64 KB
# of LDS are passed at 32,384 entries for 128 names), and 32-bit ones, for bit
# words in registers (at most 128 names) and in memory
FORMS = [(128, 2698, 12000, "16", 65520), (128, 2699, 12000, "16", 65544), (128, 2730, 12000, "16", 66288),
         (600, 2730, 3000, "16", 68176), (128, 2731, 16000, "32", 256), (128, 3600, 16000, "32", 256),
         (300, 2731, 3000, "32", 256)]


def test_forms_are_the_ones_named(form_of):
    for k, states, n, kind, lds in FORMS:
        rng = random.Random(k + states)
        got = form_of(n, names_with(rng, k, LETTERS, states))
        assert got == (kind, 12 * states, lds), (k, states)


@pytest.mark.gpu
@pytest.mark.parametrize("k,states,n,kind,lds", FORMS)
def test_forms(gpu_ctx, form_of, k, states, n, kind, lds):
    from immunodbscan_amd.interlink import gene_bitsets_gpu

    rng = random.Random(k + states)
    names = names_with(rng, k, LETTERS, states)
    assert form_of(n, names)[0] == kind
    calls = calls_of(rng, n, names, LETTERS)
    print(f"case genes {kind} bit, {k} names, {states} states, {lds} bytes of LDS", flush=True)
    got, _ = gene_bitsets_gpu(calls, names)
    assert np.array_equal(got, O.gene_bitsets(calls, names))


@pytest.mark.gpu
def test_names_that_cannot_match_cost_no_walk(gpu_ctx):
    """Only empty and too long names: no bits, and no pass over long calls (the
    walk with every lane started at its string's first byte took 59 ms)."""
    import time

    from immunodbscan_amd.interlink import gene_bitsets_gpu

    names = [b""] * 20 + [b"x" * 1100] * 20
    calls = [b"x" * 6000] * 1000
    best = 1e9
    for _ in range(4):
        t0 = time.perf_counter()
        got, _ = gene_bitsets_gpu(calls, names)
        best = min(best, time.perf_counter() - t0)
    assert got.shape == (1000, 2) and not got.any()
    assert best < 0.03  # with 6 MB of calls packed and copied


AB = b"ABCDEFGHIJKLMNOPQRSTUVWXYZ"


def arrays_of(calls, names, width):
    from immunodbscan_amd.interlink import pack_strings

    return pack_strings(calls), pack_strings(names), np.zeros((len(calls), width), np.int32)


def scan(ctx, calls, names, out):
    from immunodbscan_amd import _lib

    ctx.check(_lib.lib.idb_gene_bitsets_gpu(ctx.handle, _lib.IDB_MEM_HOST, len(calls[2]), *(a.ctypes.data for a in calls),
                                            len(names[2]), *(a.ctypes.data for a in names), out.ctypes.data,
                                            out.shape[1]))


def gene_names(*lists):
    return [ln for x in lists for ln in open(os.path.join(ROOT, "tests", "golden", x + "genes.txt"), "rb").read().split(b"\n")
            if ln]


# calls around a wave's 64 rows and a block's; every 50th string is a long one
@pytest.mark.gpu
@pytest.mark.parametrize("lists", [("VH",), ("VH", "DH")])
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 2047, 2048, 2049, 4097, 20_000, 140_001])
def test_some_long_strings(gpu_ctx, form_of, lists, n):
    rng = random.Random(n)
    names = gene_names(*lists)
    assert form_of(n, names)[0] == "16"
    pool = calls_of(rng, 250, names, AB)
    for i in range(0, 250, 50):
        pool[i] = (pool[i] + b"~" * 2100 + rng.choice(names)) * 2
    calls = [pool[i % 250] for i in range(n)]
    want = O.gene_bitsets(pool, names)
    cs, ns, out = arrays_of(calls, names, (len(names) + 31) // 32)
    scan(gpu_ctx, cs, ns, out)
    assert np.array_equal(out, want[np.arange(n) % 250])


# waves of 1 to 64 long strings: by the wave and a lane each, on both sides of the rule
@pytest.mark.gpu
@pytest.mark.parametrize("lists", [("VH",), ("VH", "DH")])
@pytest.mark.parametrize("m", [1, 10, 20, 22, 23, 24, 26, 30, 40, 63, 64])
def test_waves_of_long_strings(gpu_ctx, form_of, lists, m):
    rng = random.Random(m)
    names = gene_names(*lists)
    pool = calls_of(rng, 64, names, AB)
    for i in rng.sample(range(64), m):
        c = bytearray(b"~" * rng.choice([2049, 2100, 3000]))
        for _ in range(40):
            g = rng.choice(names)
            p = rng.randrange(0, len(c) - len(g) + 1)
            c[p:p + len(g)] = g
        pool[i] = bytes(c)
    assert form_of(len(pool) * 3, names)[0] == "16"
    want = O.gene_bitsets(pool, names)
    cs, ns, out = arrays_of(pool * 3, names, (len(names) + 31) // 32)
    scan(gpu_ctx, cs, ns, out)
    assert np.array_equal(out, np.concatenate([want] * 3))


@pytest.mark.gpu
def test_many_long_strings_run_beside_each_other(gpu_ctx, form_of):
    """A hundred strings of 2,100 bytes, a lane each, against one that its whole
    wave walks (64 of them one after the other took 14 times as long as one)."""
    import time

    rng = random.Random(2)
    names = gene_names("VH")
    string = bytes(rng.choice(AB) for _ in range(2100))
    assert form_of(1, names)[0] == form_of(100, names)[0] == "16"

    def best(n):
        cs, ns, out = arrays_of([string] * n, names, 4)
        t = 1e9
        for _ in range(20):
            t0 = time.perf_counter()
            scan(gpu_ctx, cs, ns, out)
            t = min(t, time.perf_counter() - t0)
        return t

    one, many = best(1), best(100)
    print(f"one {one * 1e6:.0f} us, a hundred {many * 1e6:.0f}", flush=True)
    assert many < 8 * one
