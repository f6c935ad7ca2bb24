"""The fused embedding kernel's packing: rows are packed back to back into
tiles of 256 activation rows, in windows of 1,024 rows.  At the edges (empty
rows, rows that fill a tile exactly, rows of the encoder's full width and
longer, a window's last row) every embedding matches the oracle's forward
pass, and does not depend on the rows packed beside it."""
from __future__ import annotations

import numpy as np
import pytest

from immunodbscan_amd import configs, synth
from oracle import learned as Lr


def _lengths(kind: str, P: int) -> np.ndarray:
    rng = np.random.default_rng(3)
    if kind == "empty":
        return np.zeros(1300, np.int64)                       # 129 rows fill a tile
    if kind == "full":
        return np.full(40, P)
    if kind == "exact":
        return np.resize([14] * 16 + [P, 254 % P, 1, 0, 2], 90)   # 16 rows of 14: 256 rows with their gaps
    if kind == "window":
        return rng.integers(0, 20, 1025)
    return np.minimum(rng.integers(0, 2 * P, 60), 150)        # longer than the encoder reads: cut


@pytest.mark.gpu
@pytest.mark.parametrize("P", [32, 160])
@pytest.mark.parametrize("kind", ["empty", "full", "exact", "window", "long"])
def test_packed_embeddings(gpu_ctx, kind, P):
    from immunodbscan_amd import learned

    lens = _lengths(kind, P).astype(np.uint32)
    nt = P == 160
    rng = np.random.default_rng(9)
    letters = np.frombuffer(synth.LETTERS[synth.NT if nt else synth.AA], np.uint8)
    off = np.zeros(len(lens), np.uint64)
    off[1:] = np.cumsum(lens[:-1])
    seq = letters[rng.integers(0, len(letters), int(lens.sum()))]
    zero = np.zeros((len(lens), 1), np.int32)
    rep = synth.Repertoire(seq, off, lens, zero, zero, np.zeros(len(lens), np.uint32))
    enc = learned.Encoder(learned.vocab_for(letters.tobytes()), seed=5, positions=P)
    z = enc.embed(rep)
    rows = np.unique(np.concatenate([np.arange(min(40, rep.n)), np.arange(max(0, rep.n - 4), rep.n)]))
    tok, ln = Lr.tokens_of([rep.row(int(i)) for i in rows], enc.vocab, positions=P)
    ref = Lr.forward(enc.get_params(), tok, ln, emulate_bf16=True)["z"]
    assert np.abs(z[rows] - ref).max() < 1e-2 and np.abs(z[rows] - ref).mean() < 1e-3
    for i in rows[::5]:
        alone = enc.embed(rep.subset(np.array([i])))
        assert np.array_equal(alone[0].view(np.uint32), z[i].view(np.uint32)), int(i)


@pytest.mark.gpu
def test_embeddings_follow_new_parameters(gpu_ctx):
    """The packed weights are those of the current parameters."""
    from immunodbscan_amd import learned

    rep = synth.generate(configs.c2_params(n_rows=300, n_seeds=30, seed=8))
    vocab = learned.vocab_for(synth.LETTERS[synth.AA])
    a, b = learned.Encoder(vocab, seed=1), learned.Encoder(vocab, seed=2)
    za, zb = a.embed(rep), b.embed(rep)
    assert not np.array_equal(za, zb)
    a.set_params(b.get_params())
    assert np.array_equal(a.embed(rep), zb)
    pairs = np.stack([np.arange(0, 200), np.arange(100, 300)], 1).astype(np.uint32)
    a.train(rep, pairs, (np.arange(200) % 2).astype(np.float32), learned.TrainParams(epochs=1, batch_pairs=100, lr=1e-2))
    b.set_params(a.get_params())
    zt = a.embed(rep)
    assert np.array_equal(zt, b.embed(rep)) and not np.array_equal(zt, zb)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [4096, 4097, 40_961])
def test_segmented_embeddings(gpu_ctx, n):
    """Calls of one segment, of a last segment of one row, and of more
    segments than are staged at a time: bit for bit those of short calls."""
    from immunodbscan_amd import learned

    rep = synth.generate(configs.c2_params(n_rows=n, n_seeds=n // 10, seed=12))
    enc = learned.Encoder(learned.vocab_for(synth.LETTERS[synth.AA]), seed=3)
    z = enc.embed(rep)
    part = learned.Encoder(learned.vocab_for(synth.LETTERS[synth.AA]), seed=3)
    for a in range(0, n, 3000):
        rows = np.arange(a, min(n, a + 3000))
        assert np.array_equal(part.embed(rep.subset(rows)), z[rows]), a
    assert np.array_equal(enc.embed(rep), z)
