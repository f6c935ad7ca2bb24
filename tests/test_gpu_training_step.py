"""The packed training step at its edges: one pair, rows without letters, rows
that fill a tile exactly, rows of the encoder's full width and longer, and
batches over several packing windows and splits of the weight gradients' rows,
each against the oracle's loss and gradients (the bounds of a bfloat16
forward and backward pass, as for the ordinary batches)."""
from __future__ import annotations

import numpy as np
import pytest

from immunodbscan_amd import synth
from oracle import learned as Lr


def _batch(kind, P):
    rng = np.random.default_rng(11)
    if kind == "one":
        return np.array([P - 3, 5]), np.array([[0, 1]])
    if kind == "empty":  # most rows without letters: a tile of 129 rows' worth of gaps
        lens = np.zeros(300, np.int64)
        lens[::50] = 9
        return lens, rng.integers(0, 300, (200, 2))
    if kind == "exact":  # 16 rows of 14 letters and their gaps are 256 rows; then full rows and odd ones
        lens = np.resize([14] * 16 + [P, 254 % P, 1, 0, 2], 84)
        return lens, np.arange(84).reshape(42, 2)
    if kind == "full":
        return np.full(30, P + 7), rng.integers(0, 30, (17, 2))
    lens = rng.integers(1, 20, 700)  # 1,402 sequences: two windows
    return lens, np.concatenate([np.arange(700).reshape(350, 2), rng.integers(0, 700, (351, 2))])


@pytest.mark.gpu
@pytest.mark.parametrize("P", [32, 160])
@pytest.mark.parametrize("kind", ["one", "empty", "exact", "full", "windows"])
def test_loss_and_gradients(gpu_ctx, kind, P):
    from immunodbscan_amd import learned

    lens, pairs = _batch(kind, P)
    letters = np.frombuffer(synth.LETTERS[synth.NT if P == 160 else synth.AA], np.uint8)
    rng = np.random.default_rng(4)
    off = np.zeros(len(lens), np.uint64)
    off[1:] = np.cumsum(lens[:-1])
    seq = letters[rng.integers(0, len(letters), max(1, int(lens.sum())))]
    zero = np.zeros((len(lens), 1), np.int32)
    rep = synth.Repertoire(seq, off, lens.astype(np.uint32), zero, zero, np.zeros(len(lens), np.uint32))
    enc = learned.Encoder(learned.vocab_for(letters.tobytes()), seed=5, positions=P)
    pairs = pairs.astype(np.uint32)
    labels = (np.arange(len(pairs)) % 3 != 0).astype(np.float32)
    tok, ln = Lr.tokens_of([rep.row(i) for i in range(rep.n)], enc.vocab, positions=P)
    a, b = pairs[:, 0].astype(np.int64), pairs[:, 1].astype(np.int64)
    lref, gref, _ = Lr.loss_and_grad(enc.get_params(), tok, ln, a, b, labels, 0.9, emulate_bf16=True)
    offs = np.cumsum([0] + [int(np.prod(s)) for _, s in Lr.SHAPES])
    for turn in range(2):  # the second pass reuses the workspace, after a larger or smaller batch
        loss, g = enc.loss_grad(rep, pairs, labels, 0.9)
        assert abs(loss - lref) <= 1e-3 * abs(lref) + 1e-6
        for k, (name, _) in enumerate(Lr.SHAPES):
            x, y = g[offs[k]:offs[k + 1]], gref[offs[k]:offs[k + 1]]
            assert np.linalg.norm(x - y) <= 2e-2 * np.linalg.norm(y) + 1e-7, (name, turn)
        enc.loss_grad(rep, pairs[:1] if turn else np.resize(pairs, (2 * len(pairs), 2)),
                      labels[:1] if turn else np.resize(labels, 2 * len(labels)), 0.9)
