"""Labels below zero and labels that are no numbers: the pair counts in the
mean, and has no loss and no gradient."""
from __future__ import annotations

import numpy as np
import pytest

from immunodbscan_amd import configs, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("label", [-1.0, -0.25, float("nan")])
def test_pairs_without_a_label(gpu_ctx, label):
    from immunodbscan_amd import learned

    rep = synth.generate(configs.c2_params(2_000, 200, 8))
    rng = np.random.default_rng(3)
    enc = learned.Encoder(learned.vocab_for(synth.LETTERS[synth.AA]), seed=5, positions=32)
    pairs = rng.integers(0, rep.n, (128, 2)).astype(np.uint32)
    y = (rng.random(128) < 0.5).astype(np.float32)
    loss, grad = enc.loss_grad(rep, pairs, y, 0.9)
    # every other pair without a label: half the mean, exactly half of every
    # rounded value on the way (a power of two); sums differ in their order
    both = np.empty((256, 2), np.uint32)
    both[0::2], both[1::2] = pairs, rng.integers(0, rep.n, (128, 2))
    yy = np.full(256, label, np.float32)
    yy[0::2] = y
    loss2, grad2 = enc.loss_grad(rep, both, yy, 0.9)
    assert abs(2 * loss2 - loss) <= 1e-5 * abs(loss)
    assert np.linalg.norm(2 * grad2 - grad) <= 1e-4 * np.linalg.norm(grad) and np.linalg.norm(grad) > 0
