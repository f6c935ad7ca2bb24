"""Gene bitsets wider than four words of more calls than run at once, into a
device array at any word offset: every bit is there, from 16-bit and 32-bit
tables, and no word beside the output is touched."""
from __future__ import annotations

import os
import random

import numpy as np
import pytest

from oracle import oracle as O

GOLDEN = os.path.join(os.path.dirname(__file__), "golden")


@pytest.mark.gpu
@pytest.mark.parametrize("extra", [0, 160])
def test_every_bit_of_many_calls(gpu_ctx, extra):
    from immunodbscan_amd import _lib
    from immunodbscan_amd.hip import DeviceBuffer
    from immunodbscan_amd.interlink import pack_strings

    rng = random.Random(extra)
    names = [ln for x in ("VH", "DH") for ln in open(os.path.join(GOLDEN, x + "genes.txt"), "rb").read().split(b"\n") if ln]
    # (more names: the 32-bit table)
    names += [bytes(rng.choice(b"abcdefghijklmnopqrstuvwxyz") for _ in range(12)) for _ in range(extra)]
    pool = [b"".join(rng.choice(names) + b"*01 " for _ in range(rng.randrange(1, 4))) for _ in range(1000)]
    n, width = 400_000, (len(names) + 31) // 32
    pick = np.random.default_rng(1).integers(0, len(pool), n)
    want = O.gene_bitsets(pool, names)[pick]
    pd, po, pl = pack_strings(pool)
    arrays = [DeviceBuffer.from_array(x) for x in (pd, po[pick], pl[pick])]
    genes = pack_strings(names)
    blank = np.full(n * width + 64, -1, np.int32)
    for word in [0, 1, 2, 3, 5, 8, 13, 16, 21, 31, 32] * 3:
        out = DeviceBuffer.from_array(blank)
        gpu_ctx.check(_lib.lib.idb_gene_bitsets_gpu(
            gpu_ctx.handle, _lib.IDB_MEM_DEVICE, n, *(x.data_ptr() for x in arrays), len(names),
            *(g.ctypes.data for g in genes), out.data_ptr() + 4 * word, width))
        whole = out.to_numpy(np.int32, len(blank))
        bad = (whole[word:word + n * width].reshape(n, width) != want).any(1).sum()
        assert bad == 0, (word, bad)
        assert (whole[:word] == -1).all() and (whole[word + n * width:] == -1).all(), word
