"""What a user of this framework has it do, as cases that can be timed and compared.

A case is a dict of plain values.  `prepare` makes what a program has in hand
before the call, `run` is one pass through the public entry points and returns
its whole outputs, `work` states what the pass cannot do without, and `exact`
gives the encoder's outputs in 64 bits.

The sizes follow immunodbscan_amd/configs.py and bench.py: the 2,000-row
Hamming repertoire, the 200,000- and 2,000,000-row protein repertoires, the
batch of uneven nucleotide repertoires, the long nucleotide repertoire (at
2,000,000 rows), the gene-call tables and the learned filter's encoder; the
relative-threshold Levenshtein run is the reference program's default
configuration (tests/golden/psdbscan.conf).
"""
import math
import os
import random

import numpy as np
import torch  # first: the native library then shares its HIP runtime

from immunodbscan_amd import _lib, configs, engine, learned, synth

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# clustering runs ------------------------------------------------------------
# gen: which generator makes the rows
#   clones   nucleotide rows of 30-75 letters in steps of 3, substitutions
#   protein  amino-acid rows of 8-25 letters, 1-3 edits per clone member
#   long     nucleotide rows of 24-150 letters, substitutions and indels
# rows per clone seed as in the configurations above
MEAN_LEN = {"clones": 52.5, "protein": 15.0, "long": 87.0}
ROWS_PER_SEED = {"clones": 10, "protein": 10, "long": 200}


def _cluster(gen, rows, hamming, eps, abs_k, min_pts, host, reps=0):
    return {"kind": "cluster", "gen": gen, "rows": rows, "hamming": hamming, "eps": eps, "abs_k": abs_k,
            "min_pts": min_pts, "host": host, "reps": reps}


def listed():
    return [
        # The smallest call: one small table from host arrays, as psdbscan
        # makes it for a file of a few thousand rows.
        {"name": "hamming_nt_2k_host", **_cluster("clones", 2_000, True, 0.15, -1, 2, True)},
        # The reference's default settings: Levenshtein with a relative
        # threshold, an ordinary table.
        {"name": "lev_nt_20k_relative_host", **_cluster("clones", 20_000, False, 0.15, -1, 2, True)},
        # Amino-acid Hamming with a relative threshold (5-bit letters).
        {"name": "hamming_aa_100k_host", **_cluster("protein", 100_000, True, 0.15, -1, 2, True)},
        # The headline workload: one protein repertoire from host arrays.
        {"name": "lev_aa_200k_host", **_cluster("protein", 200_000, False, 0.0, 2, 3, True)},
        # A deep protein repertoire that is already in HBM.
        {"name": "lev_aa_2m", **_cluster("protein", 2_000_000, False, 0.0, 2, 3, False)},
        # A deep nucleotide repertoire of long rows, in HBM.
        {"name": "lev_nt_2m_long", **_cluster("long", 2_000_000, False, 0.0, 3, 3, False)},
        # Many uneven repertoires in one call, in HBM.
        {"name": "batch_nt_128", **_cluster("clones", 2_560_000, True, 0.15, -1, 2, False, reps=128)},
        # Gene calls of a table against the reference's V gene names, in HBM.
        {"name": "genes_1m", "kind": "genes", "rows": 1_000_000, "names": "VH", "host": False},
        # Embeddings of a protein repertoire, and of nucleotide rows (which
        # need the 160-position encoder), for threshold tuning.
        {"name": "embed_aa_100k", "kind": "embed", "rows": 100_000, "positions": 32},
        {"name": "embed_nt_20k", "kind": "embed", "rows": 20_000, "positions": 160},
        # The training step's forward and backward passes over one batch of
        # pairs.
        {"name": "grad_aa_4k", "kind": "grad", "pairs": 4_096, "rows": 20_000, "positions": 32},
        # The learned run: embeddings, proposals and their exact checks.
        {"name": "learned_aa_200k", "kind": "learned", "rows": 200_000, "min_sim": 0.85},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    which = rng.random()
    if which < 0.20:  # short nucleotide tables, both distances
        ham = rng.random() < 0.5
        return _cluster("clones", _log(rng, 200, 200_000 if ham else 60_000), ham, rng.choice([0.1, 0.15, 0.2]), -1,
                        rng.choice([2, 3]), rng.random() < 0.7)
    if which < 0.40:  # protein repertoires, fixed and relative thresholds
        rows = _log(rng, 1_000, 1_500_000)
        if rows < 300_000 and rng.random() < 0.4:
            return _cluster("protein", rows, rng.random() < 0.5, rng.choice([0.1, 0.15, 0.2]), -1, rng.choice([2, 3]),
                            rng.random() < 0.7)
        return _cluster("protein", rows, False, 0.0, rng.choice([1, 2]), rng.choice([2, 3, 4]), rng.random() < 0.5)
    if which < 0.52:  # long nucleotide rows
        return _cluster("long", _log(rng, 5_000, 1_500_000), False, 0.0, rng.choice([2, 3, 4]), 3, rng.random() < 0.3)
    if which < 0.64:  # batches
        reps = _log(rng, 3, 160)
        return _cluster("clones", reps * _log(rng, 2_000, 16_000), True, 0.15, -1, 2, rng.random() < 0.3, reps=reps)
    if which < 0.76:  # gene calls
        return {"kind": "genes", "rows": _log(rng, 2_000, 1_500_000), "names": rng.choice(["VH", "VH", "JH", "DH"]),
                "host": rng.random() < 0.4}
    if which < 0.88:  # embeddings
        if rng.random() < 0.6:
            return {"kind": "embed", "rows": _log(rng, 1_000, 150_000), "positions": 32}
        return {"kind": "embed", "rows": _log(rng, 500, 30_000), "positions": 160}
    if which < 0.94:  # training steps
        if rng.random() < 0.7:
            return {"kind": "grad", "pairs": _log(rng, 256, 6_000), "rows": 20_000, "positions": 32}
        return {"kind": "grad", "pairs": _log(rng, 128, 1_500), "rows": 5_000, "positions": 160}
    return {"kind": "learned", "rows": _log(rng, 10_000, 300_000), "min_sim": rng.choice([0.8, 0.85, 0.9])}


# ---------------------------------------------------------------------------
def _sizes(case, seed):
    """Repertoire sizes of a batch: 200 rows each and lognormal shares of the
    rest of the case's rows (the workload's sigma)."""
    reps = case["reps"]
    w = np.exp(1.82 * np.random.default_rng(seed).standard_normal(reps))
    w = np.minimum(w, 40.0 * np.median(w))
    ends = np.round((case["rows"] - 200 * reps) * np.cumsum(w) / w.sum()).astype(np.int64)
    return 200 + np.diff(ends, prepend=0)


def _repertoire(gen, rows, seed, v_zipf=0.0):
    seeds = max(1, rows // ROWS_PER_SEED[gen])
    if gen == "clones":
        return synth.generate(configs.c1_params(rows, seeds, seed, v_zipf))
    if gen == "protein":
        return synth.generate(configs.c2_params(rows, seeds, seed))
    return synth.generate(configs.c5_params(rows, seeds, seed))


def _rows_of(case, seed):
    if not case.get("reps"):
        return _repertoire(case["gen"], case["rows"], seed)
    sizes = _sizes(case, seed)
    return synth.concat([_repertoire(case["gen"], int(n), seed * 1_000_003 + r, 1.1) for r, n in enumerate(sizes)])


def _up(a):
    """An array in HBM (unsigned words as signed ones of the same bits)."""
    a = np.ascontiguousarray(a)
    a = a.view({"u4": np.int32, "u8": np.int64}.get(a.dtype.str[1:], a.dtype))
    return torch.from_numpy(a).cuda()


def _resident(rep):
    """The rows in HBM, as the entry points take them, with output buffers."""
    keep = [_up(x) for x in (rep.seq, rep.off, rep.length, rep.vbits, rep.jbits)]
    outs = [torch.empty(rep.n, dtype=torch.int32, device="cuda") for _ in range(5)]
    ds = _lib.make_dataset(rep.n, *keep[:4], rep.vw, keep[4], rep.jw, mem=_lib.IDB_MEM_DEVICE, seq_bytes=len(rep.seq))
    return keep, outs, ds, _lib.make_outputs(*outs, mem=_lib.IDB_MEM_DEVICE)


def _host(rep):
    """The rows in host memory, with host output arrays (HostRun's layout,
    for a single repertoire or a batch)."""
    keep = [np.ascontiguousarray(x) for x in (rep.seq, rep.off, rep.length, rep.vbits, rep.jbits)]
    outs = [np.zeros(rep.n, np.int32 if k == 1 else np.uint32) for k in range(5)]
    ds = _lib.make_dataset(rep.n, *keep[:4], rep.vw, keep[4], rep.jw, seq_bytes=len(rep.seq))
    return keep, outs, ds, _lib.make_outputs(*outs)


def _prepare_cluster(case, seed):
    rep = _rows_of(case, seed)
    keep, outs, ds, od = _host(rep) if case["host"] else _resident(rep)
    prm = _lib.make_params(case["eps"], case["abs_k"], case["min_pts"], case["hamming"])
    s = {"kind": "cluster", "ctx": engine.default_context(), "keep": keep, "outs": outs, "ds": ds, "od": od,
         "prm": prm, "st": _lib.IdbStats(), "starts": None}
    if case["reps"]:
        s["starts"] = np.ascontiguousarray(rep.rep_start, np.uint32)
        s["nu"] = np.zeros(case["reps"], np.uint32)
    return s


def _run_cluster(s):
    ctx = s["ctx"]
    if s["starts"] is None:
        ctx.check(_lib.lib.idb_dbscan(ctx.handle, s["ds"], s["prm"], s["od"], s["st"]))
        return [*s["outs"], int(s["st"].n_uniques), int(s["st"].n_clusters)]
    ctx.check(_lib.lib.idb_dbscan_batch(ctx.handle, s["ds"], s["starts"].ctypes.data, len(s["nu"]), s["prm"],
                                        s["od"], s["nu"].ctypes.data, s["st"]))
    return [*s["outs"], s["nu"], int(s["st"].n_clusters)]


# gene calls -----------------------------------------------------------------
def _names(which):
    """The reference's gene lists (a name ends in the allele separator)."""
    with open(os.path.join(ROOT, "tests", "golden", which + "genes.txt"), "rb") as f:
        return [ln for ln in f.read().split(b"\n") if ln]


def _prepare_genes(case, seed):
    from immunodbscan_amd.interlink import pack_strings

    names = _names(case["names"])
    rng = random.Random(seed)
    # IMGT-style calls: 1-3 alleles of the list's genes
    pool = [b", or ".join(b"Homsap " + rng.choice(names)[:-1] + b"*0%d F" % rng.randrange(1, 9)
                          for _ in range(rng.randrange(1, 4))) for _ in range(4096)]
    pd, po, pl = pack_strings(pool)
    n = case["rows"]
    pick = np.random.default_rng(seed).integers(0, len(pool), n)
    lens = pl[pick].astype(np.uint32)
    off = np.zeros(n, np.uint64)
    off[1:] = np.cumsum(lens[:-1], dtype=np.uint64)
    src = np.repeat(po[pick].astype(np.int64) - off.astype(np.int64), lens)
    data = pd[src + np.arange(len(src))]
    width = (len(names) + 31) // 32
    genes = pack_strings(names)
    if case["host"]:
        keep, out, mem = [data, off, lens], np.zeros((n, width), np.int32), _lib.IDB_MEM_HOST
    else:
        keep, out, mem = [_up(x) for x in (data, off, lens)], torch.empty((n, width), dtype=torch.int32,
                                                                          device="cuda"), _lib.IDB_MEM_DEVICE
    return {"kind": "genes", "ctx": engine.default_context(), "n": n, "calls": keep, "genes": genes,
            "n_genes": len(names), "width": width, "out": out, "mem": mem}


def _run_genes(s):
    ctx = s["ctx"]
    ctx.check(_lib.lib.idb_gene_bitsets_gpu(ctx.handle, s["mem"], s["n"], *(_lib._ptr(x) for x in s["calls"]),
                                            s["n_genes"], *(_lib._ptr(x) for x in s["genes"]), _lib._ptr(s["out"]),
                                            s["width"]))
    return s["out"]


# the learned filter ---------------------------------------------------------
def _encoder(positions):
    letters = synth.LETTERS[synth.AA if positions == 32 else synth.NT]
    return learned.Encoder(learned.vocab_for(letters), seed=2, positions=positions)


def _encoder_rows(case, seed):
    return _repertoire("protein" if case["positions"] == 32 else "long", case["rows"], seed)


def _pairs(case, rep, seed):
    """Half pairs of one clone, half arbitrary pairs, with their labels."""
    rng = np.random.default_rng(seed + 7)
    n = case["pairs"]
    order = np.argsort(rep.clone_of, kind="stable")
    i = rng.integers(0, rep.n - 1, n)
    a, b = order[i], order[i + 1]
    far = rng.random(n) < 0.5
    b = np.where(far, rng.integers(0, rep.n, n), b)
    return np.stack([a, b], 1).astype(np.uint32), (rep.clone_of[a] == rep.clone_of[b]).astype(np.float32)


def prepare(case, seed):
    if case["kind"] == "cluster":
        return _prepare_cluster(case, seed)
    if case["kind"] == "genes":
        return _prepare_genes(case, seed)
    if case["kind"] == "learned":
        rep = _repertoire("protein", case["rows"], seed)
        keep, outs, ds, od = _resident(rep)
        return {"kind": "learned", "ctx": engine.default_context(), "enc": _encoder(32), "min_sim": case["min_sim"],
                "keep": keep, "outs": outs, "ds": ds, "od": od, "prm": _lib.make_params(0.0, 2, 3, False),
                "st": _lib.IdbStats()}
    rep = _encoder_rows(case, seed)
    s = {"kind": case["kind"], "enc": _encoder(case["positions"]), "rep": rep}
    if case["kind"] == "grad":
        s["pairs"], s["labels"] = _pairs(case, rep, seed)
    return s


def run(state):
    kind = state["kind"]
    if kind == "cluster":
        return _run_cluster(state)
    if kind == "genes":
        return _run_genes(state)
    if kind == "embed":
        return state["enc"].embed(state["rep"])
    if kind == "grad":
        loss, grad = state["enc"].loss_grad(state["rep"], state["pairs"], state["labels"], 0.9)
        return [loss, grad]
    ctx = state["ctx"]
    ctx.check(_lib.lib.idb_dbscan_learned(ctx.handle, state["enc"].handle, state["min_sim"], state["ds"],
                                          state["prm"], state["od"], state["st"]))
    return [*state["outs"], int(state["st"].n_clusters)]


# floating-point operations of the encoder per letter: three convolutions of
# five taps (32 -> 128 -> 128 -> 128 channels)
CONV_FLOPS = 2 * 5 * (32 * 128 + 2 * 128 * 128)


def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind == "genes":
        names = _names(case["names"])
        # about two alleles of "Homsap IGHV1-18*01 F" per call
        return {"bytes": rows * (46.7 + 12 + 4 * ((len(names) + 31) // 32)), "flops": 0}
    if kind == "cluster":
        vw, jw = 2, 1
        return {"bytes": rows * (MEAN_LEN[case["gen"]] + 12 + 4 * (vw + jw) + 20), "flops": 0}
    if kind == "learned":
        return {"bytes": rows * (15 + 12 + 12 + 20), "flops": rows * 15 * CONV_FLOPS}
    mean = 15.0 if case["positions"] == 32 else 87.0
    if kind == "embed":
        return {"bytes": rows * (mean + 12 + 256), "flops": rows * mean * CONV_FLOPS}
    seqs = 2 * case["pairs"]
    return {"bytes": case["pairs"] * 12 + rows * (mean + 12) + 8 * _lib.IDB_ENC_PARAMS,
            "flops": 3 * seqs * mean * CONV_FLOPS}


# 64-bit values --------------------------------------------------------------
def _tokens(rep, positions):
    """Token of each row's first letters (positions past the end: 31)."""
    letters = synth.LETTERS[synth.AA if positions == 32 else synth.NT]
    lut = np.full(256, 31, np.int64)
    lut[np.frombuffer(letters, np.uint8)] = np.arange(len(letters))
    tok = np.full((rep.n, positions), 31, np.int64)
    n = np.minimum(rep.length, positions).astype(np.int64)
    r = np.repeat(np.arange(rep.n), n)
    p = np.arange(len(r)) - np.repeat(np.cumsum(n) - n, n)
    tok[r, p] = lut[rep.seq[rep.off.astype(np.int64)[r] + p]]
    return tok, n


def _weights(params):
    """The flat parameters by name; the weights are bfloat16 by definition."""
    flat = torch.from_numpy(params).bfloat16().double().cuda()
    shapes = [("emb", (32, 32)), ("w1", (128, 160)), ("b1", (128,)), ("w2", (128, 640)), ("b2", (128,)),
              ("w3", (128, 640)), ("b3", (128,)), ("wp", (64, 128)), ("bp", (64,))]
    out, at = {}, 0
    for name, shape in shapes:
        n = math.prod(shape)
        out[name] = flat[at:at + n].reshape(shape).clone().requires_grad_(True)
        at += n
    return out


def _forward(w, tok, length):
    tok, length = torch.from_numpy(tok).cuda(), torch.from_numpy(length).cuda()
    P = tok.shape[1]
    mask = (torch.arange(P, device="cuda")[None, :] < length[:, None]).double()[:, :, None]
    x = w["emb"][tok] * mask
    for k in "123":
        padded = torch.nn.functional.pad(x, (0, 0, 2, 2))
        win = torch.cat([padded[:, t:t + P] for t in range(5)], dim=2)
        h = win.reshape(-1, win.shape[2]) @ w["w" + k].t() + w["b" + k]
        h = 0.5 * h * (1 + torch.tanh(math.sqrt(2 / math.pi) * (h + 0.044715 * h ** 3)))
        x = h.reshape(tok.shape[0], P, -1) * mask
    pool = x.sum(1) / length.clamp(min=1)[:, None]
    u = pool @ w["wp"].t() + w["bp"]
    return u / u.norm(dim=1, keepdim=True).clamp(min=1e-6)


def exact(case, seed):
    if case["kind"] not in ("embed", "grad"):
        return None  # whole numbers
    positions = case["positions"]
    rep = _encoder_rows(case, seed)
    w = _weights(_encoder(positions).get_params())
    tok, length = _tokens(rep, positions)
    step = 131_072 // positions
    if case["kind"] == "embed":
        with torch.no_grad():
            return np.concatenate([_forward(w, tok[a:a + step], length[a:a + step]).cpu().numpy()
                                   for a in range(0, rep.n, step)])
    pairs, labels = _pairs(case, rep, seed)
    total = 0.0
    for a in range(0, len(pairs), step // 2):
        p = pairs[a:a + step // 2].astype(np.int64)
        y = torch.from_numpy(labels[a:a + step // 2]).double().cuda()
        z1, z2 = _forward(w, tok[p[:, 0]], length[p[:, 0]]), _forward(w, tok[p[:, 1]], length[p[:, 1]])
        d2 = ((z1 - z2) ** 2).sum(1)
        hinge = (0.9 - (d2 + 1e-12).sqrt()).clamp(min=0)
        loss = (y * d2 + (1 - y) * hinge ** 2).sum() / len(pairs)
        loss.backward()
        total += float(loss)
    return [total, torch.cat([w[k].grad.reshape(-1) for k in w]).cpu().numpy()]
