"""Workloads that the correction engine is timed on, through its public entry points.

``listed()`` names them; ``draw(rng)`` gives further ones of the same ranges;
``prepare(case, seed)`` makes what a program holds before the call (reads simulated from
the seed, an engine with the reads resident and the tables built, a classifier handle);
``run(state)`` is one pass; ``work(case)`` states the bytes and operations a pass cannot
do without; ``exact(case, seed)`` is the 64-bit value of computed numbers (only the
classifier's training has such; corrected reads are bytes).

Kinds of a case:
  correct  one correction pass over resident reads and tables (CareEngine.correct): what a
           program runs per option set, and the stage the throughput is quoted on
  setup    the whole stage on new reads in a kept engine: upload, minhash tables, one pass
  fastq    FASTQ text to device read storage, records to corrected FASTQ text
  train    the seam classifier: Adam steps over device rows, then logits of those rows
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rabbitqcplus_amd import engine, learned, reads, sim

_BASE = dict(kind="correct", paired=0, quality=1, learned=0, seeded=0, candidates=0, maps=48, kmer=20,
             coverage=30.0, repeat_fraction=0.0, repeat_copies=0, q_first=36.0, q_last=28.0)


def _case(name=None, **kw):
    c = dict(_BASE, **kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # a first look at a handful of reads: launches and host work
        _case("correct_se150_6k", genome=30_000, lmin=150, lmax=150, q_first=28.0, q_last=20.0),
        # a plasmid or amplicon pool, 150 bp single end
        _case("correct_se150_40k", genome=200_000, lmin=150, lmax=150),
        # a bacterial genome, 150 bp single end, 30x: the ordinary call
        _case("correct_se150_1m", genome=5_000_000, lmin=150, lmax=150, repeat_fraction=0.02, repeat_copies=3),
        # trimmed reads of 100..250 bp with repeat families: the shape of the largest workload
        _case("correct_varlen_1m", genome=6_000_000, lmin=100, lmax=250, repeat_fraction=0.08, repeat_copies=10),
        # read pairs with 20-copy repeats and a steeper quality drop
        _case("correct_pe150_500k_pairs", genome=5_000_000, lmin=150, lmax=150, paired=1, repeat_fraction=0.10,
              repeat_copies=20, q_last=24.0),
        # short old-chemistry reads of odd length, no quality scores, higher error
        _case("correct_se101_noq_600k", genome=2_000_000, lmin=101, lmax=101, quality=0, q_first=26.0, q_last=16.0),
        # merged pairs / long amplicons of 360..450 bp
        _case("correct_long_60k", genome=810_000, lmin=360, lmax=450, kmer=32, q_first=32.0, q_last=22.0),
        # candidate correction (--candidateCorrection)
        _case("correct_candidates_200k", genome=1_000_000, lmin=150, lmax=150, candidates=1, q_first=30.0, q_last=20.0),
        # the fast learned form: seeded alignment and the classifier seam
        _case("correct_learned_seeded_500k", genome=3_000_000, lmin=100, lmax=250, learned=1, seeded=1,
              repeat_fraction=0.08, repeat_copies=10),
        # new reads into a kept engine: upload, tables, pass
        _case("setup_se150_400k", kind="setup", genome=2_000_000, lmin=150, lmax=150),
        # FASTQ in, corrected FASTQ out
        _case("fastq_varlen_300k", kind="fastq", genome=1_750_000, lmin=100, lmax=250),
        # classifier training on decision columns, full-batch Adam, then scoring
        dict(name="train_seam_65k", kind="train", rows=65536, epochs=8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["correct"] * 6 + ["setup", "fastq", "train"])
    if kind == "train":
        return dict(kind="train", rows=_log(rng, 500, 65536), epochs=rng.randint(1, 8))
    c = dict(kind=kind, maps=rng.choice([16, 32, 48, 48]), kmer=rng.choice([17, 20, 20, 24, 32]),
             quality=rng.choice([0, 1, 1]), coverage=round(rng.uniform(15.0, 30.0), 1),
             q_first=round(rng.uniform(26.0, 38.0), 1), q_last=round(rng.uniform(16.0, 28.0), 1),
             repeat_fraction=round(rng.choice([0.0, rng.uniform(0.0, 0.1)]), 3), repeat_copies=rng.randint(2, 20))
    shape = rng.choice(["fixed", "fixed", "varlen", "long"])
    if shape == "fixed":
        c["lmin"] = c["lmax"] = rng.choice([75, 100, 101, 125, 150, 151, 250])
    elif shape == "varlen":
        c["lmin"] = rng.randint(50, 150)
        c["lmax"] = rng.randint(c["lmin"], 300)
    else:
        c["lmin"] = rng.randint(200, 400)
        c["lmax"] = rng.randint(c["lmin"], 700)
    bases = _log(rng, 400_000, 60_000_000)          # bases sequenced
    if c["lmax"] > 300:
        bases = min(bases, 20_000_000)
    c["genome"] = max(20_000, int(bases / c["coverage"]))
    if kind == "correct":
        c["paired"] = rng.choice([0, 0, 1])
        if c["lmax"] <= 340:
            c["learned"] = rng.choice([0, 0, 0, 1])
            c["seeded"] = c["learned"] and rng.choice([0, 1])
            c["candidates"] = 0 if c["learned"] else rng.choice([0, 0, 0, 0, 1])
    return _case(**c)


# ---- inputs

_DEV = "cuda"


def _num_reads(case):
    n = max(int(case["coverage"] * case["genome"] / (0.5 * (case["lmin"] + case["lmax"]))), 4)
    return n & ~1 if case["paired"] else n


def _genome(case, g):
    """Uniform bases, part of them covered by copies of repeat units at 1% divergence."""
    size = case["genome"]
    seq = torch.randint(0, 4, (size,), generator=g, device=_DEV, dtype=torch.uint8)
    unit = 2000
    copies = case["repeat_copies"]
    families = int(case["repeat_fraction"] * size / (unit * copies)) if copies else 0
    if families and size > 4 * unit:
        units = torch.randint(0, 4, (families, 1, unit), generator=g, device=_DEV, dtype=torch.uint8)
        differ = torch.rand((families, copies, unit), generator=g, device=_DEV) < 0.01
        step = torch.randint(1, 4, (families, copies, unit), generator=g, device=_DEV, dtype=torch.uint8)
        rows = ((units + differ * step) & 3).reshape(-1, unit)
        slots = torch.randperm(size // unit, generator=g, device=_DEV)[:rows.shape[0]]
        seq[: (size // unit) * unit].view(-1, unit)[slots] = rows[: slots.numel()]
    return seq


def _simulate(case, seed):
    """Codes uint8 [n, lmax] (0 past a read), qualities uint8 Phred+33 [n, lmax], lengths."""
    g = torch.Generator(device=_DEV).manual_seed(seed)
    seq = _genome(case, g)
    n, lmin, lmax, size = _num_reads(case), case["lmin"], case["lmax"], case["genome"]
    # every length equally often, in an order of the seed (texts of one case have one size)
    length = (lmin + torch.arange(n, device=_DEV) % (lmax - lmin + 1))[torch.randperm(n, generator=g, device=_DEV)]
    reverse = torch.rand((n,), generator=g, device=_DEV) < 0.5
    start = (torch.rand((n,), generator=g, device=_DEV, dtype=torch.float64) * (size - lmax)).long()
    if case["paired"]:
        # mates: first read forward at the start of an insert N(350, 50), second reverse at its end
        m = n // 2
        insert = (350 + 50 * torch.randn((m,), generator=g, device=_DEV)).long().clamp(min=lmax, max=max(lmax, size // 4))
        left = (torch.rand((m,), generator=g, device=_DEV, dtype=torch.float64) * (size - insert)).long()
        start[0::2], start[1::2] = left, left + insert - length[1::2]
        reverse[1::2] = ~reverse[0::2]
    codes = torch.zeros((n, lmax), dtype=torch.uint8, device=_DEV)
    quals = torch.zeros((n, lmax), dtype=torch.uint8, device=_DEV)
    pos = torch.arange(lmax, device=_DEV)
    for a in range(0, n, 1 << 18):
        b = min(n, a + (1 << 18))
        L = length[a:b, None]
        rev = reverse[a:b, None]
        at = start[a:b, None] + torch.where(rev, L - 1 - pos, pos)
        base = seq[at.clamp(0, size - 1)]
        base = torch.where(rev, 3 - base, base)
        q = case["q_first"] + (case["q_last"] - case["q_first"]) * pos / (L - 1).clamp(min=1)
        q = (q + 2.0 * torch.randn((b - a, lmax), generator=g, device=_DEV)).round().clamp(2, 41)
        wrong = torch.rand((b - a, lmax), generator=g, device=_DEV) < 10.0 ** (-q / 10.0)
        other = torch.randint(1, 4, (b - a, lmax), generator=g, device=_DEV, dtype=torch.uint8)
        inside = pos < L
        codes[a:b] = ((base + wrong * other) & 3) * inside
        quals[a:b] = (q + 33).to(torch.uint8) * inside
    return codes, quals, length.to(torch.int32)


def _storage(case, seed):
    codes, quals, length = _simulate(case, seed)
    n, lmax = codes.shape
    words = reads.ints_per_row(int(length.max()))
    padded = torch.zeros((n, words * 16), dtype=torch.int64, device=_DEV)
    padded[:, : min(lmax, words * 16)] = codes[:, : words * 16]
    shift = 30 - 2 * torch.arange(16, device=_DEV)
    enc = (padded.view(n, words, 16) << shift).sum(-1).cpu().numpy().astype(np.uint32)
    q = quals[:, : int(length.max())].contiguous().cpu().numpy() if case["quality"] else None
    return reads.ReadStorage(enc, length.cpu().numpy(), q, np.zeros(n, np.uint8), bool(case["paired"]))


def _texts(case, seed):
    codes, quals, length = _simulate(case, seed)
    seqs = torch.tensor(list(b"ACGT"), dtype=torch.uint8, device=_DEV)[codes.long()].cpu().numpy()
    s = sim.SimReads(seqs, quals.cpu().numpy(), seqs, length.cpu().numpy(), None, None, bool(case["paired"]))
    return sim.fastq_texts(s)


def _rows(case, seed):
    """Standardized decision columns, labels of a random teacher, starting parameters."""
    rng = np.random.default_rng(seed)
    n = case["rows"]
    X = rng.standard_normal((n, 16)).astype(np.float32)
    X[:, ::5] = (X[:, ::5] > 1.0) * np.float32(2.0)
    y = (X @ rng.standard_normal(16) + 0.7 * rng.standard_normal(n) > -1.0).astype(np.float32)
    p = np.zeros(engine.MLP_PARAMS, np.float32)
    p[:1024] = rng.uniform(-0.6, 0.6, 1024)
    p[1088:5184] = rng.uniform(-0.3, 0.3, 4096)
    p[5248:5312] = rng.uniform(-0.3, 0.3, 64)
    return X, y, p


def _engine(case):
    opts = dict(kmerlength=case["kmer"], num_hash_maps=case["maps"], estimated_coverage=float(case["coverage"]),
                use_quality_scores=case["quality"], paired=case["paired"], correction_type=case["learned"],
                seeded_alignment=int(case["seeded"]), correct_candidates=case["candidates"])
    eng = engine.CareEngine(0, **opts)
    if case["learned"]:
        eng.set_classifier(learned.load_classifier()[0])
    return eng


def prepare(case, seed):
    kind = case["kind"]
    if kind == "train":
        X, y, p = _rows(case, seed)
        return dict(kind=kind, mlp=learned.Mlp(0), X=X, y=y, params=p, epochs=case["epochs"])
    eng = _engine(case)
    if kind == "fastq":
        texts = _texts(case, seed)
        eng.set_reads_fastq(*texts)
        eng.build_tables()
        _, records = eng.correct()
        return dict(kind=kind, engine=eng, texts=texts, records=records)
    storage = _storage(case, seed)
    if kind == "correct":
        eng.set_reads(storage)
        eng.build_tables()
    # the records of a pass go into one buffer of the program, zero past them
    per_read = 32 + case["lmax"] // 4 + (768 if case["candidates"] else 0)
    return dict(kind=kind, engine=eng, storage=storage, records=np.zeros(storage.n * per_read + 4096, np.uint8))


def run(state):
    kind = state["kind"]
    if kind == "train":
        mlp = state["mlp"]
        mlp.set_params(state["params"])
        mlp.reset_optimizer()
        mlp.set_data(state["X"], state["y"])
        losses = mlp.train(state["epochs"], batch=len(state["X"]), lr=1e-3, seed=1)
        return [mlp.get_params(), losses, mlp.forward(state["X"])]
    eng = state["engine"]
    if kind == "fastq":
        eng.set_reads_fastq(*state["texts"])
        return [eng.write_fastq(state["records"], file=f, as_array=True) for f in range(len(state["texts"]))]
    if kind == "setup":
        eng.set_reads(state["storage"])
        eng.build_tables()
    count, records = eng.correct()
    state["records"][: len(records)] = np.frombuffer(records, np.uint8)
    return [count, len(records), state["records"]]


def work(case):
    if case["kind"] == "train":
        n, e = case["rows"], case["epochs"]
        macs = 16 * 64 + 64 * 64 + 64
        # forward and backward (twice the forward) per epoch, then one forward
        return dict(bytes=float(n * 68 + n * 4 + 2 * engine.MLP_PARAMS * 4), flops=2.0 * n * macs * (3 * e + 1))
    n, L = _num_reads(case), 0.5 * (case["lmin"] + case["lmax"])
    if case["kind"] == "fastq":
        return dict(bytes=2.0 * n * (2 * L + 15), flops=0.0)
    rows = n * (4.0 * reads.ints_per_row(case["lmax"]) + 4 + (L if case["quality"] else 0))
    tables = 4.0 * n * case["maps"]
    # about 1.55 overlapping reads per unit of coverage; one comparison and two additions
    # per base of an aligned pair
    return dict(bytes=rows + (0.0 if case["kind"] == "setup" else tables) + 8.0 * n,
                flops=1.55 * case["coverage"] * n * L * 3.0)


def exact(case, seed):
    if case["kind"] != "train":
        return None
    X32, y32, p32 = _rows(case, seed)
    X, y, p = X32.astype(np.float64), y32.astype(np.float64), p32.astype(np.float64)
    cuts = [0, 1024, 1088, 5184, 5248, 5312, 5313]
    shapes = [(64, 16), (64,), (64, 64), (64,), (64,), ()]

    def unpack(v):
        return [v[a:b].reshape(s) for a, b, s in zip(cuts, cuts[1:], shapes)]

    def forward(v):
        W1, b1, W2, b2, W3, b3 = unpack(v)
        h1 = np.maximum(X @ W1.T + b1, 0.0)
        h2 = np.maximum(h1 @ W2.T + b2, 0.0)
        return h1, h2, h2 @ W3 + b3

    m, s, losses = np.zeros_like(p), np.zeros_like(p), []
    for t in range(1, case["epochs"] + 1):
        W1, b1, W2, b2, W3, b3 = unpack(p)
        h1, h2, z = forward(p)
        losses.append(np.mean(np.maximum(z, 0.0) - z * y + np.log1p(np.exp(-np.abs(z)))))
        dz = (1.0 / (1.0 + np.exp(-z)) - y) / len(y)
        d2 = np.outer(dz, W3) * (h2 > 0)
        d1 = (d2 @ W2) * (h1 > 0)
        grad = np.concatenate([(d1.T @ X).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), h2.T @ dz, [dz.sum()]])
        m = 0.9 * m + 0.1 * grad
        s = 0.999 * s + 0.001 * grad * grad
        p = p - float(np.float32(1e-3)) * (m / (1 - 0.9 ** t)) / (np.sqrt(s / (1 - 0.999 ** t)) + 1e-8)
    return [p, np.array(losses), forward(p)[2]]
