"""GPU tests of the matrix-core alignment filter (the default alignment of a staged batch).

Bar: every candidate's alignments of both orientations and the chosen orientation equal
those of the wavefront-per-pair kernel (``align_variant=1``, itself checked against the
oracle in tests/test_gpu_parity.py), over read lengths at the edges of its 32-shift and
64-position tiles, mixed lengths, every length class of its dispatch, low-complexity reads
(anchors handed to the lane scan), and the error rates and overlaps that move its filter
bound or take the batch to the lane scan. Integer results: equality, no tolerance.
"""
import numpy as np
import pytest

from rabbitqcplus_amd import engine, reads, sim

pytestmark = pytest.mark.gpu

LENGTHS = [(30, 33), (63, 65), (64, 64), (96, 97), (127, 129), (160, 161), (191, 193), (20, 250), (256, 257), (320, 352),
           (353, 385), (500, 513), (640, 770), (1000, 1024)]
OPTIONS = [dict(max_error_rate=0.0), dict(max_error_rate=0.05), dict(max_error_rate=0.3), dict(max_error_rate=0.31),
           dict(max_error_rate=0.45), dict(min_overlap=1, min_overlap_ratio=0.0), dict(min_overlap=0, min_overlap_ratio=0.0),
           dict(min_overlap=120, min_overlap_ratio=0.0), dict(min_overlap_ratio=0.9)]


def alignments(rs, variant, **opts):
    eng = engine.CareEngine(0, align_variant=variant, keep_intermediates=1, kmerlength=16, estimated_coverage=20.0, **opts)
    eng.set_reads(rs)
    eng.build_tables()
    eng.correct()
    b = eng.inspect_batch()
    eng.close()
    assert b.n == rs.n
    return b


def compare(rs, **opts):
    m, w = alignments(rs, 0, **opts), alignments(rs, 1, **opts)
    assert np.array_equal(m.candidate_ids, w.candidate_ids)
    assert m.candidate_ids.size > 100
    assert np.array_equal(m.alignments, w.alignments)
    return m


def storage(lmin, lmax, seed=31, **kw):
    length = 0.5 * (lmin + lmax)
    s = sim.simulate(genome_length=int(max(2000, 12 * length)), read_length_min=lmin, read_length_max=lmax,
                     coverage=20.0, q_first=26.0, q_last=16.0, seed=seed, **kw)
    return reads.storage_from_sim(s, use_qualities=False)


@pytest.mark.parametrize("lmin,lmax", LENGTHS)
def test_lengths(lmin, lmax):
    rs = storage(lmin, lmax)
    print(f"[lengths {lmin}..{lmax}] reads={rs.n}", flush=True)
    compare(rs)


@pytest.mark.parametrize("opts", OPTIONS, ids=lambda o: "-".join(f"{k}={v}" for k, v in o.items()))
def test_error_rates_and_overlaps(opts):
    rs = storage(60, 200, seed=32)
    print(f"[options {opts}] reads={rs.n}", flush=True)
    compare(rs, **opts)


@pytest.mark.parametrize("lmin,lmax", [(150, 150), (100, 250), (400, 420)])
def test_low_complexity(lmin, lmax):
    rs = storage(lmin, lmax, seed=33, tandem_fraction=0.9, tandem_period_max=2)
    print(f"[tandem {lmin}..{lmax}] reads={rs.n}", flush=True)
    compare(rs)
