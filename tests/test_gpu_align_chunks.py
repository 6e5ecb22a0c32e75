"""GPU tests of the matrix alignment's second and third chunk of 64 candidates: ordinary reads at
coverages that fill them, for every class of lengths of its dispatch. Bar: every candidate's
alignments equal those of the wavefront-per-pair kernel (integers)."""
import numpy as np
import pytest

from rabbitqcplus_amd import engine, reads, sim

pytestmark = pytest.mark.gpu


def batch(rs, variant):
    eng = engine.CareEngine(0, align_variant=variant, keep_intermediates=1, kmerlength=16, estimated_coverage=150.0)
    eng.set_reads(rs)
    eng.build_tables()
    eng.correct()
    b = eng.inspect_batch()
    eng.close()
    assert b.n == rs.n
    return b


@pytest.mark.parametrize("lmin,lmax", [(64, 64), (120, 128), (150, 150), (190, 192), (250, 256), (340, 352), (370, 384), (500, 512),
                                       (700, 768), (1000, 1024)])
def test_lists_of_several_chunks(lmin, lmax):
    s = sim.simulate(genome_length=4 * lmax, read_length_min=lmin, read_length_max=lmax, coverage=150.0, q_first=28.0,
                     q_last=18.0, seed=34)
    rs = reads.storage_from_sim(s, use_qualities=False)
    m, w = batch(rs, 0), batch(rs, 1)
    longest = int(np.diff(m.offsets).max())
    print(f"[lengths {lmin}..{lmax}] reads={rs.n} longest list {longest}", flush=True)
    assert longest > 128
    assert np.array_equal(m.candidate_ids, w.candidate_ids)
    assert np.array_equal(m.alignments, w.alignments)
