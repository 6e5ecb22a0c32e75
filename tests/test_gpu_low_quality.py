"""Reads of low quality (GPU): anchors whose candidates differ from them in more places than they have
bases leave the high-quality test before it has done anything. Bar: the records equal those
of the same pass with intermediates kept, which builds every anchor's whole MSA (bytes)."""
import pytest

from rabbitqcplus_amd import engine, reads, sim

pytestmark = pytest.mark.gpu


# coverage 25: lists of at most 64 candidates; 120: longer ones
@pytest.mark.parametrize("coverage", [25.0, 120.0])
@pytest.mark.parametrize("qualities", [True, False])
@pytest.mark.parametrize("q_last", [10.0, 16.0])
def test_records_equal_whole_msa(coverage, qualities, q_last):
    s = sim.simulate(genome_length=20_000, read_length_min=100, read_length_max=150, coverage=coverage, q_first=20.0,
                     q_last=q_last, seed=71)
    rs = reads.storage_from_sim(s, use_qualities=qualities)
    print(f"[coverage {coverage} qualities {qualities} {q_last}] reads={rs.n}", flush=True)
    out = []
    for keep in (0, 1):
        eng = engine.CareEngine(0, kmerlength=16, estimated_coverage=coverage, use_quality_scores=int(qualities),
                                keep_intermediates=keep)
        eng.set_reads(rs)
        eng.build_tables()
        out.append(eng.correct())
        eng.close()
    assert out[0][0] > 100 and out[0] == out[1]
