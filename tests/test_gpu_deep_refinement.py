"""Refinement rounds at depths where a subtracted column's error is no longer small (GPU): copies of
repeats at coverage 250 and 600, with qualities down to the lowest. Bar: the records equal
those of the same pass with intermediates kept, which builds the whole MSA each round (bytes)."""
import numpy as np
import pytest

from rabbitqcplus_amd import engine, reads, sim

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("coverage,maps", [(250.0, 32), (600.0, 8)])
@pytest.mark.parametrize("qualities", ["simulated", "lowest at the ends", None])
def test_records_equal_whole_msa(coverage, maps, qualities):
    s = sim.simulate(genome_length=4000, read_length_min=90, read_length_max=150, coverage=coverage, q_first=34.0, q_last=22.0,
                     seed=81, repeat_fraction=0.6, repeat_unit_length=400, repeat_copies=3, repeat_divergence=0.01)
    rs = reads.storage_from_sim(s, use_qualities=qualities is not None)
    if qualities == "lowest at the ends":
        at = np.arange(rs.max_length)[None, :]
        rs.quals[(at < 20) | ((at >= rs.lengths[:, None] - 20) & (at < rs.lengths[:, None]))] = 33
    print(f"[coverage {coverage} {qualities}] reads={rs.n}", flush=True)
    out = []
    for keep in (0, 1):
        eng = engine.CareEngine(0, kmerlength=20, num_hash_maps=maps, estimated_coverage=coverage,
                                use_quality_scores=int(qualities is not None), keep_intermediates=keep)
        eng.set_reads(rs)
        eng.build_tables()
        out.append(eng.correct())
        candidates = eng.timings()["candidates"]
        eng.close()
    print(f"{candidates / rs.n:.0f} candidates per anchor, {out[0][0]} records", flush=True)
    assert out[0] == out[1]
