"""Table build over groups of maps (GPU): the kept buckets of every map equal those of numpy over the
engine's signatures, with groups of all maps, an uneven last group, and the groups of one map
of k-mers whose signatures leave no bits for the map's number. Values and keys: equality."""
import numpy as np
import pytest

from rabbitqcplus_amd import engine, reads, sim
from tests.test_gpu_tables import parse_table_file

pytestmark = pytest.mark.gpu

# (k, maps, reads): groups hold 2^24 (map, read) pairs; 360,000 reads leave 46 maps, then 2
CASES = [(16, 48, 3000), (17, 1, 3000), (20, 48, 360_000), (29, 48, 3000), (30, 48, 3000), (32, 48, 3000), (31, 5, 3000)]


@pytest.mark.parametrize("k,maps,n", CASES)
def test_kept_buckets(k, maps, n, tmp_path):
    length = 33
    s = sim.simulate(genome_length=max(2000, n * length // 12), read_length_min=length, read_length_max=length, coverage=12.0,
                     q_first=38.0, q_last=30.0, seed=61)
    rs = reads.storage_from_sim(s, use_qualities=False)
    print(f"[k {k} maps {maps}] reads={rs.n}", flush=True)
    assert abs(rs.n - n) < 0.02 * n
    eng = engine.CareEngine(0, kmerlength=k, num_hash_maps=maps, estimated_coverage=12.0)
    eng.set_reads(rs)
    assert eng.build_tables() == maps
    sig = eng.signatures()
    path = str(tmp_path / "tables.bin")
    eng.save_tables(path)
    eng.close()
    (fk, thr, _, fmaps), tables = parse_table_file(path)
    assert (fk, fmaps) == (k, maps) and len(tables) == maps
    for m, t in enumerate(tables):
        order = np.argsort(sig[:, m], kind="stable")
        keys, first, counts = np.unique(sig[order, m], return_index=True, return_counts=True)
        kept = (counts >= 2) & (counts <= thr)
        assert t["num_keys"] == kept.sum() > 0
        in_kept = np.repeat(kept, counts)
        assert np.array_equal(t["values"], order[in_kept].astype(np.uint32)), m
        used = t["counts"] != 0
        by_key = np.argsort(t["keys"][used])
        assert np.array_equal(t["keys"][used][by_key], keys[kept]), m
        assert np.array_equal(t["counts"][used][by_key], counts[kept]), m
