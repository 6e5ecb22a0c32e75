"""GPU tests of what spares the MSA stage whole builds: the high-quality test in front of the MSA
(anchors certain to be corrected as high quality end before their MSA is built) and the
refinement rounds (removed candidates are taken out of the columns).

Bar: the records equal those of the same pass with intermediates kept, which builds every
anchor's whole MSA (and is checked against the oracle in tests/test_gpu_parity.py), over the
thresholds the test compares its bounds with, quality rows whose least value says nothing
or everything, mixed lengths (reverse-complement candidates then read past their read),
lists of more than 64 candidates, pairs and the learned seam. Bytes: equality.
"""
import numpy as np
import pytest

from rabbitqcplus_amd import engine, learned, reads, sim

pytestmark = pytest.mark.gpu

FIXED = dict(read_length_min=150, read_length_max=150)
MIXED = dict(read_length_min=60, read_length_max=250)
# name -> (simulator options, quality rule, engine options)
CASES = {
    "plain": (FIXED, "as simulated", {}),
    "no_quality": (FIXED, None, {}),
    "mixed": (MIXED, "as simulated", {}),
    "mixed_bytes_past_reads": (MIXED, "random past reads", {}),
    "all_lowest": (FIXED, "lowest", {}),
    "below_phred_33": (FIXED, "zeros", {}),
    "one_low_base": (FIXED, "one low", {}),
    "errorrate_0": (FIXED, "as simulated", dict(estimated_errorrate=0.0)),
    "errorrate_0.02": (FIXED, "as simulated", dict(estimated_errorrate=0.02)),
    "errorrate_0.3": (MIXED, "as simulated", dict(estimated_errorrate=0.3)),
    "coverage_bound": (FIXED, "as simulated", dict(m_coverage=4.0)),
    "coverage_bound_0": (MIXED, None, dict(m_coverage=0.0)),
    "many_candidates": (dict(FIXED, coverage=150.0), "as simulated", {}),
    "repeats": (dict(FIXED, repeat_fraction=0.3, repeat_unit_length=800, repeat_copies=6, repeat_divergence=0.02),
                "as simulated", {}),
    "n_bases": (dict(FIXED, n_rate=0.001), "as simulated", {}),
    "pairs": (dict(FIXED, paired=1, insert_mean=350.0, insert_sd=50.0), "as simulated", dict(paired=1)),
    "length_64_columns": (dict(read_length_min=128, read_length_max=128), "as simulated", {}),
    "long": (dict(read_length_min=500, read_length_max=640), "as simulated", {}),
}


def storage(simkw, rule, seed):
    kw = dict(genome_length=25_000, coverage=30.0, q_first=34.0, q_last=20.0, seed=seed)
    kw.update(simkw)
    s = sim.simulate(**kw)
    rs = reads.storage_from_sim(s, use_qualities=rule is not None)
    rng = np.random.default_rng(seed)
    inside = np.arange(rs.max_length)[None, :] < rs.lengths[:, None]
    if rule == "random past reads":
        rs.quals[~inside] = rng.integers(0, 75, int((~inside).sum()))
    elif rule == "lowest":
        rs.quals[inside] = 35
    elif rule == "zeros":
        rs.quals[:] = 0
    elif rule == "one low":
        rs.quals[np.arange(rs.n), rng.integers(0, rs.lengths)] = 35
    return rs


def records(rs, classifier=None, **opts):
    o = dict(kmerlength=20, use_quality_scores=int(rs.quals is not None))
    o.update(opts)
    eng = engine.CareEngine(0, **o)
    if classifier is not None:
        eng.set_classifier(classifier)
    eng.set_reads(rs)
    eng.build_tables()
    out = eng.correct()
    eng.close()
    return out


@pytest.mark.parametrize("name", CASES)
def test_records_equal_whole_msa(name):
    simkw, rule, opts = CASES[name]
    rs = storage(simkw, rule, 41)
    print(f"[case {name}] reads={rs.n}", flush=True)
    n, d = records(rs, **opts)
    n_w, d_w = records(rs, keep_intermediates=1, **opts)
    assert n == n_w and d == d_w


def test_learned_records_equal_whole_msa():
    rs = storage(MIXED, "as simulated", 42)
    params, _ = learned.load_classifier()
    assert records(rs, params, correction_type=1) == records(rs, params, correction_type=1, keep_intermediates=1)


REFINED = dict(genome_length=20_000, repeat_fraction=0.5, repeat_unit_length=1000, repeat_copies=5)


@pytest.mark.parametrize("rule", ["as simulated", None, "lowest"])
@pytest.mark.parametrize("lengths", [(101, 101), (150, 150), (100, 250), (260, 330), (400, 500)])
@pytest.mark.parametrize("divergence", [0.004, 0.03])
def test_refined_records_equal_whole_msa(lengths, rule, divergence):
    # copies close enough to be each other's candidates: rounds that remove one base's reads
    rs = storage(dict(REFINED, read_length_min=lengths[0], read_length_max=lengths[1], repeat_divergence=divergence,
                      coverage=40.0), rule, 43)
    print(f"[refined {lengths} {rule} {divergence}] reads={rs.n}", flush=True)
    assert records(rs, estimated_coverage=40.0) == records(rs, estimated_coverage=40.0, keep_intermediates=1)


def test_refined_learned_records_equal_whole_msa():
    rs = storage(dict(REFINED, **MIXED, repeat_divergence=0.01, coverage=40.0), "as simulated", 44)
    params, _ = learned.load_classifier()
    opts = dict(correction_type=1, estimated_coverage=40.0)
    assert records(rs, params, **opts) == records(rs, params, keep_intermediates=1, **opts)
