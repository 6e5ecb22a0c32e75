"""GPU tests of the anchors that the matrix alignment lists for a scan of every shift (reads of low
complexity): batches around the number of lists, against the wavefront-per-pair scan
(``align_variant=1``; bytes: equality), and the time of the alignment of such reads."""
import pytest

from rabbitqcplus_amd import engine, reads, sim

pytestmark = pytest.mark.gpu


def tandem(lmin, lmax, genome_length, seed=51):
    s = sim.simulate(genome_length=genome_length, read_length_min=lmin, read_length_max=lmax, coverage=30.0, q_first=32.0,
                     q_last=22.0, seed=seed, tandem_fraction=0.9, tandem_period_max=2)
    return reads.storage_from_sim(s, use_qualities=False)


def context(rs, variant, **opts):
    eng = engine.CareEngine(0, kmerlength=20, align_variant=variant, **opts)
    eng.set_reads(rs)
    eng.build_tables()
    return eng


@pytest.mark.parametrize("lengths", [(150, 150), (340, 352), (400, 420)])
def test_small_batches_of_listed_anchors(lengths):
    rs = tandem(*lengths, genome_length=12_000)
    m, w = context(rs, 0), context(rs, 1)
    for first, n in [(0, 1), (3, 5), (7, 63), (0, 64), (1, 65), (50, 129), (0, rs.n)]:
        print(f"[{lengths} anchors {first}+{n}]", flush=True)
        assert m.correct(first, n) == w.correct(first, n)
    m.close()
    w.close()


@pytest.mark.parametrize("opts", [dict(use_graphs=1), dict(use_graphs=1, batch_size=500), dict(batch_size=500),
                                  dict(batch_size=500, pipeline_capacity=4), dict(sync_batches=1), dict(correct_candidates=1)],
                         ids=lambda o: "-".join(f"{k}={v}" for k, v in o.items()))
def test_listed_anchors_on_every_schedule(opts):
    # repeated passes: the lists are emptied before each batch, in captured batches too
    rs = tandem(150, 150, genome_length=12_000, seed=52)
    print(f"[{opts}] reads={rs.n}", flush=True)
    w = context(rs, 1, correct_candidates=opts.get("correct_candidates", 0))
    want = w.correct()
    w.close()
    m = context(rs, 0, **opts)
    for _ in range(4):
        assert m.correct() == want
    m.close()


def test_long_reads_of_low_complexity_cost_what_the_scan_costs():
    # 18,000 reads of 600..700 bases, nearly all of them listed: the filter that listed them and
    # their scan within 1.2 of the scan alone
    rs = tandem(600, 700, genome_length=400_000)
    ms = {}
    for variant in (0, 1):
        eng = context(rs, variant)
        times = []
        for _ in range(6):
            eng.correct()
            times.append(eng.timings()["align_kernel_ms"])
        eng.close()
        ms[variant] = min(times)
    print(f"[reads={rs.n}] listed {ms[0]:.2f} ms, scan {ms[1]:.2f} ms", flush=True)
    assert ms[0] <= 1.2 * ms[1]
