"""Number of records that a pass reports (GPU): that of the records in its stream, whichever kernels
count them, for batches of every schedule and ranges around their sizes."""
import pytest

from rabbitqcplus_amd import engine
from tests import helpers

pytestmark = pytest.mark.gpu

SCHEDULES = [dict(), dict(sync_batches=1), dict(batch_size=777, sync_batches=1), dict(batch_size=777, pipeline_capacity=4),
             dict(engine=2), dict(engine=2, use_graphs=1), dict(correct_candidates=1),
             dict(correct_candidates=1, batch_size=1000), dict(keep_intermediates=1), dict(align_variant=1)]


@pytest.mark.parametrize("opts", SCHEDULES, ids=lambda o: "-".join(f"{k}={v}" for k, v in o.items()) or "default")
def test_count_equals_records(opts):
    s, rs, o = helpers.case("se_higherr_q")
    print(f"[{opts}] reads={rs.n}", flush=True)
    eng = engine.CareEngine(0, **{**o, **opts})
    eng.set_reads(rs)
    eng.build_tables()
    for first, n in [(0, rs.n), (0, 1), (5, 63), (100, 1024), (0, rs.n)]:
        count, data = eng.correct(first, n)
        assert count == len(helpers.parse_records(data)), (first, n)
        assert count == eng.timings()["records"]
    assert count > 1000
    eng.close()
