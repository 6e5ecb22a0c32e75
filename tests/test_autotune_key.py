"""The autotuner's cache key (no GPU): a choice cached for other kernels, or for options that
select other kernels or another schedule, is not taken for this call's."""
import json
from types import SimpleNamespace

import pytest

from rabbitqcplus_amd import autotune, engine

STORAGE = SimpleNamespace(max_length=400, n=10, paired=False, quals=None)
# the key of a choice timed while align_variant 0 was one lane per candidate (one wavefront
# per pair above 352 bases) and the automatic tile 20
OLD_KEY = "MI355X|cu256|len416|q0|v3|pe0|maps48|k20"
OTHER = [dict(use_quality_scores=1), dict(paired=1), dict(num_hash_maps=16), dict(kmerlength=24), dict(correction_type=1),
         dict(correct_candidates=1), dict(seeded_alignment=1), dict(max_error_rate=0.35), dict(min_overlap=100),
         dict(min_overlap_ratio=0.9), dict(batch_size=1000), dict(use_graphs=1), dict(sync_batches=1)]


@pytest.fixture(autouse=True)
def device(monkeypatch):
    monkeypatch.setattr(engine, "device_info", lambda device=0: ("MI355X", 256))


@pytest.mark.parametrize("opts", OTHER, ids=lambda o: next(iter(o)))
def test_options_that_select_kernels_are_in_the_key(opts):
    base = dict(kmerlength=20)
    assert autotune.shape_key(STORAGE, **base) == autotune.shape_key(STORAGE, **base)
    assert autotune.shape_key(STORAGE, **{**base, **opts}) != autotune.shape_key(STORAGE, **base)


def test_defaults_and_given_defaults_share_a_key():
    given = dict(min_overlap=30, correction_type=0, num_hash_maps=48)
    assert autotune.shape_key(STORAGE, **given) == autotune.shape_key(STORAGE)


def test_choice_of_other_kernels_is_not_replayed(tmp_path):
    cache = tmp_path / "tune.json"
    cache.write_text(json.dumps({OLD_KEY: {"choice": {"engine": 1, "align_variant": 1}, "timings_ms": []}}))
    key = autotune.shape_key(STORAGE, kmerlength=20, use_quality_scores=0, paired=0)
    assert key not in json.loads(cache.read_text())


def test_swept_tiles_leave_out_the_default():
    assert 16 not in autotune.TILES_Q and 64 not in autotune.TILES_NOQ
    assert 20 in autotune.TILES_Q
    assert all(t % 4 == 0 and 4 <= t <= 64 for t in autotune.TILES_Q + autotune.TILES_NOQ)
