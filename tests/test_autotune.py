"""The autotuner's candidates hold the automatic shapes for every path-pool
size, so that tuning a batch is never slower than leaving it alone, and it takes
them unless a chosen shape is more than a hundredth faster."""
import dataclasses

import pytest

from rise_amd import autotune, pt_scene


def test_automatic_shapes_are_candidates():
    got = list(autotune.candidates(max_paths=(1 << 22, 1 << 24)))
    for m in (1 << 22, 1 << 24):
        assert {"persistent": 0, "trace_block": 0, "max_paths": m, "stack": 0} in got
    assert len(got) == len({tuple(sorted(t.items())) for t in got}) == 26


@pytest.mark.parametrize("chosen_ms,automatic", [(9.95, True), (9.0, False), (11.0, True)])
def test_automatic_shapes_before_a_tie(monkeypatch, chosen_ms, automatic):
    space = list(autotune.candidates(max_paths=(1 << 22,)))
    monkeypatch.setattr(autotune, "time_batch", lambda items, tn, repeats: chosen_ms if tn["persistent"] else 10.0)
    r = dataclasses.replace(pt_scene.cornell_box()[1], spp=4)
    best, results = autotune.tune([(None, r)], space=space)
    assert len(results) == len(space) and (best["persistent"] == 0) == automatic
