"""The autotuner's candidates hold the automatic shapes for every path-pool
size, so that tuning a batch is never slower than leaving it alone."""
from rise_amd import autotune


def test_automatic_shapes_are_candidates():
    got = list(autotune.candidates(max_paths=(1 << 22, 1 << 24)))
    for m in (1 << 22, 1 << 24):
        assert {"persistent": 0, "trace_block": 0, "max_paths": m, "stack": 0} in got
    assert len(got) == len({tuple(sorted(t.items())) for t in got}) == 26
