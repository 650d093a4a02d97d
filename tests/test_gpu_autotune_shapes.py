"""The autotuners change only what makes a difference to what they time:
parameters that no launch of the size reads stay as they are, and candidates
that launch the same share one time."""
import json

import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu

KEYS = ("low_bits", "tiles_per_lane", "block", "class_bits", "class_min_nh", "grid_mult", "packed",
        "batch_block", "batch_wg_per_cu", "use_graph", "streams")


def shape(ctx):
    return {k: ctx.get_param("dp." + k) for k in KEYS}


@pytest.mark.parametrize("n", [8, 16, 19, 24])
@pytest.mark.parametrize("low_bits", [2, 5])
def test_small_sizes_leave_the_context_alone(tmp_path, n, low_bits):
    ctx = api.Context()
    ctx.set_param("dp.low_bits", low_bits)
    ctx.set_param("dp.block", 256)
    before = shape(ctx)
    cache = tmp_path / "tune.jsonl"
    print("tune", n, flush=True)
    best = ctx.autotune(n, cache)
    assert shape(ctx) == before
    lines = [json.loads(x) for x in cache.read_text().splitlines()]
    times = {x["level_ms"] for x in lines}
    assert len(times) == 1 and times.pop() == pytest.approx(best, abs=1e-4)
    # a cached line does not change it either
    cache.write_text(cache.read_text().replace('"low_bits":%d' % low_bits, '"low_bits":4'))
    assert ctx.autotune(n, cache) == pytest.approx(best, abs=1e-4) and shape(ctx) == before
    ctx.close()


@pytest.mark.parametrize("n", [25, 28])
def test_equal_launches_share_a_time(tmp_path, n):
    ctx = api.Context()
    ctx.set_param("dp.low_bits", 5)
    ctx.set_param("dp.class_bits", 3)
    before = shape(ctx)
    cache = tmp_path / "tune.jsonl"
    print("tune", n, flush=True)
    ctx.autotune(n, cache)
    after = shape(ctx)
    assert {k for k in KEYS if before[k] != after[k]} <= {"tiles_per_lane", "block", "grid_mult",
                                                         *(["low_bits"] if n > 27 else [])}
    if n == 28:  # two words a tile at most: 4 and 5 are alike, and 5 was there
        assert after["low_bits"] in (3, 5)
    times = {}
    for x in map(json.loads, cache.read_text().splitlines()):
        words = min(x["low_bits"] - 3, n - 27) if n > 27 else 0
        times.setdefault((words, x["tiles_per_lane"], x["block"], x["grid_mult"]),
                         set()).add(x["level_ms"])
    assert all(len(t) == 1 for t in times.values()), times
    ctx.close()


def test_batch_without_a_persistent_launch():
    ctx = api.Context()
    before = shape(ctx)
    print("tune batch", flush=True)
    api.dp_autotune_batch(ctx, [G.gnp(n, 0.3, n) for n in (5, 9, 14, 18, 20)])
    assert shape(ctx) == before
    ctx.close()
