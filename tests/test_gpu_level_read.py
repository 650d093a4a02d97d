"""Reads of whole levels: four subsets to a lane with every remainder, levels
on both sides of the 4 MiB up to which the kernel writes to host memory itself,
each graph size class; single reads go by another unranking."""
import random
from math import comb

import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 4, 5, 7, 18, 19, 24, 25, 26])
def test_level_equals_single_reads(n):
    print("level read", n, flush=True)
    rng = random.Random(n)
    with api.Context(0) as ctx:
        dp = api.DynamicGPU(ctx)
        dp(G.gnp(n, 0.3, n + 1))
        for k in (range(n + 1) if n < 8 else (0, 1, 2, n // 2, n - 1, n)):
            level = dp.level(k)
            count = comb(n, k)
            assert len(level) == count
            some = set(range(min(count, 6))) | set(range(max(0, count - 6), count))
            some |= {rng.randrange(count) for _ in range(12)}
            for code in some:
                assert dp.GetTreedepth(n, k, code) == level[code], (k, code)
        assert dp.level(n)[0] == dp.treedepth
