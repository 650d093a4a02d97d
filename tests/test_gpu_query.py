"""Queries over tables of two and four words to a tile, and of every number of
three-vertex steps: a subset's treedepth equals its entry of the level read."""
import math
import random

import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,low_bits", [(3, 4), (20, 4), (27, 4), (28, 4), (29, 5)])
def test_single_reads_equal_level(n, low_bits):
    ctx = api.Context()
    ctx.set_param("dp.low_bits", low_bits)
    dp = api.DynamicGPU(ctx)
    rng = random.Random(n)
    dp(G.gnp(n, 0.3, n))
    for k in [k for k in (0, 1, 2, 3, 4, n - 4, n - 3, n - 1, n) if 0 <= k <= n]:
        print("level", n, k, flush=True)
        level = dp.level(k)
        for code in {0, len(level) - 1, rng.randrange(len(level)), rng.randrange(len(level))}:
            assert dp.GetTreedepth(n, k, code) == level[code], (k, code)
    assert math.comb(n, n) == 1 and dp.GetTreedepth(n, n, 0) == dp.treedepth
    ctx.close()
