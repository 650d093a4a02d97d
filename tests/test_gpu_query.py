"""Queries over tables of every kind: a subset's treedepth (every number of
three-vertex steps, two and four words to a tile) equals its entry of the level
read, and the eliminations of sparse, mostly disconnected sets are the
reference's."""
import math
import random

import numpy as np
import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G
from test_gpu_dp import mask_of, ref_elimination

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


@pytest.mark.parametrize("n,p", [(16, 0.1), (22, 0.09), (25, 0.08), (25, 0.2)])
def test_elimination_of_disconnected_sets(ctx, oracle, n, p):
    g = G.gnp(n, p, n + 1)
    levels = oracle.dp_fast(g, levels=True)[2]
    dp = api.DynamicGPU(ctx)
    dp(g)
    rng = random.Random(n)
    for k in (1, 2, 3, 5, n // 2, n - 2, n):
        code = rng.randrange(math.comb(n, k))
        S = mask_of(oracle.decode(n, k, code))
        print("eliminate", n, k, code, flush=True)
        assert dp.GetElimination(n, k, code) == ref_elimination(g, levels, S, k)


# 4 MiB of a level at a time: the last whole part, two parts, three
@pytest.mark.parametrize("n,ks", [(24, (11, 12)), (25, (11, 12)), (26, (12, 13))])
def test_levels_in_parts(ctx, oracle, n, ks):
    g = G.gnp(n, 0.2, n)
    levels = oracle.dp_fast(g, levels=True)[2]
    dp = api.DynamicGPU(ctx)
    dp(g)
    for k in ks:
        print("level", n, k, flush=True)
        at = sum(math.comb(n, i) for i in range(k))
        assert np.array_equal(dp.level(k), levels[at: at + math.comb(n, k)])
