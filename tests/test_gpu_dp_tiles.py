"""Words per tile of the single-graph level kernels: the sizes at which a
graph changes from tiles of one word to two and four (n = 27, 28, 29),
against the oracle's treedepth, tree and level tables."""
import math

import numpy as np
import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [27, 28, 29])
def test_tile_widths_at_the_boundaries(ctx, oracle, n):
    g = G.gnp(n, 0.2, n)
    td, par, lv = oracle.dp_fast(g, levels=True)
    off = [0]
    for k in range(n + 1):
        off.append(off[-1] + math.comb(n, k))
    saved = ctx.get_param("dp.low_bits")
    try:
        for low_bits in (3, 4, 5):
            print("tiles n", n, "low_bits", low_bits, flush=True)
            ctx.set_param("dp.low_bits", low_bits)
            dp = api.DynamicGPU(ctx)
            dp(g)
            assert (dp.treedepth, dp.parent) == (td, par)
            for k in (0, 1, 2, 7, n // 2, n - 1, n):
                assert np.array_equal(dp.level(k), lv[off[k]: off[k + 1]]), (low_bits, k)
    finally:
        ctx.set_param("dp.low_bits", saved)
