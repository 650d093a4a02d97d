"""Bottom-up levels wide enough for the workgroups of 1024 (more than 65536
subsets: the middle ones from n = 19 on), in each record width: every
entry of the history equals the oracle's."""
from math import comb

import numpy as np
import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G
from oracle_lib import Oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("make", [
    lambda: G.gnp(19, 0.2, 3),       # 92378 subsets at most, ragged slices
    lambda: G.gnp(20, 0.12, 1),      # 12-byte records at the widest levels
    lambda: G.gnp(21, 0.5, 4),       # 3 to 4 planes at wide levels
    lambda: G.complete(20),          # 3, 4, 8 planes: heights are the sizes
    lambda: G.edgeless(20),          # every component a single vertex
    lambda: G.relabeled(G.path(21), 5),
])
def test_wide_levels(make):
    g = make()
    print("bu wide", g.name, flush=True)
    td, order, parent, root, last, height = Oracle().bottom_up(g)
    c = api.Context(0)
    bu = api.BottomUpHeuristicGPU(c)
    bu(g)
    assert (bu.treedepth, bu.parent) == (td, parent)
    assert bu.GetElimination(g.n, g.n, 0) == order
    off = 0
    for k in range(g.n + 1):
        gl, gh = bu.level(k)
        end = off + comb(g.n, k)
        assert np.array_equal(gl, last[off:end]), k
        assert np.array_equal(gh, height[off:end]), k
        off = end
    c.close()
