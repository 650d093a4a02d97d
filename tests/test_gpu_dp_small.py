"""Graphs of at most 24 vertices, which a single solve resolves in one launch:
in one workgroup's LDS (n <= 18) or in several workgroups that pass finished
words on (n = 19..24), against the oracle's treedepth, tree and level tables;
the same kernels in batch calls; and the way back to the level kernels where
a wait is given up or the byte budget has no room for the published words."""
import math
import random

import numpy as np
import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


def check_levels(dp, g, lv, ks):
    off = [0]
    for k in range(g.n + 1):
        off.append(off[-1] + math.comb(g.n, k))
    for k in ks:
        assert np.array_equal(dp.level(k), lv[off[k]: off[k + 1]]), (g.name, k)


# every size: workgroups of 64 to 1024 threads up to 18, then 8 to 256
# workgroups; complete graphs have the deepest tables, sparse ones the most
# disconnected sets
@pytest.mark.parametrize("n", list(range(1, 25)))
def test_every_size(ctx, oracle, n):
    rng = random.Random(n)
    dp = api.DynamicGPU(ctx)
    graphs = [G.gnp(n, rng.uniform(0.1, 0.5), rng.getrandbits(32)), G.complete(n),
              G.edgeless(n), G.path(n)]
    for g in graphs[: 4 if n <= 20 else 2]:
        print("one launch", g.name, flush=True)
        td, par, lv = oracle.dp_fast(g, levels=True)
        dp(g)
        assert (dp.treedepth, dp.parent) == (td, par), g.name
        check_levels(dp, g, lv, range(n + 1) if n <= 18 else (0, 1, 2, 5, n // 2, n - 1, n))
        S = rng.getrandbits(n) | 1
        k = bin(S).count("1")
        code, i = 0, 0
        for v in range(n):
            if S >> v & 1:
                i += 1
                code += math.comb(v, i)
        order = dp.GetElimination(n, k, code)
        assert sorted(order) == [v for v in range(n) if S >> v & 1]


def test_batch_shares_out_by_size(ctx, oracle):
    """Few graphs of 19..24 vertices (several workgroups each, one launch or
    more), with smaller ones; with larger ones beside them; and many."""
    rng = random.Random(3)

    def draw(sizes):
        return [G.gnp(n, rng.uniform(0.15, 0.5), rng.getrandbits(32)) for n in sizes]

    batches = {"one launch": draw([19, 24, 7, 18, 1, 12]),
               "several launches": draw([24, 24, 23, 22, 21, 20, 19, 19, 16]),
               "with larger": draw([25, 22, 19, 14, 18]),
               "many": draw([19] * 60 + [20] * 40 + [9] * 300)}
    for name, graphs in batches.items():
        print("batch", name, flush=True)
        want = [oracle.dp_fast(g) for g in graphs]
        for rep in range(2):
            tds, pars, st = api.dp_solve_batch(ctx, graphs, 0)
            assert list(zip(tds, pars)) == want, (name, rep)
        assert st.graphs == len(graphs) and st.level_kernels == 1


def test_waits_given_up(oracle):
    """dp.flow_spin = 0: every wait is given up at once, the kernel ends by
    itself, and the level kernels answer (single solves and a batch)."""
    ctx = api.Context()
    ctx.set_param("dp.flow_spin", 0)
    dp = api.DynamicGPU(ctx)
    graphs = [G.gnp(22, 0.3, 5), G.gnp(19, 0.2, 4), G.gnp(9, 0.3, 2)]
    for g in graphs:
        print("given up", g.name, flush=True)
        td, par, lv = oracle.dp_fast(g, levels=True)
        dp(g)
        assert (dp.treedepth, dp.parent) == (td, par)
        check_levels(dp, g, lv, (1, g.n // 2, g.n))
    tds, pars, _ = api.dp_solve_batch(ctx, graphs, 0)
    assert list(zip(tds, pars)) == [oracle.dp_fast(g) for g in graphs]
    ctx.close()


def test_no_room_for_published_words(oracle):
    """A byte budget that holds the table (one byte per subset) and little
    more: the level kernels solve the graph; and the published words give way
    to a larger graph's table."""
    g = G.gnp(22, 0.3, 5)
    want = oracle.dp_fast(g)
    tight = api.Context(mem_budget_bytes=(1 << 22) + (1 << 20))
    dp = api.DynamicGPU(tight)
    print("no room", flush=True)
    dp(g)
    assert (dp.treedepth, dp.parent) == want
    tight.close()
    room = api.Context(mem_budget_bytes=(1 << 24) + (1 << 20))
    dp = api.DynamicGPU(room)
    dp(g)
    assert (dp.treedepth, dp.parent) == want
    h = G.gnp(24, 0.25, 11)
    dp(h)
    assert (dp.treedepth, dp.parent) == oracle.dp_fast(h)
    dp(g)
    assert (dp.treedepth, dp.parent) == want
    room.close()
