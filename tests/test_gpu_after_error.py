"""A call that fails after it has launched something leaves nothing behind that
the next call's staging memory could meet."""
import ctypes as C

import numpy as np
import pytest

from gisbdw_amd import api, learn
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [8, 512])
def test_call_after_no_memory(oracle, count):
    """The gradient's rows (about 100 KB a graph) do not fit the budget when the
    graphs are on their way already; the same memory then stages a solve's
    record and the next scores."""
    graphs = [G.tree_plus_edges(20 + i % 40, 0.1, i) for i in range(count)]
    ns, adj = learn.pad_adj(graphs)
    tgt = np.ones(count, np.uint64)
    g = G.gnp(25, 0.2, 3)
    want = oracle.dp_fast(g)
    with api.Context() as free:
        prop = learn.Proposal(free)
        prop.init(1)
        scores = prop.scores_padded(ns, adj)
    # the solve's table, the other DP and network buffers, 1548 bytes a graph
    ctx = api.Context(mem_budget_bytes=(1 << 25) + 650000 + 1600 * count)
    prop = learn.Proposal(ctx)
    prop.init(1)
    dp = api.DynamicGPU(ctx)
    dp(g)
    for rep in range(4):
        print("no memory", count, rep, flush=True)
        with pytest.raises(api.TDError) as e:
            prop.loss_grad(ns, adj, tgt)
        assert e.value.code == api.TD_E_NOMEM
        dp(g)
        assert (dp.treedepth, dp.parent) == want
        assert np.array_equal(prop.scores_padded(ns, adj), scores)
    ctx.close()


def test_invalid_graph_comes_before_no_memory():
    ctx = api.Context(mem_budget_bytes=1 << 20)
    prop = learn.Proposal(ctx)
    prop.init(1)
    ns, adj = learn.pad_adj([G.path(9) for _ in range(2000)])
    tgt = np.ones(2000, np.uint64)
    calls = {"features": lambda: prop.features(ns, adj),
             "scores": lambda: prop.scores_padded(ns, adj),
             "gradient": lambda: prop.loss_grad(ns, adj, tgt),
             "train": lambda: prop.train(ns, adj, tgt, 1, 256)}
    for code in (api.TD_E_NOMEM, api.TD_E_INVALID):
        for name, call in calls.items():
            print(name, code, flush=True)
            with pytest.raises(api.TDError) as e:
                call()
            assert e.value.code == code, name
        adj[1500, 3] |= np.uint64(1 << 3)  # a self loop
    ctx.close()


@pytest.mark.parametrize("n", [9, 20, 24, 26])
def test_solve_after_an_error_of_another_call(oracle, n):
    """An error that an earlier HIP call of the thread has left may end a solve
    at its launch check; the solves after it are right."""
    hip = C.CDLL("libamdhip64.so.7")
    g = G.gnp(n, 0.25, n)
    want = oracle.dp_fast(g)
    ctx = api.Context()
    dp = api.DynamicGPU(ctx)
    for rep in range(3):
        print("left-over error", n, rep, flush=True)
        assert hip.hipSetDevice(1 << 20) != 0
        try:
            dp(g)
        except api.TDError as e:
            assert e.code == api.TD_E_HIP
        for _ in range(2):
            dp(g)
            assert (dp.treedepth, dp.parent) == want
        assert api.dp_solve_batch(ctx, [g, g], 0)[0] == [want[0]] * 2
    ctx.close()
