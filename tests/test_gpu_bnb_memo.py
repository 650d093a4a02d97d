"""The search's common memo: wave counts from one to the most, also odd ones
(lanes past the waves' entries), and tables from the smallest, where buckets
fill up and entries are replaced, agree with the subset DP."""
import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu

BUDGET = 100000


def graphs():
    return [G.tree_plus_edges(26, 0.3, 5), G.tree_plus_edges(28, 0.15, 6),
            G.tree_plus_edges(29, 0.1, 7), G.gnp(25, 0.12, 9),
            G.relabeled(G.grid(5, 5), 2), G.path(27), G.complete(25)]


@pytest.fixture(scope="module")
def exact():
    with api.Context(0) as c:
        dp = api.DynamicGPU(c)
        return [dp(g).treedepth for g in graphs()]


@pytest.mark.parametrize("waves", [1, 3, 7, 16])
@pytest.mark.parametrize("memo_log2", [8, 0])
def test_common_memo(exact, oracle, waves, memo_log2):
    print("bnb memo", waves, memo_log2, flush=True)
    gs = graphs()
    with api.Context(0) as c:
        c.set_param("bnb.waves_per_graph", waves)
        c.set_param("bnb.memo_log2", memo_log2)
        c.set_param("bnb.node_budget", BUDGET)
        for _ in range(2):  # the second call finds the first one's entries
            tds, pars, cert, _ = api.bnb_solve_batch(c, gs)
            heur, lb, nodes = api.bnb_last_details(c, len(gs))
            for i, g in enumerate(gs):
                assert oracle.certify(g, pars[i], tds[i]), g.name
                assert lb[i] <= exact[i] <= tds[i] <= heur[i], g.name
                # settled, or the budget is spent
                assert cert[i] or int(nodes[i]) >= BUDGET, g.name
                assert not cert[i] or tds[i] == lb[i] == exact[i], g.name
