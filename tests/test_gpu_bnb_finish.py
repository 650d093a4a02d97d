"""Small graphs (n <= 24) that the search leaves unsettled after 1024 nodes are
finished by the subset DP: certified answers equal to the oracle's, the last
single solve's queries stay, budgets up to 32768 nodes search as before, and a
byte budget without room for the DP goes back to the search."""
import random

import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


def hard_small():
    rng = random.Random(19)
    gs = [G.gnp(n, 0.6, rng.getrandbits(32)) for n in (18, 19, 22, 24)]
    gs += [G.random_cubic(20, 5), G.random_cubic(24, 6)]
    return gs + [G.tree_plus_edges(40, 0.1, 3), G.path(5), G.gnp(25, 0.15, 4)]


def test_finished_by_the_dp(oracle):
    ctx = api.Context()
    gs = hard_small()
    dp = api.DynamicGPU(ctx)
    g = G.gnp(13, 0.3, 5)
    dp(g)
    level = dp.level(6).tobytes()
    print("finish", flush=True)
    tds, pars, cert, st = api.bnb_solve_batch(ctx, gs)
    heur, lb, nodes = api.bnb_last_details(ctx, len(gs))
    for i, h in enumerate(gs):
        assert oracle.certify(h, pars[i], tds[i]) and lb[i] <= tds[i] <= heur[i]
        if h.n <= 24:
            assert cert[i] and tds[i] == oracle.dp_fast(h)[0] and lb[i] == tds[i], h.name
            assert int(nodes[i]) <= 1024 + 16 * 64
    assert st.certified == sum(cert) and st.kernel_ms > 0
    # the single solve's tables are still there to query
    assert dp.level(6).tobytes() == level and dp.GetTreedepth(13, 13, 0) == dp.treedepth
    b = api.BnBGPU(ctx)
    assert b(gs[2], 0) == tds[2] and b.certified
    # a budget that the early stop does not apply to
    ctx.set_param("bnb.node_budget", 20000)
    _, _, cert2, _ = api.bnb_solve_batch(ctx, [gs[3]])
    assert not cert2[0]
    ctx.close()


def test_no_room_for_the_dp(oracle):
    """The DP would claim 2^22 bytes; this budget leaves the search alone."""
    g = G.gnp(22, 0.15, 8)
    ctx = api.Context(mem_budget_bytes=(1 << 22) - 1)
    ctx.set_param("bnb.waves_per_graph", 1)
    ctx.set_param("bnb.memo_log2", 10)
    print("no room", flush=True)
    tds, pars, cert, _ = api.bnb_solve_batch(ctx, [g])
    heur, lb, nodes = api.bnb_last_details(ctx, 1)
    want = oracle.dp_fast(g)[0]
    assert oracle.certify(g, pars[0], tds[0]) and tds[0] >= want and lb[0] <= want
    assert not cert[0] or tds[0] == want
    assert int(nodes[0]) > 1024 or cert[0]
    ctx.close()
