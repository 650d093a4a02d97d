"""What a byte budget admits: calls that fit it exactly, one after another."""
import math

import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


def least(calls, high):
    """The smallest budget (to 16 bytes) that admits calls(context)."""
    low = 0
    while high - low > 16:
        mid = (low + high) // 2
        ctx = api.Context(mem_budget_bytes=mid)
        try:
            calls(ctx)
            high = mid
        except api.TDError as e:
            assert e.code == api.TD_E_NOMEM
            low = mid
        finally:
            ctx.close()
    return high


@pytest.mark.parametrize("n", [6, 16, 20, 25])
def test_treedepth_query_needs_no_room(oracle, n):
    """A subset's treedepth is read within the budget of the solve itself."""
    g = G.gnp(n, 0.3, n)
    print("query", n, flush=True)
    ctx = api.Context(mem_budget_bytes=least(lambda c: api.DynamicGPU(c)(g), 1 << 26))
    dp = api.DynamicGPU(ctx)
    dp(g)
    assert dp.GetTreedepth(n, n, 0) == dp.treedepth == oracle.dp_fast(g)[0]
    ctx.close()


# Bytes that a table of one byte per subset takes in tiles of 2^low subsets,
# each level of tiles padded to 256 bytes, with the buffers beside it.
def byte_table(n, low):
    high, pad, tiles = max(n - low, 0), max(1, 256 >> low), 0
    for h in range(high + 1):
        tiles += -(-math.comb(high, h) // pad) * pad
    return tiles << low


RECORD, PASCAL = 4648, 139648


@pytest.mark.parametrize("low_bits", [2, 3, 4, 5])
def test_small_graphs_fit_where_byte_tables_did(oracle, low_bits):
    """Padding of the bit planes' levels does not outgrow the byte tables."""
    for n in range(1, 13):
        g = G.gnp(n, 0.4, n)
        want = oracle.dp_fast(g)
        print("budget", low_bits, n, flush=True)
        ctx = api.Context(mem_budget_bytes=byte_table(n, low_bits) + RECORD + 24 + PASCAL + 80)
        ctx.set_param("dp.low_bits", low_bits)
        dp = api.DynamicGPU(ctx)
        dp(g)
        assert (dp.treedepth, dp.parent) == want
        ctx.close()
        count = 16
        for mode in (0, 1, 2):
            rows = -(-byte_table(n, low_bits) // 256) * 256 + RECORD + 72
            chunks = 16 * (max(n - low_bits, 0) + 1) if mode == 1 else 0
            ctx = api.Context(mem_budget_bytes=count * (rows + chunks) + PASCAL + 256)
            ctx.set_param("dp.low_bits", low_bits)
            tds, pars, _ = api.dp_solve_batch(ctx, [g] * count, mode)
            assert list(zip(tds, pars)) == [want] * count, mode
            ctx.close()


@pytest.mark.parametrize("low_bits", [3, 4])
def test_packed_claim_at_32_vertices(low_bits):
    """17/32 of a byte per subset, as tiles of 16 subsets and more took."""
    n = 32
    ctx = api.Context(mem_budget_bytes=(17 << 27) + (1 << 20) + (64 << 20))
    for k, v in (("low_bits", low_bits), ("class_bits", 4), ("packed", 1)):
        ctx.set_param("dp." + k, v)
    dp = api.DynamicGPU(ctx)
    print("packed", low_bits, flush=True)
    dp(G.path(n))
    assert dp.treedepth == 6
    ctx.close()


def test_bottom_up_has_the_room_of_published_words(oracle):
    """The words that a solve of 19..24 vertices publishes are no claim on the
    budget: the bottom-up heuristic still gets all its levels."""
    g, h = G.gnp(20, 0.3, 20), G.gnp(16, 0.3, 1)
    want = oracle.dp_fast(g)[0]
    single = (1 << 20) + RECORD + 24 + PASCAL + 80
    bottom_up = least(lambda c: api.BottomUpHeuristicGPU(c)(h, h.n + 1), 1 << 24)
    for iterations in (-1, h.n + 1):
        # what is left over is less than the 0.5 MB of published words
        ctx = api.Context(mem_budget_bytes=single + bottom_up + (8 << 10))
        dp = api.DynamicGPU(ctx)
        print("bottom up", iterations, flush=True)
        dp(g)
        bu = api.BottomUpHeuristicGPU(ctx)
        bu(h, iterations)
        assert bu.GetIterationsPerformed() == h.n + 1
        dp(g)
        assert dp.treedepth == want
        ctx.close()


def test_search_gives_the_dp_s_memory_back(oracle):
    """Small graphs that the search hands to the subset DP leave nothing of it
    on the budget: what fits after a search without the DP still fits."""
    hard = [G.random_cubic(20, 5), G.gnp(18, 0.6, 3)]
    g = G.gnp(21, 0.25, 8)
    want = oracle.dp_fast(g)

    def search(ctx, nodes):
        for k, v in (("waves_per_graph", 1), ("memo_log2", 10), ("node_budget", nodes)):
            ctx.set_param("bnb." + k, v)
        return api.bnb_solve_batch(ctx, hard)

    def alone(ctx):
        search(ctx, 20000)  # too few for the DP to step in
        api.DynamicGPU(ctx)(g)

    ctx = api.Context(mem_budget_bytes=least(alone, 1 << 24))
    dp = api.DynamicGPU(ctx)
    print("search, then solve", flush=True)
    tds, _, cert, _ = search(ctx, 50000)
    assert all(cert) and tds == [oracle.dp_fast(h)[0] for h in hard]
    dp(g)
    assert (dp.treedepth, dp.parent) == want
    # beside a solve that fills the budget the search does without the DP, and
    # the solve's queries go on
    tds, pars, _, _ = search(ctx, 50000)
    assert all(oracle.certify(h, p, t) for h, p, t in zip(hard, pars, tds))
    assert dp.GetTreedepth(g.n, g.n, 0) == want[0]
    ctx.close()
