"""Waits between workgroups that are given up (dp.flow_spin = 0: on the second
read of a word that is not there yet): that they are, who solves the graphs
then, and what the call reports."""
import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


def graphs():
    return [G.gnp(22, 0.3, 5), G.gnp(19, 0.2, 4), G.gnp(9, 0.3, 2)]


def test_single_solve_reports_the_level_kernels(oracle):
    """The flow path counts as one level kernel; the level kernels that take
    over are more."""
    ctx = api.Context()
    ctx.set_param("dp.flow_spin", 0)
    dp = api.DynamicGPU(ctx)
    for g, small in zip(graphs(), (False, False, True)):
        print("given up", g.name, flush=True)
        dp(g)
        assert (dp.treedepth, dp.parent) == oracle.dp_fast(g)
        st = dp.stats
        assert (st.level_kernels == 1) == small and (st.launches == 1) == small
    ctx.close()


def test_batch_reports_both_launches(oracle):
    ctx = api.Context()
    want = [oracle.dp_fast(g) for g in graphs()]
    print("batch", flush=True)
    for _ in range(2):  # the first call also loads and captures
        tds, pars, st = api.dp_solve_batch(ctx, graphs(), 0)
        assert list(zip(tds, pars)) == want and st.level_kernels == 1
    ctx.set_param("dp.flow_spin", 0)
    for _ in range(2):
        tds, pars, late = api.dp_solve_batch(ctx, graphs(), 0)
        assert list(zip(tds, pars)) == want
    assert late.level_kernels == 2 and late.launches >= st.launches + 2
    # the persistent kernel's time is in it: a workgroup by itself takes more
    # than 256 workgroups took
    assert late.level_ms > st.level_ms and late.total_ms >= late.level_ms + late.tree_ms
    ctx.close()


def test_batch_needs_no_more_room(oracle):
    """The graphs are solved in the batch's own memory, and the last single
    solve's queries stay where a search calls for the batch."""
    gs = [G.gnp(22, 0.3, 5), G.gnp(21, 0.2, 4)]
    want = [oracle.dp_fast(g) for g in gs]
    # tables, records, binomials, queue, and 2.1 + 1.1 MB of published words
    ctx = api.Context(mem_budget_bytes=(1 << 22) + (1 << 21) + (7 << 19) + (1 << 18))
    ctx.set_param("dp.flow_spin", 0)
    print("budget", flush=True)
    tds, pars, st = api.dp_solve_batch(ctx, gs, 0)
    assert list(zip(tds, pars)) == want and st.level_kernels == 2
    ctx.close()
    ctx = api.Context()
    ctx.set_param("dp.flow_spin", 0)
    dp = api.DynamicGPU(ctx)
    dp(G.gnp(13, 0.3, 5))
    level = dp.level(6).tobytes()
    hard = [G.random_cubic(20, 5), G.gnp(22, 0.6, 3)]
    print("search", flush=True)
    tds, _, cert, _ = api.bnb_solve_batch(ctx, hard)
    assert tds == [oracle.dp_fast(g)[0] for g in hard] and all(cert)
    assert dp.level(6).tobytes() == level
    ctx.close()
