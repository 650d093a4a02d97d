"""What a byte budget admits: calls that fit it exactly, one after another."""
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
