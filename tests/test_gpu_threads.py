"""Contexts in several host threads, one each: some capture their launch
sequences anew for every solve, others make their first uses and read tables."""
import threading

import pytest

from gisbdw_amd import api
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


def test_contexts_in_threads(oracle):
    graphs = [G.gnp(n, 0.3, n) for n in (9, 18, 20, 24, 25)]
    want = [oracle.dp_fast(g) for g in graphs]
    errors, done = [], threading.Event()

    def guarded(f):
        def run(i):
            try:
                f(i)
            except BaseException as e:  # noqa: BLE001
                errors.append(repr(e))
                done.set()
        return run

    @guarded
    def capture(i):
        with api.Context() as ctx:
            dp = api.DynamicGPU(ctx)
            for r in range(60):
                ctx.set_param("dp.grid_mult", 4 + r % 2)  # drops captured launches
                dp(graphs[-1])
                assert (dp.treedepth, dp.parent) == want[-1]
                if done.is_set():
                    return

    @guarded
    def read(i):
        while not done.is_set():
            with api.Context() as ctx:
                dp = api.DynamicGPU(ctx)
                bu = api.BottomUpHeuristicGPU(ctx)
                bu(G.path(11))
                for k, g in enumerate(graphs):
                    dp(g)
                    assert (dp.treedepth, dp.parent) == want[k]
                    assert dp.GetTreedepth(g.n, g.n, 0) == want[k][0]
                    for _ in range(20):
                        assert bu.GetTreedepth(11, 1, 3) == 1

    readers = [threading.Thread(target=read, args=(i,)) for i in range(2)]
    captures = [threading.Thread(target=capture, args=(i,)) for i in range(2)]
    print("threads", flush=True)
    for t in readers + captures:
        t.start()
    for t in captures:
        t.join()
    done.set()
    for t in readers:
        t.join()
    assert not errors, errors
