"""Batches that the device checks and takes from page-locked memory
(td_mlp_scores, td_mlp_loss_grad, td_mlp_train, td_heuristic_batch): an
invalid graph anywhere is the error the host check gives, for the lowest one,
and no result is written; and calls of more graphs than one staging chunk
(4096) equal the same graphs in smaller calls."""
import ctypes as C

import numpy as np
import pytest

from gisbdw_amd import api, learn
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu

BAD = {
    "asymmetric": ({0: 0b110}, "asymmetric"),
    "self loop": ({2: 0b1110}, "self loop"),
    "vertex >= n": ({1: 0b101 | 1 << 20}, "names a vertex"),
    "row beyond n": ({40: 1}, "rows beyond n"),
}


@pytest.mark.parametrize("kind", list(BAD))
def test_invalid_graph_is_refused(kind):
    ctx = api.Context()
    prop = learn.Proposal(ctx)
    prop.init(1)
    before = prop.get_weights()
    ns, adj = learn.pad_adj([G.path(9) for _ in range(70)])
    tgt = np.ones(70, np.uint64)
    rows, word = BAD[kind]
    for at in (66, 31):
        for v, r in rows.items():
            adj[at, v] = r
    print("invalid", kind, flush=True)
    P = C.POINTER
    out = np.full((70, 64), 7.0, np.float32)
    grad = np.full(prop.nparams, 7.0, np.float32)
    loss = C.c_float(7.0)
    p = lambda a, t: a.ctypes.data_as(P(t))  # noqa: E731
    calls = [
        lambda: ctx.lib.td_mlp_scores(ctx.h, 70, p(ns, C.c_int32), p(adj, C.c_uint64),
                                      p(out, C.c_float)),
        lambda: ctx.lib.td_mlp_loss_grad(ctx.h, 70, p(ns, C.c_int32), p(adj, C.c_uint64),
                                         p(tgt, C.c_uint64), C.byref(loss), p(grad, C.c_float)),
        lambda: ctx.lib.td_mlp_train(ctx.h, 70, p(ns, C.c_int32), p(adj, C.c_uint64),
                                     p(tgt, C.c_uint64), 1, 16, 1e-3, 1, None),
    ]
    for call in calls:
        assert call() == api.TD_E_INVALID
        assert word in ctx.lib.td_last_error(ctx.h).decode()
    assert (out == 7.0).all() and (grad == 7.0).all() and loss.value == 7.0
    assert np.array_equal(prop.get_weights(), before)
    if kind != "row beyond n":  # heuristics take packed rows
        packed = np.concatenate([adj[i, :9] for i in range(70)])
        td = np.full(70, 7, np.int32)
        rc = ctx.lib.td_heuristic_batch(ctx.h, 70, p(ns, C.c_int32), p(packed, C.c_uint64), 1,
                                        p(td, C.c_int32), None)
        assert rc == api.TD_E_INVALID and (td == 7).all()
        assert word in ctx.lib.td_last_error(ctx.h).decode()
    ns[5] = 65
    assert calls[0]() == api.TD_E_INVALID
    # and the context still works
    s = prop.scores([G.path(9)])[0]
    assert np.isfinite(s).all()
    ctx.close()


def test_more_graphs_than_one_chunk():
    ctx = api.Context()
    prop = learn.Proposal(ctx)
    prop.init(1)
    graphs = [G.tree_plus_edges(3 + i % 20, 0.1, i) for i in range(4099)]
    ns, adj = learn.pad_adj(graphs)
    print("chunks", flush=True)
    whole = prop.scores_padded(ns, adj)
    parts = np.concatenate([prop.scores_padded(ns[a:a + 1500], adj[a:a + 1500])
                            for a in range(0, 4099, 1500)])
    assert np.array_equal(whole, parts)
    tds, pars = api.heuristic_batch(ctx, graphs, "chain")
    again = [api.heuristic_batch(ctx, graphs[a:a + 1500], "chain") for a in range(0, 4099, 1500)]
    assert tds == sum((a[0] for a in again), [])
    assert pars == sum((a[1] for a in again), [])
    loss, grad = prop.loss_grad(ns, adj, np.ones(4099, np.uint64))
    assert np.isfinite(loss) and np.isfinite(grad).all()
    ctx.close()
