"""Output pointers that a call cannot do without: null is an error, and the
context goes on working."""
import ctypes as C

import numpy as np
import pytest

from gisbdw_amd import api, learn
from gisbdw_amd import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("call", ["td_mlp_features", "td_mlp_scores"])
def test_null_output(call):
    ctx = api.Context()
    prop = learn.Proposal(ctx)
    prop.init(1)
    ns, adj = learn.pad_adj([G.path(9), G.cycle(12)])
    p = lambda a, t: a.ctypes.data_as(C.POINTER(t))  # noqa: E731
    print("null", call, flush=True)
    rc = getattr(ctx.lib, call)(ctx.h, 2, p(ns, C.c_int32), p(adj, C.c_uint64), None)
    assert rc == api.TD_E_INVALID
    assert np.isfinite(prop.scores([G.path(9)])[0]).all()
    ctx.close()
