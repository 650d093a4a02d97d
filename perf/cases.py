"""What a program of this library has it do, as measurable cases.

A case is a dict of plain values; `kind` names the path:

  solve      one graph through DynamicGPU: treedepth and decomposition
  query      one graph through DynamicGPU, then one level table read back
  batch      many graphs in one batched subset-DP call
  bottom_up  the bottom-up heuristic on one graph
  heuristic  the reference's heuristic chain on a batch of sparse graphs
  search     the batched branch-and-bound on sparse graphs
  scores     the learned proposal's forward pass on a batch of graphs
  gradient   its forward and backward pass (what training repeats)

Graphs go in and trees come out in host memory, so inputs are host arrays and
every pass is a whole synchronous call.  Sizes and families are those of the
library's workloads (gisbdw_amd/graphs.py, bench.py, tests).
"""
import ctypes as C
import math
import random

import numpy as np

from gisbdw_amd import api, learn
from gisbdw_amd import graphs as G

HIDDEN = 64
MATRIX = HIDDEN * HIDDEN


def listed():
    return [
        # the smallest call: one small graph, where latency and launches count
        {"name": "solve 9", "kind": "solve", "n": 9, "density": 0.35},
        # the single-graph workload: G(20, 0.3)
        {"name": "solve 20", "kind": "solve", "n": 20, "density": 0.3},
        # a large single graph of odd size, in the default launch shape
        {"name": "solve 29", "kind": "solve", "n": 29, "density": 0.2},
        # a solve followed by a read of its largest level table
        {"name": "query 23", "kind": "query", "n": 23, "density": 0.25},
        # the headline workload: eight n = 30 graphs (G(n, 0.2) and grids with
        # a tenth of their edges dropped) in the launch shape that
        # td_dp_autotune picks for n = 30
        {"name": "batch 8 x 30", "kind": "batch", "count": 8, "low": 30, "high": 30,
         "tuned": True},
        # the batched workload: G(n, p), n in 12..24, p in 0.15..0.5, in the
        # shape that td_dp_autotune_batch picks for it
        {"name": "batch 4096", "kind": "batch", "count": 4096, "low": 12, "high": 24,
         "tuned": True},
        # a small ragged batch in the default shape
        {"name": "batch 200", "kind": "batch", "count": 200, "low": 5, "high": 19,
         "tuned": False},
        # the bottom-up heuristic, all levels
        {"name": "bottom_up 25", "kind": "bottom_up", "n": 25, "density": 0.15},
        # upper bounds for the search workload: cubic graphs, grids, near-trees
        {"name": "heuristic 1024", "kind": "heuristic", "count": 1024},
        # branch-and-bound on the families it certifies
        {"name": "search 256", "kind": "search", "count": 256, "high": 50},
        # the learned order for the search workload
        {"name": "scores 1024", "kind": "scores", "count": 1024},
        # one training minibatch
        {"name": "gradient 512", "kind": "gradient", "count": 512},
    ]


def _spread(rng, low, high):
    """A whole number from low to high, uniform in its logarithm."""
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    kind = rng.choice(["solve", "solve", "solve", "query", "batch", "batch", "batch",
                       "bottom_up", "heuristic", "search", "scores", "gradient"])
    if kind == "solve":
        return {"kind": kind, "n": rng.randint(6, 30), "density": round(rng.uniform(0.12, 0.5), 3)}
    if kind == "query":
        return {"kind": kind, "n": rng.randint(12, 24), "density": round(rng.uniform(0.15, 0.5), 3)}
    if kind == "batch":
        if rng.random() < 0.3:
            low = rng.randint(27, 29)
            return {"kind": kind, "count": rng.randint(2, 8), "low": low,
                    "high": rng.randint(low, 30), "tuned": rng.random() < 0.5}
        low = rng.randint(4, 16)
        return {"kind": kind, "count": _spread(rng, 16, 4096), "low": low,
                "high": rng.randint(low + 2, 24), "tuned": rng.random() < 0.5}
    if kind == "bottom_up":
        return {"kind": kind, "n": rng.randint(12, 25), "density": round(rng.uniform(0.1, 0.35), 3)}
    if kind == "search":
        return {"kind": kind, "count": _spread(rng, 24, 256), "high": rng.randint(42, 50)}
    return {"kind": kind, "count": _spread(rng, 32, 512 if kind == "gradient" else 1024)}


# ---- inputs ---------------------------------------------------------------
def _gnp_rows(rng, n, p):
    """Adjacency rows of one G(n, p), as uint64."""
    a = np.triu(rng.random((n, n)) < p, 1)
    a = (a | a.T).astype(np.uint64)
    return (a << np.arange(n, dtype=np.uint64)[None, :]).sum(1, dtype=np.uint64)


def _graph(rng, n, p):
    return G.Graph(n, [int(x) for x in _gnp_rows(rng, n, p)])


def _padded(rows_list):
    ns = np.array([len(r) for r in rows_list], np.int32)
    adj = np.zeros((len(rows_list), 64), np.uint64)
    for i, r in enumerate(rows_list):
        adj[i, : len(r)] = r
    return ns, adj


def _sizes(case, low, high):
    """Vertex counts of a batch, spread evenly over low..high, in an order that
    belongs to the case (the seed draws the graphs, not their sizes)."""
    sizes = [low + i % (high - low + 1) for i in range(case["count"])]
    random.Random(case["count"]).shuffle(sizes)
    return sizes


def _batch_graphs(case, seed):
    """Rows of the graphs of a batch case."""
    rng = np.random.default_rng(seed)
    rows = []
    for i, n in enumerate(_sizes(case, case["low"], case["high"])):
        if case["low"] <= 26:
            rows.append(_gnp_rows(rng, n, rng.uniform(0.15, 0.5)))
        elif i % 2 and (n % 5 == 0 or n % 6 == 0):  # grids where one fits, else G(n, 0.2)
            side = 5 if n % 5 == 0 else 6
            g = G.grid_dropped(side, n // side, 0.10, int(rng.integers(1 << 31)))
            rows.append(g.adj_array())
        else:
            rows.append(_gnp_rows(rng, n, 0.2))
    return rows


def _sparse_graphs(case, seed):
    """The search workload's mix for n in 40..64: a quarter random cubic, a
    quarter relabelled 7 x 7 and 8 x 8 grids, half near-trees."""
    rng = random.Random(seed)
    gs = []
    for i, n in enumerate(_sizes(case, 40, 64)):
        s = rng.getrandbits(32)
        if i % 4 == 0:
            gs.append(G.random_cubic(n + n % 2, s))
        elif i % 4 == 1:
            gs.append(G.relabeled(G.grid(7, 7) if i % 8 == 1 else G.grid(8, 8), s))
        else:
            gs.append(G.tree_plus_edges(n, 0.10, s))
    return gs


def _search_graphs(case, seed):
    """Near-trees with n in 40..high and small random cubic graphs, which the
    search certifies within its default budget."""
    rng = random.Random(seed)
    gs = []
    for i, n in enumerate(_sizes(case, 40, case["high"])):
        s = rng.getrandbits(32)
        gs.append(G.random_cubic(14 + 2 * (n % 4), s) if i % 4 == 3
                  else G.tree_plus_edges(n, 0.10, s))
    return gs


def _learn_inputs(case, seed):
    rng = np.random.default_rng(seed)
    if case["kind"] == "scores":
        return learn.pad_adj(_sparse_graphs(case, seed)), None
    rows = [_gnp_rows(rng, n, rng.uniform(0.1, 0.5)) for n in _sizes(case, 8, 24)]
    targets = np.zeros(len(rows), np.uint64)
    for i, r in enumerate(rows):  # about 0.6 of the vertices are optimal roots
        n = len(r)
        pick = rng.random(n) < 0.6
        pick[int(rng.integers(n))] = True
        targets[i] = (pick.astype(np.uint64) << np.arange(n, dtype=np.uint64)).sum()
    return _padded(rows), targets


def _weights(seed):
    """Weights as td_mlp_init draws them (uniform, scaled by the fan-in), with
    nonzero biases."""
    rng = np.random.default_rng(seed + 77)

    def layer(out, fan):
        return [rng.uniform(-1, 1, out * fan) * math.sqrt(6 / fan), rng.uniform(-0.1, 0.1, out)]

    parts = layer(HIDDEN, 4)
    for matrices in (2, 2, 1, 1):
        for _ in range(matrices):
            w, b = layer(HIDDEN, HIDDEN)
            parts.append(w)
        parts.append(b)
    parts += layer(1, HIDDEN)
    return np.concatenate(parts).astype(np.float32)


# the launch shapes that the autotuner keeps for the two batch workloads
TUNED_LARGE = {"dp.class_bits": 4, "dp.low_bits": 5, "dp.block": 256, "dp.grid_mult": 2}
TUNED_SMALL = {"dp.low_bits": 5, "dp.batch_block": 512, "dp.batch_wg_per_cu": 8}


def prepare(case, seed):
    kind = case["kind"]
    ctx = api.Context(0)
    state = {"kind": kind, "ctx": ctx}
    if kind in ("solve", "query", "bottom_up"):
        state["graph"] = _graph(np.random.default_rng(seed), case["n"], case["density"])
        state["solver"] = (api.BottomUpHeuristicGPU if kind == "bottom_up"
                           else api.DynamicGPU)(ctx)
    elif kind == "batch":
        rows = _batch_graphs(case, seed)
        state["ns"] = np.array([len(r) for r in rows], np.int32)
        state["adj"] = np.concatenate(rows)
        if case["tuned"]:
            for k, v in (TUNED_LARGE if case["low"] > 26 else TUNED_SMALL).items():
                ctx.set_param(k, v)
    elif kind == "heuristic":
        state["ns"], state["adj"] = api.pack_graphs(_sparse_graphs(case, seed))
    elif kind == "search":
        state["ns"], state["adj"] = api.pack_graphs(_search_graphs(case, seed))
    else:
        (state["ns"], state["adj"]), state["targets"] = _learn_inputs(case, seed)
        state["net"] = learn.Proposal(ctx)
        state["net"].set_weights(_weights(seed))
    return state


# ---- one pass -------------------------------------------------------------
def _heuristic(state):
    """td_heuristic_batch on packed arrays, through the C interface."""
    ns, adj, ctx = state["ns"], state["adj"], state["ctx"]
    depth = np.zeros(len(ns), np.int32)
    parent = np.zeros(int(ns.sum()), np.int8)
    ctx.check(ctx.lib.td_heuristic_batch(
        ctx.h, len(ns), ns.ctypes.data_as(C.POINTER(C.c_int32)),
        adj.ctypes.data_as(C.POINTER(C.c_uint64)), api.HEURISTIC_KINDS["chain"],
        depth.ctypes.data_as(C.POINTER(C.c_int32)), parent.ctypes.data_as(C.POINTER(C.c_int8))))
    return {"depth": depth, "parent": parent}


def run(state):
    kind = state["kind"]
    if kind in ("solve", "query", "bottom_up"):
        solver, g = state["solver"], state["graph"]
        solver(g)
        out = {"treedepth": solver.treedepth, "parent": np.array(solver.parent, np.int8)}
        if kind == "query":
            out["level"] = solver.level(g.n // 2)
        return out
    if kind == "batch":
        td, parent, _ = api.dp_solve_batch_arrays(state["ctx"], state["ns"], state["adj"], 0)
        return {"treedepth": td, "parent": parent}
    if kind == "heuristic":
        return _heuristic(state)
    if kind == "search":
        # the tree returned with a certified treedepth is whichever optimal one
        # the graph's waves found first: only the answers are the same each time
        td, _, certified, _ = api.bnb_solve_batch_arrays(state["ctx"], state["ns"], state["adj"])
        return {"treedepth": td, "certified": certified.astype(np.uint8)}
    if kind == "scores":
        return {"scores": state["net"].scores_padded(state["ns"], state["adj"])}
    loss, gradient = state["net"].loss_grad(state["ns"], state["adj"], state["targets"])
    return {"loss": np.float32(loss), "gradient": gradient}


# ---- what a pass cannot do without ------------------------------------------
def work(case):
    """Bytes: inputs and outputs once, and for a single solve one byte for
    each subset's treedepth, which the queries read afterwards.  Operations:
    one comparison for every vertex of every subset (the subset DP and the
    bottom-up heuristic), the multiply-adds of the network, or (heuristics and
    search, whose least work is not known) one pass over every graph's rows
    for each vertex that leaves it."""
    kind = case["kind"]
    if kind in ("solve", "query", "bottom_up"):
        n = case["n"]
        out = math.comb(n, n // 2) if kind == "query" else 0
        return {"bytes": 9 * n + (1 << n) + 2 * out, "flops": n << (n - 1)}
    count = case["count"]
    if kind == "batch":
        sizes = range(case["low"], case["high"] + 1)
        mean = sum(n << (n - 1) for n in sizes) / len(sizes)
        return {"bytes": count * (9 * sum(sizes) / len(sizes) + 5), "flops": count * mean}
    if kind in ("heuristic", "search"):
        n = 52 if kind == "heuristic" else 0.75 * (40 + case["high"]) / 2 + 0.25 * 17
        return {"bytes": count * (9 * n + 6), "flops": count * n * n}
    n = 52 if kind == "scores" else 16
    forward = 2 * n * (6 * MATRIX + 5 * HIDDEN)
    weights = 4 * (6 * MATRIX + 10 * HIDDEN + 1)
    if kind == "scores":
        return {"bytes": weights + count * (512 + 256), "flops": count * forward}
    return {"bytes": 2 * weights + count * (512 + 8), "flops": 3 * count * forward}


# ---- the network in 64 bits ---------------------------------------------------
def _features(ns, adj):
    """deg/4, core number/4, vertices within distance 2 / 16, eccentricity/8,
    and the adjacency matrices (rows beyond n are zero)."""
    bits = (adj[:, :, None] >> np.arange(64, dtype=np.uint64)) & np.uint64(1)
    A = bits.astype(np.float64)
    inside = np.arange(64)[None, :] < ns[:, None]
    core = np.zeros(inside.shape)
    for k in range(1, 64):
        alive = inside.copy()
        while True:
            keep = alive & ((A @ alive[:, :, None].astype(float))[:, :, 0] >= k)
            if (keep == alive).all():
                break
            alive = keep
        if not alive.any():
            break
        core[alive] = k
    eye = np.eye(64)[None]
    two = ((A @ A + A) > 0) & (eye == 0)
    seen = np.broadcast_to(eye, A.shape) > 0
    front, ecc = seen, np.zeros(inside.shape)
    while True:
        front = ((front.astype(float) @ A) > 0) & ~seen
        grew = front.any(2)
        if not grew.any():
            break
        ecc += grew
        seen = seen | front
    x = np.stack([A.sum(2) / 4, core / 4, two.sum(2) / 16, ecc / 8], 2) * inside[:, :, None]
    return x, A, inside


def exact(case, seed):
    """Scores, loss and gradient in 64 bits; the other outputs are whole numbers."""
    kind = case["kind"]
    if kind not in ("scores", "gradient"):
        return None
    (ns, adj), targets = _learn_inputs(case, seed)
    x, A, inside = _features(ns, adj)
    flat = _weights(seed).astype(np.float64)
    at, shapes = 0, [(HIDDEN, 4), (HIDDEN,)]
    for matrices in (2, 2, 1, 1):
        shapes += [(HIDDEN, HIDDEN)] * matrices + [(HIDDEN,)]
    shapes += [(1, HIDDEN), (1,)]
    P = []
    for s in shapes:
        P.append(flat[at: at + math.prod(s)].reshape(s))
        at += math.prod(s)
    W0, b0, S1, N1, b1, S2, N2, b2, W3, b3, W4, b4, w5, b5 = P
    degree = A.sum(2)
    mean = A / np.maximum(degree, 1)[:, :, None]
    h0 = np.maximum(x @ W0.T + b0, 0)
    m1 = mean @ h0
    h1 = np.maximum(h0 @ S1.T + m1 @ N1.T + b1, 0)
    m2 = mean @ h1
    h2 = np.maximum(h1 @ S2.T + m2 @ N2.T + b2, 0)
    z1 = np.maximum(h2 @ W3.T + b3, 0)
    z2 = np.maximum(z1 @ W4.T + b4, 0)
    s = (z2 @ w5.T)[:, :, 0] + b5
    if kind == "scores":
        return {"scores": np.where(inside, s, 0.0)}
    s = np.where(inside, s, -np.inf)
    e = np.exp(s - s.max(1, keepdims=True))
    p = e / e.sum(1, keepdims=True)
    t = ((targets[:, None] >> np.arange(64, dtype=np.uint64)) & np.uint64(1)).astype(np.float64)
    t /= t.sum(1, keepdims=True)
    loss = -(t * np.log(np.where(inside, p, 1.0))).sum(1).mean()
    ds = ((p - t) * inside / len(ns))[:, :, None]

    def product(g, y):
        return np.einsum("gvo,gvi->oi", g, y, optimize=True)

    def column(g):
        return g.sum((0, 1))

    back = [column(ds), product(ds, z2)]
    g = ds * w5 * (z2 > 0)
    back += [column(g), product(g, z1)]
    g = g @ W4 * (z1 > 0)
    back += [column(g), product(g, h2)]
    g = g @ W3 * (h2 > 0)
    transposed = mean.transpose(0, 2, 1)
    for own, near, y, m in ((S2, N2, h1, m2), (S1, N1, h0, m1)):
        back += [column(g), product(g, m), product(g, y)]
        g = (g @ own + transposed @ (g @ near)) * (y > 0)
    back += [column(g), product(g, x)]
    return {"loss": loss, "gradient": np.concatenate([b.ravel() for b in reversed(back)])}
