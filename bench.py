#!/usr/bin/env python3
"""Benchmark of the MI355X treedepth solver; prints ONE JSON line.

Default workload (the n = 30 subset-DP configuration): 8 graphs, 4 x G(30,0.2)
seeds 0-3 and 4 x 5x6 grids with 5 of their 49 edges dropped, seeds 0-3.  One
step = one td_dp_solve_batch call on the 8 graphs: the full subset DP (all
2^30 subsets) and the decomposition of each graph, the level kernels those of
td_dp_solve, two graphs' level sequences in flight at once on two streams
(each starting when the previous graph is half done; dp.streams = 2, or one
graph at a time with --streams 1), each graph's decomposition on a third
stream.  value = subsets resolved per second over the timed steps (wall
clock; every call is synchronous).

roofline: the level kernels against HBM peak, with achieved = compulsory
bytes / GPU time of the level launches (HIP events on the level streams
around each graph's level sequence; the union of those intervals, so time
in which two graphs' levels overlap counts once, and avg_launch_ms is that
time over the launches: the period of one launch at the achieved rate, not
the duration of a single kernel, which runs beside another graph's
kernels), compulsory bytes = 0.75 * 2^n per graph
(every level table, three bits per subset, written once and read back once by
the next level).  The
per-subset model of k one-byte reads of level k-1 plus one write, 2^(n-1)
(n+2) bytes per graph, counts reads that the kernel serves from registers
and caches; its rate is reported beside as model_GBps, not as the roofline.
A graph's levels run as DPLevelKernel launches, except the runs of small levels
at either end, which one DPSmallLevelsKernel workgroup does per run.  Per-launch
figures divide by that launch count.
traffic is NOT measured by this run: it is the rocprofv3 --pmc figure (read
and write bytes per launch from the L2's request counts by size) that the
committed summary profiles/dp_level_kernel_n30_traffic.md holds for the
launch shape that ran (null if it has none); traffic_over_compulsory divides
it by the compulsory bytes per launch.

Launch shape: td_dp_autotune picks (low_bits, tiles_per_lane, grid_mult, block) for n before the warm-up, unless --no-autotune or an
explicit shape flag is given.

cpu_baseline: the oracle's flat-table DP (OpenMP over each level) timed on the
host on a bounded sample: the subgraph induced by the first m vertices of the
first workload graph, m chosen so the run takes about 10-20 s.

extra: copy bandwidth; branch-and-bound certified graphs/s on the 256- and
1024-graph sparse workloads (plain and learned order, proposal trained here);
the single G(20,0.3) graph end to end and the 4096-graph batch before and
after td_dp_autotune_batch; and the oracle's CPU paths for the same
configurations (faithful DynamicCPU, flat-table DP, BranchAndBound) on
bounded samples.

Other workloads: --workload dp20 | dpbatch | bottomup | bnb.  bnb: the
1024-graph sparse workload (n in [40,64]), learned-ordered against plain
branch-and-bound at 5e4 nodes per graph in the launch shape
td_bnb_autotune_batch picks for the batch, the proposal trained first on the
GPU; value = certified graphs/s of the learned search.
"""
from __future__ import annotations

import argparse
import json
import math
import os
import random
import sys
import time
from pathlib import Path

ROOT = Path(__file__).resolve().parent
sys.path.insert(0, str(ROOT))

HBM_PEAK_GBPS = 8000.0


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=3)
    ap.add_argument("--warmup", type=int, default=1)
    ap.add_argument("--workload", default="dp30",
                    choices=["dp30", "dp20", "dpbatch", "bottomup", "bnb"])
    ap.add_argument("--no-cpu", action="store_true", help="skip the CPU baseline leg")
    ap.add_argument("--batch-mode", type=int, default=0)
    ap.add_argument("--low-bits", type=int, default=None)
    ap.add_argument("--tiles-per-lane", type=int, default=None)
    ap.add_argument("--block", type=int, default=None)
    ap.add_argument("--xcd-remap", type=int, default=None, choices=[0, 1])
    ap.add_argument("--class-bits", type=int, default=None, choices=[0, 3, 4])
    ap.add_argument("--grid-mult", type=int, default=None)
    ap.add_argument("--packed", type=int, default=None, choices=[0, 1],
                    help="kept for older command lines; without effect")
    ap.add_argument("--streams", type=int, default=None, choices=[1, 2, 3],
                    help="large graphs of a batch call: level sequences in flight at once")
    ap.add_argument("--batch-block", type=int, default=None)
    ap.add_argument("--batch-wg-per-cu", type=int, default=None)
    ap.add_argument("--no-autotune", action="store_true",
                    help="keep the default launch shape instead of td_dp_autotune's pick")
    ap.add_argument("--no-bnb", action="store_true",
                    help="skip the branch-and-bound / learned-proposal extra figures")
    ap.add_argument("--no-extra", action="store_true",
                    help="only the timed workload (no copy, B&B, other-configuration or CPU "
                         "figures): the form used for kernel profiles")
    ap.add_argument("--calibrate-copy", type=int, default=0, metavar="MIB",
                    help="only run the plain copy kernel over MIB MiB (rocprof calibration)")
    return ap.parse_args()


def bnb_extra(ctx, budget=50000):
    """Branch-and-bound figures for the extra block: the 256-graph sparse
    workload with the plain search, then 1024 graphs of the same distribution
    plain vs learned (proposal trained here on the GPU on DP labels).
    certified graphs/s = graphs proven optimal / wall time of the call, on
    inputs packed beforehand (a learned call's time includes scoring the
    graphs on the GPU)."""
    from gisbdw_amd import api, learn
    from gisbdw_amd import graphs as G

    ctx.set_param("bnb.node_budget", budget)
    out = {"node_budget_per_graph": budget}

    def families(W, cert):
        fam = {}
        for g, c in zip(W, cert):
            k = g.name.split("#")[0].rstrip("0123456789+-x.~")
            k = "cubic" if k.startswith("cubic") else ("grid" if k.startswith("grid") else "tree+edges")
            a = fam.setdefault(k, [0, 0])
            a[0] += int(c)
            a[1] += 1
        return {k: f"{v[0]}/{v[1]}" for k, v in fam.items()}
    shape_keys = ("bnb.waves_per_graph", "bnb.groups", "bnb.memo_log2")
    W = G.workload_bnb(256, 0)
    P = PackedBatch(W)
    # launch shape tuned on this batch (the sweep also warms the memo and the
    # captured launch), then one timed call on inputs packed beforehand
    api.bnb_autotune_batch(ctx, W)
    t0 = time.perf_counter()
    tds, pars, cert, st = P.solve(ctx)
    wall = time.perf_counter() - t0
    out["bnb256_plain"] = {"certified": int(sum(cert)), "graphs": len(W), "wall_s": wall,
                           "certified_graphs_per_s": sum(cert) / wall, "nodes": st.nodes,
                           "kernel_ms": st.kernel_ms, "certified_by_family": families(W, cert),
                           "shape": {k: ctx.get_param(k) for k in shape_keys}}
    prop = learn.Proposal(ctx)
    prop.init(1)
    t0 = time.perf_counter()
    ns, adj, tg, _ = learn.make_dataset(ctx, 800, 250, seed=11, nmin=8, nmax=24)
    t1 = time.perf_counter()
    curve = prop.train(ns, adj, tg, epochs=6, batch=512, lr=2e-3, seed=3)
    t2 = time.perf_counter()
    out["proposal_training"] = {"labels": int(len(ns)), "label_graphs": "800 G(n, p), n 8-24, "
                                "p 0.1-0.5 (the learned configuration's)", "label_s": t1 - t0,
                                "train_s": t2 - t1, "epoch_loss": [round(x, 4) for x in curve]}
    W = G.workload_bnb(1024, 1000)
    # launch shape for this batch and budget (waves per graph, workgroups,
    # memo size): td_bnb_autotune_batch, then every search below uses it
    t0 = time.perf_counter()
    tuned_rate = api.bnb_autotune_batch(ctx, W)
    out["bnb1024_autotune"] = {
        "s": time.perf_counter() - t0, "certified_per_kernel_s": tuned_rate,
        "shape": {k: ctx.get_param(k) for k in shape_keys}}
    P = PackedBatch(W)
    t0 = time.perf_counter()
    tds, pars, cert, st = P.solve(ctx)
    wall_p = time.perf_counter() - t0
    heur_gpu, _, _ = api.bnb_last_details(ctx, len(W))
    out["bnb1024_accounting"] = bnb_accounting(ctx, W, tds, cert)
    # the reference's heuristic chain HighestDegree(SpanningTree(Variance)) on
    # the GPU, as an alternative upper-bound seed
    t0 = time.perf_counter()
    chain_td, _ = api.heuristic_batch(ctx, W, "chain")
    chain_s = time.perf_counter() - t0
    t0 = time.perf_counter()
    tdc, _, certc, _ = P.solve(ctx, ub_seed=chain_td)
    wall_c = time.perf_counter() - t0 + chain_s
    cert_td = [t for t, c in zip(tds, cert) if c]
    out["ub_seeds"] = {
        "reference_chain_mean_depth": sum(chain_td) / len(W),
        "reference_chain_ms_1024_graphs": chain_s * 1e3,
        "gpu_seed_trees_mean_depth": float(sum(heur_gpu)) / len(W),
        "certified_graphs": len(cert_td),
        "certified_mean_td": sum(cert_td) / max(len(cert_td), 1),
        "reference_chain_mean_depth_on_certified": sum(h for h, c in zip(chain_td, cert) if c) / max(len(cert_td), 1),
        "gpu_seed_mean_depth_on_certified": float(sum(h for h, c in zip(heur_gpu, cert) if c)) / max(len(cert_td), 1),
        "bnb_with_reference_chain_seed": {"certified": int(sum(certc)), "wall_s": wall_c,
                                          "certified_graphs_per_s": sum(certc) / wall_c},
    }
    t0 = time.perf_counter()
    scores = P.scores(prop)
    tdl, parl, certl, stl = P.solve(ctx, scores=scores)
    wall_l = time.perf_counter() - t0
    agree = all(a == b for a, b, c, d in zip(tds, tdl, cert, certl) if c and d)
    out["bnb1024"] = {
        "plain": {"certified": int(sum(cert)), "wall_s": wall_p,
                  "certified_graphs_per_s": sum(cert) / wall_p, "nodes": st.nodes,
                  "certified_by_family": families(W, cert)},
        "learned": {"certified": int(sum(certl)), "wall_s": wall_l,
                    "certified_graphs_per_s": sum(certl) / wall_l, "nodes": stl.nodes,
                    "includes_scoring": True},
        "learned_over_plain": (sum(certl) / wall_l) / max(sum(cert) / wall_p, 1e-9),
        "certified_answers_agree": agree,
    }
    acct_l = bnb_accounting(ctx, W, tdl, certl)
    out["bnb1024_learned_family_trained"] = family_trained_run(
        ctx, W, P, out["bnb1024_accounting"], acct_l, sum(cert) / wall_p)
    # the same comparison over per-graph node budgets (scores computed once)
    sweep = []
    for b in (1000, 3000, 10000, 30000, 100000):
        ctx.set_param("bnb.node_budget", b)
        row = {"node_budget_per_graph": b}
        for name, sc in (("plain", None), ("learned", scores)):
            t0 = time.perf_counter()
            _, _, c, s = P.solve(ctx, scores=sc)
            wall = time.perf_counter() - t0
            row[name] = {"certified": int(sum(c)), "wall_s": round(wall, 4),
                         "certified_graphs_per_s": round(sum(c) / wall, 1)}
        row["learned_over_plain"] = round(row["learned"]["certified_graphs_per_s"] /
                                          max(row["plain"]["certified_graphs_per_s"], 1e-9), 3)
        sweep.append(row)
    ctx.set_param("bnb.node_budget", budget)
    out["bnb1024_budget_sweep"] = sweep
    return out


def descent_nodes(acct, family="tree+edges"):
    """Nodes of the descent's feasible calls of one family (all nodes but
    those of the last k, the refutation of td - 1 for a certified graph)."""
    a = acct[family]
    return a["nodes"] - a["last_k_nodes"]


def family_trained_run(ctx, W, P, acct_plain, acct_learned, plain_rate):
    """A second network, trained on DP labels of graphs like the certified
    family (random trees + 10% edges, n 16-28), ordering the same search:
    certified graphs/s and the tree+edges descent nodes beside the plain
    order's and the configuration-trained network's."""
    from gisbdw_amd import api, learn

    prop = learn.Proposal(ctx)
    prop.init(1)
    t0 = time.perf_counter()
    ns, adj, tg, _ = learn.make_dataset(ctx, 800, 250, seed=11, nmin=16, nmax=28,
                                        family="tree+edges")
    prop.train(ns, adj, tg, epochs=6, batch=512, lr=2e-3, seed=3)
    train_s = time.perf_counter() - t0
    t0 = time.perf_counter()
    tdf, _, certf, stf = P.solve(ctx, scores=P.scores(prop))
    wall = time.perf_counter() - t0
    acct_f = bnb_accounting(ctx, W, tdf, certf)
    rate = sum(certf) / wall
    return {"label_graphs": "800 random trees + 10% edges, n 16-28", "labels_and_train_s": train_s,
            "certified": int(sum(certf)), "wall_s": wall, "certified_graphs_per_s": rate,
            "over_plain": rate / max(plain_rate, 1e-9), "nodes": stf.nodes,
            "tree_edges_descent_nodes": {"plain": descent_nodes(acct_plain),
                                         "learned_configuration": descent_nodes(acct_learned),
                                         "learned_family": descent_nodes(acct_f)},
            "mean_ub": {"plain": {f: acct_plain[f]["mean_ub"] for f in acct_plain},
                        "learned_family": {f: acct_f[f]["mean_ub"] for f in acct_f}}}


class PackedBatch:
    """A search batch packed once, outside any timing: counts and rows as the
    C ABI takes them, the 64-row padded form the proposal scores, and the
    mask that picks each graph's vertices out of the padded scores."""

    def __init__(self, graphs):
        import numpy as np
        from gisbdw_amd import api, learn

        self.ns, self.adj = api.pack_graphs(graphs)
        self.ns_pad, self.adj_pad = learn.pad_adj(graphs)
        self.vmask = np.arange(64)[None, :] < self.ns[:, None]

    def scores(self, prop):
        return prop.scores_padded(self.ns_pad, self.adj_pad)[self.vmask]

    def solve(self, ctx, scores=None, ub_seed=None):
        from gisbdw_amd import api

        return api.bnb_solve_batch_arrays(ctx, self.ns, self.adj, ub_seed, scores)


def family_of(g):
    return "cubic" if g.name.startswith("cubic") else (
        "grid" if g.name.startswith("grid") else "tree+edges")


def bnb_accounting(ctx, W, tds, cert):
    """Per family, after a search call on W: the initial upper bound (best
    seed tree), the final upper bound (returned tree), the proven lower
    bound, the gap between the two bounds, and the search nodes, all of them
    and those spent on the last k the descent tried (for a certified graph
    the refutation of td - 1; for the others the attempt the budget cut)."""
    from gisbdw_amd import api

    heur, lb, nodes = api.bnb_last_details(ctx, len(W))
    last_k, last_nodes = api.bnb_last_search(ctx, len(W))
    fam = {}
    for i, g in enumerate(W):
        a = fam.setdefault(family_of(g), {"graphs": 0, "certified": 0, "seed_ub": 0, "ub": 0,
                                          "lb": 0, "gap_max": 0, "nodes": 0, "last_k_nodes": 0})
        a["graphs"] += 1
        a["certified"] += int(cert[i])
        a["seed_ub"] += int(heur[i])
        a["ub"] += int(tds[i])
        a["lb"] += int(lb[i])
        a["gap_max"] = max(a["gap_max"], int(tds[i]) - int(lb[i]))
        a["nodes"] += int(nodes[i])
        a["last_k_nodes"] += int(last_nodes[i])
    for a in fam.values():
        g = a["graphs"]
        a["mean_seed_ub"] = round(a.pop("seed_ub") / g, 3)
        a["mean_ub"] = round(a.pop("ub") / g, 3)
        a["mean_lb"] = round(a.pop("lb") / g, 3)
        a["mean_gap"] = round(a["mean_ub"] - a["mean_lb"], 3)
        a["last_k_node_share"] = round(a["last_k_nodes"] / max(a["nodes"], 1), 4)
    return fam


def cpu_baseline_dp(g, target_s=12.0):
    """Oracle flat-table DP on the subgraph induced by the first m vertices."""
    sys.path.insert(0, str(ROOT / "tests"))
    import oracle_lib
    from gisbdw_amd import graphs as G

    o = oracle_lib.Oracle()
    threads = min(os.cpu_count() or 1, 16)

    def induced(m):
        mask = (1 << m) - 1
        return G.Graph(m, [g.adj[v] & mask for v in range(m)], f"{g.name}[:{m}]")

    m = 22
    t0 = time.perf_counter()
    o.dp_fast(induced(m), threads=threads)
    dt = time.perf_counter() - t0
    rate = (1 << m) / dt
    # pick the largest m <= n whose estimated time fits the target
    while m < g.n and (1 << (m + 1)) / rate * 1.15 < target_s:
        m += 1
    t0 = time.perf_counter()
    o.dp_fast(induced(m), threads=threads)
    dt = time.perf_counter() - t0
    return {"value": (1 << m) / dt, "unit": "subsets/s", "cores": threads, "kind": "port",
            "sample": f"oracle flat-table DP (faithful recurrence of dynamic_gpu.cu, OpenMP "
                      f"within each level) on the subgraph induced by vertices 0..{m - 1} of "
                      f"{g.name}: 2^{m} subsets in {dt:.2f} s"}


def gpu_configs_extra(ctx):
    """GPU side of the single-graph (G(20,0.3) seed 0) and batched (4096
    graphs, n in [12,24]) configurations, for comparison with cpu_extra."""
    from gisbdw_amd import api
    from gisbdw_amd import graphs as G

    g = G.workload_dp_single(0)
    dp = api.DynamicGPU(ctx)
    dp(g)
    c1_td = dp.treedepth
    reps = 20
    t0 = time.perf_counter()
    for _ in range(reps):
        dp(g)
    c1_ms = (time.perf_counter() - t0) / reps * 1e3
    batch = G.workload_dp_batch(4096, 0)
    ns, adj = api.pack_graphs(batch)
    keys = ("dp.low_bits", "dp.tiles_per_lane", "dp.batch_block", "dp.batch_wg_per_cu")
    saved = {k: ctx.get_param(k) for k in keys}

    def timed():
        api.dp_solve_batch_arrays(ctx, ns, adj, 0)
        t0 = time.perf_counter()
        api.dp_solve_batch_arrays(ctx, ns, adj, 0)
        return time.perf_counter() - t0

    c3_default = timed()
    t0 = time.perf_counter()
    api.dp_autotune_batch(ctx, batch)
    tune_s = time.perf_counter() - t0
    chosen = {k: ctx.get_param(k) for k in keys}
    c3_tuned = timed()
    for k, v in saved.items():
        ctx.set_param(k, v)
    # the bottom-up heuristic (BottomUpHeuristicGPU) on the same G(20,0.3)
    # and on a G(26,0.15): every level, then the walk and the forest
    bu = api.BottomUpHeuristicGPU(ctx)
    bu_out = {}
    for name, gb in (("g20", g), ("g26", G.gnp(26, 0.15, 1))):
        bu(gb)
        reps = 5 if gb.n <= 20 else 2
        t0 = time.perf_counter()
        for _ in range(reps):
            bu(gb)
        ms = (time.perf_counter() - t0) / reps * 1e3
        dp(gb)
        bu_out[name] = {"graph": gb.name, "n": gb.n, "ms_end_to_end": ms,
                        "subsets_per_s": (1 << gb.n) / (ms * 1e-3),
                        "bottom_up_td": bu.treedepth, "exact_td": dp.treedepth}
    return {"dp_n20_single": {"graph": g.name, "treedepth": c1_td,
                              "ms_per_graph_end_to_end": c1_ms},
            "bottom_up": bu_out,
            "dp_batch4096": {"graphs_per_s_before_tuning": len(batch) / c3_default,
                             "before_tuning": saved,
                             "graphs_per_s_autotuned": len(batch) / c3_tuned,
                             "autotuned": chosen, "autotune_s": tune_s}}


def cpu_extra(threads):
    """The oracle's CPU paths on bounded samples of the single-graph, batched
    and branch-and-bound configurations, timed on this host:
    - G(20,0.3) seed 0: the faithful DynamicCPU restatement (std::map per
      level, dynamic_cpu.cpp:14-107) on one core over the subgraph induced by
      the first m vertices (m picked for about 8 s), and the flat-table DP on
      the whole graph with 1 and `threads` threads;
    - 4096-graph batch: the flat-table DP, one graph per thread, on the first
      256 graphs;
    - 256 sparse graphs n in [40,64]: the BranchAndBound restatement with
      EdgeLowerBound and the HighestDegree(SpanningTree(Variance)) seed chain
      (branch_and_bound.cpp:9-115), graph-parallel, on every 4th graph with a
      budget of 2e6 search nodes per graph."""
    from concurrent.futures import ThreadPoolExecutor

    sys.path.insert(0, str(ROOT / "tests"))
    import oracle_lib
    from gisbdw_amd import graphs as G

    o = oracle_lib.Oracle()
    out = {"cores": threads}
    g = G.workload_dp_single(0)

    def induced(m):
        mask = (1 << m) - 1
        return G.Graph(m, [g.adj[v] & mask for v in range(m)], f"{g.name}[:{m}]")

    m = 15
    t0 = time.perf_counter()
    o.dyncpu(induced(m))
    dt = time.perf_counter() - t0
    while m < g.n and dt * 2.4 < 8.0:
        m += 1
        dt *= 2.4
    t0 = time.perf_counter()
    o.dyncpu(induced(m))
    dt = time.perf_counter() - t0
    t0 = time.perf_counter()
    o.dp_fast(g, threads=1)
    flat1 = time.perf_counter() - t0
    t0 = time.perf_counter()
    o.dp_fast(g, threads=threads)
    flatn = time.perf_counter() - t0
    out["dp_n20_single"] = {
        "faithful_dyncpu_1core": {"vertices": m, "s": dt, "subsets_per_s": (1 << m) / dt},
        "flat_dp_1core_ms": flat1 * 1e3, f"flat_dp_{threads}cores_ms": flatn * 1e3}
    # the bottom-up heuristic's restatement (union-find arrays per subset,
    # bottom_up_heuristic_gpu_algorithm.cu:57-95) on one core, same graph
    t0 = time.perf_counter()
    o.bottom_up(g, history=False)
    dt = time.perf_counter() - t0
    out["bottom_up_g20_1core"] = {"s": dt, "subsets_per_s": (1 << g.n) / dt}

    sample = G.workload_dp_batch(4096, 0)[:256]
    t0 = time.perf_counter()
    with ThreadPoolExecutor(threads) as ex:
        list(ex.map(lambda h: o.dp_fast(h, threads=1), sample))
    dt = time.perf_counter() - t0
    out["dp_batch4096"] = {"sample_graphs": len(sample), "s": dt, "graphs_per_s": len(sample) / dt}

    sample = G.workload_bnb(256, 0)[::4]
    budget = 2_000_000
    t0 = time.perf_counter()
    with ThreadPoolExecutor(threads) as ex:
        res = list(ex.map(lambda h: o.bnb(h, 0, 1, budget), sample))
    dt = time.perf_counter() - t0
    cert = sum(1 for r in res if r[3])
    out["bnb256"] = {"sample_graphs": len(sample), "node_budget_per_graph": budget, "s": dt,
                     "certified": cert, "certified_graphs_per_s": cert / dt,
                     "nodes_per_s": sum(r[4] for r in res) / dt}
    return out


def cpu_baseline_bnb(threads):
    """The oracle's BranchAndBound restatement (EdgeLowerBound, the
    HighestDegree(SpanningTree(Variance)) seed chain, branch_and_bound.cpp:
    9-115), graph-parallel on every 16th graph of the 1024-graph workload with
    2e6 search nodes per graph."""
    from concurrent.futures import ThreadPoolExecutor

    sys.path.insert(0, str(ROOT / "tests"))
    import oracle_lib
    from gisbdw_amd import graphs as G

    o = oracle_lib.Oracle()
    sample = G.workload_bnb(1024, 1000)[::16]
    budget = 2_000_000
    t0 = time.perf_counter()
    with ThreadPoolExecutor(threads) as ex:
        res = list(ex.map(lambda h: o.bnb(h, 0, 1, budget), sample))
    dt = time.perf_counter() - t0
    cert = sum(1 for r in res if r[3])
    return {"value": cert / dt, "unit": "certified graphs/s", "cores": threads, "kind": "port",
            "sample": f"oracle BranchAndBound restatement on {len(sample)} of the 1024 graphs "
                      f"(every 16th), {budget} nodes per graph: {cert} certified in {dt:.2f} s, "
                      f"{sum(r[4] for r in res) / dt:.3g} nodes/s"}


def cpu_baseline_bottom_up(g):
    """The oracle's BottomUpHeuristicGPU restatement (union-find arrays per
    subset, bottom_up_heuristic_gpu_algorithm.cu:57-95) on one core, over the
    subgraph induced by the first m vertices of g (m picked for about 10 s)."""
    sys.path.insert(0, str(ROOT / "tests"))
    import oracle_lib
    from gisbdw_amd import graphs as G

    o = oracle_lib.Oracle()

    def induced(m):
        mask = (1 << m) - 1
        return G.Graph(m, [g.adj[v] & mask for v in range(m)], f"{g.name}[:{m}]")

    m = 16
    t0 = time.perf_counter()
    o.bottom_up(induced(m), history=False)
    dt = time.perf_counter() - t0
    while m < g.n and dt * 2.3 < 10.0:
        m += 1
        dt *= 2.3
    t0 = time.perf_counter()
    o.bottom_up(induced(m), history=False)
    dt = time.perf_counter() - t0
    return {"value": (1 << m) / dt, "unit": "subsets/s", "cores": 1, "kind": "port",
            "sample": f"oracle bottom-up restatement on the subgraph induced by vertices "
                      f"0..{m - 1} of {g.name}: 2^{m} subsets in {dt:.2f} s"}


def shape_key(ctx):
    """The DP launch shape, as the traffic summary keys its lines."""
    return "low_bits={} tiles_per_lane={} block={} grid_mult={}".format(
        *(ctx.get_param("dp." + k) for k in ("low_bits", "tiles_per_lane", "block", "grid_mult")))


def profile_traffic(key):
    """HBM bytes per level launch for this launch shape from the committed
    rocprofv3 --pmc summary (profiles/dp_level_kernel_n30_traffic.md,
    calibrated against a plain copy of known size), or None when the summary
    has no line for the shape."""
    p = ROOT / "profiles" / "dp_level_kernel_n30_traffic.md"
    if p.exists():
        want = f"traffic_bytes_per_launch [{key}]:"
        for line in p.read_text().splitlines():
            if line.startswith(want):
                return int(line.split(":")[1])
    return None


def main():
    args = parse()
    if args.gpus != 1:
        print(f"bench.py runs on one GPU only (asked for {args.gpus}): graphs would be "
              "sharded one process per GPU, which this build does not implement",
              file=sys.stderr)
        sys.exit(2)
    from gisbdw_amd import api
    from gisbdw_amd import graphs as G

    ctx = api.Context(0)
    if args.calibrate_copy:
        gbps = ctx.copy_bench(args.calibrate_copy << 20, 3)
        print(json.dumps({"copy_MiB": args.calibrate_copy, "launches": 4, "GBps": gbps}))
        return
    if args.low_bits:
        ctx.set_param("dp.low_bits", args.low_bits)
    if args.tiles_per_lane:
        ctx.set_param("dp.tiles_per_lane", args.tiles_per_lane)
    if args.block:
        ctx.set_param("dp.block", args.block)
    if args.xcd_remap is not None:
        ctx.set_param("dp.xcd_remap", args.xcd_remap)
    if args.class_bits is not None:
        ctx.set_param("dp.class_bits", args.class_bits)
    if args.grid_mult:
        ctx.set_param("dp.grid_mult", args.grid_mult)
    if args.packed is not None:
        ctx.set_param("dp.packed", args.packed)
    if args.streams:
        ctx.set_param("dp.streams", args.streams)
    if args.batch_block:
        ctx.set_param("dp.batch_block", args.batch_block)
    if args.batch_wg_per_cu:
        ctx.set_param("dp.batch_wg_per_cu", args.batch_wg_per_cu)

    explicit = args.low_bits or args.tiles_per_lane or args.block or args.batch_block or \
        args.batch_wg_per_cu or args.class_bits is not None or args.grid_mult or \
        args.packed is not None
    tuned_ms = None
    if args.workload in ("dp30", "dp20"):
        graphs = G.workload_dp_n30() if args.workload == "dp30" else [G.workload_dp_single(0)]
        if not explicit and not args.no_autotune:
            tuned_ms = ctx.autotune(graphs[0].n)
            print(f"[bench] autotuned: {shape_key(ctx)}", file=sys.stderr, flush=True)
        dp = api.DynamicGPU(ctx)
        ns, adj = api.pack_graphs(graphs)  # inputs packed once, outside the timing

        kernels = [0]

        def step():
            if len(graphs) > 1:
                # the eight graphs in one td_dp_solve_batch call: the same
                # level kernels as td_dp_solve, each graph's decomposition
                # overlapped with the next graph's levels
                _, _, st = api.dp_solve_batch_arrays(ctx, ns, adj, 0)
                kernels[0] += st.level_kernels
                return st.level_ms, st.alg_bytes, st.subsets
            lvl_ms = 0.0
            alg = 0
            sub = 0
            for g in graphs:
                dp(g)
                lvl_ms += dp.stats.level_ms
                alg += dp.stats.alg_bytes
                sub += dp.stats.subsets
                kernels[0] += dp.stats.level_kernels
            return lvl_ms, alg, sub

        for _ in range(args.warmup):
            step()
        print(f"[bench] warmup done ({args.warmup} steps)", file=sys.stderr, flush=True)
        kernels[0] = 0
        t0 = time.perf_counter()
        lvl_ms = 0.0
        alg = sub = 0
        launches = 0
        for i in range(args.steps):
            a, b, c = step()
            lvl_ms += a
            alg += b
            sub += c
            print(f"[bench] step {i} level_ms={a:.3f}", file=sys.stderr, flush=True)
        wall = time.perf_counter() - t0
        nlev = kernels[0]  # level-kernel executions in the timed steps
        # compulsory bytes: three bits per subset, written once, read once
        comp = 0.75 * sub
        achieved = comp / (lvl_ms * 1e-3) / 1e9
        n = graphs[0].n
        traffic = profile_traffic(shape_key(ctx))
        out = {
            "metric": f"DP subsets/sec (exact subset DP, n={n})",
            "value": sub / wall,
            "unit": "subsets/s",
            "n_gpus": 1,
            "steps": args.steps,
            "warmup": args.warmup,
            "ms_per_step": wall / args.steps * 1e3,
            "higher_is_better": True,
            "scaling": "weak",
            "vs_baseline": None,
            "dtype": "u8",
            "data": "synthetic",
            "config": {
                "workload": ("dp-n30: 4 x G(30,0.2) seeds 0-3 + 4 x 5x6 grid minus 5 of 49 "
                             "edges seeds 0-3" if args.workload == "dp30" else
                             "dp-n20: one G(20,0.3) seed 0 (reseeded until connected)"),
                "graphs": len(graphs),
                "n": n,
                "low_bits": ctx.get_param("dp.low_bits"),
                "tiles_per_lane": ctx.get_param("dp.tiles_per_lane"),
                "block": ctx.get_param("dp.block"),
                "grid_mult": ctx.get_param("dp.grid_mult"),
                "streams": ctx.get_param("dp.streams"),
                "autotuned": tuned_ms is not None,
            },
            "roofline": {
                "bound": "hbm",
                "achieved": achieved,
                "peak": HBM_PEAK_GBPS,
                "unit": "GB/s",
                "frac": achieved / HBM_PEAK_GBPS,
                "traffic": traffic,
                "traffic_source": "profiles/dp_level_kernel_n30_traffic.md (rocprofv3 --pmc "
                                  "TCC_EA0_RDREQ_{32B,64B,128B} and TCC_EA0_WRREQ(_64B) "
                                  "request counts, not this run)",
                "traffic_over_compulsory": (traffic / (comp / nlev)) if traffic else None,
                "kernel": "DPLevelKernel",
                "bytes_basis": "compulsory: 0.75 * 2^n per graph (3 bits per subset)",
                "compulsory_bytes_per_launch": comp / nlev,
                "avg_launch_ms": lvl_ms / nlev,
                "launches": nlev,
                "model_bytes_per_launch": alg / nlev,
                "model_GBps": alg / (lvl_ms * 1e-3) / 1e9,
            },
            "extra": {
                "graphs_per_s": len(graphs) * args.steps / wall,
                "level_kernel_ms_per_step": lvl_ms / args.steps,
                "subsets_per_s_kernel": sub / (lvl_ms * 1e-3),
            },
        }
    elif args.workload == "bottomup":
        # BottomUpHeuristicGPU on one G(26,0.15): every level, then the walk
        # and the forest.  Algorithmic bytes per subset S (|S| = k), one byte
        # per height: the kept forest's 32 slots read and 34 bytes written
        # (its 32 slots, the vertex added last, the height), plus the k
        # heights of S \ v and 2|E(S)| neighbour slots read; over all subsets
        # 66 * 2^n + (n + m) * 2^(n-1).  The kernel packs slots into 3 or 4
        # bits where the heights allow, so it moves fewer bytes than this.
        g = G.gnp(26, 0.15, 1)
        graphs = [g]
        m = sum(bin(r).count("1") for r in g.adj) // 2
        alg_bytes = 66 * (1 << g.n) + (g.n + m) * (1 << (g.n - 1))
        bu = api.BottomUpHeuristicGPU(ctx)
        for _ in range(args.warmup):
            bu(g)
        t0 = time.perf_counter()
        for i in range(args.steps):
            bu(g)
            print(f"[bench] step {i} td={bu.treedepth}", file=sys.stderr, flush=True)
        wall = time.perf_counter() - t0
        achieved = alg_bytes * args.steps / wall / 1e9
        out = {
            "metric": "bottom-up heuristic subsets/sec (n=26)",
            "value": (1 << g.n) * args.steps / wall,
            "unit": "subsets/s",
            "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
            "ms_per_step": wall / args.steps * 1e3,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "u8", "data": "synthetic",
            "config": {"workload": f"bottom-up heuristic: {g.name}, {m} edges, all 27 levels",
                       "graphs": 1, "n": g.n},
            "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBPS,
                         "unit": "GB/s", "frac": achieved / HBM_PEAK_GBPS, "traffic": None,
                         "kernel": "BottomUpLevelKernel", "alg_bytes_per_step": alg_bytes,
                         "timing": "wall clock of the whole call"},
            "extra": {"treedepth": bu.treedepth},
        }
    elif args.workload == "bnb":
        # 1024 sparse graphs, n in [40,64]: the proposal is trained on the GPU
        # (DP labels of G(n <= 24, p in [0.1, 0.5]), 6 epochs, as the learned
        # configuration states), then each step runs the plain search and the
        # learned-ordered one (scoring included) on the whole batch
        from gisbdw_amd import learn

        graphs = G.workload_bnb(1024, 1000)
        ctx.set_param("bnb.node_budget", 50000)
        ctx.set_param("bnb.waves_per_graph", 8)
        prop = learn.Proposal(ctx)
        prop.init(1)
        t0 = time.perf_counter()
        ns, adj, tg, _ = learn.make_dataset(ctx, 800, 250, seed=11, nmin=8, nmax=24)
        prop.train(ns, adj, tg, epochs=6, batch=512, lr=2e-3, seed=3)
        train_s = time.perf_counter() - t0

        tune_t0 = time.perf_counter()
        api.bnb_autotune_batch(ctx, graphs)
        tune_s = time.perf_counter() - tune_t0
        shape = {k: ctx.get_param(k) for k in
                 ("bnb.waves_per_graph", "bnb.groups", "bnb.memo_log2")}
        print(f"[bench] autotuned search shape {shape}", file=sys.stderr, flush=True)

        # inputs packed once, outside the timing (as for the DP workloads);
        # the learned call's time includes scoring the graphs on the GPU
        P = PackedBatch(graphs)

        def run(learned):
            t = time.perf_counter()
            sc = P.scores(prop) if learned else None
            td, _, cert, st = P.solve(ctx, scores=sc)
            return time.perf_counter() - t, td, cert, st

        for _ in range(args.warmup):
            run(False)
            run(True)
        tot = {False: [0.0, 0, 0], True: [0.0, 0, 0]}
        answers = {}
        for i in range(args.steps):
            for learned in (False, True):
                dt, td, cert, st = run(learned)
                a = tot[learned]
                a[0] += dt
                a[1] += int(sum(cert))
                a[2] += st.nodes
                answers[learned] = (td, cert)
            print(f"[bench] step {i} certified plain {tot[False][1]} learned {tot[True][1]}",
                  file=sys.stderr, flush=True)
        agree = all(a == b for a, b, c, d in zip(answers[False][0], answers[True][0],
                                                   answers[False][1], answers[True][1]) if c and d)
        # per-family bounds and nodes of the last (learned) call, and of a
        # plain call
        acct_learned = bnb_accounting(ctx, graphs, *answers[True])
        t_p, td_p, cert_p, _ = run(False)
        acct_plain = bnb_accounting(ctx, graphs, td_p, cert_p)
        family = family_trained_run(ctx, graphs, P, acct_plain, acct_learned,
                                    sum(cert_p) / t_p)
        # 256 dense small graphs (n in [20,24], p in [0.5,0.8]): the plain
        # search, the search with components of at most 12 vertices answered
        # by its in-wave subset DP (bnb.dp_small = 12), and the whole graphs
        # routed to the batched subset DP (bnb.dp_max_n = 24)
        rng = random.Random(17)
        dense = [G.gnp(rng.randint(20, 24), rng.uniform(0.5, 0.8), rng.getrandbits(32))
                 for _ in range(256)]
        routing = {}
        Pd = PackedBatch(dense)
        for name, dps, dpn in (("search_only", 0, 0), ("in_search_dp12", 12, 0),
                               ("dp_routing", 0, 24)):
            ctx.set_param("bnb.dp_small", dps)
            ctx.set_param("bnb.dp_max_n", dpn)
            Pd.solve(ctx)
            t = time.perf_counter()
            _, _, cert_d, st_d = Pd.solve(ctx)
            wall_d = time.perf_counter() - t
            routing[name] = {
                "certified": int(sum(cert_d)), "wall_s": wall_d, "nodes": st_d.nodes,
                "certified_graphs_per_s": sum(cert_d) / wall_d}
        ctx.set_param("bnb.dp_small", 0)
        ctx.set_param("bnb.dp_max_n", 0)
        rate = {k: v[1] / v[0] for k, v in tot.items()}
        out = {
            "metric": "certified graphs/sec (learned-ordered B&B, 1024 graphs, n in [40,64])",
            "value": rate[True],
            "unit": "certified graphs/s",
            "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
            "ms_per_step": (tot[False][0] + tot[True][0]) / args.steps * 1e3,
            "higher_is_better": True, "scaling": "weak",
            "vs_baseline": None, "dtype": "int32", "data": "synthetic",
            "config": {"workload": "bnb-1024: 256 random cubic, 128 7x7 + 128 8x8 grids "
                                   "relabelled, 512 random trees + 10% edges; seed 1000",
                       "graphs": len(graphs), "node_budget_per_graph": 50000,
                       "waves_per_graph": shape["bnb.waves_per_graph"],
                       "groups": shape["bnb.groups"], "memo_log2": shape["bnb.memo_log2"],
                       "autotuned": True},
            "roofline": None,
            "extra": {
                "roofline_note": "latency-bound search: no streaming roofline; nodes/s below",
                "plain_certified_graphs_per_s": rate[False],
                "learned_over_plain": rate[True] / max(rate[False], 1e-9),
                "certified_per_step": {"plain": tot[False][1] // args.steps,
                                       "learned": tot[True][1] // args.steps},
                "nodes_per_s": {"plain": tot[False][2] / tot[False][0],
                                "learned": tot[True][2] / tot[True][0]},
                "certified_answers_agree": agree,
                "proposal_training_s": train_s,
                "autotune_s": tune_s,
                "accounting": {"plain": acct_plain, "learned": acct_learned},
                "learned_family_trained": family,
                "dense_n20_24_256_graphs": routing,
            },
        }
    else:
        graphs = G.workload_dp_batch(4096, 0)
        ns, adj = api.pack_graphs(graphs)  # inputs packed once, outside the timing
        if not explicit and not args.no_autotune:
            tuned_ms = api.dp_autotune_batch(ctx, graphs)

        def step():
            td, par, st = api.dp_solve_batch_arrays(ctx, ns, adj, args.batch_mode)
            return st

        for _ in range(args.warmup):
            step()
        t0 = time.perf_counter()
        lvl_ms = 0.0
        alg = sub = 0
        for i in range(args.steps):
            st = step()
            lvl_ms += st.level_ms
            alg += st.alg_bytes
            sub += st.subsets
            print(f"[bench] step {i} level_ms={st.level_ms:.3f}", file=sys.stderr, flush=True)
        wall = time.perf_counter() - t0
        achieved = 0.75 * sub / (lvl_ms * 1e-3) / 1e9  # three bits per subset, twice
        out = {
            "metric": "DP graphs/sec (batched exact subset DP)",
            "value": len(graphs) * args.steps / wall,
            "unit": "graphs/s",
            "n_gpus": 1, "steps": args.steps, "warmup": args.warmup,
            "ms_per_step": wall / args.steps * 1e3,
            "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
            "dtype": "u8", "data": "synthetic",
            "config": {"workload": "dp-batch: 4096 G(n,p), n~U{12..24}, p~U[0.15,0.5], seed 0",
                       "graphs": len(graphs), "mode": args.batch_mode,
                       "batch_block": ctx.get_param("dp.batch_block"),
                       "batch_wg_per_cu": ctx.get_param("dp.batch_wg_per_cu"),
                       "low_bits": ctx.get_param("dp.low_bits"),
                       "tiles_per_lane": ctx.get_param("dp.tiles_per_lane"),
                       "autotuned": tuned_ms is not None},
            "roofline": {"bound": "hbm", "achieved": achieved, "peak": HBM_PEAK_GBPS,
                         "unit": "GB/s", "frac": achieved / HBM_PEAK_GBPS, "traffic": None,
                         "kernel": "DPPersistentKernel",
                         "bytes_basis": "compulsory: 0.75 * 2^n per graph (3 bits per subset)",
                         "model_GBps": alg / (lvl_ms * 1e-3) / 1e9},
            "extra": {"subsets_per_s": sub / wall},
        }
    if args.no_extra:
        args.no_bnb = args.no_cpu = True
    else:
        out["extra"]["copy_GBps_2GiB"] = ctx.copy_bench(2 << 30, 3)
    if not args.no_bnb and args.workload == "dp30":
        print("[bench] branch-and-bound extra", file=sys.stderr, flush=True)
        out["extra"]["bnb"] = bnb_extra(ctx)
    if args.workload == "dp30" and not args.no_extra:
        out["extra"]["gpu_configs"] = gpu_configs_extra(ctx)
    if not args.no_cpu and args.workload == "bottomup":
        print("[bench] cpu baseline", file=sys.stderr, flush=True)
        out["cpu_baseline"] = cpu_baseline_bottom_up(graphs[0])
    elif not args.no_cpu and args.workload == "bnb":
        print("[bench] cpu baseline", file=sys.stderr, flush=True)
        out["cpu_baseline"] = cpu_baseline_bnb(min(os.cpu_count() or 1, 16))
    elif not args.no_cpu:
        g0 = graphs[0]
        print("[bench] cpu baseline", file=sys.stderr, flush=True)
        out["cpu_baseline"] = cpu_baseline_dp(g0)
        if args.workload == "dp30":
            print("[bench] cpu paths of the other configurations", file=sys.stderr, flush=True)
            out["extra"]["cpu_configs"] = cpu_extra(out["cpu_baseline"]["cores"])
    else:
        out["cpu_baseline"] = None
    print(json.dumps(out), flush=True)


if __name__ == "__main__":
    main()
