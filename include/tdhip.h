/*
 * tdhip.h -- C ABI of the MI355X exact treedepth library (libtdhip.so).
 *
 * The reference (Zackere/GiSBDW) exposes its GPU paths as C++ classes over
 * Boost graphs; this header is the flat boundary those classes are rebuilt
 * on.  Each entry point names the reference interface it replaces.
 *
 * Graph input everywhere: n vertices 0..n-1, adjacency as n uint64 bitmask
 * rows (bit u of row v set <=> edge {u,v}); rows must be symmetric with no
 * self loops and no bits >= n.  The caller owns every host buffer; the
 * context owns every device buffer.  Calls are synchronous.  One context per
 * host thread; the library holds no global mutable state across contexts.
 * No C++ exception crosses this boundary: every call returns a td_status.
 */
#ifndef TDHIP_H_
#define TDHIP_H_
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

typedef enum td_status {
  TD_OK = 0,
  TD_E_INVALID = 1, /* bad argument or graph (self loop, asymmetric, n)   */
  TD_E_NOMEM = 2,   /* the context's byte budget or the device is full    */
  TD_E_HIP = 3,     /* a HIP runtime call failed                          */
  TD_E_BUDGET = 4,  /* search stopped by its node/time budget (uncertified) */
  TD_E_STATE = 5    /* query before any solve, or out-of-range query      */
} td_status;

typedef struct td_ctx td_ctx;

/* Context: owns a HIP stream, a device arena and the tuning parameters.
 * mem_budget_bytes = 0 means "whatever the device has".
 * Replaces the implicit device-0 + Thrust allocations of
 * Treedepth/src/dynamic_gpu/dynamic_gpu.cu:171-201 and
 * Treedepth/src/bnb_gpu/bnb_gpu.cu:264-285. */
int td_ctx_create(td_ctx** out, int device, uint64_t mem_budget_bytes);
void td_ctx_destroy(td_ctx* ctx);
/* Last error message of this context ("" if none). */
const char* td_last_error(const td_ctx* ctx);
/* Tuning knobs (see td_dp_autotune): "dp.low_bits" (2..5, default 4: level
 * tables in tiles of 1, 1, 2 or 4 words of 32 subsets; a single graph takes
 * fewer words where larger tiles would leave lanes idle),
 * "dp.tiles_per_lane" (1..64, default 1), "dp.block" (64..1024, default 512),
 * "dp.grid_mult" (1..64, default 4: level launches use at most this many
 * times the workgroups the device holds at once),
 * "dp.batch_wg_per_cu", "dp.use_graph" (0/1), "dp.streams" (1..3, default 2:
 * graphs above 26 vertices in a td_dp_solve_batch call run their level
 * sequences that many at a time on that many streams, each graph starting
 * when the previous one has done the first 1/streams of its subsets; 1: one
 * graph at a time), "dp.flow_spin" (0..2^30, default 2^17: how often a
 * workgroup of a graph of 19..24 vertices reads a word that another one has
 * to publish, before the call is solved without such waits).  "dp.class_bits" (0, 3 or 4, default 0),
 * "dp.class_min_nh" (5..32, default 16), "dp.packed" (0/1, default 0) and
 * "dp.xcd_remap" (0/1) are accepted and kept for callers and tuning caches
 * that set them: one table layout, three bits per subset and contiguous
 * slices per XCD, serves all of them.  A table claims one byte per subset of
 * the byte budget, or 17/32 with class_bits and packed both set.
 * "bnb.node_budget"
 * (per graph, default 2e6), "bnb.waves_per_graph" (1..16; 0, the
 * default: 16 for batches of at most one graph per CU, 12 for up to two,
 * else 8),
 * "bnb.groups" (workgroups in flight; 0, the default: 4 per CU),
 * "bnb.memo_log2" (memo buckets per wave, 4 entries of 16 bytes each; 0, the
 * default: sized to the per-wave node budget within [2^10, 2^17]),
 * "bnb.dp_small" (0..12, default 0: components of at most that many
 * vertices are decided inside the search by a subset DP in the wave's LDS,
 * the in-search half of the DP + B&B hybrid), "bnb.use_graph" (0/1,
 * default 1: replay the search launch from a hipGraph). */
int td_ctx_set_param(td_ctx* ctx, const char* key, int64_t value);
int td_ctx_get_param(const td_ctx* ctx, const char* key, int64_t* value);

/* Streaming copy of `bytes` (read + write), reps times: returns the achieved
 * GB/s (2 * bytes * reps / time).  No reference counterpart: it measures the
 * device's practical HBM bandwidth and is the known-size kernel used to scale
 * rocprofv3's FETCH_SIZE / WRITE_SIZE counters. */
int td_ctx_copy_bench(td_ctx* ctx, uint64_t bytes, int32_t reps, double* gbps_out);

/* ---------------------------------------------------------------------- */
/* Subset DP                                                               */
/* ---------------------------------------------------------------------- */
typedef struct td_dp_stats {
  uint64_t graphs;       /* graphs solved by the call                    */
  uint64_t subsets;      /* sum over graphs of 2^n                        */
  uint64_t alg_bytes;    /* sum over graphs of 2^(n-1) (n+2)              */
  uint64_t launches;     /* kernel launches (or graph replays)            */
  double level_ms;       /* GPU time of the level kernels (HIP events, or the
                            device's clock for single graphs of at most 24
                            vertices, which one launch resolves;
                            with two graphs' levels in flight, the union of
                            the graphs' level intervals)                  */
  double tree_ms;        /* GPU time of the decomposition (tree) kernel   */
  double total_ms;       /* host wall time of the whole call              */
  uint64_t level_kernels; /* level-kernel executions behind level_ms (a batch
                            call's graphs of at most 26 vertices count as
                            one in mode 0)                                */
} td_dp_stats;

/* DynamicGPU::operator()(g) + GetElimination(n, n, 0) + EliminationTree +
 * Decompose (Treedepth/src/dynamic_gpu/dynamic_gpu.hpp:38-64,
 * Treedepth/main.cpp:187-195).  n <= 32.  Writes the treedepth and the
 * canonical decomposition as a parent array (-1 = root).  A disconnected
 * input yields a forest: one canonical tree per component, roots -1, and
 * treedepth = the largest tree's depth (the reference rejects such input).
 * The level tables stay on the device for the queries below. stats nullable. */
int td_dp_solve(td_ctx* ctx, int32_t n, const uint64_t* adj,
                uint8_t* treedepth_out, int8_t* parent_out,
                td_dp_stats* stats);

/* td_dp_solve for callers that cannot allocate device memory (code under
 * HIP graph capture, tight serving loops, harnesses that forbid hipMalloc).
 * No counterpart in the reference.  Same inputs, outputs and results as
 * td_dp_solve, for n <= 24: the descriptor, Pascal tables, level tables and
 * tree output live in one fixed device array of 17,104,896 bytes that the library's code object holds on each
 * device it runs on until the process ends.  The call allocates no device or
 * page-locked memory and captures no graph (its level kernels launch
 * directly).  n > 24 is TD_E_INVALID.  Every call on one device shares that
 * device's array: calls that overlap on one device (several contexts or
 * threads) race and must be serialized by the caller.  Nothing in the array
 * needs to start at zero; each call overwrites what it reads.  Afterwards the
 * td_dp_get_* queries return TD_E_STATE until the next td_dp_solve. */
int td_dp_solve_noalloc(td_ctx* ctx, int32_t n, const uint64_t* adj,
                        uint8_t* treedepth_out, int8_t* parent_out,
                        td_dp_stats* stats);

/* DynamicCPU::GetTreedepth(nverts, subset_size, subset_code)
 * (Treedepth/src/dynamic_cpu/dynamic_cpu.hpp:34-36, .cpp:29-39) over the
 * last td_dp_solve: treedepth of the subset with this colex code.  Unlike
 * the reference, disconnected subsets are answered too. */
int td_dp_get_treedepth(td_ctx* ctx, int32_t subset_size,
                        uint64_t subset_code, uint32_t* td_out);

/* The level-k table of the last td_dp_solve in colex order:
 * out[code] = td of the k-subset with that code, out_len >= C(n, k).
 * (The reference keeps these as history_, dynamic_gpu.hpp:33-35.) */
int td_dp_get_level(td_ctx* ctx, int32_t k, uint8_t* out, uint64_t out_len);

/* DynamicGPU::GetElimination<V>(nverts, subset_size, subset_code)
 * (Treedepth/src/dynamic_gpu/dynamic_gpu.hpp:49-64): the elimination order
 * of that subset, subset_size vertices written to order_out. */
int td_dp_get_elimination(td_ctx* ctx, int32_t nverts, int32_t subset_size,
                          uint64_t subset_code, int32_t* order_out);

/* Many graphs in one call (no reference counterpart: the reference loops
 * over input files one at a time, Treedepth/main.cpp:130).  n[i] <= 32;
 * adj_concat holds the rows of graph 0, then graph 1, ...; parent_concat
 * likewise (sum n[i] entries).  For the graphs of at most 26 vertices, mode:
 * 0 = one persistent launch (graphs pulled from a device queue, all levels
 * inside; graphs of at most 18 vertices in LDS, a workgroup each, and few
 * graphs of 19..24 vertices in several workgroups each), 1 = level-synchronous launches over the whole batch, 2 = one
 * launch per graph and level (the baseline the persistent launch is
 * measured against).  Larger graphs go one after another through
 * td_dp_solve's level kernels, each graph's decomposition on a second stream
 * while the next graph's levels run (two tables of the largest such graph
 * are held).  Results equal td_dp_solve's for every graph; afterwards the
 * td_dp_get_* queries return TD_E_STATE until the next td_dp_solve. */
int td_dp_solve_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                      const uint64_t* adj_concat, uint8_t* treedepth_out,
                      int8_t* parent_concat, int32_t mode,
                      td_dp_stats* stats);

/* Autotuner: times every candidate (low_bits, tiles_per_lane, grid_mult,
 * block) on a seeded G(n, 0.25) graph and keeps the best in the
 * context: the level kernels for n > 26 (such graphs also run in batch
 * calls, where the tree kernel is hidden), the level kernels plus the tree
 * kernel for smaller n.  Candidates that launch the same share a time, and a
 * parameter that makes no difference to the best launch stays as it is; so do
 * "dp.class_bits" and "dp.packed", and for n <= 24, whose one launch reads
 * none of these parameters, all of them.  With a non-null cache_path (JSON
 * lines), a "best" line for this n and device arch is applied (n > 24) without
 * timing anything; otherwise the sweep runs and every candidate plus the best
 * are appended.
 * best_ms_out (nullable) receives the best time.  No reference counterpart:
 * the reference hard-codes 4096 x 128 threads per chunk
 * (Treedepth/src/dynamic_gpu/dynamic_gpu.cu:123-124). */
int td_dp_autotune(td_ctx* ctx, int32_t n, const char* cache_path,
                   double* best_ms_out);
/* Autotuner of the persistent batch launch (td_dp_solve_batch mode 0):
 * sweeps (low_bits, tiles_per_lane, batch_block, batch_wg_per_cu) on the
 * given batch itself and keeps the best (the present ones for a batch whose
 * graphs all go to other kernels); the cache key is the batch's
 * (graph count, largest n, sum of n).  Same cache rules as td_dp_autotune. */
int td_dp_autotune_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                         const uint64_t* adj_concat, const char* cache_path,
                         double* best_ms_out);

/* ---------------------------------------------------------------------- */
/* Upper-bound heuristics                                                  */
/* ---------------------------------------------------------------------- */
/* The reference's elimination-tree heuristics on the GPU, one graph per
 * wave, for ngraphs graphs of n[i] <= 64 vertices (rows concatenated):
 *   kind 1: HighestDegree(SpanningTree(Variance(1.0, 0.2, 0.8))), the
 *           decorator chain keeping an inner result only when strictly
 *           shallower (the heuristics/ headers; BranchAndBound's Heuristic::Get,
 *           Treedepth/src/branch_and_bound/branch_and_bound.hpp:38-42);
 *   kind 2: HighestDegreeHeuristic::Get (highest_degree_heuristic.hpp:19-45);
 *   kind 3: SpanningTreeHeuristic::Get (spanning_tree_heuristic.hpp:20-83);
 *   kind 4: VarianceHeuristic::Get (variance_heuristic.hpp:24-78);
 *   kind 5: HighestDegree(SpanningTree(Variance(BottomUpHeuristicGPU))), the
 *           bnbCPU chain of Treedepth/main.cpp:172-176;
 *   kind 6: HighestDegree(Variance(BottomUpHeuristicGPU)), the bnbGPU chain
 *           of Treedepth/main.cpp:180-183.
 * In kinds 5 and 6 the bottom-up link is td_bottom_up for graphs of at most
 * 32 vertices and absent (the reference's UINT_MAX) above; the context's
 * td_bottom_up queries then refer to the last such graph of the batch.
 * td_out[i] = depth of the tree, parent_concat (nullable) its parent array
 * (-1 = root).  Upper bounds, not proofs. */
int td_heuristic_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                       const uint64_t* adj_concat, int32_t kind, int32_t* td_out,
                       int8_t* parent_concat);

/* BottomUpHeuristicGPU::Get (Treedepth/src/branch_and_bound/heuristics/
 * bottom_up_heuristic.hpp:17-31) over BottomUpHeuristicGPUAlgorithm::
 * operator()(g, k) (bottom_up_heuristic_gpu_algorithm.hpp:67-90): levels
 * 0..k-1 of the bottom-up union-find DP for a graph of n <= 32 vertices,
 * with k = iterations, or with iterations = -1 as many levels as memory
 * holds (GetMaxIterations, bottom_up_heuristic_gpu_algorithm.cu:152-175; here
 * the context budget or the device's free memory).  *iterations_out
 * (nullable) = levels run (GetIterationsPerformed).  With all n + 1 levels,
 * *treedepth_out = depth of the elimination forest of GetElimination(n, n, 0)
 * and parent_out (nullable, n entries, -1 = root) that forest; otherwise
 * *treedepth_out = -1 (the reference's UINT_MAX).  An upper bound. */
int td_bottom_up(td_ctx* ctx, int32_t n, const uint64_t* adj, int32_t iterations,
                 int32_t* treedepth_out, int8_t* parent_out, int32_t* iterations_out);
/* BottomUpHeuristicGPUAlgorithm::GetTreedepth(nverts, subset_size,
 * subset_code) (bottom_up_heuristic_gpu_algorithm.cu:181-188) over the last
 * td_bottom_up: the kept forest's height for that subset (0 for the empty
 * set, and 0 for a size whose level was not run, like the reference). */
int td_bottom_up_get_treedepth(td_ctx* ctx, int32_t subset_size, uint64_t subset_code,
                               uint32_t* td_out);
/* Level k of the last td_bottom_up's history in colex order (history_,
 * bottom_up_heuristic_gpu_algorithm.hpp:60-61): the vertex added last and
 * the height of every k-subset (nullable outputs, out_len >= C(n, k)). */
int td_bottom_up_get_level(td_ctx* ctx, int32_t k, int8_t* last_out, uint8_t* height_out,
                           uint64_t out_len);
/* BottomUpHeuristicGPUAlgorithm::GetElimination(nverts, subset_size,
 * subset_code) (bottom_up_heuristic_gpu_algorithm.hpp:92-108): subset_size
 * vertices into order_out.  A size whose level was not run is TD_E_STATE
 * (the reference returns an empty list, or reads past its history at
 * subset_size == levels run). */
int td_bottom_up_get_elimination(td_ctx* ctx, int32_t subset_size, uint64_t subset_code,
                                 int32_t* order_out);

/* ---------------------------------------------------------------------- */
/* Branch-and-bound                                                        */
/* ---------------------------------------------------------------------- */
typedef struct td_bnb_stats {
  uint64_t graphs;     /* graphs in the call                              */
  uint64_t certified;  /* graphs whose treedepth was proven (LB = UB)     */
  uint64_t nodes;      /* search nodes expanded, all graphs               */
  uint64_t memo_hits;  /* nodes answered by the memo                      */
  double kernel_ms;    /* GPU time of the search kernel (HIP events)      */
  double total_ms;     /* host wall time of the whole call                */
} td_bnb_stats;

/* BnBGPU::operator()(g, heur_td) (Treedepth/src/bnb_gpu/bnb_gpu.hpp:13-31,
 * bnb_gpu.cu:264-380): exact treedepth by branch-and-bound, n <= 64.
 * heur_td is the caller's upper bound (the reference seeds best_td with it);
 * it is used only if a tree of that depth is found, so a wrong seed cannot
 * produce a wrong answer.  Unlike the reference, a decomposition is returned
 * (parent array) and certified_out = 1 iff the search completed (the search
 * stops after the "bnb.node_budget" parameter's node count, default 2e6). */
int td_bnb_solve(td_ctx* ctx, int32_t n, const uint64_t* adj, int32_t heur_td,
                 int32_t* treedepth_out, int8_t* parent_out,
                 uint8_t* certified_out);

/* Many graphs in one persistent launch, one wavefront per graph taken from a
 * device queue (no reference counterpart; the reference solves one graph
 * per process run).  ub_seed (nullable): per-graph upper bounds like
 * heur_td.  vertex_scores (nullable, sum n[i] floats): a learned proposal;
 * higher score = tried first as a root and used for an extra greedy upper
 * bound.  Scores only order the search; they never prune.
 * A graph of at most 24 vertices that 1,024 nodes have not settled is finished
 * by the subset DP (certified; its details count the search's nodes and end at
 * the k it had reached) if "bnb.node_budget" is above 32,768 or 0, none.
 * td_out / certified_out: ngraphs bytes; parent_concat: sum n[i] bytes.
 * With the context parameter "bnb.dp_max_n" = m > 0 (default 0), graphs of
 * at most m <= 32 vertices are answered by td_dp_solve_batch instead
 * (certified, td_dp_solve's tree; their details read heuristic = lower
 * bound = td, 0 nodes), the DP+B&B hybrid the reference proposes but does
 * not build (docs/introductory_documentation/our_approach/main.tex:181).
 * td_bnb_solve takes the same route.  Its in-search half is
 * "bnb.dp_small": components met by the search with at most that many
 * vertices are decided by a subset DP over their induced subgraph. */
int td_bnb_solve_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                       const uint64_t* adj_concat, const int32_t* ub_seed,
                       const float* vertex_scores, uint8_t* td_out,
                       int8_t* parent_concat, uint8_t* certified_out,
                       td_bnb_stats* stats);

/* Per-graph details of the last td_bnb_solve / td_bnb_solve_batch call on
 * this context (no reference counterpart; for analysis): the depth of the
 * initial heuristic tree, the proven lower bound and the search nodes.
 * Output arrays are nullable; count <= graphs of that call. */
int td_bnb_last_details(td_ctx* ctx, int32_t count, int32_t* heur_td_out,
                        int32_t* lower_bound_out, uint64_t* nodes_out);

/* How the last td_bnb_* call's descent ended, per graph (no reference
 * counterpart; for analysis): the last k it tried (td(C) <= k for every
 * component), -1 if it tried none, and the search nodes spent on that k --
 * the refutation of td - 1 when certified, the unfinished attempt when the
 * budget ran out.  Outputs nullable; count <= graphs of that call. */
int td_bnb_last_search(td_ctx* ctx, int32_t count, int32_t* last_k_out,
                       uint64_t* last_k_nodes_out);

/* Autotuner of the batched search launch (no reference counterpart: the
 * reference hard-codes its grid, Treedepth/src/bnb_gpu/bnb_gpu.cu:15-17):
 * times td_bnb_solve_batch's search on the given batch (scores nullable, as
 * there) under 4 or 8 waves per graph, 1/2/4/8 workgroups per CU and three
 * memo sizes around the default for the context's node budget, and keeps in
 * the context ("bnb.waves_per_graph", "bnb.groups", "bnb.memo_log2") the
 * shape with the most certified graphs per second of kernel time.  Cache
 * rules as td_dp_autotune; the key is the batch's (graph count, largest n,
 * sum of n), the node budget and whether scores were given.  The waves of a
 * graph share its node budget, so the shape can change which graphs are
 * certified within it, never a certified answer.  best_rate_out (nullable)
 * receives that rate.  The search launch itself (queue reset + persistent
 * kernel) is captured once per shape and buffers into a hipGraph and
 * replayed ("bnb.use_graph" = 0 launches it directly). */
int td_bnb_autotune_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                          const uint64_t* adj_concat, const float* vertex_scores,
                          const char* cache_path, double* best_rate_out);

/* ---------------------------------------------------------------------- */
/* Learned proposal (no reference counterpart: it feeds the reference's     */
/* LowerBoundInfo::attempt_order and Heuristic::Get extension points,       */
/* Treedepth/src/branch_and_bound/branch_and_bound.hpp:21-24, :38-42)       */
/* ---------------------------------------------------------------------- */
/* A message-passing MLP over per-vertex features (degree, core number,
 * vertices within distance 2, BFS eccentricity): 4 -> 64, two rounds of
 * mean aggregation (64+64 -> 64), then 64 -> 64 -> 64 -> 1.  BF16 weights and
 * activations on MFMA, FP32 accumulation, FP32 master weights + Adam.
 * Graph batches use 64 adjacency rows per graph (rows >= n zero). */
int td_mlp_num_params(void);
int td_mlp_init(td_ctx* ctx, uint64_t seed);
int td_mlp_set_weights(td_ctx* ctx, const float* w, int64_t count);
int td_mlp_get_weights(td_ctx* ctx, float* w, int64_t count);
/* features_out: ngraphs x 64 x 4 floats (rows >= n zero) */
int td_mlp_features(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                    const uint64_t* adj64, float* features_out);
/* scores_out: ngraphs x 64 floats (higher = better root) */
int td_mlp_scores(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                  const uint64_t* adj64, float* scores_out);
/* targets[i]: mask of optimal roots of graph i.  loss_out = mean
 * cross-entropy; grad_out (nullable): its gradient, td_mlp_num_params()
 * floats, ordered like the weights. */
int td_mlp_loss_grad(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                     const uint64_t* adj64, const uint64_t* targets,
                     float* loss_out, float* grad_out);
/* Adam on shuffled minibatches, entirely on the device. */
int td_mlp_train(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                 const uint64_t* adj64, const uint64_t* targets, int32_t epochs,
                 int32_t batch, float lr, uint64_t seed,
                 float* epoch_loss_out);
/* Labelled samples from the last td_dp_solve: random connected vertex sets S
 * (induced graph relabelled, 64 rows each), their optimal-root masks
 * {v : td(S \ v) = td(S) - 1} and td(S). */
int td_mlp_make_samples(td_ctx* ctx, int32_t count, uint64_t seed,
                        int32_t* n_out, uint64_t* adj64_out,
                        uint64_t* targets_out, uint8_t* td_out);

#ifdef __cplusplus
}
#endif
#endif /* TDHIP_H_ */
