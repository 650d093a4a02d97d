// bnb.hip -- exact treedepth by branch-and-bound over elimination orderings,
// one wavefront per graph, lanes = vertices (n <= 64), on gfx950.
//
// Reference path: BnBGPU (Treedepth/src/bnb_gpu/bnb_gpu.cu:167-380) and the
// CPU BranchAndBound it restates (Treedepth/src/branch_and_bound/
// branch_and_bound.cpp:51-115): choose a root of a component, recurse on the
// components left behind, prune when depth + lower bound cannot beat the best
// tree.  Here the search is the decision form
//   feasible(C, k)  <=>  td(C) <= k      (C connected)
//   = |C| <= k  or  exists v in C: feasible(D, k-1) for every component D of C-v
// run for k = UB-1, UB-2, ... until it fails, so the last failure proves
// td = UB.  Every answer is certified by an exhausted search, never by a
// heuristic.  Pruning uses proven bounds only:
//   * |C| <= k (path decomposition),
//   * EdgeLowerBound in its exact integer form: smallest d with
//     (d-1)(2|C|-d) >= 2|E(C)| (edge_lower_bound.hpp:13-20),
//   * k-core: a nonempty k-core of C means td(C) - 1 >= degeneracy >= k,
//   * path: a BFS from a peripheral vertex exposes a shortest path of e+1
//     vertices, and td(P_m) = ceil(log2(m+1)),
//   * a memo in HBM of proven facts per vertex set: lb (td(C) >= lb) and
//     sol (td(C) <= solk with root r).
// The wave holds one DFS stack in LDS; every set operation is a 64-bit mask
// and every neighbourhood is one ballot: lane u votes (adj[u] & F) != 0, so
// ballot = N(F).
#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <map>
#include <string>
#include <vector>

#include "ctx.hpp"

namespace tdhip {
namespace {

constexpr int kMaxBnBN = 64;
constexpr int kTagWord = 16;  // queue word holding the memo tag base (own 64 bytes)
constexpr int kStack = 72;  // Feasible(C, k) nests at most k + 1 <= 65 frames
// A graph of at most kFinishMaxN vertices that kFinishNodes search nodes have
// not settled is finished by the subset DP, where the node budget is above
// kFinishBudget (or 0, none).  The DP's 2^n subsets cost the same whatever the
// graph: 30 us on one CU for n = 18, 95 us on the device for n = 24, what a
// workgroup of 16 waves spends on 100 to 400 nodes, while a refutation on 20
// vertices of a random cubic graph takes 3e5 nodes (80 ms).  Past 1024 nodes
// (0.3 ms) the search is the worse bet.  Fewer would be faster on dense graphs
// (256 of 20..24 vertices: 7.0 ms, and 1.6 with the DP at once, which
// bnb.dp_max_n asks for), but sparse ones are settled by then, with the search's
// own trees and details.  kFinishBudget is no speed limit: a budget of some
// thousand nodes asks for an answer that may be uncertified after that much
// search (sweeps of the budget use 1e3 to 3e4), and keeps that meaning; the line
// lies between those and the budgets meant for certificates (5e4 and up).
constexpr int kFinishMaxN = 24;
constexpr uint64_t kFinishNodes = 1024, kFinishBudget = 32768;
constexpr uint32_t kBudgetChunk = 64;  // search nodes a wave takes from its graph's budget at once

struct BnBGraph {
  uint32_t n;
  int32_t ub_seed;   // caller's upper bound (<= 0: none)
  uint32_t use_scores;
  uint32_t pad;
  uint64_t adj[64];
  float score[64];
};

struct BnBOut {
  int32_t td;
  int32_t lb;        // proven lower bound (== td when certified)
  uint32_t certified;
  uint32_t heur_td;  // depth of the initial heuristic tree
  uint64_t nodes;
  uint64_t memo_hits;
  uint64_t last_nodes;  // nodes of the last k tried (the refutation when certified)
  int32_t last_k;       // that k, or -1 when no k was tried
  int32_t pad;
  int8_t parent[64];
};

struct Frame {
  uint64_t C, cand, pending, curD;
  int32_t k, v, state, pad;
};

enum : int { kNextRoot = 1, kNextComp = 2, kAfterChild = 3 };

// Orders this wave's LDS writes before its later reads by other lanes of
// the same wave (LDS operations of one wave execute in order; the fence
// keeps the compiler from moving them).  Workgroup-wide points use
// __syncthreads() explicitly.
__device__ __forceinline__ void Sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

__device__ __forceinline__ uint64_t Ballot(bool p) {
  return static_cast<uint64_t>(__ballot(p));
}

__device__ __forceinline__ uint64_t Uniform64(uint64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(x));
  const uint32_t hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(x >> 32));
  return (static_cast<uint64_t>(hi) << 32) | lo;
}

__device__ __forceinline__ int Uniform32(int x) {
  return __builtin_amdgcn_readfirstlane(x);
}

// Wave-wide sum and maximum of a 32-bit value by DPP: row shifts by 1, 2, 4
// and 8 leave each row's total in its lane 15; row broadcasts of lanes 15
// and 31 then bring rows 0-2 into lane 63, which is read back.  A lane whose
// DPP source lies outside its row (or in a row the mask leaves out) keeps
// `old`: 0 for the sum, its own value for the maximum.  Every lane of the
// wave must be active.
template <int kCtrl, int kRows>
__device__ __forceinline__ uint32_t Dpp(uint32_t old, uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_update_dpp(
      static_cast<int>(old), static_cast<int>(v), kCtrl, kRows, 0xf, false));
}

constexpr int kRowShr1 = 0x111, kRowShr2 = 0x112, kRowShr4 = 0x114, kRowShr8 = 0x118;
constexpr int kRowBcast15 = 0x142, kRowBcast31 = 0x143;

__device__ __forceinline__ uint32_t WaveSum(uint32_t v) {
  v += Dpp<kRowShr1, 0xf>(0u, v);
  v += Dpp<kRowShr2, 0xf>(0u, v);
  v += Dpp<kRowShr4, 0xf>(0u, v);
  v += Dpp<kRowShr8, 0xf>(0u, v);
  v += Dpp<kRowBcast15, 0xa>(0u, v);
  v += Dpp<kRowBcast31, 0xc>(0u, v);
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

__device__ __forceinline__ uint32_t WaveMaxU32(uint32_t v) {
  v = max(v, Dpp<kRowShr1, 0xf>(v, v));
  v = max(v, Dpp<kRowShr2, 0xf>(v, v));
  v = max(v, Dpp<kRowShr4, 0xf>(v, v));
  v = max(v, Dpp<kRowShr8, 0xf>(v, v));
  v = max(v, Dpp<kRowBcast15, 0xa>(v, v));
  v = max(v, Dpp<kRowBcast31, 0xc>(v, v));
  return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

// The lane of the largest key among the lanes of `set` (nonempty), ties to
// the lowest lane; key below 2^24.
__device__ __forceinline__ int ArgMaxLane(uint64_t set, uint32_t key, uint32_t* best) {
  const uint32_t lane = threadIdx.x & 63;
  const uint32_t K = ((set >> lane) & 1ull) ? (1u << 30) | (key << 6) | (63u - lane) : 0u;
  const uint32_t m = WaveMaxU32(K);
  if (best) *best = (m >> 6) & 0xFFFFFFu;
  return 63 - static_cast<int>(m & 63u);
}

// Component of `from` inside X (from in X): frontier grows by one ballot a
// round.  rounds = eccentricity of `from` in the component; last = the last
// nonempty frontier.  (The loop ends on an empty frontier, and comp takes
// the new frontier without the mask: ten instructions a round.)
__device__ __forceinline__ uint64_t Component(uint64_t myadj, uint64_t X,
                                              uint64_t from, int* rounds,
                                              uint64_t* last) {
  uint64_t comp = from, front = from, prev;
  int r = -1;
  do {
    prev = front;
    ++r;
    front = Ballot((myadj & front) != 0ull) & X & ~comp;
    comp |= front;
  } while (front);
  if (rounds) *rounds = r;
  if (last) *last = prev;
  return comp;
}

// smallest d with (d-1)(2n-d) >= 2e (EdgeLowerBound in integers)
__device__ __forceinline__ int EdgeLB(int n, int e) {
  int d = 1;
  if (e > 0) {
    // start near the root of (d-1)(2n-d) = 2e, then settle exactly: the
    // predicate is monotone in d on [1, n]
    const float est = n + 0.5f - sqrtf(fmaxf((n - 0.5f) * (n - 0.5f) - 2.0f * e, 0.f));
    d = min(max(static_cast<int>(est) - 1, 1), max(n, 1));
    while (d > 1 && (d - 2) * (2 * n - d + 1) >= 2 * e) --d;
    while ((d - 1) * (2 * n - d) < 2 * e) ++d;
  }
  return d;
}

// EdgeLB(n, e) > k for 0 <= k < n, without the root: (d - 1)(2n - d)
// increases with d on [1, n], so the smallest d reaching 2e exceeds k
// exactly when d = k falls short (at k = 0 both hold)
__device__ __forceinline__ bool EdgeLBAbove(int n, int e, int k) {
  return (k - 1) * (2 * n - k) < 2 * e;
}

__device__ __forceinline__ int CeilLog2(int x) {  // x >= 1
  return x <= 1 ? 0 : 32 - __builtin_clz(static_cast<uint32_t>(x - 1));
}

// Treedepth of a tree, exactly: the optimal vertex ranking of Schaeffer
// (1989), computed bottom-up over the BFS tree of C rooted at its lowest
// vertex.  Each vertex keeps its critical set L(v) (bit r-1 = rank r is
// visible from above v).  For v with children c_i:
//   U = union of L(c_i), D = ranks present in two or more L(c_i),
//   rank(v) = the smallest rank above max(D) that is not in U,
//   L(v) = {rank(v)} u {x in U : x > rank(v)};
// the largest rank is the treedepth of the tree and its vertex is unique.
// For a connected C with |E(C)| = |C| - 1 the BFS tree is C: the result is
// td(C) and *top an optimal root.  For any other connected C the BFS tree is
// a spanning subgraph, so the result is a lower bound on td(C).
// A tree of at most 64 vertices has an optimal ranking with at most 7
// ranks, so every L, U and D fits 32 bits.
// sU / sD: this wave's LDS scratch (64 entries each) for U and D; a child
// adds its L to its parent's entries with LDS atomics (the value an OR
// returns shows the bits an earlier child already brought, which go to D).
__device__ __forceinline__ int TreeRank(uint64_t myadj, uint64_t C, int* top, uint32_t* sU, uint32_t* sD) {
  const int lane = threadIdx.x & 63;
  const uint64_t root = C & (0ull - C);
  int mylvl = (root >> lane) & 1ull ? 0 : -1;
  int mypar = -1;
  uint64_t seen = root, front = root;
  int depth = 0;
  sU[lane] = 0;
  sD[lane] = 0;
  for (;;) {
    const uint64_t nb = Ballot((myadj & front) != 0ull) & C & ~seen;
    if (!nb) break;
    ++depth;
    if ((nb >> lane) & 1ull) {
      mylvl = depth;
      mypar = __builtin_ctzll(myadj & front);
    }
    seen |= nb;
    front = nb;
  }
  Sync();
  int rank = 0;
  uint32_t myL = 0;
  for (int l = depth; l >= 0; --l) {
    if (mylvl == l + 1) {
      const uint32_t old = atomicOr(sU + mypar, myL);
      if (old & myL) atomicOr(sD + mypar, old & myL);
    }
    Sync();
    if (mylvl == l) {
      const uint32_t U = sU[lane], dup = sD[lane];
      // ranks above the highest duplicated one (all when none); U and dup
      // use bits 0-6, so a free bit exists below bit 8
      const uint32_t above = dup ? ~0u << (32 - __builtin_clz(dup)) : ~0u;
      const int b = __builtin_ctz(~U & above);
      rank = b + 1;
      myL = (1u << b) | (U & (~1u << b));
    }
  }
  // largest rank (<= 64) and its (unique) vertex
  uint32_t best;
  const int v = ArgMaxLane(C, static_cast<uint32_t>(rank), &best);
  if (top) *top = v;
  return static_cast<int>(best);
}

// Lower bound on td(C), C connected, all from proven facts.
// Cheapest bound first: returns as soon as one exceeds k (k >= 0).
// e = |E(C)|, or -1 to count it here; ecc1 / last1: the rounds and last
// front of the BFS from C's lowest vertex if the caller ran it, else
// ecc1 = -1.  With decide set the caller only
// compares the result with k: bounds that cannot exceed k are skipped, so a
// result above k is the same, and a result of at most k only says that no
// bound exceeds k.
// *height (if non-null) receives the eccentricity of C's lowest vertex, the
// height of the BFS tree TreeRank ranks (0 when the BFS was not reached; a
// decision skips it for k at or above the bit length of |C|).
__device__ __forceinline__ int LowerBound(uint64_t myadj, bool in_c, uint64_t C,
                                          int k, int e = -1, int* height = nullptr,
                                          bool decide = false, int ecc1 = -1,
                                          uint64_t last1 = 0) {
  const int n = __builtin_popcountll(C);
  if (e < 0) {
    const int deg = in_c ? __builtin_popcountll(myadj & C) : 0;
    e = static_cast<int>(WaveSum(static_cast<uint32_t>(deg))) / 2;
  }
  int lb = 1;
  if (k < n) {
    if (EdgeLBAbove(n, e, k)) return EdgeLB(n, e);
    if (!decide) lb = EdgeLB(n, e);
  } else {
    lb = EdgeLB(n, e);
  }
  // path: double sweep BFS from the lowest vertex.  ceil(log2(ecc + 2)) is
  // at most the bit length of n (ecc <= n - 1), so it cannot exceed a k at
  // or above that length.
  if (!decide || k < 32 - __builtin_clz(static_cast<uint32_t>(n))) {
    int ecc = ecc1;
    uint64_t last = last1;
    if (ecc1 < 0) Component(myadj, C, C & (0ull - C), &ecc, &last);
    if (height) *height = ecc;
    Component(myadj, C, last & (0ull - last), &ecc, nullptr);
    lb = max(lb, CeilLog2(ecc + 2));
    if (lb > k) return lb;
  }
  // k-core of C nonempty => degeneracy >= k => td >= k+1
  if (k >= 1) {
    uint64_t X = C;
    for (;;) {
      const bool in = (X >> (threadIdx.x & 63)) & 1ull;
      const int d = in ? __builtin_popcountll(myadj & X) : 0;
      const uint64_t keep = Ballot(in && d >= k);
      if (keep == X) break;
      X = keep;
      if (!X) break;
    }
    if (X) lb = max(lb, k + 1);
  }
  return lb;
}

// degeneracy of X: largest d whose d-core is nonempty (parallel peeling)
__device__ __forceinline__ int Degeneracy(uint64_t myadj, uint64_t X0) {
  const int lane = threadIdx.x & 63;
  int d = 0;
  for (int t = 1; t < 64; ++t) {
    uint64_t X = X0;
    for (;;) {
      const bool in = (X >> lane) & 1ull;
      const int dd = in ? __builtin_popcountll(myadj & X) : 0;
      const uint64_t keep = Ballot(in && dd >= t);
      if (keep == X) break;
      X = keep;
    }
    if (!X) break;
    d = t;
  }
  return d;
}

// ---- memo: a table of 2^log2 buckets, 4 entries of 16 bytes a wave in each --
// entry = {key = the set, val}; val: bits 0-7 lb, 8-15 solk (0 = none), 16-23
// root, 32-63 tag = graph serial + 1 (0 = empty), so a new graph needs no
// clearing.  A wave writes its own four entries of a bucket and reads those of
// every wave of its workgroup, which are next to each other: what one wave has
// proven settles the set for all (with a table to each wave, 16 waves spent 1.8
// times the nodes of one on the same refutation: 21200 and 11400 on a near-tree
// of 49 vertices).
//
// Entries 0-2 get their key once for a tag: key, then (release) the val with
// the tag.  So a reader that has seen the val may take the facts of another
// wave if the key, read again after an acquire, is the set's.  Entry 3 is the
// one replaced when a bucket is full; only its own wave reads it.
struct MemoEntry {
  uint64_t key, val;
};

struct Memo {
  MemoEntry* table;  // the workgroup's
  uint32_t mask;     // buckets - 1
  uint32_t tag;
  uint32_t waves, wave;
};

__device__ __forceinline__ uint32_t BucketOf(uint64_t C, uint32_t mask) {
  return static_cast<uint32_t>((C * 0x9E3779B97F4A7C15ull) >> 40) & mask;
}

template <typename T>
__device__ __forceinline__ T MemoLoad(const T* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Lane 4 w + e reads entry e of wave w's part of C's bucket (lanes past the
// waves read along and take no part).  The lane that reads one of this wave's
// entries is the one that writes it, so its program order keeps every probe
// after every earlier store of the wave.  MemoIssue loads C's bucket so the
// latency can overlap other work; MemoResolve returns all that is known of C
// (0: nothing) and the entry to store at: C's own one of this wave, or else
// -1 - the first unused one (3 if none is).
struct Bucket {
  const MemoEntry* p;
  uint64_t key, val;
};

__device__ __forceinline__ Bucket MemoIssue(const Memo& m, uint64_t C) {
  Bucket b;
  const uint32_t at = min(threadIdx.x & 63u, 4u * m.waves - 1u);
  b.p = m.table + static_cast<size_t>(BucketOf(C, m.mask)) * (4u * m.waves) + at;
  b.val = MemoLoad(&b.p->val);
  b.key = MemoLoad(&b.p->key);
  return b;
}

__device__ __forceinline__ uint32_t MemoResolve(const Memo& m, uint64_t C,
                                                const Bucket& b, int* slot) {
  const uint32_t lane = threadIdx.x & 63;
  const bool own = lane >> 2 == m.wave;
  const bool live = static_cast<uint32_t>(b.val >> 32) == m.tag && lane < 4 * m.waves;
  bool hit = live && b.key == C && (own || (lane & 3) != 3);
  uint64_t hits = Ballot(hit);
  const uint64_t mine = 15ull << (4 * m.wave);
  if (hits & ~mine) {
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    hit = hit && (own || MemoLoad(&b.p->key) == C);
    hits = Ballot(hit);
  }
  const uint64_t known = hits & mine;
  const uint64_t frees = Ballot(own && !live);
  *slot = known ? static_cast<int>(__builtin_ctzll(known) & 3)
                : -1 - (frees ? static_cast<int>(__builtin_ctzll(frees) & 3) : 3);
  uint32_t data = 0;
  for (; hits; hits &= hits - 1) {  // the best of every wave's facts
    const uint32_t d = static_cast<uint32_t>(__builtin_amdgcn_readlane(
        static_cast<int>(static_cast<uint32_t>(b.val)), __builtin_ctzll(hits)));
    const uint32_t lb = max(data & 0xFFu, d & 0xFFu);
    const uint32_t have = data >> 8 & 0xFFu, more = d >> 8 & 0xFFu;
    const uint32_t sol = more && (!have || more < have) ? d : data;
    data = lb | (sol & 0xFFFF00u);
  }
  return data;
}

__device__ __forceinline__ uint32_t MemoProbe(const Memo& m, uint64_t C,
                                              int* slot) {
  const Bucket b = MemoIssue(m, C);
  return MemoResolve(m, C, b, slot);
}

// Adds to the facts known of C (`old`, the result of the probe that gave slot).
__device__ __forceinline__ void MemoStore(const Memo& m, uint64_t C, int slot,
                                          uint32_t old, uint32_t lb, uint32_t solk,
                                          uint32_t root) {
  const uint32_t osk = old >> 8 & 0xFFu;
  const uint32_t nlb = max(old & 0xFFu, lb);
  uint32_t sol = old & 0xFFFF00u;
  if (solk && (!osk || solk < osk)) sol = solk << 8 | root << 16;
  const uint32_t s = static_cast<uint32_t>(slot < 0 ? -1 - slot : slot);
  if ((threadIdx.x & 63) == 4 * m.wave + s) {  // the entry's owner
    MemoEntry* p = m.table + static_cast<size_t>(BucketOf(C, m.mask)) * (4u * m.waves) +
                   (4 * m.wave + s);
    if (slot < 0) {
      __hip_atomic_store(&p->key, C, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    }
    __hip_atomic_store(&p->val, static_cast<uint64_t>(m.tag) << 32 | sol | nlb,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  }
}

// Highest key among cand (nonempty), ties to the lowest vertex: plain =
// degree inside C, learned = the top 16 bits of the vertex score's
// order-preserving image.
__device__ __forceinline__ int PickRoot(bool use_scores, float score,
                                        uint64_t myadj, uint64_t C,
                                        uint64_t cand) {
  uint32_t key;
  if (use_scores) {
    const uint32_t u = __float_as_uint(score);
    key = ((u & 0x80000000u) ? ~u : (u | 0x80000000u)) >> 16;  // order-preserving
  } else {
    key = static_cast<uint32_t>(__builtin_popcountll(myadj & C));
  }
  return ArgMaxLane(cand, key, nullptr);
}

// Roots worth trying in C.  Root v dominates root u when
// N_C(u) \ {v} is a subset of N_C(v) \ {u}: then C \ v is isomorphic to a
// subgraph of C \ u (u -> v), so td(C \ v) <= td(C \ u) and u may be
// skipped.  Domination implies deg_C(u) <= deg_C(v) with equality only for
// twins; u is skipped only for a dominator of higher degree, or of equal
// degree and lower id, so every chain of skips ends at a root that is tried.
// A dominator of u is u's lowest neighbour w in C or a neighbour of w (w is
// in N_C(u) \ {v}, hence in N_C(v), unless v = w), so each lane tests only
// those, reading their rows from the graph's copy in LDS.
__device__ __forceinline__ uint64_t Undominated(uint64_t myadj, const uint64_t* adj,
                                                uint64_t C) {
  const int lane = threadIdx.x & 63;
  const bool in = (C >> lane) & 1ull;
  const uint64_t Nu = myadj & C;
  const int du = __builtin_popcountll(Nu);
  uint64_t cand = 0;
  if (in) {
    if (Nu) {
      const int w = __builtin_ctzll(Nu);
      cand = (adj[w] & C) | (1ull << w);
    } else {
      cand = C;
    }
    cand &= ~(1ull << lane);
  }
  bool dominated = false;
  for (uint64_t m = cand; m && !dominated; m &= m - 1) {
    const int v = __builtin_ctzll(m);
    const uint64_t Nv = adj[v] & C;
    const int dv = __builtin_popcountll(Nv);
    const bool sub = ((Nu & ~(1ull << v)) & ~(Nv & ~(1ull << lane))) == 0ull;
    const bool higher = dv > du || (dv == du && v < lane);
    dominated = sub && higher;
  }
  return C & ~Ballot(dominated);
}

// One wave's search.  Every function that takes it by reference is inlined: with
// one of them out of line the state lives in memory and the LDS pointers in it
// become generic ones, 5.0 us a node instead of 3.7 for a wave alone.
struct Search {
  Frame* st;  // LDS stack
  uint64_t myadj;
  const uint64_t* adj;  // the graph's rows in LDS (shared by the workgroup)
  float score;
  bool use_scores;
  Memo memo;
  uint64_t nodes, hits;
  // node budget of the graph, shared by its waves: each wave takes chunks of
  // kBudgetChunk nodes from the workgroup's LDS counter *pool (nodes handed
  // out so far) and `left` counts what remains of its chunk; budget = 0
  // turns the limit off
  uint64_t budget;
  unsigned long long* pool;
  uint32_t left;
  bool aborted;          // node budget exhausted: results are not proofs
  const int* cancel;     // LDS flag set when another wave of the graph succeeded
  uint32_t* tu;          // TreeRank scratch (this wave's LDS): unions
  uint32_t* tdup;        // and duplicated ranks per parent
  bool building;         // inside Build: every decided set must leave a root
  // components of at most dp_small vertices are answered by SmallDP, in this
  // wave's LDS table sdp (2^dp_small bytes) and rows sdp_rows (0: off)
  int dp_small;
  uint8_t* sdp;
  uint16_t* sdp_rows;
};

// ---- the DP + B&B hybrid: exact treedepth of a small component ----------
constexpr int kSmallDPMax = 12;
constexpr size_t kSmallDPBytes = (1u << kSmallDPMax) + 32;  // table + rows

// C(x, j) for 0 <= x, j <= kSmallDPMax (0 for j > x)
__constant__ uint16_t kSmallBinom[kSmallDPMax + 1][kSmallDPMax + 1] = {
    {1, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {1, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {1, 2, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {1, 3, 3, 1, 0, 0, 0, 0, 0, 0, 0, 0, 0},
    {1, 4, 6, 4, 1, 0, 0, 0, 0, 0, 0, 0, 0},
    {1, 5, 10, 10, 5, 1, 0, 0, 0, 0, 0, 0, 0},
    {1, 6, 15, 20, 15, 6, 1, 0, 0, 0, 0, 0, 0},
    {1, 7, 21, 35, 35, 21, 7, 1, 0, 0, 0, 0, 0},
    {1, 8, 28, 56, 70, 56, 28, 8, 1, 0, 0, 0, 0},
    {1, 9, 36, 84, 126, 126, 84, 36, 9, 1, 0, 0, 0},
    {1, 10, 45, 120, 210, 252, 210, 120, 45, 10, 1, 0, 0},
    {1, 11, 55, 165, 330, 462, 462, 330, 165, 55, 11, 1, 0},
    {1, 12, 66, 220, 495, 792, 924, 792, 495, 220, 66, 12, 1}};
__device__ __forceinline__ uint32_t SmallBinom(int x, int j) { return kSmallBinom[x][j]; }

// Exact treedepth of a connected set C of n <= kSmallDPMax vertices by the
// subset DP over C's induced subgraph, its vertices renumbered 0..n-1 in
// increasing order: T[S] = 2 td(S) + [S connected] for every S, level by
// level (|S| = 1, 2, ...), each lane taking a contiguous run of a level's
// subsets in colex order.  td(S) = 1 + min over v of td(S \ v) if S is
// connected, else the max over v (some component stays whole); S is
// connected iff it is a single vertex, or none of its vertices is isolated
// in S and some S \ v is connected.  Returns td(C) and in *root the lowest
// vertex v of C with td(C \ v) = td(C) - 1.
__device__ __attribute__((noinline)) int SmallDP(const Search& S, uint64_t C, int n,
                                                int* root) {
  const int lane = threadIdx.x & 63;
  uint8_t* T = S.sdp;
  uint16_t* rows = S.sdp_rows;
  const bool in_c = (C >> lane) & 1ull;
  const uint64_t below = (1ull << lane) - 1ull;  // lane < 64
  const int r = __builtin_popcountll(C & below);
  if (in_c) {
    uint32_t row = 0;
    for (uint64_t a = S.myadj & C; a; a &= a - 1) {
      const int u = __builtin_ctzll(a);
      row |= 1u << __builtin_popcountll(C & ((1ull << u) - 1ull));
    }
    rows[r] = static_cast<uint16_t>(row);
  }
  if (lane == 0) T[0] = 0;
  Sync();
  for (int k = 1; k <= n; ++k) {
    const uint32_t cnt = SmallBinom(n, k);
    const uint32_t per = (cnt + 63u) / 64u;
    const uint32_t i0 = static_cast<uint32_t>(lane) * per;
    const uint32_t i1 = min(cnt, i0 + per);
    if (i0 < i1) {
      // colex unrank of i0 among the k-subsets of {0..n-1}
      uint32_t X = 0, rem = i0;
      for (int x = n - 1, kk = k; x >= 0 && kk > 0; --x) {
        const uint32_t c = SmallBinom(x, kk);
        if (rem >= c) {
          X |= 1u << x;
          rem -= c;
          --kk;
        }
      }
      for (uint32_t i = i0;;) {
        uint32_t mn = 0xFFu, mx = 0u;
        bool sub_conn = false, iso = false;
        for (uint32_t b = X; b; b &= b - 1) {
          const int v = __builtin_ctz(b);
          const uint32_t t = T[X ^ (1u << v)];
          mn = min(mn, t >> 1);
          mx = max(mx, t >> 1);
          sub_conn |= (t & 1u) != 0;
          iso |= (rows[v] & X) == 0;
        }
        const bool conn = k == 1 || (!iso && sub_conn);
        T[X] = static_cast<uint8_t>(((conn ? mn + 1u : mx) << 1) | (conn ? 1u : 0u));
        if (++i >= i1) break;
        // next k-subset in colex (numeric) order
        const uint32_t t = X | (X - 1u);
        X = (t + 1u) | (((~t & (0u - ~t)) - 1u) >> (__builtin_ctz(X) + 1));
      }
    }
    Sync();
  }
  const uint32_t full = (1u << n) - 1u;
  const int td = static_cast<int>(T[full] >> 1);
  // lanes outside C read T[full], inside the table
  const uint32_t without = in_c ? (full ^ (1u << r)) : full;
  const bool cand = in_c && static_cast<int>(T[without] >> 1) == td - 1;
  const uint64_t roots = Ballot(cand);
  *root = __builtin_ctzll(roots);
  Sync();  // the table is free for the next call
  return td;
}

// A halted search (budget or cancellation) returns false without storing a
// lower bound, so the memo only ever holds proven facts.
__device__ __forceinline__ bool Halted(Search& S) {
  if (S.aborted) return true;
  if (S.cancel) {
    const int c = __atomic_load_n(S.cancel, __ATOMIC_RELAXED);
    if (Uniform32(c)) {
      S.aborted = true;
      return true;
    }
  }
  return false;
}

// One search node: entering (C, k) with |C| > k >= 1, C connected.  Counts
// the node, then decides it from the memo and the bounds where it can:
// returns 1 (td(C) <= k), 0 (td(C) > k, or the search halted) or -1 (not
// decided: *roots holds the roots to try).  e = |E(C)| or -1; ecc / last:
// the BFS from C's lowest vertex (its rounds and last front) when the caller
// has run it, else ecc = -1.
__device__ __forceinline__ int Enter(Search& S, uint64_t C, int k, int e, int ecc, uint64_t last,
                     uint64_t* roots) {
  const int lane = threadIdx.x & 63;
  const int n = __builtin_popcountll(C);
  if (Halted(S)) return 0;
  ++S.nodes;
  if (S.budget) {
    if (S.left == 0) {  // the next chunk of the graph's budget
      uint32_t got = 0;
      if (lane == 0) {
        const unsigned long long chunk = kBudgetChunk;
        const unsigned long long old = atomicAdd(S.pool, chunk);
        if (old < S.budget) got = static_cast<uint32_t>(min(chunk, S.budget - old));
      }
      S.left = Uniform32(__shfl(got, 0));
      if (S.left == 0) {
        S.aborted = true;
        return 0;
      }
    }
    --S.left;
  }
  const Bucket me = MemoIssue(S.memo, C);
  const bool in_c = (C >> lane) & 1ull;
  const int ecount =
      e >= 0 ? e : static_cast<int>(WaveSum(in_c ? __builtin_popcountll(S.myadj & C) : 0)) / 2;
  if (ecount == n - 1) {
    // a tree: td <= 1 + floor(log2 |C|), so k at least that decides it
    // without ranking (Build, which needs the root, ranks it)
    if (!S.building && k >= 32 - __builtin_clz(static_cast<uint32_t>(n))) return 1;
    // exact treedepth and an optimal root, no search
    int top;
    const int t = TreeRank(S.myadj, C, &top, S.tu, S.tdup);
    int slot;
    const uint32_t md = MemoResolve(S.memo, C, me, &slot);
    MemoStore(S.memo, C, slot, md, static_cast<uint32_t>(t), static_cast<uint32_t>(t),
              static_cast<uint32_t>(top));
    return t <= k ? 1 : 0;
  }
  // a memo entry decides before any bound is computed (about a third of
  // the nodes of sparse graphs)
  int slot;
  const uint32_t md = MemoResolve(S.memo, C, me, &slot);
  {
    const uint32_t mlb = md & 0xFF, sk = (md >> 8) & 0xFF;
    if (sk && sk <= static_cast<uint32_t>(k)) { ++S.hits; return 1; }
    if (mlb > static_cast<uint32_t>(k)) { ++S.hits; return 0; }
  }
  // the DP + B&B hybrid: a small component's exact treedepth and an optimal
  // root from a subset DP, instead of a search below it
  if (n <= S.dp_small) {
    int top;
    const int t = SmallDP(S, C, n, &top);
    MemoStore(S.memo, C, slot, md, static_cast<uint32_t>(t), static_cast<uint32_t>(t),
              static_cast<uint32_t>(top));
    return t <= k ? 1 : 0;
  }
  int height = 0;
  int lb = LowerBound(S.myadj, in_c, C, k, ecount, &height, true, ecc, last);
  // the BFS spanning tree of C has treedepth <= 1 + floor(log2 |C|) (a
  // centroid leaves parts of at most half the vertices) and <= its height
  // + 1, so its ranking can only exceed k when k is below both
  if (lb <= k && ecount - (n - 1) <= 12 && k < 32 - __builtin_clz(static_cast<uint32_t>(n)) &&
      k <= height)
    lb = max(lb, TreeRank(S.myadj, C, nullptr, S.tu, S.tdup));
  if (lb > k) {
    MemoStore(S.memo, C, slot, md, static_cast<uint32_t>(lb), 0, 0);
    return 0;
  }
  *roots = n >= 4 ? Undominated(S.myadj, S.adj, C) : C;
  return -1;
}

// Decision search td(C0) <= k0 ?  Uniform across the wave.  Stack frames
// are written by lane 0 and read back through readfirstlane (lane 0's own
// view), so no barrier is needed between a frame update and its use.  A
// child that its node decides at once (most of them: a bound or the memo)
// gets no frame; a frame is pushed only for a child whose roots are tried.
__device__ __forceinline__ bool Feasible(Search& S, uint64_t C0, int k0) {
  const int lane = threadIdx.x & 63;
  {
    const int n0 = __builtin_popcountll(C0);
    if (n0 <= k0) return true;
    if (k0 <= 0) return false;
  }
  int sp = 0;
  bool ret = false;
  // a node to enter before the next frame step (one call site for Enter):
  // (eC, ek) with its edge count and first BFS, as a child of the top
  // frame (whose pending / trivial sets are given) or as the root
  bool entering = true;
  uint64_t eC = C0, e_pending = 0, e_trivial = 0, e_last = 0;
  int ek = k0, e_e = -1, e_ecc = -1;
  for (;;) {
    if (entering) {
      entering = false;
      uint64_t roots = 0;
      const int r = Enter(S, eC, ek, e_e, e_ecc, e_last, &roots);
      if (sp == 0) {  // the root
        if (r >= 0) return r != 0;
      } else if (r >= 0) {
        // a child decided at once: continue as on its return
        ret = r != 0;
        if (lane == 0) {
          Frame* P = &S.st[sp - 1];
          if (ret) {
            P->pending = e_pending & ~e_trivial & ~eC;
            P->state = kNextComp;
          } else {
            P->state = kNextRoot;
          }
        }
        continue;
      } else {
        if (lane == 0) {
          Frame* P = &S.st[sp - 1];
          P->pending = e_pending & ~e_trivial;
          P->curD = eC;
          P->state = kAfterChild;
        }
      }
      if (sp >= kStack) {  // cannot happen: Feasible(C, k) nests at most k + 1 frames
        S.aborted = true;
        ret = false;
        if (sp == 0) return false;
        continue;
      }
      if (lane == 0) {
        Frame f;
        f.C = eC;
        f.k = ek;
        f.state = kNextRoot;
        f.cand = roots;
        f.pending = f.curD = 0;
        f.v = -1;
        f.pad = 0;
        S.st[sp] = f;
      }
      ++sp;
      continue;
    }
    if (sp == 0) break;
    Frame* F = &S.st[sp - 1];
    const uint64_t C = Uniform64(F->C);
    const int k = Uniform32(F->k);
    const int state = Uniform32(F->state);
    if (state == kNextRoot) {
      const uint64_t cand = Uniform64(F->cand);
      if (cand == 0 || S.aborted) {
        if (!S.aborted) {
          int slot;
          const uint32_t md = MemoProbe(S.memo, C, &slot);
          MemoStore(S.memo, C, slot, md, static_cast<uint32_t>(k + 1), 0, 0);
        }
        ret = false;
        --sp;
        continue;
      }
      const int v = PickRoot(S.use_scores, S.score, S.myadj, C, cand);
      if (lane == 0) {
        F->cand = cand & ~(1ull << v);
        F->v = v;
        F->pending = C & ~(1ull << v);
        F->state = kNextComp;
      }
      continue;
    }
    if (state == kNextComp) {
      const uint64_t pending = Uniform64(F->pending);
      if (pending == 0) {
        const int v = Uniform32(F->v);
        int slot;
        const uint32_t md = MemoProbe(S.memo, C, &slot);
        MemoStore(S.memo, C, slot, md, 0, static_cast<uint32_t>(k),
                  static_cast<uint32_t>(v));
        ret = true;
        --sp;
        continue;
      }
      // every component of C - v still unverified: one with a proven bound
      // above k-1 rejects v now; components of at most k-1 vertices pass; the
      // largest remaining one is searched next.  Each component is found by
      // a BFS from its lowest vertex, the BFS its node's path bound starts
      // with, so the largest one's rounds and last front go along.
      uint64_t rest = pending, D = 0, trivial = 0, bestlast = 0;
      int bestn = 0, beste = 0, bestecc = 0;
      bool reject = false;
      while (rest) {
        int ecc;
        uint64_t last;
        const uint64_t Dc = Component(S.myadj, rest, rest & (0ull - rest), &ecc, &last);
        rest &= ~Dc;
        const int nd = __builtin_popcountll(Dc);
        if (nd <= k - 1) {
          trivial |= Dc;
          continue;
        }
        const bool in_d = (Dc >> lane) & 1ull;
        const int dd = in_d ? __builtin_popcountll(S.myadj & Dc) : 0;
        const int ed = static_cast<int>(WaveSum(static_cast<uint32_t>(dd))) / 2;
        if (EdgeLBAbove(nd, ed, k - 1)) {  // k - 1 < nd
          reject = true;
          break;
        }
        if (ed == nd - 1) {  // a tree: decided exactly here
          if (TreeRank(S.myadj, Dc, nullptr, S.tu, S.tdup) > k - 1) {
            reject = true;
            break;
          }
          trivial |= Dc;
          continue;
        }
        if (nd > bestn) {
          bestn = nd;
          beste = ed;
          bestecc = ecc;
          bestlast = last;
          D = Dc;
        }
      }
      if (reject) {
        if (lane == 0) F->state = kNextRoot;
        continue;
      }
      if (!D) {  // only trivial components left
        if (lane == 0) F->pending = 0;
        continue;
      }
      // the child's node (|D| > k - 1 >= 1 here: k - 1 = 0 rejects above)
      entering = true;
      eC = D;
      ek = k - 1;
      e_e = beste;
      e_ecc = bestecc;
      e_last = bestlast;
      e_pending = pending;
      e_trivial = trivial;
      continue;
    }
    // kAfterChild
    if (lane == 0) {
      if (ret) {
        F->pending &= ~F->curD;
        F->state = kNextComp;
      } else {
        F->state = kNextRoot;
      }
    }
  }
  return ret;
}

// Rebuild a tree of depth <= k for connected C from the memo's roots,
// re-running the search for a set whose entry was evicted.  parent[] in LDS.
__device__ __forceinline__ void Build(Search& S, uint64_t C0, int k0, int par0, int8_t* parent,
                      uint64_t* bst, int* bk, int* bpar) {
  const int lane = threadIdx.x & 63;
  int sp = 0;
  auto push = [&](uint64_t C, int k, int par) {
    if (lane == 0) {
      bst[sp] = C;
      bk[sp] = k;
      bpar[sp] = par;
    }
    ++sp;
    Sync();
  };
  push(C0, k0, par0);
  while (sp > 0) {
    --sp;
    const uint64_t C = Uniform64(bst[sp]);
    const int k = Uniform32(bk[sp]);
    const int par = Uniform32(bpar[sp]);
    const int n = __builtin_popcountll(C);
    if (n <= k) {  // chain in ascending id order
      int prev = par;
      for (uint64_t m = C; m; m &= m - 1) {
        const int u = __builtin_ctzll(m);
        if (lane == 0) parent[u] = static_cast<int8_t>(prev);
        prev = u;
      }
      Sync();
      continue;
    }
    int slot;
    uint32_t md = MemoProbe(S.memo, C, &slot);
    uint32_t sk = (md >> 8) & 0xFF;
    if (!(sk && sk <= static_cast<uint32_t>(k))) {
      const uint64_t saved_budget = S.budget;
      S.budget = 0;  // the set is known feasible: finish the search
      S.building = true;
      Feasible(S, C, k);
      S.building = false;
      S.budget = saved_budget;
      md = MemoProbe(S.memo, C, &slot);
      sk = (md >> 8) & 0xFF;
      if (!(sk && sk <= static_cast<uint32_t>(k))) {
        // no tree can be rebuilt: report the call as uncertified and keep
        // the previous best tree
        S.aborted = true;
        return;
      }
    }
    const int v = static_cast<int>((md >> 16) & 0xFF);
    if (lane == 0) parent[v] = static_cast<int8_t>(par);
    Sync();
    uint64_t rest = C & ~(1ull << v);
    while (rest) {
      const uint64_t D = Component(S.myadj, rest, rest & (0ull - rest), nullptr, nullptr);
      rest &= ~D;
      push(D, static_cast<int>(sk) - 1, v);
    }
  }
}

// Greedy top-down tree: root of each component = best key (degree inside
// the component, or the learned score).  Returns its depth; parent in LDS.
__device__ int GreedyTree(Search& S, uint64_t V, bool use_scores, int8_t* parent,
                          uint64_t* bst, int* bk, int* bpar) {
  const int lane = threadIdx.x & 63;
  int sp = 0, depth = 0;
  uint64_t rest = V;
  while (rest) {
    const uint64_t D = Component(S.myadj, rest, rest & (0ull - rest), nullptr, nullptr);
    rest &= ~D;
    if (lane == 0) { bst[sp] = D; bk[sp] = 1; bpar[sp] = -1; }
    ++sp;
  }
  Sync();
  while (sp > 0) {
    --sp;
    const uint64_t C = Uniform64(bst[sp]);
    const int d = Uniform32(bk[sp]);
    const int par = Uniform32(bpar[sp]);
    depth = max(depth, d);
    const int v = PickRoot(use_scores, S.score, S.myadj, C, C);
    if (lane == 0) parent[v] = static_cast<int8_t>(par);
    uint64_t r = C & ~(1ull << v);
    while (r) {
      const uint64_t D = Component(S.myadj, r, r & (0ull - r), nullptr, nullptr);
      r &= ~D;
      if (lane == 0) { bst[sp] = D; bk[sp] = d + 1; bpar[sp] = v; }
      ++sp;
    }
    Sync();
  }
  return depth;
}

// Minimum-degree elimination ordering with fill-in; the elimination tree of
// the filled graph (parent = the neighbour eliminated next) is a treedepth
// decomposition.  Sequential over vertices, lanes hold the filled rows.
__device__ int MinDegreeTree(uint64_t myadj, uint64_t V, int8_t* parent,
                             int* depth_tmp) {
  const int lane = threadIdx.x & 63;
  uint64_t fill = myadj;
  uint64_t remain = V;
  // elimination index per vertex, kept by its lane
  int idx = 1 << 20;
  int step = 0;
  while (remain) {
    const bool in = (remain >> lane) & 1ull;
    const int d = in ? __builtin_popcountll(fill & remain) : 1 << 20;
    // min degree, ties lowest id
    uint64_t key = in ? (static_cast<uint64_t>(d) << 8) | static_cast<uint64_t>(lane) : ~0ull;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const uint64_t o = __shfl_xor(key, off);
      key = o < key ? o : key;
    }
    const int v = static_cast<int>(key & 0xFF);
    const uint64_t nv =
        Uniform64(static_cast<uint64_t>(__shfl(static_cast<unsigned long long>(fill), v))) &
        remain & ~(1ull << v);
    // make N(v) a clique among the remaining vertices
    if ((nv >> lane) & 1ull) fill |= nv & ~(1ull << lane);
    if (lane == v) idx = step;
    remain &= ~(1ull << v);
    ++step;
  }
  // parent(v) = neighbour (in the filled graph) with the smallest later
  // index; a uniform loop so every lane takes part in each shuffle
  const bool in = (V >> lane) & 1ull;
  int p = -1, best = 1 << 21;
  for (int u = 0; u < 64; ++u) {
    const int iu = __shfl(idx, u);
    if (in && ((fill >> u) & 1ull) && ((V >> u) & 1ull) && iu > idx && iu < best) {
      best = iu;
      p = u;
    }
  }
  if (in) parent[lane] = static_cast<int8_t>(p);
  Sync();
  // depth: iterate parent pointers (depth_tmp in LDS)
  int dep = 0;
  if (in) {
    int u = lane;
    dep = 1;
    while (parent[u] >= 0 && dep <= 64) {
      u = parent[u];
      ++dep;
    }
  }
  (void)depth_tmp;
  uint32_t mx = in ? static_cast<uint32_t>(dep) : 0u;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = max(mx, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mx), off)));
  return static_cast<int>(mx);
}

// One workgroup of W waves per graph, graphs taken from a device queue.
// Wave 0 computes the upper-bound trees and the static bound; then for each
// k = UB-1, UB-2, ... the W waves share out the top-level root candidates (in
// key order, each wave claiming the next one when it is free), each
// searching its candidates with the waves' common memo and drawing on the graph's
// node budget in chunks.  A wave that finds a decomposition raises s_found
// and the others stop; if none does and the budget did not run out, td > k
// is proven.
constexpr int kMaxWaves = 16;
// dynamic LDS per wave: its frame stack, then its two 64-entry rank arrays,
// then (with the small-component DP on) the DP table and rows
constexpr size_t kWaveLds = kStack * sizeof(Frame) + 2 * 64 * sizeof(uint32_t);
__host__ __device__ constexpr size_t WaveLds(int dp_small) {
  return kWaveLds + (dp_small > 0 ? kSmallDPBytes : 0);
}

// 80 VGPRs (6 waves per SIMD): the search is latency-bound, and measured on
// the 1024-graph batch 8 waves per graph at this occupancy resolve 1.5x the
// nodes per second of 4 waves at 93 VGPRs (5 per SIMD).  The per-wave LDS is
// sized by the launch's wave count, so 8-wave workgroups still fit three to
// a CU and 12-wave ones two (24 waves either way); a 16-wave workgroup is
// alone on its CU, for batches with fewer graphs than CUs.
__global__ __launch_bounds__(64 * kMaxWaves)
__attribute__((amdgpu_waves_per_eu(6, 6))) void BnBKernel(
    const BnBGraph* __restrict__ gs, BnBOut* __restrict__ outs,
    MemoEntry* __restrict__ memo_base, int memo_log2, uint64_t node_budget, uint64_t small_budget,
    int dp_small, int ngraphs, uint32_t* __restrict__ queue) {
  // queue[0]: the next graph; queue[kTagWord]: this call's memo tag base,
  // written before the launch (a captured launch replays with new tags)
  const uint32_t tag_base = queue[kTagWord];
  extern __shared__ uint4 s_waves[];  // W x WaveLds(dp_small) bytes
  __shared__ int8_t s_parent[64], s_best[64];
  __shared__ uint64_t s_bst[130];
  __shared__ int s_bk[130], s_bpar[130];
  __shared__ uint64_t s_comps[64];
  __shared__ uint64_t s_adj[64];
  __shared__ int s_gi, s_ub, s_lb, s_heur, s_ncomp;
  __shared__ int s_found, s_winner, s_wroot, s_abort;
  __shared__ unsigned long long s_nodes, s_hits, s_last_nodes, s_pool;
  __shared__ int s_next;  // next top-level root candidate to hand out
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int W = blockDim.x >> 6;
  Search S;
  S.building = false;
  {
    uint8_t* mine = reinterpret_cast<uint8_t*>(s_waves) + static_cast<size_t>(wid) * WaveLds(dp_small);
    S.st = reinterpret_cast<Frame*>(mine);
    S.tu = reinterpret_cast<uint32_t*>(mine + kStack * sizeof(Frame));
    S.tdup = S.tu + 64;
    S.dp_small = dp_small;
    S.sdp = mine + kWaveLds;
    S.sdp_rows = reinterpret_cast<uint16_t*>(S.sdp + (1u << kSmallDPMax));
  }
  S.memo.table =
      memo_base + (static_cast<size_t>(blockIdx.x * W) << (memo_log2 + 2));
  S.memo.waves = static_cast<uint32_t>(W);
  S.memo.wave = static_cast<uint32_t>(Uniform32(wid));
  S.memo.mask = (1u << memo_log2) - 1u;
  for (;;) {
    if (threadIdx.x == 0) s_gi = static_cast<int>(atomicAdd(queue, 1u));
    __syncthreads();
    const int gi = s_gi;
    if (gi >= ngraphs) break;  // uniform across the workgroup
    const BnBGraph* g = gs + gi;
    const int n = static_cast<int>(g->n);
    const uint64_t V = n >= 64 ? ~0ull : ((1ull << n) - 1ull);
    S.myadj = lane < n ? g->adj[lane] : 0ull;
    // every wave has left the previous graph (barrier above)
    if (wid == 0) s_adj[lane] = S.myadj;
    __syncthreads();
    S.adj = s_adj;
    S.score = lane < n ? g->score[lane] : 0.f;
    S.use_scores = g->use_scores != 0;
    S.memo.tag = tag_base + static_cast<uint32_t>(gi) + 1u;
    S.nodes = 0;
    S.hits = 0;
    // the node budget is per graph; the waves draw on it in chunks
    S.budget = n <= kFinishMaxN ? small_budget : node_budget;
    S.pool = &s_pool;
    S.left = 0;
    S.aborted = false;
    S.cancel = nullptr;
    if (threadIdx.x == 0) {
      s_nodes = 0;
      s_hits = 0;
      s_last_nodes = 0;
      s_pool = 0;
      s_abort = 0;
    }
    if (wid == 0) {
      // ---- initial upper bound: best of the greedy trees ----------------
      int ub = GreedyTree(S, V, false, s_best, s_bst, s_bk, s_bpar);
      if (S.use_scores) {
        const int t = GreedyTree(S, V, true, s_parent, s_bst, s_bk, s_bpar);
        if (t < ub) {
          ub = t;
          s_best[lane] = s_parent[lane];
        }
      }
      {
        const int t = MinDegreeTree(S.myadj, V, s_parent, nullptr);
        if (t < ub) {
          ub = t;
          s_best[lane] = s_parent[lane];
        }
      }
      Sync();
      const int heur = ub;
      int ncomp = 0;
      {
        uint64_t rest = V;
        while (rest) {
          const uint64_t D = Component(S.myadj, rest, rest & (0ull - rest), nullptr, nullptr);
          if (lane == 0) s_comps[ncomp] = D;
          ++ncomp;
          rest &= ~D;
        }
      }
      // caller's seed: accept it only with a tree of that depth
      const int seed = g->ub_seed;
      if (seed > 0 && seed < ub) {
        bool ok = true;
        for (int c = 0; c < ncomp && ok; ++c) ok = Feasible(S, Uniform64(s_comps[c]), seed);
        if (ok && !S.aborted) {
          s_parent[lane] = -1;
          Sync();
          for (int c = 0; c < ncomp && !S.aborted; ++c)
            Build(S, Uniform64(s_comps[c]), seed, -1, s_parent, s_bst, s_bk, s_bpar);
          if (!S.aborted) {
            ub = seed;
            s_best[lane] = s_parent[lane];
            Sync();
          }
        }
        S.aborted = false;  // the seed check does not decide certification
      }
      int lb = 1;
      for (int c = 0; c < ncomp; ++c) {
        const uint64_t Cc = Uniform64(s_comps[c]);
        lb = max(lb, LowerBound(S.myadj, (Cc >> lane) & 1ull, Cc, 1 << 10));
      }
      lb = max(lb, Degeneracy(S.myadj, V) + 1);
      if (lane == 0) {
        s_ub = ub;
        s_lb = lb;
        s_heur = heur;
        s_ncomp = ncomp;
      }
    }
    __syncthreads();
    int ub = s_ub, lb = s_lb;
    const int ncomp = s_ncomp;
    bool uncertain = false;
    // this wave's node count when the last k began, and that k
    uint64_t nodes_k0 = S.nodes;
    int last_k = -1;
    // ---- descend: k = ub-1 until it fails -------------------------------
    while (ub - 1 >= lb) {
      const int k = ub - 1;
      nodes_k0 = S.nodes;
      last_k = k;
      bool all_ok = true;
      for (int c = 0; c < ncomp && all_ok; ++c) {
        const uint64_t C = s_comps[c];
        const int nc = __builtin_popcountll(C);
        if (nc <= k) continue;
        if (threadIdx.x == 0) {
          s_found = 0;
          s_winner = -1;
          s_wroot = -1;
          s_next = 0;
        }
        __syncthreads();
        S.cancel = &s_found;
        const bool in_c = (C >> lane) & 1ull;
        const bool lb_fail = LowerBound(S.myadj, in_c, C, k, -1, nullptr, true) > k;
        if (!lb_fail) {
          // the top-level roots in key order, handed out one at a time: a
          // wave claims the next index when it is free
          auto claim = [&] {
            int t = 0;
            if (lane == 0) t = atomicAdd(&s_next, 1);
            return Uniform32(__shfl(t, 0));
          };
          uint64_t cand = nc >= 4 ? Undominated(S.myadj, S.adj, C) : C;
          int mine = claim();
          for (int i = 0; cand; ++i) {
            const int v = PickRoot(S.use_scores, S.score, S.myadj, C, cand);
            cand &= ~(1ull << v);
            if (i != mine) continue;
            if (Halted(S)) break;
            bool ok = true;
            uint64_t rest = C & ~(1ull << v);
            while (rest && ok) {
              const uint64_t D = Component(S.myadj, rest, rest & (0ull - rest), nullptr, nullptr);
              rest &= ~D;
              if (__builtin_popcountll(D) > k - 1) ok = Feasible(S, D, k - 1);
            }
            if (ok && !S.aborted) {
              if (lane == 0 && atomicCAS(&s_found, 0, 1) == 0) {
                s_winner = wid;
                s_wroot = v;
              }
              break;
            }
            mine = claim();
          }
        }
        if (S.aborted && !__atomic_load_n(&s_found, __ATOMIC_RELAXED) && lane == 0)
          atomicOr(&s_abort, 1);
        S.cancel = nullptr;
        __syncthreads();
        const bool found = s_found != 0;
        if (!found) {
          all_ok = false;
          if (s_abort) uncertain = true;
          break;
        }
        // the winning wave rebuilds this component's tree with its memo
        if (wid == s_winner) {
          const int v = s_wroot;
          if (c == 0) s_parent[lane] = -1;
          Sync();
          if (lane == 0) s_parent[v] = -1;
          Sync();
          S.aborted = false;
          uint64_t rest = C & ~(1ull << v);
          while (rest && !S.aborted) {
            const uint64_t D = Component(S.myadj, rest, rest & (0ull - rest), nullptr, nullptr);
            rest &= ~D;
            Build(S, D, k - 1, v, s_parent, s_bst, s_bk, s_bpar);
          }
          if (S.aborted && lane == 0) atomicOr(&s_abort, 2);
        }
        __syncthreads();
        if (s_abort & 2) {  // no tree could be rebuilt: keep the previous best
          all_ok = false;
          uncertain = true;
          break;
        }
        // reset per-wave halt state for the next component / k
        S.aborted = false;
        if (threadIdx.x == 0) s_abort = 0;
        __syncthreads();
      }
      if (!all_ok) {
        if (!uncertain) lb = ub;
        break;
      }
      // components that fit in k are chained (path decomposition)
      if (wid == 0) {
        for (int c = 0; c < ncomp; ++c) {
          const uint64_t C = Uniform64(s_comps[c]);
          if (__builtin_popcountll(C) > k) continue;
          int prev = -1;
          for (uint64_t m = C; m; m &= m - 1) {
            const int u = __builtin_ctzll(m);
            if (lane == 0) s_parent[u] = static_cast<int8_t>(prev);
            prev = u;
          }
        }
        Sync();
        s_best[lane] = s_parent[lane];
      }
      ub = k;
      __syncthreads();
    }
    if (ub - 1 < lb) lb = ub;
    // totals over the waves
    if (lane == 0) {
      atomicAdd(&s_nodes, static_cast<unsigned long long>(S.nodes));
      atomicAdd(&s_hits, static_cast<unsigned long long>(S.hits));
      atomicAdd(&s_last_nodes, static_cast<unsigned long long>(S.nodes - nodes_k0));
    }
    __syncthreads();
    BnBOut* o = outs + gi;
    if (wid == 0) {
      if (lane < n) o->parent[lane] = s_best[lane];
      if (lane == 0) {
        o->td = ub;
        o->lb = lb;
        o->certified = (!uncertain && lb == ub) ? 1u : 0u;
        o->heur_td = static_cast<uint32_t>(s_heur);
        o->nodes = s_nodes;
        o->memo_hits = s_hits;
        o->last_nodes = s_last_nodes;
        o->last_k = last_k;
      }
    }
    __syncthreads();
  }
}

__global__ void BnBResetQueue(uint32_t* q) {
  if (threadIdx.x == 0) *q = 0u;
}

int64_t Param(td_ctx* ctx, const char* k, int64_t dflt) {
  auto it = ctx->params.find(k);
  return it == ctx->params.end() ? dflt : it->second;
}

void SolveBnBSearch(td_ctx* ctx, int ngraphs, const int32_t* ns, const uint64_t* adj_concat,
                    const int32_t* ub_seed, const float* scores, uint8_t* td_out,
                    int8_t* parent_concat, uint8_t* certified_out, td_bnb_stats* stats,
                    bool finish = true);

// Device buffers of td_dp_solve_batch for graphs of at most 26 vertices.
constexpr const char* kBatchBuffers[] = {"dp.batch_arena", "dp.batch_graphs", "dp.batch_queue",
                                         "dp.pascal", "dp.flow"};

// The graphs of at most kFinishMaxN vertices that the search has left
// uncertified, by the subset DP (whose single-solve tables and queries stay
// as they are), in calls of at most 2^30 subsets; where the device or the
// byte budget has no room for that, by the search without its early stop.
void FinishSmall(td_ctx* ctx, const int32_t* ns, const uint64_t* adj_concat,
                 const std::vector<size_t>& off, const int32_t* ub_seed, const float* scores,
                 std::vector<BnBOut>& out, double* ms) {
  std::vector<int> left;
  for (size_t i = 0; i < out.size(); ++i)
    if (ns[i] <= kFinishMaxN && !out[i].certified) left.push_back(static_cast<int>(i));
  if (left.empty()) return;
  std::map<std::string, size_t> held;
  for (const char* k : kBatchBuffers) held[k] = ctx->Held(k);
  for (size_t at = 0; at < left.size();) {
    std::vector<int32_t> n, seed;
    std::vector<uint64_t> adj;
    std::vector<float> score;
    uint64_t subsets = 0;
    size_t end = at;
    for (; end < left.size(); ++end) {
      const int i = left[end];
      if (end > at && subsets + (1ull << ns[i]) > (1ull << 30)) break;
      subsets += 1ull << ns[i];
      n.push_back(ns[i]);
      adj.insert(adj.end(), adj_concat + off[i], adj_concat + off[i + 1]);
      seed.push_back(ub_seed ? ub_seed[i] : 0);
      if (scores) score.insert(score.end(), scores + off[i], scores + off[i + 1]);
    }
    const int count = static_cast<int>(n.size());
    std::vector<uint8_t> td(count);
    std::vector<int8_t> par(adj.size());
    td_dp_stats st{};
    const int rc = KeepDP(ctx, [&] {
      return td_dp_solve_batch(ctx, count, n.data(), adj.data(), td.data(), par.data(), 0, &st);
    });
    if (rc == TD_OK) {
      *ms += st.level_ms + st.tree_ms;
      size_t r = 0;
      for (int j = 0; j < count; ++j) {
        BnBOut& o = out[left[at + j]];
        o.td = o.lb = td[j];
        o.certified = 1;
        std::memcpy(o.parent, par.data() + r, n[j]);
        r += n[j];
      }
    } else {
      TD_REQUIRE(rc == TD_E_NOMEM, rc, ctx->err);
      std::vector<uint8_t> cert(count);
      td_bnb_stats bst{};
      SolveBnBSearch(ctx, count, n.data(), adj.data(), ub_seed ? seed.data() : nullptr,
                     scores ? score.data() : nullptr, td.data(), par.data(), cert.data(), &bst,
                     false);
      *ms += bst.kernel_ms;
      size_t r = 0;
      for (int j = 0; j < count; ++j) {
        BnBOut& o = out[left[at + j]];
        const td_ctx::BnBDetail& d = ctx->bnb_last[j];
        o.td = td[j];
        o.lb = d.lb;
        o.certified = cert[j];
        o.nodes += d.nodes;
        o.last_k = d.last_k;
        o.last_nodes = d.last_nodes;
        std::memcpy(o.parent, par.data() + r, n[j]);
        r += n[j];
      }
    }
    at = end;
  }
  // a byte budget is the caller's to spend on other calls: what the DP has taken
  // goes back, and captured launches with it, which know its addresses
  if (!ctx->budget) return;
  bool released = false;
  for (const char* k : kBatchBuffers)
    if (ctx->Held(k) > held[k]) {
      ctx->Release(k);
      released = true;
    }
  if (released) ctx->DropDPGraphs();
}

void SolveBnBSearch(td_ctx* ctx, int ngraphs, const int32_t* ns, const uint64_t* adj_concat,
                    const int32_t* ub_seed, const float* scores, uint8_t* td_out,
                    int8_t* parent_concat, uint8_t* certified_out, td_bnb_stats* stats,
                    bool finish) {
  const auto t0 = std::chrono::steady_clock::now();
  TD_REQUIRE(ngraphs >= 1 && ns && adj_concat, TD_E_INVALID, "empty batch or null pointer");
  std::vector<size_t> off(ngraphs + 1, 0);
  for (int i = 0; i < ngraphs; ++i) {
    TD_REQUIRE(ns[i] >= 1 && ns[i] <= kMaxBnBN, TD_E_INVALID, "n must be in [1, 64]");
    off[i + 1] = off[i] + ns[i];
  }
  std::vector<BnBGraph> hg(ngraphs);
  for (int i = 0; i < ngraphs; ++i) {
    ValidateGraph(ns[i], adj_concat + off[i], kMaxBnBN);
    BnBGraph& G = hg[i];
    std::memset(&G, 0, sizeof(G));
    G.n = ns[i];
    G.ub_seed = ub_seed ? ub_seed[i] : 0;
    G.use_scores = scores ? 1u : 0u;
    for (int v = 0; v < ns[i]; ++v) {
      G.adj[v] = adj_concat[off[i] + v];
      G.score[v] = scores ? scores[off[i] + v] : 0.f;
    }
  }
  const uint64_t budget = static_cast<uint64_t>(Param(ctx, "bnb.node_budget", 2000000));
  if (budget != 0 && budget <= kFinishBudget) finish = false;
  const uint64_t small_budget = finish ? kFinishNodes : budget;
  // waves per graph; 0 (the default): as many as keep 24 waves on each CU
  // when every graph has its own workgroup slot (16 for at most one graph
  // per CU, 12 for two), else 8 (three 8-wave workgroups per CU)
  int W = static_cast<int>(Param(ctx, "bnb.waves_per_graph", 0));
  if (W == 0) {
    const int cus = ctx->prop.multiProcessorCount;
    W = ngraphs <= cus ? 16 : ngraphs <= 2 * cus ? 12 : 8;
  }
  TD_REQUIRE(W >= 1 && W <= kMaxWaves, TD_E_INVALID, "bnb.waves_per_graph in [1, 16]");
  const int dp_small = static_cast<int>(Param(ctx, "bnb.dp_small", 0));
  TD_REQUIRE(dp_small >= 0 && dp_small <= kSmallDPMax, TD_E_INVALID,
             "bnb.dp_small in [0, 12]");
  // memo buckets per wave: by default 2^ceil(log2(nodes per wave / 2)) in
  // [2^10, 2^17] (4 entries of 16 bytes each), with a wave's share of the
  // graph's budget taken as budget / W, so the table holds about two facts
  // per node the wave expands; "bnb.memo_log2" overrides it
  int memo_auto = 17;
  if (budget > 0) {
    const uint64_t per_wave = (budget + W - 1) / W;
    memo_auto = 10;
    while (memo_auto < 17 && (1ull << memo_auto) < per_wave / 2) ++memo_auto;
  }
  int memo_log2 = static_cast<int>(Param(ctx, "bnb.memo_log2", 0));
  if (memo_log2 == 0) memo_log2 = memo_auto;  // 0: sized to the budget
  TD_REQUIRE(memo_log2 >= 8 && memo_log2 <= 24, TD_E_INVALID, "bnb.memo_log2 in [8, 24]");
  int groups_cap = static_cast<int>(Param(ctx, "bnb.groups", 0));
  if (groups_cap <= 0) groups_cap = ctx->prop.multiProcessorCount * 4;  // 0: 4 per CU
  const int groups = std::max(1, std::min(ngraphs, groups_cap));
  const size_t waves = static_cast<size_t>(groups) * W;
  const size_t memo_bytes = (waves << (memo_log2 + 2)) * sizeof(MemoEntry);
  auto* dG = static_cast<BnBGraph*>(ctx->Buffer("bnb.graphs", sizeof(BnBGraph) * ngraphs));
  auto* dO = static_cast<BnBOut*>(ctx->Buffer("bnb.out", sizeof(BnBOut) * ngraphs));
  auto* dM = static_cast<MemoEntry*>(ctx->Buffer("bnb.memo", memo_bytes));
  auto* dQ = static_cast<uint32_t*>(ctx->Buffer("bnb.queue", 256));
  // Entries carry the tag of the graph that wrote them (a serial that grows
  // across calls), so a table is cleared only when it is (re)allocated.
  if (ctx->bnb_memo_ptr != dM || ctx->bnb_memo_bytes != memo_bytes ||
      ctx->bnb_tag > 0xF0000000u - static_cast<uint32_t>(ngraphs)) {
    TD_HIP(hipMemsetAsync(dM, 0, memo_bytes, ctx->stream));
    ctx->bnb_memo_ptr = dM;
    ctx->bnb_memo_bytes = memo_bytes;
    ctx->bnb_tag = 0;
  }
  const uint32_t tag_base = ctx->bnb_tag;
  ctx->bnb_tag += static_cast<uint32_t>(ngraphs);
  TD_HIP(hipMemcpyAsync(dG, hg.data(), sizeof(BnBGraph) * ngraphs, hipMemcpyHostToDevice,
                        ctx->stream));
  TD_HIP(hipMemcpyAsync(dQ + kTagWord, &tag_base, 4, hipMemcpyHostToDevice, ctx->stream));
  TD_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
  // queue reset (a kernel, so the pair can be captured) and the persistent
  // search, replayed from a hipGraph cached per launch shape and buffers
  auto launch = [&] {
    hipLaunchKernelGGL(BnBResetQueue, dim3(1), dim3(64), 0, ctx->stream, dQ);
    hipLaunchKernelGGL(BnBKernel, dim3(groups), dim3(64 * W), W * WaveLds(dp_small),
                       ctx->stream, dG, dO, dM, memo_log2, budget, small_budget, dp_small, ngraphs,
                       dQ);
  };
  if (Param(ctx, "bnb.use_graph", 1) == 0) {
    launch();
  } else {
    const std::vector<uint64_t> key = {
        static_cast<uint64_t>(groups), static_cast<uint64_t>(W), static_cast<uint64_t>(dp_small),
        static_cast<uint64_t>(memo_log2), budget, small_budget, static_cast<uint64_t>(ngraphs),
        reinterpret_cast<uint64_t>(dG), reinterpret_cast<uint64_t>(dO),
        reinterpret_cast<uint64_t>(dM), reinterpret_cast<uint64_t>(dQ)};
    if (ctx->bnb_graph && ctx->bnb_graph_key != key) {
      (void)hipGraphExecDestroy(ctx->bnb_graph);
      ctx->bnb_graph = nullptr;
    }
    if (!ctx->bnb_graph) {
      hipGraph_t graph;
      TD_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
      launch();
      TD_HIP(hipStreamEndCapture(ctx->stream, &graph));
      hipGraphExec_t exec;
      const hipError_t e = hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0);
      (void)hipGraphDestroy(graph);
      TD_HIP(e);
      ctx->bnb_graph = exec;
      ctx->bnb_graph_key = key;
    }
    TD_HIP(hipGraphLaunch(ctx->bnb_graph, ctx->stream));
  }
  TD_HIP(hipGetLastError());
  TD_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
  std::vector<BnBOut> ho(ngraphs);
  TD_HIP(hipMemcpyAsync(ho.data(), dO, sizeof(BnBOut) * ngraphs, hipMemcpyDeviceToHost,
                        ctx->stream));
  TD_HIP(hipStreamSynchronize(ctx->stream));
  float search_ms = 0.f;
  TD_HIP(hipEventElapsedTime(&search_ms, ctx->ev[0], ctx->ev[1]));
  double finish_ms = 0.0;
  if (finish) FinishSmall(ctx, ns, adj_concat, off, ub_seed, scores, ho, &finish_ms);
  ctx->bnb_last.assign(ngraphs, {0, 0, 0, -1, 0});
  uint64_t cert = 0, nodes = 0, hits = 0;
  for (int i = 0; i < ngraphs; ++i) {
    ctx->bnb_last[i] = {ho[i].heur_td, ho[i].lb, ho[i].nodes, ho[i].last_k, ho[i].last_nodes};
    if (td_out) td_out[i] = static_cast<uint8_t>(ho[i].td);
    if (certified_out) certified_out[i] = static_cast<uint8_t>(ho[i].certified);
    if (parent_concat) std::memcpy(parent_concat + off[i], ho[i].parent, ns[i]);
    cert += ho[i].certified;
    nodes += ho[i].nodes;
    hits += ho[i].memo_hits;
  }
  if (stats) {
    stats->graphs = static_cast<uint64_t>(ngraphs);
    stats->certified = cert;
    stats->nodes = nodes;
    stats->memo_hits = hits;
    stats->kernel_ms = search_ms + finish_ms;
    stats->total_ms = std::chrono::duration<double, std::milli>(
                          std::chrono::steady_clock::now() - t0)
                          .count();
  }
}

// Graphs of at most "bnb.dp_max_n" vertices (0, the default: none) are
// answered by the batched subset DP (td_dp_solve_batch): exact, certified,
// with the DP's canonical tree; the others go to the search.  The DP does
// 2^n work however dense the graph is, where the search's refutation can
// grow far faster on dense small graphs.
void SolveBnB(td_ctx* ctx, int ngraphs, const int32_t* ns, const uint64_t* adj_concat,
              const int32_t* ub_seed, const float* scores, uint8_t* td_out,
              int8_t* parent_concat, uint8_t* certified_out, td_bnb_stats* stats) {
  const int dp_max_n = static_cast<int>(Param(ctx, "bnb.dp_max_n", 0));
  TD_REQUIRE(dp_max_n >= 0 && dp_max_n <= 32, TD_E_INVALID, "bnb.dp_max_n in [0, 32]");
  TD_REQUIRE(ngraphs >= 1 && ns && adj_concat, TD_E_INVALID, "empty batch or null pointer");
  std::vector<int> dpi, rest;
  for (int i = 0; i < ngraphs; ++i) {
    TD_REQUIRE(ns[i] >= 1 && ns[i] <= kMaxBnBN, TD_E_INVALID, "n must be in [1, 64]");
    (ns[i] <= dp_max_n ? dpi : rest).push_back(i);
  }
  if (dpi.empty()) {
    SolveBnBSearch(ctx, ngraphs, ns, adj_concat, ub_seed, scores, td_out, parent_concat,
                   certified_out, stats);
    return;
  }
  const auto t0 = std::chrono::steady_clock::now();
  std::vector<size_t> off(ngraphs + 1, 0);
  for (int i = 0; i < ngraphs; ++i) off[i + 1] = off[i] + ns[i];
  // one side's graphs packed in input order; results scattered back
  struct Part {
    std::vector<int32_t> n, seed;
    std::vector<uint64_t> adj;
    std::vector<float> score;
    std::vector<uint8_t> td, cert;
    std::vector<int8_t> par;
  };
  auto pack = [&](const std::vector<int>& idx, Part& P) {
    for (int i : idx) {
      P.n.push_back(ns[i]);
      P.seed.push_back(ub_seed ? ub_seed[i] : 0);
      P.adj.insert(P.adj.end(), adj_concat + off[i], adj_concat + off[i + 1]);
      if (scores) P.score.insert(P.score.end(), scores + off[i], scores + off[i + 1]);
    }
    P.td.assign(idx.size(), 0);
    P.cert.assign(idx.size(), 0);
    P.par.assign(P.adj.size(), 0);
  };
  Part D, B;
  pack(dpi, D);
  pack(rest, B);
  td_dp_stats dst{};
  const int rc = td_dp_solve_batch(ctx, static_cast<int32_t>(dpi.size()), D.n.data(),
                                   D.adj.data(), D.td.data(), D.par.data(), 0, &dst);
  TD_REQUIRE(rc == TD_OK, rc, ctx->err);
  td_bnb_stats bst{};
  if (!rest.empty())
    SolveBnBSearch(ctx, static_cast<int>(rest.size()), B.n.data(), B.adj.data(),
                   ub_seed ? B.seed.data() : nullptr, scores ? B.score.data() : nullptr,
                   B.td.data(), B.par.data(), B.cert.data(), &bst);
  const std::vector<td_ctx::BnBDetail> bdet = ctx->bnb_last;  // the search's graphs
  ctx->bnb_last.assign(ngraphs, {0, 0, 0, -1, 0});
  auto scatter = [&](const std::vector<int>& idx, const Part& P, bool exact) {
    size_t r = 0;
    for (size_t j = 0; j < idx.size(); ++j) {
      const int i = idx[j];
      if (td_out) td_out[i] = P.td[j];
      if (certified_out) certified_out[i] = exact ? 1 : P.cert[j];
      if (parent_concat) std::memcpy(parent_concat + off[i], P.par.data() + r, ns[i]);
      r += ns[i];
      ctx->bnb_last[i] = exact ? td_ctx::BnBDetail{P.td[j], P.td[j], 0, -1, 0} : bdet[j];
    }
  };
  scatter(dpi, D, true);
  scatter(rest, B, false);
  if (stats) {
    stats->graphs = static_cast<uint64_t>(ngraphs);
    stats->certified = dpi.size() + bst.certified;
    stats->nodes = bst.nodes;
    stats->memo_hits = bst.memo_hits;
    stats->kernel_ms = bst.kernel_ms + dst.level_ms + dst.tree_ms;
    stats->total_ms = std::chrono::duration<double, std::milli>(
                          std::chrono::steady_clock::now() - t0)
                          .count();
  }
}

// ---------------------------------------------------------------------------
// Autotuner of the batched search launch: waves per graph, workgroups in
// flight and memo buckets per wave, timed on the batch itself.  The score is
// certified graphs per second of kernel time (the waves of a graph share its
// node budget, so the shape can change what is certified, never a certified
// answer).  Results are kept as JSON lines like the DP autotuner's.
// ---------------------------------------------------------------------------
struct BnBShape {
  int waves, groups, memo_log2;
};

std::string BnBJsonLine(const std::string& key, const BnBShape& c, double rate, double ms,
                        uint64_t cert, bool best, const char* arch) {
  char line[400];
  std::snprintf(line, sizeof(line),
                "{\"key\":\"%s\",\"best\":%s,\"waves_per_graph\":%d,\"groups\":%d,"
                "\"memo_log2\":%d,\"certified\":%llu,\"kernel_ms\":%.4f,"
                "\"certified_per_s\":%.2f,\"arch\":\"%s\"}\n",
                key.c_str(), best ? "true" : "false", c.waves, c.groups, c.memo_log2,
                static_cast<unsigned long long>(cert), ms, rate, arch);
  return line;
}

bool BnBJsonInt(const std::string& line, const char* name, long long* v) {
  const std::string k = std::string("\"") + name + "\":";
  const size_t p = line.find(k);
  return p != std::string::npos && std::sscanf(line.c_str() + p + k.size(), "%lld", v) == 1;
}

bool BnBJsonDouble(const std::string& line, const char* name, double* v) {
  const std::string k = std::string("\"") + name + "\":";
  const size_t p = line.find(k);
  return p != std::string::npos && std::sscanf(line.c_str() + p + k.size(), "%lf", v) == 1;
}

bool BnBCacheLookup(const char* path, const std::string& key, const char* arch,
                    BnBShape* out, double* rate) {
  if (!path) return false;
  std::ifstream f(path);
  if (!f) return false;
  const std::string want_key = "\"key\":\"" + key + "\"";
  const std::string want_arch = std::string("\"arch\":\"") + arch + "\"";
  bool found = false;
  std::string line;
  while (std::getline(f, line)) {
    if (line.find(want_key) == std::string::npos ||
        line.find("\"best\":true") == std::string::npos ||
        line.find(want_arch) == std::string::npos)
      continue;
    long long w = 0, g = 0, m = 0;
    double r = 0;
    if (BnBJsonInt(line, "waves_per_graph", &w) && BnBJsonInt(line, "groups", &g) &&
        BnBJsonInt(line, "memo_log2", &m) && BnBJsonDouble(line, "certified_per_s", &r) &&
        w >= 1 && w <= kMaxWaves && g >= 1 && m >= 8 && m <= 24) {
      *out = {static_cast<int>(w), static_cast<int>(g), static_cast<int>(m)};
      *rate = r;
      found = true;
    }
  }
  return found;
}

void AutotuneBnB(td_ctx* ctx, int ngraphs, const int32_t* ns, const uint64_t* adj_concat,
                 const float* scores, const char* cache_path, double* best_rate_out) {
  TD_REQUIRE(ngraphs >= 1 && ns && adj_concat, TD_E_INVALID, "empty batch or null pointer");
  int maxn = 0;
  long long sumn = 0;
  for (int i = 0; i < ngraphs; ++i) {
    TD_REQUIRE(ns[i] >= 1 && ns[i] <= kMaxBnBN, TD_E_INVALID, "n must be in [1, 64]");
    maxn = std::max(maxn, static_cast<int>(ns[i]));
    sumn += ns[i];
  }
  const uint64_t budget = static_cast<uint64_t>(Param(ctx, "bnb.node_budget", 2000000));
  const std::string key = "bnb g=" + std::to_string(ngraphs) + " maxn=" + std::to_string(maxn) +
                          " sumn=" + std::to_string(sumn) + " budget=" +
                          std::to_string(budget) + " scores=" + (scores ? "1" : "0");
  const char* arch = ctx->prop.gcnArchName;
  auto apply = [&](const BnBShape& c) {
    ctx->params["bnb.waves_per_graph"] = c.waves;
    ctx->params["bnb.groups"] = c.groups;
    ctx->params["bnb.memo_log2"] = c.memo_log2;
  };
  BnBShape best{};
  double best_rate = -1.0;
  if (BnBCacheLookup(cache_path, key, arch, &best, &best_rate)) {
    apply(best);
    if (best_rate_out) *best_rate_out = best_rate;
    return;
  }
  // the three tuned parameters as they are now, restored on an error
  std::map<std::string, int64_t> saved;
  for (const char* k : {"bnb.waves_per_graph", "bnb.groups", "bnb.memo_log2"}) {
    auto it = ctx->params.find(k);
    if (it != ctx->params.end()) saved[k] = it->second;
  }
  const int cus = ctx->prop.multiProcessorCount;
  std::vector<uint8_t> td(ngraphs), cert(ngraphs);
  std::string log;
  double best_ms = 0;
  // candidates: 4, 8, 12 or 16 waves per graph; 1, 2, 4 or 8 workgroups per CU
  // (at most one per graph); the default memo size for the per-wave budget,
  // halved, as is, or doubled; memo tables above 8 GiB in all are skipped
  std::vector<BnBShape> cands;
  for (int W : {4, 8, 12, 16})
    for (int mult : {1, 2, 4, 8}) {
      const int groups = std::min(cus * mult, ngraphs);
      if (mult > 1 && groups == std::min(cus * (mult / 2), ngraphs)) continue;
      int memo = 17;
      if (budget > 0) {
        const uint64_t per_wave = (budget + W - 1) / W;
        memo = 10;
        while (memo < 17 && (1ull << memo) < per_wave / 2) ++memo;
      }
      for (int dm : {-1, 0, 1}) {
        const int m = std::max(8, std::min(24, memo + dm));
        const uint64_t bytes = (static_cast<uint64_t>(groups) * W << (m + 2)) * 16ull;
        if (bytes <= (8ull << 30)) cands.push_back({W, groups, m});
      }
    }
  TD_REQUIRE(!cands.empty(), TD_E_NOMEM, "no launch shape fits the memo limit");
  try {
    for (const BnBShape& c : cands) {
      apply(c);
      td_bnb_stats st{};
      SolveBnBSearch(ctx, ngraphs, ns, adj_concat, nullptr, scores, td.data(), nullptr,
                     cert.data(), &st);  // warm-up (memo allocation, capture)
      double ms = 0;
      uint64_t certified = 0;
      for (int rep = 0; rep < 2; ++rep) {
        SolveBnBSearch(ctx, ngraphs, ns, adj_concat, nullptr, scores, td.data(), nullptr,
                       cert.data(), &st);
        ms += st.kernel_ms;
        certified += st.certified;
      }
      ms /= 2;
      const double rate = (certified / 2.0) / (ms * 1e-3);
      log += BnBJsonLine(key, c, rate, ms, certified / 2, false, arch);
      if (rate > best_rate) {
        best_rate = rate;
        best = c;
        best_ms = ms;
      }
    }
  } catch (...) {
    for (const char* k : {"bnb.waves_per_graph", "bnb.groups", "bnb.memo_log2"}) {
      auto it = saved.find(k);
      if (it == saved.end()) ctx->params.erase(k);
      else ctx->params[k] = it->second;
    }
    throw;
  }
  apply(best);
  // the sweep's largest memo table is not needed any more
  ctx->Release("bnb.memo");
  ctx->bnb_memo_ptr = nullptr;
  if (cache_path) {
    std::ofstream f(cache_path, std::ios::app);
    f << log << BnBJsonLine(key, best, best_rate, best_ms, 0, true, arch);
    TD_REQUIRE(f.good(), TD_E_INVALID, "cannot write the autotune cache file");
  }
  if (best_rate_out) *best_rate_out = best_rate;
}

}  // namespace
}  // namespace tdhip

using namespace tdhip;  // NOLINT

extern "C" {

int td_bnb_solve_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                       const uint64_t* adj_concat, const int32_t* ub_seed,
                       const float* vertex_scores, uint8_t* td_out,
                       int8_t* parent_concat, uint8_t* certified_out,
                       td_bnb_stats* stats) {
  return Guard(ctx, [&] {
    SolveBnB(ctx, ngraphs, n, adj_concat, ub_seed, vertex_scores, td_out, parent_concat,
             certified_out, stats);
  });
}

int td_bnb_last_details(td_ctx* ctx, int32_t count, int32_t* heur_td_out,
                        int32_t* lower_bound_out, uint64_t* nodes_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(count >= 0 && static_cast<size_t>(count) <= ctx->bnb_last.size(), TD_E_STATE,
               "count exceeds the graphs of the last branch-and-bound call");
    for (int i = 0; i < count; ++i) {
      if (heur_td_out) heur_td_out[i] = static_cast<int32_t>(ctx->bnb_last[i].heur);
      if (lower_bound_out) lower_bound_out[i] = ctx->bnb_last[i].lb;
      if (nodes_out) nodes_out[i] = ctx->bnb_last[i].nodes;
    }
  });
}

int td_bnb_last_search(td_ctx* ctx, int32_t count, int32_t* last_k_out,
                       uint64_t* last_k_nodes_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(count >= 0 && static_cast<size_t>(count) <= ctx->bnb_last.size(), TD_E_STATE,
               "count exceeds the graphs of the last branch-and-bound call");
    for (int i = 0; i < count; ++i) {
      if (last_k_out) last_k_out[i] = ctx->bnb_last[i].last_k;
      if (last_k_nodes_out) last_k_nodes_out[i] = ctx->bnb_last[i].last_nodes;
    }
  });
}

int td_bnb_autotune_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                          const uint64_t* adj_concat, const float* vertex_scores,
                          const char* cache_path, double* best_rate_out) {
  return Guard(ctx, [&] {
    AutotuneBnB(ctx, ngraphs, n, adj_concat, vertex_scores, cache_path, best_rate_out);
  });
}

int td_bnb_solve(td_ctx* ctx, int32_t n, const uint64_t* adj, int32_t heur_td,
                 int32_t* treedepth_out, int8_t* parent_out, uint8_t* certified_out) {
  return Guard(ctx, [&] {
    uint8_t td = 0, cert = 0;
    const int32_t seed = heur_td;
    SolveBnB(ctx, 1, &n, adj, &seed, nullptr, &td, parent_out, &cert, nullptr);
    if (treedepth_out) *treedepth_out = td;
    if (certified_out) *certified_out = cert;
  });
}

}  // extern "C"
