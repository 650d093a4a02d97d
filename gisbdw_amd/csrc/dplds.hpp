// dplds.hpp -- the subset DP of one graph of at most 24 vertices in one launch,
// with the words (dpword.hpp) in LDS: DPLdsKernel (n <= 18) in one workgroup,
// with the decomposition; DPFlowKernel (n = 19..24) in 2^T workgroups that
// pass finished words on to each other.
//
// Such a graph has at most 2^13 words of 12 bytes, 96 of a CU's 160 KiB, so
// a level step is a barrier and a few LDS reads (0.5 us for a level that fits
// the workgroup) where a level kernel of its own costs 5 us and more.  Words
// are indexed by H itself (bit x = vertex 5 + x), so neighbours need no ranks;
// only the order of work comes from the table of the 16-bit k-subsets.  The
// tree's lookups are LDS reads, too.
#pragma once
#include "dpword.hpp"

namespace tdhip {
namespace {

constexpr int kLdsMaxN = 18;

// A graph in the kernel's arguments: no copy has to go ahead of the launch.
struct LdsGraph {
  uint32_t n;
  uint32_t adj[kLdsMaxN];
};

// LDS in front of the words: adjacency rows, level sizes C(nh, k), first
// entries of the k-subsets in the order table, N(H) and isolation tables by
// 7-bit chunks (2 chunks cover 13 vertices).
constexpr int kLdsAdj = 0, kLdsSize = 32, kLdsOff = 48, kLdsNbh = 64, kLdsIsoH = 64 + 192,
              kLdsIsoL = 64 + 384, kLdsHead = 64 + 416;
constexpr size_t LdsBytes(int n) {
  return 4 * static_cast<size_t>(kLdsHead) + (12ull << (n > 5 ? n - 5 : 0));
}
// Threads for one graph: a wave up to n = 13 (at 13 one level, of 70 words,
// takes two passes); else about the largest level, at most 1024.
constexpr int LdsThreads(int n) {
  return n <= 13 ? 64 : n == 14 ? 128 : n == 15 ? 256 : n == 16 ? 512 : 1024;
}

// Everything this wave has written, and what other waves had written before a
// barrier, is in memory: clock[3] = 1, which the host waits for.
__device__ __forceinline__ void PublishDone(unsigned long long* clock) {
  __threadfence_system();
  if ((threadIdx.x & 63) == 0)
    __hip_atomic_store(clock + 3, 1ull, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// the L of a word that meet the low set T
__device__ __forceinline__ uint32_t Meets(uint32_t T) {
  return ((T & 1u) ? 0xAAAAAAAAu : 0u) | ((T & 2u) ? 0xCCCCCCCCu : 0u) |
         ((T & 4u) ? 0xF0F0F0F0u : 0u) | ((T & 8u) ? 0xFF00FF00u : 0u) |
         ((T & 16u) ? 0xFFFF0000u : 0u);
}

// N(H) by chunks, the L that give every vertex of a chunk a neighbour, and the
// L in which every y of Y n L has one (see DPGraph), for the entries that nh
// high vertices use.
__device__ __forceinline__ void BuildLdsTables(uint32_t* s, int nh) {
  const int c0 = 1 << (nh < 7 ? nh : 7), c1 = 1 << (nh > 7 ? nh - 7 : 0);
  for (int i = threadIdx.x; i < c0 + c1 + 32; i += blockDim.x) {
    if (i < c0 + c1) {
      const bool second = i >= c0;
      const uint32_t* row = s + kLdsAdj + (second ? 12 : 5);
      uint32_t nb = 0u, iso = ~0u;
      for (uint32_t ch = second ? i - c0 : i; ch; ch &= ch - 1) {
        const uint32_t r = row[__builtin_ctz(ch)];
        nb |= r;
        iso &= Meets(r & 31u);
      }
      const int at = second ? 128 + i - c0 : i;
      s[kLdsNbh + at] = nb;
      s[kLdsIsoH + at] = iso;
    } else {
      const uint32_t Y = static_cast<uint32_t>(i - c0 - c1);
      uint32_t m = ~0u;
      for (uint32_t yy = Y; yy; yy &= yy - 1) {
        const int y = __builtin_ctz(yy);
        m &= ~Meets(1u << y) | Meets(s[kLdsAdj + y] & 31u);
      }
      s[kLdsIsoL + Y] = m;
    }
  }
}

// Word H (|H| = h) from the words of H \ x.
template <bool kTiny>
__device__ __forceinline__ DPWord LdsWord(const uint32_t* s, const uint32_t* w, int N, uint32_t H,
                                          int h) {
  DPFold f;
  auto at = [&](uint32_t G) { return DPWord{w[G], w[N + G], w[2 * N + G]}; };
  uint32_t rem = H;
  int i = 0;
  for (; i + 2 <= h; i += 2) {
    const uint32_t a = rem & (0u - rem);
    rem ^= a;
    const uint32_t b = rem & (0u - rem);
    rem ^= b;
    f.Add2(at(H ^ a), at(H ^ b));
  }
  if (i < h) {
    const DPWord v = at(H ^ rem);
    f.Add(v.g0, v.g1, v.c);
  }
  const uint32_t NH = s[kLdsNbh + (H & 127u)] | s[kLdsNbh + 128 + (H >> 7)];
  const uint32_t I = H & ~(NH >> 5);
  const uint32_t fine = s[kLdsIsoL + (~NH & 31u)] & s[kLdsIsoH + (I & 127u)] &
                        s[kLdsIsoH + 128 + (I >> 7)];
  const uint32_t single = !kTiny ? 0u : h == 0 ? 0x00010116u : 1u;
  return SolveWord(f, fine, single, kTiny && h == 0, AnyLane());
}

// One graph per workgroup.  gs: the batch's graphs (host memory, read once),
// or null for the graph in `one`.  table (nullable): takes the graph's three planes
// (2^nh words each, word H at H: DPGraph::direct), for later queries.
// Results: 64 parents and the depth per graph; clock (nullable): the device's
// clock at the start, after the levels and at the end, then PublishDone once
// every wave has written its part of everything.
__global__ __launch_bounds__(1024) void DPLdsKernel(
    const LdsGraph* __restrict__ gs, const LdsGraph one, const uint32_t* __restrict__ g_cb,
    uint32_t* __restrict__ table, int8_t* __restrict__ parent_out, int32_t* __restrict__ td_out,
    unsigned long long* __restrict__ clock) {
  extern __shared__ uint32_t s[];
  const unsigned long long t0 = clock ? wall_clock64() : 0ull;
  const int tid = threadIdx.x;
  const LdsGraph* g = gs ? gs + blockIdx.x : nullptr;
  const int n = static_cast<int>(g ? g->n : one.n);
  const int nh = n > 5 ? n - 5 : 0;
  const int N = 1 << nh;
  uint32_t* w = s + kLdsHead;
  const uint16_t* order = reinterpret_cast<const uint16_t*>(g_cb + kTailWord);
  if (tid < 32)
    s[kLdsAdj + tid] = tid >= n ? 0u : g ? g->adj[tid] : one.adj[tid];
  else if (tid < 48)
    s[kLdsSize + tid - 32] = g_cb[nh * kCbStride + tid - 32];
  else if (tid < 64)
    s[kLdsOff + tid - 48] = g_cb[kCbOffs + tid - 48];
  __syncthreads();
  BuildLdsTables(s, nh);
  __syncthreads();
  // The order entry of a lane's first word of a level is read before the
  // barrier that starts the level.
  uint32_t next = 0u;
  for (int h = 0; h <= nh; ++h) {
    const int count = static_cast<int>(s[kLdsSize + h]);
    const uint16_t* sets = order + s[kLdsOff + h];
    for (int t = tid; t < count; t += blockDim.x) {
      const uint32_t H = t == tid ? next : sets[t];
      const DPWord r = h <= 1 ? LdsWord<true>(s, w, N, H, h) : LdsWord<false>(s, w, N, H, h);
      w[H] = r.g0;
      w[N + H] = r.g1;
      w[2 * N + H] = r.c;
    }
    if (h < nh && tid < static_cast<int>(s[kLdsSize + h + 1]))
      next = order[s[kLdsOff + h + 1] + tid];
    __syncthreads();
  }
  if (table) {
    for (int i = tid; i < 3 * N; i += blockDim.x) table[i] = w[i];
    // a wave's part is written before the barrier that "done" waits for, not
    // on its way (wave 0's own part: PublishDone)
    if (tid >= 64) __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
  }
  if (tid < 64) {
    const unsigned long long t1 = clock ? wall_clock64() : 0ull;
    int depth = 0;
    const int parent =
        DecomposeWave(s[kLdsAdj + (tid & 31)], n >= 32 ? ~0u : (1u << n) - 1u, &depth,
                      [&](uint32_t A, uint32_t B) {
                        const uint32_t *a = w + (A >> 5), *b = w + (B >> 5);
                        const uint32_t x = a[0], y = a[N], u = b[0], v = b[N];
                        return (((x >> (A & 31u)) ^ (u >> (B & 31u))) |
                                ((y >> (A & 31u)) ^ (v >> (B & 31u)))) & 1u;
                      });
    if (tid < n)
      parent_out[64 * static_cast<size_t>(blockIdx.x) + tid] = static_cast<int8_t>(parent);
    if (tid == 0) {
      td_out[blockIdx.x] = depth;
      if (clock) {
        clock[0] = t0;
        clock[1] = t1;
        clock[2] = wall_clock64();
      }
    }
  }
  if (!clock) return;
  // "done" stands for the tables too, whichever wave wrote them (they are
  // written while wave 0 decomposes: 47 us a call at n = 18 with and without)
  __syncthreads();
  if (tid < 64) PublishDone(clock);
}

// ---------------------------------------------------------------------------
// Graphs of 19..24 vertices, each in 2^T workgroups.  The 11 vertices above
// the word's five are a workgroup's own; workgroup P of a graph stands for the
// subset P of the T = n - 16 vertices above those, keeps the 2^11 words of P
// in LDS and resolves them level by level like DPLdsKernel.  A word also needs
// the same word of every workgroup P \ x: those are published, one by one, in
// a buffer that both sides index by the order of work, so reads and writes
// coalesce.
//
// A published word is two 64-bit atomics, 16 bits of the call's tag in each:
// (tag, c's low half, g0) and (tag, c's high half, g1).  Data and tag arrive
// together, so there is no fence, no flag and no barrier between workgroups:
// a reader that finds another tag reads again.  Workgroup P only waits for
// smaller P of its graph, and P comes from a ticket taken when the workgroup
// starts, so what a workgroup waits for is already running; a lane that has
// still not seen its word after `spin` reads gives up and marks the result,
// and the host solves the call again without this kernel.  With more than one
// workgroup per CU a reader was seen to keep getting an old copy of a line
// from its L2 (tag and all, so it only waits); the acquire fence after every
// 128 reads drops such copies, and the host launches at most one workgroup
// per CU.
//
// P runs one hand-over (4 to 5 us) behind its predecessors, not behind their
// whole tables: the chain is 12 level steps and T hand-overs, where level
// kernels take n - 4 launches of 5 us and more.  A lane reads the
// predecessors' words of its next level before it computes the present one.
// Levels of one graph with this kernel / with level kernels, us: n = 19
// 36 / 62, n = 20 40 / 70, n = 22 49 / 84, n = 24 65 / 103; n = 25 114 / 114
// (512 workgroups, which no longer run all at once).  10 and 12 own vertices:
// n = 20 40 and 42, n = 24 - and 71.
constexpr int kFlowMinN = 19, kFlowMaxN = 24, kFlowDims = 11;
constexpr int kFlowClasses = kFlowMaxN - kFlowMinN + 1;
constexpr int FlowTop(int n) { return n - 5 - kFlowDims; }
// A workgroup's entries start 2^11 + 32 apart: at 2^11, 16 KiB, the entries
// that many workgroups poll at once (every P's first, for one) fall on the
// same memory channels.
constexpr uint32_t kFlowStride = (1u << kFlowDims) + 32u;
// published words and planes of one graph, bytes
constexpr size_t FlowBytes(int n) { return (16ull * kFlowStride) << FlowTop(n); }
constexpr size_t DirectBytes(int n) { return 12ull << (n > 5 ? n - 5 : 0); }

struct FlowGraph {
  uint32_t adj[kFlowMaxN];
};
// The graphs of one n in a call: their first ticket, first graph, and offsets
// of the first one's published words (8 bytes each) and planes (4 bytes each).
struct FlowClass {
  uint32_t n, ticket, graph;
  uint64_t ex, table;
};
struct FlowCall {
  uint32_t classes, ticket0, tag, spin;
  FlowClass c[kFlowClasses];
  FlowGraph one;  // the graph, where there is one only
};
// class of a ticket / of a graph
__device__ __forceinline__ int FlowClassOf(const FlowCall& f, uint32_t i, bool graph) {
  int k = 0;
  while (k + 1 < static_cast<int>(f.classes) && i >= (graph ? f.c[k + 1].graph : f.c[k + 1].ticket))
    ++k;
  return k;
}

__device__ __forceinline__ unsigned long long FlowLoad(const unsigned long long* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void FlowStore(unsigned long long* p, unsigned long long v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// gs: the call's graphs (host memory, read once), or null for f.one.  ex: for
// each graph kFlowStride 2^T entries of (tag, c, g0), then as many of
// (tag, c, g1); entry kFlowStride P + position in P's order of work.  ticket: counts the
// workgroups of all calls, from f.ticket0 on in this one.  table: the planes
// (DPGraph::direct).  status: set to 1 if a wait was given up.  kT: at least T
// of every graph in the call.
template <int kT>
__global__ __launch_bounds__(512) void DPFlowKernel(
    const FlowCall f, const FlowGraph* __restrict__ gs, const uint32_t* __restrict__ g_cb,
    unsigned long long* __restrict__ ex, uint32_t* __restrict__ ticket,
    uint32_t* __restrict__ table, int32_t* __restrict__ status,
    unsigned long long* __restrict__ clock) {
  constexpr int D = kFlowDims, W = 1 << D, kThreads = 512;
  __shared__ uint32_t w[3 * W];
  __shared__ uint32_t s_tab[3 * 256 + 32];  // per chunk N and isolation, then isol
  __shared__ uint32_t s_adj[32], s_size[D + 1], s_off[D + 1], s_ticket;
  const int tid = threadIdx.x;
  const uint16_t* order = reinterpret_cast<const uint16_t*>(g_cb + kTailWord);
  if (tid == 0) {
    s_ticket = atomicAdd(ticket, 1u) - f.ticket0;
    if (clock && s_ticket == 0u) clock[0] = wall_clock64();
  }
  __syncthreads();
  const FlowClass& cl = f.c[FlowClassOf(f, s_ticket, false)];
  const int n = static_cast<int>(cl.n);
  const uint32_t T = static_cast<uint32_t>(n - 5 - D);
  const uint32_t index = (s_ticket - cl.ticket) >> T;
  const uint32_t P = (s_ticket - cl.ticket) & ((1u << T) - 1u);
  if (tid < 32) {
    const FlowGraph* g = gs ? gs + cl.graph + index : nullptr;
    s_adj[tid] = tid >= n ? 0u : g ? g->adj[tid] : f.one.adj[tid];
  }
  if (tid >= 64 && tid < 64 + D + 1) {
    s_size[tid - 64] = g_cb[D * kCbStride + tid - 64];
    s_off[tid - 64] = g_cb[kCbOffs + tid - 64];
  }
  __syncthreads();
  for (int i = tid; i < 3 * 128 + 32; i += kThreads) {
    if (i < 3 * 128) {
      uint32_t nb = 0u, iso = ~0u;
      for (uint32_t ch = i & 127; ch; ch &= ch - 1) {
        const uint32_t r = s_adj[5 + 7 * (i >> 7) + __builtin_ctz(ch)];
        nb |= r;
        iso &= Meets(r & 31u);
      }
      s_tab[(i >> 7) * 256 + (i & 127)] = nb;
      s_tab[(i >> 7) * 256 + 128 + (i & 127)] = iso;
    } else {
      const uint32_t Y = static_cast<uint32_t>(i - 3 * 128);
      uint32_t m = ~0u;
      for (uint32_t yy = Y; yy; yy &= yy - 1) {
        const int y = __builtin_ctz(yy);
        m &= ~Meets(1u << y) | Meets(s_adj[y] & 31u);
      }
      s_tab[3 * 256 + Y] = m;
    }
  }
  const int np = __builtin_popcount(P);
  const size_t plane = static_cast<size_t>(1) << (n - 5);
  const size_t half = static_cast<size_t>(kFlowStride) << T;
  unsigned long long* exa = ex + cl.ex + 2 * half * index;
  unsigned long long* exb = exa + half;
  const unsigned long long want = static_cast<unsigned long long>(f.tag) << 48;
  // the words of P \ x at position pos, as read (perhaps not there yet)
  // (no branches here, so that all loads are in flight together: an x outside
  // P reads one entry of P's own, which nobody looks at)
  unsigned long long ra[kT], rb[kT];
  auto fetch = [&](uint32_t pos) {
#pragma unroll
    for (int x = 0; x < kT; ++x) {
      const uint32_t at = P >> x & 1u ? (P ^ (1u << x)) * kFlowStride + pos : P * kFlowStride;
      ra[x] = FlowLoad(exa + at);
      rb[x] = FlowLoad(exb + at);
    }
  };
  bool dead = false;
  uint32_t base = 0u, next = 0u;  // first position of the level
  if (tid == 0) fetch(0u);
  __syncthreads();
  for (int h = 0; h <= D; ++h) {
    const uint32_t count = s_size[h];
    const bool mine = static_cast<uint32_t>(tid) < count;
    if (mine) {
      const uint32_t H = next, pos = base + tid;
      // all words that are not there yet are read again together
      for (uint32_t tries = 0; !dead; ++tries) {
        uint32_t late = 0u;
#pragma unroll
        for (int x = 0; x < kT; ++x)
          late |= static_cast<uint32_t>(((ra[x] ^ want) | (rb[x] ^ want)) >> 48) ? 1u << x : 0u;
        if (!(late & P)) break;
        if (tries > f.spin) dead = true;
        if (tries > 3) __builtin_amdgcn_s_sleep(1);
        if ((tries & 127u) == 127u) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        fetch(pos);
      }
      DPFold fold;
#pragma unroll
      for (int x = 0; x < kT; ++x)
        if (P >> x & 1u)
          fold.Add(static_cast<uint32_t>(ra[x]), static_cast<uint32_t>(rb[x]),
                (static_cast<uint32_t>(ra[x] >> 32) & 0xFFFFu) |
                    static_cast<uint32_t>(rb[x] >> 32) << 16);
      // the next level's words of the predecessors, while this one is computed
      const uint32_t then = h < D ? s_size[h + 1] : 0u;
      if (static_cast<uint32_t>(tid) < then) fetch(base + count + tid);
      auto at = [&](uint32_t G) { return DPWord{w[G], w[W + G], w[2 * W + G]}; };
      uint32_t rem = H;
      int i = 0;
      for (; i + 2 <= h; i += 2) {
        const uint32_t a = rem & (0u - rem);
        rem ^= a;
        const uint32_t b = rem & (0u - rem);
        rem ^= b;
        fold.Add2(at(H ^ a), at(H ^ b));
      }
      if (i < h) {
        const DPWord v = at(H ^ rem);
        fold.Add(v.g0, v.g1, v.c);
      }
      const uint32_t A = H | P << D;
      const uint32_t NH = s_tab[A & 127u] | s_tab[256 + (A >> 7 & 127u)] | s_tab[512 + (A >> 14)];
      const uint32_t I = A & ~(NH >> 5);
      const uint32_t fine = s_tab[3 * 256 + (~NH & 31u)] & s_tab[128 + (I & 127u)] &
                            s_tab[256 + 128 + (I >> 7 & 127u)] & s_tab[512 + 128 + (I >> 14)];
      const int size = np + h;
      DPWord r;
      if (size <= 1)
        r = SolveWord(fold, fine, size == 0 ? 0x00010116u : 1u, size == 0, AnyLane());
      else
        r = SolveWord(fold, fine, 0u, false, AnyLane());
      w[H] = r.g0;
      w[W + H] = r.g1;
      w[2 * W + H] = r.c;
      const uint32_t to = P * kFlowStride + pos;
      FlowStore(exa + to, want | static_cast<unsigned long long>(r.c & 0xFFFFu) << 32 | r.g0);
      FlowStore(exb + to, want | static_cast<unsigned long long>(r.c >> 16) << 32 | r.g1);
    } else if (h < D && static_cast<uint32_t>(tid) < s_size[h + 1]) {
      fetch(base + count + tid);
    }
    if (h < D && static_cast<uint32_t>(tid) < s_size[h + 1]) next = order[s_off[h + 1] + tid];
    base += count;
    __syncthreads();
  }
  if (dead) *status = 1;
  uint32_t* to = table + cl.table + 3 * plane * index + (static_cast<size_t>(P) << D);
  for (int i = tid; i < W; i += kThreads) {
    to[i] = w[i];
    to[plane + i] = w[W + i];
    to[2 * plane + i] = w[2 * W + i];
  }
  if (clock && tid == 0 && P == (1u << T) - 1u) clock[1] = wall_clock64();
}

// The decompositions of a call's graphs from their planes, a wave each.
__global__ __launch_bounds__(64) void DPDirectTreeKernel(
    const FlowCall f, const FlowGraph* __restrict__ gs, const uint32_t* __restrict__ table,
    int8_t* __restrict__ parent_out, int32_t* __restrict__ td_out,
    unsigned long long* __restrict__ clock) {
  const int lane = threadIdx.x;
  const FlowClass& cl = f.c[FlowClassOf(f, blockIdx.x, true)];
  const int n = static_cast<int>(cl.n);
  const size_t plane = static_cast<size_t>(1) << (n - 5);
  const uint32_t* mine = table + cl.table + 3 * plane * (blockIdx.x - cl.graph);
  const uint32_t row = lane >= n ? 0u : gs ? gs[blockIdx.x].adj[lane] : f.one.adj[lane];
  int depth = 0;
  const int parent = DecomposeWave(row, (1u << n) - 1u, &depth, [&](uint32_t A, uint32_t B) {
    const uint32_t *a = mine + (A >> 5), *b = mine + (B >> 5);
    const uint32_t x = a[0], y = a[plane], u = b[0], v = b[plane];
    return (((x >> (A & 31u)) ^ (u >> (B & 31u))) | ((y >> (A & 31u)) ^ (v >> (B & 31u)))) & 1u;
  });
  if (lane < n) parent_out[64 * static_cast<size_t>(blockIdx.x) + lane] = static_cast<int8_t>(parent);
  if (lane == 0) {
    td_out[blockIdx.x] = depth;
    if (clock) clock[2] = wall_clock64();
  }
  if (clock) PublishDone(clock);
}

}  // namespace
}  // namespace tdhip
