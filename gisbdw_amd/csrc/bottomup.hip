// bottomup.hip -- the bottom-up union-find heuristic on gfx950.
//
// Reference: BottomUpHeuristicGPU (Treedepth/src/branch_and_bound/heuristics/
// bottom_up_heuristic.hpp:11-35) over BottomUpHeuristicGPUAlgorithm
// (bottom_up_heuristic_gpu_algorithm.{hpp,cu}).  Level k holds, for every
// k-subset S of the vertices, the elimination forest of G[S] that the
// heuristic keeps: the empty set has height 1; S tries its vertices v in
// ascending order as the one added last (v becomes the parent of the roots of
// the components of its neighbours in S, DynamicStepKernel :57-95 with the
// union-find of Treedepth/src/union_find/ext_array_union_find.hpp) and keeps
// the first forest of strictly smallest height, starting from |S| + 1.
//
// Only the component heights matter for later levels (Union reads the heights
// of the two roots; Find only the root), and the components of the kept forest
// are those of G[S].  So a subset's record here holds 32 slots, one per
// vertex: slot w is the height of w's component for w in S, and the height of
// the whole forest for w outside S.  Adding v to S \ v then needs one record:
// slot v gives the height of S \ v, v's neighbours' slots the heights that v
// joins (the new component's height is 1 + their largest, 1 if none), and the
// forest height is the larger of the two.  Records are bit-sliced: plane j is
// a 32-bit mask holding bit j of every slot, so all neighbours' slots are
// compared at once and their largest is a descent over the planes.  A
// level's heights are at most k and at most 1 + the largest height of the
// level below, so a level whose heights must stay below 8 stores 3 planes
// (12-byte records), below 16 4 planes (16 bytes), any other level 8 (32
// bytes), instead of the reference's n + 2 union-find bytes; each launch finds
// the width from the largest heights the launches before it recorded.  The history keeps, per subset, the vertex
// added last and the height (history_ in the reference), 2 bytes per subset
// over all levels; the records live for two levels only.
#include <algorithm>
#include <cstring>
#include <type_traits>
#include <vector>

#include "ctx.hpp"

namespace tdhip {
namespace {

constexpr int kBuStride = 33;  // s_cb[x * 33 + j] = C(x, j)
constexpr int kRecBytes = 32;  // largest per-subset record (byte slots)
constexpr int kBuBlock = 256, kBuBlockMax = 1024;  // level kernel's workgroups
// The binomial buffer continues with O_k = sum_{j<k} C(16, j) (k = 0..16)
// and, from word kBuTailWord, the colex k-subsets of {0..15} as 16-bit masks
// (entry O_k + r is the subset of rank r).
constexpr int kBuTailBits = 16;
constexpr int kBuOffs = 32 * kBuStride;
constexpr int kBuCbWords = kBuOffs + kBuTailBits + 1;
constexpr int kBuTailWord = (kBuCbWords + 31) / 32 * 32;
constexpr int kBuPascalWords = kBuTailWord + (1 << kBuTailBits) / 2;

// Colex unrank of r among the k-subsets of {0..n-1} (set_encoder.hpp:61-73):
// greedy from the top down to vertex 16, then one table read for the rest
// (the remainder is then below C(16, k)); needs r < C(n, k).
__device__ __forceinline__ uint32_t BuUnrank(uint32_t r, int k, int n, const uint32_t* s_cb,
                                             const uint16_t* __restrict__ tail) {
  uint32_t S = 0;
  for (int x = n - 1; x >= kBuTailBits; --x) {
    const uint32_t c = s_cb[x * kBuStride + k];
    const uint32_t take = r >= c ? 1u : 0u;
    r = take ? r - c : r;
    S = 2u * S + take;
    k -= static_cast<int>(take);
  }
  return (S << kBuTailBits) | tail[s_cb[kBuOffs + k] + r];
}

// Ranks in the level kernel count units of a record's byte offset: three to a
// 12-byte record, so that the address is one shift and add (a multiply by 12
// in 64 bits takes four times its issue slots); 3 C(32, 16) fits 32 bits.
__host__ __device__ constexpr uint32_t BuUnit(int planes) { return planes == 3 ? 3u : 1u; }

// LDS tables of the level kernel, indexed by z = leading zeros of a vertex
// bit: C(31 - z, j) units at z * 33 + j and the row of vertex 31 - z; and the
// neighbours of every set of vertices 8 c .. 8 c + 7 at 256 c + set.
struct BuTables {
  uint32_t rev[32 * kBuStride];
  uint32_t row[32];
  uint32_t nbh[4 * 256];
};

// Connected component of vertex bit b in G[S]: breadth-first, a round for all
// of the front by four table reads (vertex by vertex it was a quarter of the
// level kernel's instructions).
__device__ __forceinline__ uint32_t BuComponent(const BuTables& t, uint32_t S, uint32_t b) {
  uint32_t comp = b, grown = b;
  do {
    const uint32_t f = grown;
    const uint32_t nb = t.nbh[f & 255u] | t.nbh[256 + (f >> 8 & 255u)] |
                        t.nbh[512 + (f >> 16 & 255u)] | t.nbh[768 + (f >> 24)];
    grown = nb & S & ~comp;
    comp |= grown;
  } while (grown);
  return comp;
}

// A record in registers, bit-sliced: plane j (p0..p7) holds bit j of every
// slot, slot w at bit w of each plane.  A level uses the first 3, 4 or 8 of
// them (see BuPlanes).  Named fields, not an array, so that plane selects stay
// in registers.
struct BuRec {
  uint32_t p0, p1, p2, p3, p4, p5, p6, p7;
};

template <int P>
__device__ __forceinline__ BuRec BuLoad(const uint8_t* ptr) {
  BuRec q;
  if (P == 3) {
    const uint3 x = *reinterpret_cast<const uint3*>(ptr);
    q.p0 = x.x;
    q.p1 = x.y;
    q.p2 = x.z;
    q.p3 = 0;
  } else {
    const uint4 x = reinterpret_cast<const uint4*>(ptr)[0];
    q.p0 = x.x;
    q.p1 = x.y;
    q.p2 = x.z;
    q.p3 = x.w;
  }
  q.p4 = q.p5 = q.p6 = q.p7 = 0;
  if (P == 8) {
    const uint4 y = reinterpret_cast<const uint4*>(ptr)[1];
    q.p4 = y.x;
    q.p5 = y.y;
    q.p6 = y.z;
    q.p7 = y.w;
  }
  return q;
}

__device__ __forceinline__ uint32_t BuPlane(const BuRec& q, int j) {  // j compile-time
  return j == 0 ? q.p0 : j == 1 ? q.p1 : j == 2 ? q.p2 : j == 3 ? q.p3
       : j == 4 ? q.p4 : j == 5 ? q.p5 : j == 6 ? q.p6 : q.p7;
}

// Largest slot among the vertices of M (0 for an empty M), from the top
// plane down: keep the candidates that have the bit whenever any does.
template <int P>
__device__ __forceinline__ uint32_t BuMaxSlot(const BuRec& q, uint32_t M) {
  uint32_t top = 0;
#pragma unroll
  for (int j = P - 1; j >= 0; --j) {
    const uint32_t t = M & BuPlane(q, j);
    top = 2u * top + (t != 0u ? 1u : 0u);
    M = t ? t : M;
  }
  return top;
}

// Planes of level k's records: its heights are at most 1 + the largest height
// of level k - 1, and at most k.  A 12-byte record costs an eighth fewer
// instructions a removal than one of 16 (30 and 34) and reads a quarter less.
__device__ __forceinline__ int BuPlanes(int k, const uint32_t* maxh) {
  const uint32_t most = k == 0 ? 0u : min(static_cast<uint32_t>(k), maxh[k - 1] + 1u);
  return most < 8u ? 3 : most < 16u ? 4 : 8;
}

// Every k-subset of rank r < count at one level; returns the largest height
// this lane wrote.  As workgroups go to the 8 XCDs in turn, each XCD takes a
// contiguous eighth of the ranks, so that neighbouring subsets' common
// predecessors are fetched into one L2.
template <int PIn, int POut>
__device__ __forceinline__ uint32_t BuLevel(const uint32_t* s_cb, const BuTables& tab,
                                            const uint16_t* __restrict__ tail, int n, int k,
                                            uint32_t count, const uint8_t* __restrict__ prev_rec,
                                            uint8_t* __restrict__ cur_rec,
                                            int8_t* __restrict__ cur_last,
                                            uint8_t* __restrict__ cur_height) {
  constexpr int kIn = 4 * PIn, kOut = 4 * POut;
  constexpr uint32_t kUnit = BuUnit(PIn);
  uint32_t lane_max = 0;
  constexpr uint32_t kXcds = 8;
  const uint32_t slices = gridDim.x % kXcds == 0 ? kXcds : 1u;
  const uint32_t slice = blockIdx.x % slices;
  const uint32_t end = static_cast<uint32_t>(static_cast<uint64_t>(count) * (slice + 1) / slices);
  for (uint32_t r = static_cast<uint32_t>(static_cast<uint64_t>(count) * slice / slices) +
                    blockIdx.x / slices * blockDim.x + threadIdx.x;
       r < end; r += gridDim.x / slices * blockDim.x) {
    const uint32_t S = BuUnrank(r, k, n, s_cb, tail);
    // Elements y_0 < ... < y_{k-1} of S from the top: rank(S \ y_i) =
    // r - C(y_i, i+1) - sum_{j>i} (C(y_j, j+1) - C(y_j, j)) (set_encoder.hpp:
    // 48-59); B is r less that sum, all in units of kUnit.  The candidate to
    // keep is the smallest vertex of least height (the ascending strict "<"
    // of the reference): the least key, height above vertex.  The records of
    // kGroup removals are loaded together; every lane has k elements, so the
    // groups are the same across the wave.
    constexpr int kGroup = PIn == 8 ? 2 : 4;
    uint32_t B = r * kUnit, rem = S, key = ~0u, brank = 0;
    auto next = [&](int i, uint32_t* z) {  // rank without element i; B moves on
      *z = static_cast<uint32_t>(__builtin_clz(rem));
      rem ^= 0x80000000u >> *z;
      const uint32_t* c = tab.rev + *z * kBuStride + i;
      const uint32_t rank = B - c[1];
      B = rank + c[0];
      return rank;
    };
    auto load = [&](uint32_t rank) {
      return BuLoad<PIn>(prev_rec + (static_cast<size_t>(rank) * (kIn / kUnit)));
    };
    // A component of S \ v is no higher than the forest, so v under the
    // highest neighbour component gives the forest's height, or one more if
    // a neighbour's slot holds that height.  Slot v, outside S \ v, does
    // hold it, and all neighbour slots are compared with it at once.
    auto weigh = [&](const BuRec& q, uint32_t z, uint32_t rank) {
      const uint32_t v = 31u - z;
      uint32_t top = tab.row[z] & S, mine = v;
#pragma unroll
      for (int j = 0; j < PIn; ++j) {
        const uint32_t f = static_cast<uint32_t>(
            __builtin_amdgcn_sbfe(static_cast<int>(BuPlane(q, j)), v, 1));
        top &= ~(BuPlane(q, j) ^ f);
        mine |= f & 32u << j;
      }
      mine += top != 0u ? 32u : 0u;
      brank = mine < key ? rank : brank;
      key = min(key, mine);
    };
    int i = k;
    auto group = [&](auto size) {
      constexpr int G = decltype(size)::value;
      uint32_t z[G], rank[G];
      BuRec q[G];
#pragma unroll
      for (int u = 0; u < G; ++u) rank[u] = next(--i, &z[u]);
#pragma unroll
      for (int u = 0; u < G; ++u) q[u] = load(rank[u]);
#pragma unroll
      for (int u = 0; u < G; ++u) weigh(q[u], z[u], rank[u]);
    };
    while (i >= kGroup) group(std::integral_constant<int, kGroup>());
    if (i == 3)
      group(std::integral_constant<int, 3>());
    else if (i == 2)
      group(std::integral_constant<int, 2>());
    else if (i == 1)
      group(std::integral_constant<int, 1>());
    // (the empty set's forest has height 0, its union-find state in the
    // reference 1: one vertex alone has height 1 either way)
    const uint32_t best = max(key >> 5, 1u), bv = key & 31u;
    // the planes a narrower record lacks are zero, and those a wider one has
    // beyond this level's are too
    const BuRec q = load(brank);
    // the joined component's height: 1 + the largest neighbour slot
    const uint32_t bnew = BuMaxSlot<PIn>(q, tab.row[31u - bv] & S) + 1u;
    const uint32_t comp = BuComponent(tab, S, 1u << bv);
    // kept slots: S outside v's component; v's component: bnew; outside S:
    // the forest height
    const uint32_t keep = S & ~comp, out_of_s = ~S;
    uint32_t w[8];
#pragma unroll
    for (int j = 0; j < POut; ++j)
      w[j] = (BuPlane(q, j) & keep) | ((bnew >> j) & 1 ? comp : 0u) |
             ((best >> j) & 1 ? out_of_s : 0u);
    uint8_t* dst = cur_rec + static_cast<size_t>(r) * kOut;
    if (POut == 3)
      *reinterpret_cast<uint3*>(dst) = make_uint3(w[0], w[1], w[2]);
    else
      *reinterpret_cast<uint4*>(dst) = make_uint4(w[0], w[1], w[2], w[3]);
    if (POut == 8)
      reinterpret_cast<uint4*>(dst)[1] = make_uint4(w[4], w[5], w[6], w[7]);
    cur_last[r] = static_cast<int8_t>(bv);
    cur_height[r] = static_cast<uint8_t>(best);
    lane_max = max(lane_max, best);
  }
  return lane_max;
}

// One level k (1 <= k <= n).  Bound by vector issue: 30 instructions a removal
// (9 find the vertex and its predecessor's rank, 17 weigh it) and 240 a subset
// beside them, 87% of the issue slots taken over G(25, 0.15), whose levels
// take 795 us and read 2.2 GB.  With a descent for every removal, 64-bit rank
// multiplies and the component found vertex by vertex it was 74 a removal and
// 1310 us.  maxh[j] is the largest height of level j
// (maxh[0] = 0, maxh[k] cleared before the launch); it picks the width of
// level k - 1's records and of this level's, and gets level k's maximum.
__global__ __launch_bounds__(kBuBlockMax) void BottomUpLevelKernel(
    const uint32_t* __restrict__ g_adj, const uint32_t* __restrict__ g_cb, int n, int k,
    uint32_t count, const uint8_t* __restrict__ prev_rec, uint8_t* __restrict__ cur_rec,
    int8_t* __restrict__ cur_last, uint8_t* __restrict__ cur_height,
    uint32_t* __restrict__ maxh) {
  __shared__ uint32_t s_cb[kBuCbWords];
  __shared__ BuTables tab;
  __shared__ uint32_t s_max;
  const int in = BuPlanes(k - 1, maxh), out = BuPlanes(k, maxh);
  for (int i = threadIdx.x; i < kBuCbWords; i += blockDim.x) {
    const uint32_t c = g_cb[i];
    s_cb[i] = c;
    if (i < 32 * kBuStride)
      tab.rev[(31 - i / kBuStride) * kBuStride + i % kBuStride] = c * BuUnit(in);
  }
  if (threadIdx.x < 32)
    tab.row[31 - threadIdx.x] = threadIdx.x < static_cast<unsigned>(n) ? g_adj[threadIdx.x] : 0u;
  if (threadIdx.x == 0) s_max = 0;
  __syncthreads();
  const uint32_t set = threadIdx.x & 255u;
  for (uint32_t c = threadIdx.x >> 8; c < 4; c += blockDim.x >> 8) {
    uint32_t nb = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b) nb |= set >> b & 1 ? tab.row[31 - 8 * c - b] : 0u;
    tab.nbh[256 * c + set] = nb;
  }
  __syncthreads();
  const uint16_t* tail = reinterpret_cast<const uint16_t*>(g_cb + kBuTailWord);
  uint32_t lane_max = 0;
  auto level = [&](auto pin, auto pout) {
    if (in == decltype(pin)::value && out == decltype(pout)::value)
      lane_max = BuLevel<decltype(pin)::value, decltype(pout)::value>(
          s_cb, tab, tail, n, k, count, prev_rec, cur_rec, cur_last, cur_height);
  };
  using P3 = std::integral_constant<int, 3>;
  using P4 = std::integral_constant<int, 4>;
  using P8 = std::integral_constant<int, 8>;
  level(P3(), P3());
  level(P3(), P4());
  level(P4(), P3());
  level(P4(), P4());
  level(P4(), P8());
  level(P8(), P4());
  level(P8(), P8());
  // (one level's widest height is at most one more or any less than the
  // next's: 3 planes are next to 8 only downwards)
  level(P8(), P3());
  atomicMax(&s_max, lane_max);
  __syncthreads();
  if (threadIdx.x == 0) atomicMax(&maxh[k], s_max);
}

// GetElimination (bottom_up_heuristic_gpu_algorithm.hpp:92-108): from set S,
// the vertex stored as added last, removed, `steps` times.  One wave: lane v
// holds vertex v's term of S's rank, one table read gives the next vertex
// (n = 25: 15.3 us; with one lane adding up the rank, 24.5).
__global__ __launch_bounds__(64) void BottomUpWalkKernel(
    const uint32_t* __restrict__ g_cb, const int8_t* __restrict__ last,
    const uint64_t* __restrict__ level_off, uint32_t S, int steps,
    int32_t* __restrict__ out) {
  __shared__ uint32_t s_cb[32 * kBuStride];
  __shared__ uint64_t s_off[33];
  for (int i = threadIdx.x; i < 32 * kBuStride; i += blockDim.x) s_cb[i] = g_cb[i];
  if (static_cast<int>(threadIdx.x) <= __builtin_popcount(S))
    s_off[threadIdx.x] = level_off[threadIdx.x];
  __syncthreads();
  const uint32_t v = threadIdx.x & 31u;
  for (int i = 0; i < steps; ++i) {
    const uint32_t mine = S >> v & 1u;
    uint32_t r = mine ? s_cb[v * kBuStride + __builtin_popcount(S & (2u << v) - 1u)] : 0u;
#pragma unroll
    for (int d = 16; d > 0; d >>= 1) r += __shfl_xor(r, d, 32);
    const int w = __builtin_amdgcn_readfirstlane(last[s_off[__builtin_popcount(S)] + r]);
    if (threadIdx.x == 0) out[i] = w;
    S &= ~(1u << (w & 31));
  }
}

const uint32_t* BuPascal(td_ctx* ctx) {
  auto it = ctx->bufs.find("bu.pascal");
  if (it != ctx->bufs.end() && it->second.p) return static_cast<const uint32_t*>(it->second.p);
  std::vector<uint32_t> cb(kBuPascalWords, 0);
  for (int x = 0; x < 32; ++x)
    for (int j = 0; j < kBuStride; ++j) cb[x * kBuStride + j] = static_cast<uint32_t>(Binom(x, j));
  uint16_t* tail = reinterpret_cast<uint16_t*>(cb.data() + kBuTailWord);
  uint32_t off = 0;
  for (int k = 0; k <= kBuTailBits; ++k) {
    cb[kBuOffs + k] = off;
    // the k-subsets of {0..15} in colex order = increasing integers
    for (uint32_t mask = 0; mask < (1u << kBuTailBits); ++mask)
      if (__builtin_popcount(mask) == k) tail[off++] = static_cast<uint16_t>(mask);
  }
  void* d = ctx->Buffer("bu.pascal", cb.size() * 4);
  ctx->Copy(d, cb.data(), cb.size() * 4, hipMemcpyHostToDevice);
  return static_cast<const uint32_t*>(d);
}

// Device bytes for levels 0..K-1: two record buffers sized for the largest
// level below K, the history (2 bytes per subset), offsets, adjacency, the
// binomials and the walk's output.
uint64_t BuBytes(int n, int K) {
  uint64_t maxc = 1, hist = 0;
  for (int k = 0; k < K; ++k) {
    maxc = std::max<uint64_t>(maxc, Binom(n, k));
    hist += Binom(n, k);
  }
  return 2 * maxc * kRecBytes + 2 * ((hist + 255) / 256 * 256) + 8 * 40 + 4 * 32 +
         4 * kBuPascalWords + 4 * 32 + 4 * 40;
}

uint64_t BuHeld(td_ctx* ctx) {
  uint64_t b = 0;
  for (const char* k : {"bu.rec0", "bu.rec1", "bu.last", "bu.height", "bu.off", "bu.adj",
                        "bu.pascal", "bu.walk", "bu.maxh"})
    b += ctx->Held(k);
  return b;
}

// Walks `steps` removals from S on the device; returns the vertices.
std::vector<int32_t> BuWalk(td_ctx* ctx, uint32_t S, int steps) {
  int32_t* dout = static_cast<int32_t*>(ctx->Buffer("bu.walk", 4 * 32));
  hipLaunchKernelGGL(BottomUpWalkKernel, dim3(1), dim3(64), 0, ctx->stream, BuPascal(ctx),
                     static_cast<const int8_t*>(ctx->bufs["bu.last"].p),
                     static_cast<const uint64_t*>(ctx->bufs["bu.off"].p), S, steps, dout);
  TD_HIP(hipGetLastError());
  std::vector<int32_t> order(std::max(steps, 1));
  TD_HIP(hipMemcpyAsync(order.data(), dout, 4 * steps, hipMemcpyDeviceToHost, ctx->stream));
  TD_HIP(hipStreamSynchronize(ctx->stream));
  order.resize(steps);
  return order;
}

}  // namespace
}  // namespace tdhip

using namespace tdhip;  // NOLINT

extern "C" {

int td_bottom_up(td_ctx* ctx, int32_t n, const uint64_t* adj, int32_t iterations,
                 int32_t* treedepth_out, int8_t* parent_out, int32_t* iterations_out) {
  return Guard(ctx, [&] {
    ValidateGraph(n, adj, 32);
    TD_REQUIRE(treedepth_out != nullptr, TD_E_INVALID, "treedepth_out is null");
    TD_REQUIRE(iterations == -1 || (iterations >= 1 && iterations <= n + 1), TD_E_INVALID,
               "iterations must be -1 or in [1, n + 1]");
    ctx->have_bu = false;
    // GetMaxIterations (bottom_up_heuristic_gpu_algorithm.cu:152-175): as
    // many levels as the memory holds, here the context budget or the
    // device's free memory
    const uint64_t held = BuHeld(ctx);
    uint64_t avail;
    if (ctx->budget) {
      // the subset DP's published words make room (td_ctx::Buffer)
      const uint64_t room = held + ctx->Held("dp.flow");
      avail = ctx->budget - std::min(ctx->budget, ctx->allocated - room);
    } else {
      size_t free_b = 0, total_b = 0;
      TD_HIP(hipMemGetInfo(&free_b, &total_b));
      avail = static_cast<uint64_t>((free_b + held) * 0.9);
    }
    int K = iterations;
    if (K < 0) {
      K = 1;
      while (K < n + 1 && BuBytes(n, K + 1) <= avail) ++K;
    }
    TD_REQUIRE(BuBytes(n, K) <= avail, TD_E_NOMEM,
               "bottom-up tables for " + std::to_string(K) + " levels exceed the memory");
    uint64_t maxc = 1, hist = 0;
    std::vector<uint64_t> off(n + 2, 0);
    for (int k = 0; k <= n; ++k) {
      off[k] = hist;
      if (k < K) {
        maxc = std::max<uint64_t>(maxc, Binom(n, k));
        hist += Binom(n, k);
      }
    }
    off[n + 1] = hist;
    uint8_t* rec[2] = {static_cast<uint8_t*>(ctx->Buffer("bu.rec0", maxc * kRecBytes)),
                       static_cast<uint8_t*>(ctx->Buffer("bu.rec1", maxc * kRecBytes))};
    int8_t* last = static_cast<int8_t*>(ctx->Buffer("bu.last", (hist + 255) / 256 * 256));
    uint8_t* height = static_cast<uint8_t*>(ctx->Buffer("bu.height", (hist + 255) / 256 * 256));
    uint64_t* doff = static_cast<uint64_t*>(ctx->Buffer("bu.off", 8 * 40));
    uint32_t* dadj = static_cast<uint32_t*>(ctx->Buffer("bu.adj", 4 * 32));
    uint32_t* dmaxh = static_cast<uint32_t*>(ctx->Buffer("bu.maxh", 4 * 40));
    const uint32_t* cb = BuPascal(ctx);
    uint32_t hadj[32] = {};
    for (int v = 0; v < n; ++v) hadj[v] = static_cast<uint32_t>(adj[v]);
    TD_HIP(hipMemcpyAsync(dadj, hadj, sizeof(hadj), hipMemcpyHostToDevice, ctx->stream));
    TD_HIP(hipMemcpyAsync(doff, off.data(), 8 * off.size(), hipMemcpyHostToDevice, ctx->stream));
    // level 0: the empty set, history (-1, 0) (:232-234), record all zero
    // (every slot is outside the set and holds its height, 0)
    TD_HIP(hipMemsetAsync(rec[0], 0, kRecBytes, ctx->stream));
    TD_HIP(hipMemsetAsync(last, 0xFF, 1, ctx->stream));
    TD_HIP(hipMemsetAsync(height, 0, 1, ctx->stream));
    TD_HIP(hipMemsetAsync(dmaxh, 0, 4 * 40, ctx->stream));  // largest height per level
    for (int k = 1; k < K; ++k) {
      const uint32_t count = static_cast<uint32_t>(Binom(n, k));
      // 32 waves per CU in equal passes, a multiple of 8 workgroups for the
      // slices of BuLevel.  Once every CU has a workgroup of 256, they are of
      // 1024: a quarter of the tables built and of the workgroups started
      // (n = 25, k = 7: 31 us at 256, 16 at 1024; all levels 817 and 795).
      const uint64_t cus = ctx->prop.multiProcessorCount;
      const uint64_t block = count > cus * kBuBlock ? kBuBlockMax : kBuBlock;
      const uint64_t groups = (count + block - 1) / block, once = cus * 2048 / block;
      const uint64_t passes = (groups + once - 1) / once;
      int grid = static_cast<int>((groups + passes - 1) / passes);
      if (grid >= 64) grid = (grid + 7) / 8 * 8;
      hipLaunchKernelGGL(BottomUpLevelKernel, dim3(grid), dim3(block), 0, ctx->stream, dadj,
                         cb, n, k, count, rec[(k - 1) & 1], rec[k & 1], last + off[k],
                         height + off[k], dmaxh);
      TD_HIP(hipGetLastError());
    }
    ctx->bu_n = n;
    ctx->bu_iters = K;
    ctx->bu_off = off;
    if (iterations_out) *iterations_out = K;
    if (K < n + 1) {  // BottomUpHeuristicGPU::Get returns UINT_MAX treedepth
      TD_HIP(hipStreamSynchronize(ctx->stream));
      ctx->have_bu = true;
      *treedepth_out = -1;
      return;
    }
    // GetElimination(n, n, 0), then the elimination forest of that order
    // (EliminationTree::Eliminate ... Decompose, bottom_up_heuristic.hpp:23-28);
    // the walk follows the levels on the same stream and synchronizes
    const uint32_t full = n == 32 ? 0xFFFFFFFFu : ((1u << n) - 1u);
    const std::vector<int32_t> order = BuWalk(ctx, full, n);
    ctx->have_bu = true;
    std::vector<int> parent(n, -1);
    std::vector<char> added(n, 0);
    for (int i = n - 1; i >= 0; --i) {
      const int v = order[i];
      TD_REQUIRE(v >= 0 && v < n && !added[v], TD_E_HIP, "bottom-up history is inconsistent");
      for (uint64_t m = adj[v]; m; m &= m - 1) {
        const int w = __builtin_ctzll(m);
        if (!added[w]) continue;
        int r = w;
        while (parent[r] >= 0) r = parent[r];
        if (r != v) parent[r] = v;
      }
      added[v] = 1;
    }
    int td = 0;
    for (int v = 0; v < n; ++v) {
      int d = 1;
      for (int u = v; parent[u] >= 0; u = parent[u]) ++d;
      td = std::max(td, d);
      if (parent_out) parent_out[v] = static_cast<int8_t>(parent[v]);
    }
    *treedepth_out = td;
  });
}

int td_bottom_up_get_treedepth(td_ctx* ctx, int32_t k, uint64_t code, uint32_t* td_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_bu, TD_E_STATE, "no td_bottom_up result to query");
    TD_REQUIRE(td_out != nullptr, TD_E_INVALID, "td_out is null");
    TD_REQUIRE(k >= 0 && k <= ctx->bu_n && code < Binom(ctx->bu_n, k), TD_E_INVALID,
               "subset code out of range");
    if (k >= ctx->bu_iters) {  // GetTreedepth (:181-188): 0 beyond the levels run
      *td_out = 0;
      return;
    }
    uint8_t h = 0;
    ctx->Copy(&h, static_cast<const uint8_t*>(ctx->bufs["bu.height"].p) + ctx->bu_off[k] + code, 1,
              hipMemcpyDeviceToHost);
    *td_out = h;
  });
}

int td_bottom_up_get_level(td_ctx* ctx, int32_t k, int8_t* last_out, uint8_t* height_out,
                           uint64_t out_len) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_bu, TD_E_STATE, "no td_bottom_up result to query");
    TD_REQUIRE(k >= 0 && k < ctx->bu_iters, TD_E_STATE, "level not run");
    const uint64_t cnt = Binom(ctx->bu_n, k);
    TD_REQUIRE(out_len >= cnt, TD_E_INVALID, "output shorter than the level");
    if (last_out)
      ctx->Copy(last_out, static_cast<const int8_t*>(ctx->bufs["bu.last"].p) + ctx->bu_off[k], cnt,
                hipMemcpyDeviceToHost);
    if (height_out)
      ctx->Copy(height_out, static_cast<const uint8_t*>(ctx->bufs["bu.height"].p) + ctx->bu_off[k],
                cnt, hipMemcpyDeviceToHost);
  });
}

int td_bottom_up_get_elimination(td_ctx* ctx, int32_t k, uint64_t code, int32_t* order_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_bu, TD_E_STATE, "no td_bottom_up result to query");
    TD_REQUIRE(order_out != nullptr || k == 0, TD_E_INVALID, "order_out is null");
    TD_REQUIRE(k >= 0 && k <= ctx->bu_n && code < Binom(ctx->bu_n, k), TD_E_INVALID,
               "subset code out of range");
    TD_REQUIRE(k < ctx->bu_iters, TD_E_STATE, "subset size beyond the levels run");
    if (k == 0) return;
    const std::vector<int32_t> order =
        BuWalk(ctx, static_cast<uint32_t>(UnrankColex(ctx->bu_n, k, code)), k);
    std::memcpy(order_out, order.data(), 4 * k);
  });
}

}  // extern "C"
