// dp.hip -- subset dynamic program for exact treedepth on gfx950.
//
// Reference path: DynamicGPU (Treedepth/src/dynamic_gpu/dynamic_gpu.cu:40-201,
// dynamic_gpu.hpp:38-64).  Recurrence (docs introduction/main.tex:10-15):
//   td(S) = 1 + min_{v in S} td(S \ v)   if S is connected,
//   td(S) = max over the components of S otherwise.
// For a disconnected S the second line equals max_{v in S} td(S \ v), so every
// subset of size k needs only subsets of size k-1.  Connectivity is carried in
// the table too: S (|S| >= 2) is connected iff no vertex of S is isolated in S
// and some S \ v is connected.
//
// Layout.  A subset takes three bits, in words of 32 subsets (dpword.hpp):
// the Gray code of td mod 4 and "connected".  Vertices 0..4 are a word's,
// vertices 5..lb-1 pick one of the 2^(lb-5) words of a tile (1, 2 or 4), and
// vertices lb..n-1 are "high": their subset H picks the tile.  The tiles of
// high level h = |H| are ranked by the colex rank of H among the h-subsets of
// the nh = n - lb high vertices (rank(H) = sum_i C(x_i, i+1),
// set_encoder.hpp:40-46), and the levels are concatenated, once for each of
// the three bit planes.  The tile of H is computed from the h tiles of H \ x
// (x in H, all at high level h-1) and, inside the tile, from smaller words.
// One lane owns a tile; a lane walks consecutive ranks with Gosper's
// successor (colex order = numeric order).
#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <fstream>
#include <mutex>
#include <string>
#include <thread>
#include <type_traits>
#include <vector>

#include "ctx.hpp"
#include "dpword.hpp"

namespace tdhip {
namespace {

constexpr int kCbStride = 33;  // s_cb[x * 33 + j] = C(x, j), x < 32, j <= 32
// The Pascal buffer (global) holds: C(x, j) at word x * 33 + j; the offsets
// O_k = sum_{j<k} C(16, j) (k = 0..16) at word kCbOffs + k; from word
// kTailWord the 16-bit colex unrank table of the k-subsets of {0..15} (entry
// O_k + r is the subset of rank r); from word kRevWord, C(31 - z, j) at
// z * 33 + j.
constexpr int kTailBits = 16;
constexpr int kCbOffs = 32 * kCbStride;
constexpr int kTailWord = (kCbOffs + kTailBits + 1 + 31) / 32 * 32;
constexpr int kRevWord = kTailWord + (1 << kTailBits) / 2;
constexpr int kPascalWords = kRevWord + 32 * kCbStride;
// The level kernels keep in LDS (s_lvl) C(31 - z, j) << SH at z * 33 + j
// (a tile is 2^SH bytes in each plane), indexed by z = leading zeros of a
// vertex bit, so that neighbour ranks come out as byte offsets, then O_k at
// kLvlOffs + k.  Every entry read is at most a level's bytes in one plane,
// below 2^32; entries never read may wrap.
constexpr int kLvlOffs = 32 * kCbStride;
constexpr int kLvlWords = kLvlOffs + kTailBits + 1;

// words per tile and log2 of its bytes in one plane
template <int WB>
constexpr int kTileWords = 1 << WB;
template <int WB>
constexpr int kTileShift = WB + 2;

// Colex unrank of r among the k-subsets of {0..nh-1}; greedy from the top
// (set_encoder.hpp:61-73) with the binomials read from LDS.  Needs
// r < C(nh, k): the remainder then reaches 0 exactly when k does, and
// C(x, 0) = 1 > 0 takes nothing more, so no k > 0 test is needed.  H is
// built MSB first (H = 2H + take), which keeps the loop to a compare, a
// select and two carry-style updates per x.
__device__ __forceinline__ uint32_t Unrank(uint32_t r, int k, int nh,
                                           const uint32_t* s_cb) {
  uint32_t H = 0;
  for (int x = nh - 1; x >= 0; --x) {
    const uint32_t c = s_cb[x * kCbStride + k];
    const uint32_t take = r >= c ? 1u : 0u;
    r = take ? r - c : r;
    H = 2u * H + take;
    k -= static_cast<int>(take);
  }
  return H;
}

// Unrank for the level kernels, on the shifted table: the greedy scan down
// to vertex 16 with r and the binomials scaled by 2^SH, then one read of the
// 16-bit table for the rest (the remainder is then below C(16, k)).  Same
// result as Unrank; r < C(nh, k), nh <= 32.
template <int SH>
__device__ __forceinline__ uint32_t UnrankTiles(uint32_t r, int k, int nh,
                                                const uint32_t* s_lvl,
                                                const uint16_t* __restrict__ tail) {
  uint32_t rs = r << SH;
  uint32_t H = 0;
  for (int z = 32 - nh; z < 32 - kTailBits; ++z) {  // vertex 31 - z
    const uint32_t c = s_lvl[z * kCbStride + k];
    const uint32_t take = rs >= c ? 1u : 0u;
    rs = take ? rs - c : rs;
    H = 2u * H + take;
    k -= static_cast<int>(take);
  }
  return (H << kTailBits) | tail[s_lvl[kLvlOffs + k] + (rs >> SH)];
}

// C(nh, h) from the shifted table
template <int SH>
__device__ __forceinline__ uint32_t LevelTiles(const uint32_t* s_lvl, int nh, int h) {
  return s_lvl[(31 - nh) * kCbStride + h] >> SH;
}

// Next k-subset in colex order (Gosper's hack, shift instead of divide).
__device__ __forceinline__ uint32_t NextCombination(uint32_t x) {
  const uint32_t c = x & (0u - x);
  const uint32_t r = x + c;
  return r | (((x ^ r) >> 2) >> __builtin_ctz(x));
}

// One plane of a tile (2^WB words).
template <int WB>
__device__ __forceinline__ void LoadPlane(const uint8_t* p, uint32_t (&w)[1 << WB]) {
  if constexpr (WB == 0) {
    w[0] = *reinterpret_cast<const uint32_t*>(p);
  } else if constexpr (WB == 1) {
    const uint2 v = *reinterpret_cast<const uint2*>(p);
    w[0] = v.x;
    w[1] = v.y;
  } else {
    const uint4 v = *reinterpret_cast<const uint4*>(p);
    w[0] = v.x;
    w[1] = v.y;
    w[2] = v.z;
    w[3] = v.w;
  }
}

template <int WB>
__device__ __forceinline__ void StorePlane(uint8_t* p, const uint32_t (&w)[1 << WB]) {
  if constexpr (WB == 0)
    *reinterpret_cast<uint32_t*>(p) = w[0];
  else if constexpr (WB == 1)
    *reinterpret_cast<uint2*>(p) = make_uint2(w[0], w[1]);
  else
    *reinterpret_cast<uint4*>(p) = make_uint4(w[0], w[1], w[2], w[3]);
}

template <int WB>
struct TileWords {
  uint32_t g0[1 << WB], g1[1 << WB], c[1 << WB];
  __device__ __forceinline__ DPWord At(int w) const { return {g0[w], g1[w], c[w]}; }
};

struct AnyLane {
  __device__ __forceinline__ bool operator()(uint32_t x) const {
    return __builtin_amdgcn_ballot_w64(x != 0u) != 0ull;
  }
};

// Resolve one tile: all subsets of the lb = 5 + WB low vertices joined with
// the high part H (|H| = h, t = its colex rank).  prev / cur = first tile of
// high level h-1 / h in plane 0; plane i is i * ps bytes further.
// kTiny: h <= 1, the only levels with the empty set and single vertices.
template <int WB, bool kTiny>
__device__ __forceinline__ void DPTile(const uint8_t* __restrict__ prev,
                                       uint8_t* __restrict__ cur, size_t ps, uint32_t t,
                                       uint32_t H, int h, const uint32_t* s_lvl,
                                       const uint32_t* s_tab) {
  constexpr int W = kTileWords<WB>, SH = kTileShift<WB>;
  DPFold f[W];
  // neighbour tiles H \ y_j, j = h-1 .. 0 (y_j = j-th smallest of H):
  // rank(H \ y_j) = t - C(y_j, j+1) - sum_{i>j} (C(y_i, i+1) - C(y_i, i)).
  // h is uniform across the wave, so every guard below is uniform.
  // Up to four tiles' loads are issued before they are folded, in pairs.
  // B = (t - sum_{i>j} (C(y_i, i+1) - C(y_i, i))) << SH runs down with j.  Byte
  // offsets within a level fit 32 bits, so the loads use a uniform base plus
  // a 32-bit lane offset.
  uint32_t rem = H;
  uint32_t B = t << SH;
  auto load = [&](int i, TileWords<WB>& v) {
    const int j = h - 1 - i;
    const int z = __builtin_clz(rem);  // y_j = 31 - z
    rem ^= 0x80000000u >> z;
    const uint32_t c1 = s_lvl[z * kCbStride + j + 1];
    const uint32_t c0 = s_lvl[z * kCbStride + j];
    const uint32_t off = B - c1;  // rank(H \ y_j) << SH
    B = off + c0;
    LoadPlane<WB>(prev + off, v.g0);
    LoadPlane<WB>(prev + ps + off, v.g1);
    LoadPlane<WB>(prev + 2 * ps + off, v.c);
  };
  int i = 0;
  for (; i + 4 <= h; i += 4) {
    TileWords<WB> v0, v1, v2, v3;
    load(i, v0);
    load(i + 1, v1);
    load(i + 2, v2);
    load(i + 3, v3);
#pragma unroll
    for (int w = 0; w < W; ++w) f[w].Add2(v0.At(w), v1.At(w));
#pragma unroll
    for (int w = 0; w < W; ++w) f[w].Add2(v2.At(w), v3.At(w));
  }
  if (i + 2 <= h) {
    TileWords<WB> v0, v1;
    load(i, v0);
    load(i + 1, v1);
#pragma unroll
    for (int w = 0; w < W; ++w) f[w].Add2(v0.At(w), v1.At(w));
    i += 2;
  }
  if (i < h) {
    TileWords<WB> v0;
    load(i, v0);
#pragma unroll
    for (int w = 0; w < W; ++w) f[w].Add(v0.g0[w], v0.g1[w], v0.c[w]);
  }
  // No vertex of S isolated in S, for the 32 subsets of each word, from
  // per-graph tables over 7-bit chunks of the vertices above 4:
  //   a vertex of H or of w with no neighbour there needs one in L;
  //   a vertex of L with no neighbour in H or w needs one in L.
  const uint32_t Hw = H << WB;
  const uint32_t NH = s_tab[kTabNbh + (Hw & 127u)] |
                      s_tab[kTabNbh + 128 + ((Hw >> 7) & 127u)] |
                      s_tab[kTabNbh + 256 + ((Hw >> 14) & 127u)] |
                      s_tab[kTabNbh + 384 + ((Hw >> 21) & 127u)];
  TileWords<WB> out;
#pragma unroll
  for (int w = 0; w < W; ++w) {
    const uint32_t N = w ? NH | s_tab[kTabNbh + w] : NH;
    const uint32_t I = (Hw | static_cast<uint32_t>(w)) & ~(N >> 5);
    const uint32_t fine = s_tab[kTabIsoL + (~N & 31u)] & s_tab[kTabIsoH + (I & 127u)] &
                          s_tab[kTabIsoH + 128 + ((I >> 7) & 127u)] &
                          s_tab[kTabIsoH + 256 + ((I >> 14) & 127u)] &
                          s_tab[kTabIsoH + 384 + ((I >> 21) & 127u)];
    // the words of w \ b are neighbours too
#pragma unroll
    for (int b = 0; b < WB; ++b)
      if (w >> b & 1) f[w].Add(out.g0[w ^ (1 << b)], out.g1[w ^ (1 << b)], out.c[w ^ (1 << b)]);
    uint32_t single = 0u;
    bool empty = false;
    if constexpr (kTiny) {
      const int size = h + __builtin_popcount(static_cast<unsigned>(w));
      single = size == 0 ? 0x00010116u : size == 1 ? 1u : 0u;
      empty = size == 0;
    }
    const DPWord r = SolveWord(f[w], fine, single, empty, AnyLane());
    out.g0[w] = r.g0;
    out.g1[w] = r.g1;
    out.c[w] = r.c;
  }
  StorePlane<WB>(cur + (t << SH), out.g0);
  StorePlane<WB>(cur + ps + (t << SH), out.g1);
  StorePlane<WB>(cur + 2 * ps + (t << SH), out.c);
}

template <int WB>
__device__ __forceinline__ void LoadPascal(const uint32_t* __restrict__ g_cb,
                                           uint32_t* s_lvl) {
  for (int i = threadIdx.x; i < 32 * kCbStride; i += blockDim.x)
    s_lvl[i] = g_cb[kRevWord + i] << kTileShift<WB>;
  if (threadIdx.x <= kTailBits) s_lvl[kLvlOffs + threadIdx.x] = g_cb[kCbOffs + threadIdx.x];
}

template <int WB>
__device__ __forceinline__ void LoadShared(const DPGraph* __restrict__ g,
                                           const uint32_t* __restrict__ g_cb,
                                           uint32_t* s_lvl, uint32_t* s_tab,
                                           bool load_cb) {
  if (load_cb) LoadPascal<WB>(g_cb, s_lvl);
  // nbh, isoh and isol are consecutive in DPGraph
  for (int i = threadIdx.x; i < kTabWords; i += blockDim.x) s_tab[i] = g->nbh[i];
}

// Tiles [first, end) of high level h of graph g, R consecutive per lane,
// lanes of the launch striding by `stride` tiles.
template <int WB>
__device__ __forceinline__ void DPLevelRange(const DPHead* __restrict__ g,
                                             const uint32_t* __restrict__ g_cb,
                                             uint8_t* __restrict__ arena,
                                             int h, uint32_t first,
                                             uint32_t end, uint32_t lane_id,
                                             uint32_t stride, int R,
                                             const uint32_t* s_lvl,
                                             const uint32_t* s_tab) {
  const int nh = static_cast<int>(g->nh);
  constexpr int SH = kTileShift<WB>;
  uint8_t* base = arena + g->table;
  const uint8_t* prev =
      h > 0 ? base + (static_cast<size_t>(g->lvl[h - 1]) << SH) : base;
  uint8_t* cur = base + (static_cast<size_t>(g->lvl[h]) << SH);
  const size_t ps = static_cast<size_t>(g->lvl[nh + 1]) << SH;
  const uint16_t* tail = reinterpret_cast<const uint16_t*>(g_cb + kTailWord);
  for (uint32_t t0 = first + lane_id * R; t0 < end; t0 += stride) {
    uint32_t H = UnrankTiles<kTileShift<WB>>(t0, h, nh, s_lvl, tail);
    const uint32_t tend = min(t0 + static_cast<uint32_t>(R), end);
    for (uint32_t t = t0;;) {
      if (h <= 1)
        DPTile<WB, true>(prev, cur, ps, t, H, h, s_lvl, s_tab);
      else
        DPTile<WB, false>(prev, cur, ps, t, H, h, s_lvl, s_tab);
      if (++t >= tend) break;
      H = NextCombination(H);
    }
  }
}

// One high level of one graph.
// Workgroups are dealt to the 8 XCDs round-robin (workgroup i -> XCD i % 8).
// The tile range is cut into 8 contiguous slices and XCD x works through
// slice x (where the grid is a multiple of 8, which the host sees to for
// grids of 64 and more), so the neighbour tiles that consecutive tiles share
// are fetched by one XCD's L2 instead of by all eight.  At n = 30 (two graphs
// in flight, 128-subset tiles, 256 threads) a graph takes 430 us with slices
// and 500 us without; at n <= 26 both take the same.
constexpr uint32_t kXcds = 8;

template <int WB>
__global__ __launch_bounds__(1024) void DPLevelKernel(
    const DPGraph* __restrict__ g, const uint32_t* __restrict__ g_cb,
    uint8_t* __restrict__ arena, int h, uint32_t ntiles, int R) {
  __shared__ uint32_t s_lvl[kLvlWords];
  __shared__ uint32_t s_tab[kTabWords];
  LoadShared<WB>(g, g_cb, s_lvl, s_tab, true);
  __syncthreads();
  uint32_t bid = blockIdx.x;
  if (gridDim.x % kXcds == 0)
    bid = (bid % kXcds) * (gridDim.x / kXcds) + bid / kXcds;
  const uint32_t lane_id = bid * blockDim.x + threadIdx.x;
  const uint32_t stride = gridDim.x * blockDim.x * R;
  DPLevelRange<WB>(g, g_cb, arena, h, 0, ntiles, lane_id, stride, R, s_lvl, s_tab);
}

// Level-synchronous batch: one launch per high level h over all graphs;
// each workgroup resolves one chunk (graph, tile range) of that level.
struct Chunk {
  uint32_t gi, first, end, pad;
};

template <int WB>
__global__ __launch_bounds__(1024) void DPChunkKernel(
    const DPGraph* __restrict__ gs, const uint32_t* __restrict__ g_cb,
    uint8_t* __restrict__ arena, const Chunk* __restrict__ chunks, int h,
    int R) {
  __shared__ uint32_t s_lvl[kLvlWords];
  __shared__ uint32_t s_tab[kTabWords];
  const Chunk c = chunks[blockIdx.x];
  const DPGraph* g = gs + c.gi;
  LoadShared<WB>(g, g_cb, s_lvl, s_tab, true);
  __syncthreads();
  DPLevelRange<WB>(g, g_cb, arena, h, c.first, c.end, threadIdx.x,
                   blockDim.x * R, R, s_lvl, s_tab);
}

// Persistent batch: workgroups pull whole graphs from a device queue (graphs
// pre-sorted largest first) and resolve every level of a graph with a
// workgroup barrier between levels, so no level of a graph ever waits on
// another workgroup and the graph's tables stay in one XCD's L2.
// Masks over the 32 low parts L of a word: s_m[T] = the L meeting the low set
// T (none for T = 0), s_m[32 + y] = the L without low vertex y.
constexpr int kLowMaskWords = 37;
__device__ __forceinline__ void LowMasksShared(uint32_t* s_m) {
  const uint32_t t = threadIdx.x;
  if (t < kLowMaskWords) {
    uint32_t m = 0;
    for (uint32_t L = 0; L < 32; ++L)
      if (t < 32 ? (L & t) != 0u : !(L >> (t - 32) & 1u)) m |= 1u << L;
    s_m[t] = m;
  }
}

// The N(H), isolation-by-high and isolation-by-low tables of graph g (the
// nbh / isoh / isol arrays MakeGraph builds on the host), built in LDS from
// g's adjacency rows: entry by entry the same unions and intersections over
// the bits of each chunk.  s_m from LowMasksShared.
__device__ __forceinline__ void BuildTables(const DPHead* __restrict__ g, const uint32_t* s_m,
                                            uint32_t* s_tab) {
  const int n = static_cast<int>(g->n);
  for (int i = threadIdx.x; i < kTabWords; i += blockDim.x) {
    uint32_t m;
    if (i < kTabIsoH) {  // N(chunk) = union of its vertices' rows
      const int c = i >> 7;
      m = 0;
      for (uint32_t ch = i & 127; ch; ch &= ch - 1) {
        const int x = 5 + 7 * c + __builtin_ctz(ch);
        if (x < n) m |= g->adj[x];
      }
    } else if (i < kTabIsoL) {  // the L that give every x of the chunk a neighbour
      const int j = i - kTabIsoH, c = j >> 7;
      m = ~0u;
      for (uint32_t ch = j & 127; ch; ch &= ch - 1) {
        const int x = 5 + 7 * c + __builtin_ctz(ch);
        m &= x < n ? s_m[g->adj[x] & 31u] : 0u;
      }
    } else {  // the L in which every y of Y n L has a neighbour in L
      m = ~0u;
      for (uint32_t yy = static_cast<uint32_t>(i - kTabIsoL); yy; yy &= yy - 1) {
        const int y = __builtin_ctz(yy);
        m &= s_m[32 + y] | s_m[g->adj[y] & 31u];
      }
    }
    s_tab[i] = m;
  }
}

template <int WB>
__global__ __launch_bounds__(1024) void DPPersistentKernel(
    const DPHead* __restrict__ gs, const uint32_t* __restrict__ g_cb,
    uint8_t* __restrict__ arena, int ngraphs, uint32_t* __restrict__ queue,
    int R) {
  __shared__ uint32_t s_lvl[kLvlWords];
  __shared__ uint32_t s_tab[kTabWords];
  __shared__ uint32_t s_masks[kLowMaskWords];
  __shared__ int s_gi;
  LoadPascal<WB>(g_cb, s_lvl);
  LowMasksShared(s_masks);
  for (;;) {
    if (threadIdx.x == 0) s_gi = static_cast<int>(atomicAdd(queue, 1u));
    __syncthreads();
    const int gi = s_gi;
    if (gi >= ngraphs) break;  // uniform: every thread read the same s_gi
    const DPHead* g = gs + gi;
    BuildTables(g, s_masks, s_tab);
    __syncthreads();
    const int nh = static_cast<int>(g->nh);
    for (int h = 0; h <= nh; ++h) {
      const uint32_t ntiles = LevelTiles<kTileShift<WB>>(s_lvl, nh, h);  // no padding
      DPLevelRange<WB>(g, g_cb, arena, h, 0, ntiles, threadIdx.x, blockDim.x * R, R,
                       s_lvl, s_tab);
      __syncthreads();
    }
  }
}

// A run of small high levels [h0, h1] of one graph in one workgroup, with a
// workgroup barrier between levels (the first and last levels of a large
// graph have few tiles; one launch replaces h1 - h0 + 1 of them).
template <int WB>
__global__ __launch_bounds__(1024) void DPSmallLevelsKernel(
    const DPGraph* __restrict__ g, const uint32_t* __restrict__ g_cb,
    uint8_t* __restrict__ arena, int h0, int h1) {
  __shared__ uint32_t s_lvl[kLvlWords];
  __shared__ uint32_t s_tab[kTabWords];
  LoadShared<WB>(g, g_cb, s_lvl, s_tab, true);
  __syncthreads();
  const int nh = static_cast<int>(g->nh);
  for (int h = h0; h <= h1; ++h) {
    const uint32_t ntiles = LevelTiles<kTileShift<WB>>(s_lvl, nh, h);
    DPLevelRange<WB>(g, g_cb, arena, h, 0, ntiles, threadIdx.x, blockDim.x, 1, s_lvl, s_tab);
    __syncthreads();
  }
}

__global__ void ResetCounter(uint32_t* c) {
  if (threadIdx.x == 0 && blockIdx.x == 0) *c = 0u;
}

// Binomials and the level offsets (read per lane, so LDS spares a memory
// round trip before each table read).  Ends with a barrier.
constexpr int kLookupWords = 34;
__device__ __forceinline__ void LoadLookupTables(const DPHead* __restrict__ g,
                                                 const uint32_t* __restrict__ g_cb,
                                                 uint32_t* s_cb, uint32_t* s_base) {
  for (int i = threadIdx.x; i < 32 * kCbStride; i += blockDim.x) s_cb[i] = g_cb[i];
  for (int i = threadIdx.x; i < kLookupWords; i += blockDim.x) s_base[i] = g->lvl[i];
  __syncthreads();
}

// Gray code of td(S) mod 4 (bit v of S = vertex v) from the finished tables.
__device__ __forceinline__ uint32_t LookupCode(const DPHead* __restrict__ g,
                                               const uint8_t* __restrict__ arena,
                                               const uint32_t* s_cb, const uint32_t* s_base,
                                               uint32_t S) {
  if (g->direct) {
    const size_t plane = static_cast<size_t>(1) << (g->n > 5 ? g->n - 5 : 0);
    const uint32_t* p = reinterpret_cast<const uint32_t*>(arena + g->table) + (S >> 5);
    return (p[0] >> (S & 31u) & 1u) | (p[plane] >> (S & 31u) & 1u) << 1;
  }
  const uint32_t lb = g->lb;
  uint32_t H = S >> lb;
  uint32_t tile = s_base[__builtin_popcount(H)];
  for (int i = 1; H; ++i) {
    tile += s_cb[__builtin_ctz(H) * kCbStride + i];
    H &= H - 1;
  }
  const size_t ps = static_cast<size_t>(s_base[g->nh + 1]) << (lb - 3);
  const uint8_t* p = arena + g->table + (static_cast<size_t>(tile) << (lb - 3)) +
                     4 * ((S >> 5) & ((1u << (lb - 5)) - 1u));
  const uint32_t g0 = *reinterpret_cast<const uint32_t*>(p);
  const uint32_t g1 = *reinterpret_cast<const uint32_t*>(p + ps);
  return ((g0 >> (S & 31u)) & 1u) | (((g1 >> (S & 31u)) & 1u) << 1);
}

// Whether td(A) and td(B) differ, A a set and B = A without at most one
// vertex: both ranks in one pass, four vertices of each at a time, so that
// eight reads of the binomials are in flight, then the four words together
// (one set after the other, a vertex at a time: 33 us for the tree at n = 29,
// 25 this way).
__device__ __forceinline__ bool CodesDiffer(const DPHead* __restrict__ g,
                                            const uint8_t* __restrict__ arena,
                                            const uint32_t* s_cb, const uint32_t* s_base,
                                            uint32_t A, uint32_t B) {
  if (g->direct) return LookupCode(g, arena, s_cb, s_base, A) != LookupCode(g, arena, s_cb, s_base, B);
  const uint32_t lb = g->lb;
  uint32_t Ha = A >> lb, Hb = B >> lb;
  uint32_t ta = s_base[__builtin_popcount(Ha)], tb = s_base[__builtin_popcount(Hb)];
  // the i-th vertex's binomial; past the last one C(0, 1) = 0
  auto term = [&](uint32_t* H, int i) {
    const uint32_t at = *H ? static_cast<uint32_t>(__builtin_ctz(*H)) * kCbStride + i : 1u;
    *H &= *H - 1;
    return s_cb[at];
  };
  for (int i = 1; Ha; i += 4) {  // B has no vertex that A lacks
    const uint32_t a0 = term(&Ha, i), b0 = term(&Hb, i);
    const uint32_t a1 = term(&Ha, i + 1), b1 = term(&Hb, i + 1);
    const uint32_t a2 = term(&Ha, i + 2), b2 = term(&Hb, i + 2);
    const uint32_t a3 = term(&Ha, i + 3), b3 = term(&Hb, i + 3);
    ta += a0 + a1 + a2 + a3;
    tb += b0 + b1 + b2 + b3;
  }
  const size_t ps = static_cast<size_t>(s_base[g->nh + 1]) << (lb - 3);
  const uint32_t words = (1u << (lb - 5)) - 1u;
  const uint8_t* base = arena + g->table;
  const uint8_t* pa = base + (static_cast<size_t>(ta) << (lb - 3)) + 4 * ((A >> 5) & words);
  const uint8_t* pb = base + (static_cast<size_t>(tb) << (lb - 3)) + 4 * ((B >> 5) & words);
  const uint32_t a0 = *reinterpret_cast<const uint32_t*>(pa);
  const uint32_t a1 = *reinterpret_cast<const uint32_t*>(pa + ps);
  const uint32_t b0 = *reinterpret_cast<const uint32_t*>(pb);
  const uint32_t b1 = *reinterpret_cast<const uint32_t*>(pb + ps);
  const uint32_t sa = A & 31u, sb = B & 31u;
  return (((a0 >> sa) ^ (b0 >> sb)) | ((a1 >> sa) ^ (b1 >> sb))) & 1u;
}

// td mod 4 of a Gray code
__device__ __forceinline__ uint32_t GrayValue(uint32_t code) { return code ^ (code >> 1); }

// td(S): three more vertices raise td by 0..3, which the codes mod 4 tell, so
// S is put together three vertices at a time, lowest first: one pass over its
// vertices keeps the rank, the reads do not wait for each other, and the sets
// of the lowest vertices are few and stay in the caches.
__device__ __forceinline__ uint32_t LookupTd(const DPHead* __restrict__ g,
                                             const uint8_t* __restrict__ arena,
                                             const uint32_t* s_cb, const uint32_t* s_base,
                                             uint32_t S) {
  const int lb = static_cast<int>(g->lb);
  // direct planes have tiles of one word, lb = 5
  const size_t ps = g->direct ? static_cast<size_t>(4) << (g->n > 5 ? g->n - 5 : 0)
                              : static_cast<size_t>(s_base[g->nh + 1]) << (lb - 3);
  const uint8_t* base = arena + g->table;
  const uint32_t words = (1u << (lb - 5)) - 1u;
  uint32_t td = 0, last = 0, T = 0, r = 0;
  int h = 0, since = 0;
  while (S) {
    const int v = __builtin_ctz(S);
    S &= S - 1;
    T |= 1u << v;
    if (v >= lb && !g->direct) r += s_cb[(v - lb) * kCbStride + ++h];
    if (++since == 3 || !S) {
      since = 0;
      const uint32_t tile = g->direct ? T >> 5 : s_base[h] + r;
      const uint8_t* p = base + (static_cast<size_t>(tile) << (lb - 3)) + 4 * ((T >> 5) & words);
      const uint32_t g0 = *reinterpret_cast<const uint32_t*>(p);
      const uint32_t g1 = *reinterpret_cast<const uint32_t*>(p + ps);
      const uint32_t now =
          GrayValue(((g0 >> (T & 31u)) & 1u) | (((g1 >> (T & 31u)) & 1u) << 1));
      td += (now - last) & 3u;
      last = now;
    }
  }
  return td;
}

__device__ __forceinline__ uint32_t WaveMax(uint32_t v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = max(v, __shfl_xor(v, off));
  return v;
}

// GetElimination (dynamic_gpu.hpp:49-64) from S, by one wave: pop the root
// stored for the current set and repeat, `steps` times.  The root of a connected C is
// the smallest v with td(C \ v) = td(C) - 1 (the strict < over ascending v of
// dynamic_gpu.cu:84-87); a disconnected set stores the root of its first
// component (lowest vertex order) of largest td (dynamic_gpu.cu:90-104).
__global__ __launch_bounds__(64) void DPWalkKernel(
    const DPGraph* __restrict__ g, const uint32_t* __restrict__ g_cb,
    const uint8_t* __restrict__ arena, uint32_t S, int steps, int32_t* __restrict__ out) {
  __shared__ uint32_t s_cb[32 * kCbStride];
  __shared__ uint32_t s_base[kLookupWords];
  LoadLookupTables(g, g_cb, s_cb, s_base);
  const int lane = threadIdx.x;
  const uint32_t myadj = lane < 32 ? g->adj[lane] : 0u;
  for (int step = 0; step < steps && S != 0u; ++step) {
    // C = the first component of largest td, components by ballot BFS from each
    // lowest vertex.  A td takes up to 11 reads all over the table, so it is
    // looked up only where sizes leave it open: td of a component is at most
    // its size, and at least 2 if it has an edge (an elimination of all 25
    // vertices: 67 us a call, 111 with a td for every component).
    uint32_t rest = S, C = 0u, T = 0u;  // T = td(C) once it is needed
    while (rest) {
      uint32_t comp = rest & (0u - rest), front = comp;
      for (;;) {
        const uint32_t nb =
            static_cast<uint32_t>(__ballot((myadj & front) != 0u)) & rest & ~comp;
        if (!nb) break;
        comp |= nb;
        front = nb;
      }
      rest &= ~comp;
      const int most = __builtin_popcount(comp);
      if (!C) {
        C = comp;
      } else if (most > (T ? static_cast<int>(T) : min(__builtin_popcount(C), 2))) {
        if (!T) T = LookupTd(g, arena, s_cb, s_base, C);
        const uint32_t td = LookupTd(g, arena, s_cb, s_base, comp);
        if (td > T) {
          T = td;
          C = comp;
        }
      }
    }
    // the root: the lowest v of C whose removal lowers td, that is, changes
    // the code
    const bool inC = lane < 32 && ((C >> lane) & 1u);
    const unsigned long long rb =
        __ballot(inC && CodesDiffer(g, arena, s_cb, s_base, C, C & ~(1u << lane)));
    const int root = __ffsll(static_cast<long long>(rb)) - 1;
    if (lane == 0) out[step] = root;
    S &= ~(1u << root);
  }
}

// The canonical decomposition of vertex set S by one wave (lane u holds
// adj[u] in myadj), level by level of the tree: every component of the
// vertices left takes its root (the smallest v with td(C \ v) = td(C) - 1) in
// the same round, the parent of a root is the root whose removal created its
// component, and all roots leave together.  The tree is the one
// GetElimination's order produces (each component's root depends only on the
// component), in about td rounds instead of n.  differ(C, D): whether the Gray
// codes of td(C) and td(D) mod 4 differ.  Returns lane u's parent (-1: a root); *depth_out = the tree's
// depth in every lane.
template <typename Differ>
__device__ __forceinline__ int DecomposeWave(uint32_t myadj, uint32_t S, int* depth_out,
                                             Differ differ) {
  const int lane = threadIdx.x & 63;
  if (lane >= 32) myadj = 0u;
  int creator = -1, depth = 0, parent = -1;
  // every round removes at least one vertex per component, so at most 32
  for (int round = 0; round < 32 && S; ++round) {
    const bool in = lane < 32 && ((S >> lane) & 1u);
    uint32_t rest = S, mine = 0u;
    while (rest) {
      uint32_t comp = rest & (0u - rest), front = comp;
      for (;;) {
        const uint32_t nb =
            static_cast<uint32_t>(__ballot((myadj & front) != 0u)) & rest & ~comp;
        if (!nb) break;
        comp |= nb;
        front = nb;
      }
      if ((comp >> lane) & 1u) mine = comp;
      rest &= ~comp;
    }
    // td(C \ v) is td(C) or td(C) - 1: the codes mod 4 tell which
    const uint32_t cand =
        static_cast<uint32_t>(__ballot(in && differ(mine, mine & ~(1u << (lane & 31)))));
    // a connected set always has a vertex with td(C \ v) = td(C) - 1; the
    // lowest vertex stands in only so that a damaged table cannot stall
    const uint32_t rc = cand & mine;
    const int root = in ? __builtin_ctz(rc ? rc : mine) : 0;
    const int cdepth = __shfl(depth, creator >= 0 ? creator : lane);
    if (in && root == lane) {
      parent = creator;
      depth = creator >= 0 ? cdepth + 1 : 1;
    } else if (in) {
      creator = root;
    }
    S &= ~static_cast<uint32_t>(__ballot(in && root == lane));
  }
  *depth_out = static_cast<int>(WaveMax(static_cast<uint32_t>(depth)));
  return parent;
}

// DecomposeWave for one whole graph per workgroup, from tables in memory.
// parent_out: 64 int8 per graph; td_out: the tree's depth.
template <typename Record>
__global__ __launch_bounds__(64) void DPTreeKernel(
    const Record* __restrict__ gs, const uint32_t* __restrict__ g_cb,
    const uint8_t* __restrict__ arena, int8_t* __restrict__ parent_out,
    int32_t* __restrict__ td_out) {
  __shared__ uint32_t s_cb[32 * kCbStride];
  __shared__ uint32_t s_base[kLookupWords];
  const Record* g = gs + blockIdx.x;
  LoadLookupTables(g, g_cb, s_cb, s_base);
  const int lane = threadIdx.x;
  const uint32_t S = g->n >= 32 ? ~0u : (1u << g->n) - 1u;
  int depth = 0;
  const int parent =
      DecomposeWave(lane < 32 ? g->adj[lane] : 0u, S, &depth,
                    [&](uint32_t C, uint32_t D) {
                      return CodesDiffer(g, arena, s_cb, s_base, C, D);
                    });
  int8_t* out = parent_out + static_cast<size_t>(blockIdx.x) * 64;
  if (lane < 32 && ((S >> lane) & 1u)) out[lane] = static_cast<int8_t>(parent);
  if (lane == 0) td_out[blockIdx.x] = depth;
}

// Level-k table in colex order over n vertices (td values): the `count`
// subsets from code `first` on, four consecutive ones to a lane, so that one
// unranking (half of the work of a subset alone) and one store serve four
// (C(23, 11) subsets: 16.6 us, 18.8 one to a lane).  The record's head is an
// argument: a graph solved out of LDS has none on the device.  out is aligned
// to 4 bytes.
__global__ __launch_bounds__(256) void DPExportLevelKernel(
    const DPHead g, const uint32_t* __restrict__ g_cb, const uint8_t* __restrict__ arena, int k,
    uint32_t first, uint32_t count, uint8_t* __restrict__ out) {
  __shared__ uint32_t s_cb[32 * kCbStride];
  __shared__ uint32_t s_base[kLookupWords];
  LoadLookupTables(&g, g_cb, s_cb, s_base);
  const int n = static_cast<int>(g.n);
  const uint32_t quads = count / 4 + (count % 4 ? 1 : 0);
  for (uint32_t q = blockIdx.x * blockDim.x + threadIdx.x; q < quads;
       q += gridDim.x * blockDim.x) {
    const uint32_t r = 4 * q, some = min(count - r, 4u);
    uint32_t S = Unrank(first + r, k, n, s_cb), word = 0;
    for (uint32_t i = 0; i < some; ++i) {
      if (i) S = NextCombination(S);
      word |= LookupTd(&g, arena, s_cb, s_base, S) << 8 * i;
    }
    if (some == 4)
      reinterpret_cast<uint32_t*>(out)[q] = word;
    else
      for (uint32_t i = 0; i < some; ++i) out[r + i] = static_cast<uint8_t>(word >> 8 * i);
  }
}

}  // namespace
}  // namespace tdhip

#include "dplds.hpp"

namespace tdhip {
namespace {

// td(S) for one S.  T[i] is S's first 3 (i + 1) vertices (fewer at the end):
// three more vertices raise td by 0..3, so its code mod 4 after each T[i] gives
// td (see LookupTd).  The host has worked out where each T[i]'s two bits are
// (byte offset of the word in plane 0, and bit), so a lane reads one code and
// nothing waits for a rank.  8.4 us a call at n = 12..28; through the level
// read's kernel (binomials to LDS, unranking, a stream synchronization) 17, and
// one byte copied from a table of bytes took 11.7.
constexpr int kReadSets = (32 + 2) / 3;
struct ReadAt {
  uint64_t plane;  // bytes from a plane to the next
  uint64_t word[kReadSets];
  uint8_t bit[kReadSets];
  uint8_t sets;
};
__global__ __launch_bounds__(64) void DPReadKernel(const ReadAt r,
                                                   const uint8_t* __restrict__ table,
                                                   int32_t* __restrict__ td_out,
                                                   unsigned long long* __restrict__ clock) {
  const int lane = threadIdx.x;
  uint32_t now = 0u;
  if (lane < r.sets) {
    const uint8_t* p = table + r.word[lane];
    const uint32_t g0 = *reinterpret_cast<const uint32_t*>(p) >> r.bit[lane];
    const uint32_t g1 = *reinterpret_cast<const uint32_t*>(p + r.plane) >> r.bit[lane];
    now = GrayValue((g0 & 1u) | (g1 & 1u) << 1);
  }
  const uint32_t last = __shfl_up(now, 1);
  uint32_t td = lane < r.sets ? (now - (lane ? last : 0u)) & 3u : 0u;
#pragma unroll
  for (int off = 8; off > 0; off >>= 1) td += __shfl_xor(td, off);
  if (lane == 0) *td_out = static_cast<int32_t>(td);
  PublishDone(clock);
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
constexpr int kMaxDPN = 32;
constexpr int kMaxBatchN = 26;

// Masks over the 32 low parts L of a word: the L meeting a low set T, and
// the L without low vertex y.
struct LowMasks {
  uint32_t meet[32] = {}, without[5] = {};
  LowMasks() {
    for (uint32_t L = 0; L < 32; ++L) {
      for (uint32_t T = 0; T < 32; ++T)
        if (L & T) meet[T] |= 1u << L;
      for (int y = 0; y < 5; ++y)
        if (!(L >> y & 1u)) without[y] |= 1u << L;
    }
  }
};

// Words per tile (as a power of two) of the parameter dp.low_bits.
int WordBits(int low_bits) { return low_bits >= 5 ? 2 : low_bits == 4 ? 1 : 0; }

// Tile offsets of each high level, each level padded to a 128-byte boundary
// of its plane so no cache line holds tiles of two levels (32 bytes below 8
// high vertices: such tables fit a few lines, and with more padding they
// would take more bytes than a byte per subset did).  Vertices n and
// up, where a tile has more than n, count as isolated.
DPHead MakeHead(int n, const uint64_t* adj, int wb) {
  DPHead G;
  std::memset(&G, 0, sizeof(G));
  const int lb = 5 + wb;
  G.n = n;
  G.lb = lb;
  G.nh = n > lb ? n - lb : 0;
  const uint32_t pad_tiles = (G.nh < 8 ? 32u : 128u) >> (lb - 3);
  uint64_t off = 0;
  for (uint32_t h = 0; h <= G.nh; ++h) {
    G.lvl[h] = static_cast<uint32_t>(off);
    off += Binom(G.nh, h);
    off = (off + pad_tiles - 1) / pad_tiles * pad_tiles;
  }
  G.lvl[G.nh + 1] = static_cast<uint32_t>(off);
  for (int v = 0; v < n; ++v) G.adj[v] = static_cast<uint32_t>(adj[v]);
  return G;
}

// The head and the tables; without `tables`, the head only.
DPGraph MakeGraph(int n, const uint64_t* adj, int wb, bool tables = true) {
  DPGraph G;
  static_cast<DPHead&>(G) = MakeHead(n, adj, wb);
  if (!tables) return G;
  // N(chunk) = N(chunk without its lowest bit) | N(lowest bit), and the low
  // parts that give every vertex of the chunk a neighbour
  static const LowMasks M;
  for (int c = 0; c < 4; ++c) {
    G.nbh[128 * c] = 0;
    G.isoh[128 * c] = ~0u;
    for (int chunk = 1; chunk < 128; ++chunk) {
      const int x = 5 + 7 * c + __builtin_ctz(static_cast<unsigned>(chunk));
      const uint32_t row = x < n ? G.adj[x] : 0u;
      G.nbh[128 * c + chunk] = G.nbh[128 * c + (chunk & (chunk - 1))] | row;
      G.isoh[128 * c + chunk] = G.isoh[128 * c + (chunk & (chunk - 1))] & M.meet[row & 31u];
    }
  }
  // L is fine for low vertex y iff y is not in L or L meets N(y)
  G.isol[0] = ~0u;
  for (int Y = 1; Y < 32; ++Y) {
    const int y = __builtin_ctz(static_cast<unsigned>(Y));
    G.isol[Y] = G.isol[Y & (Y - 1)] & (M.without[y] | M.meet[G.adj[y] & 31u]);
  }
  return G;
}

// Bytes of a graph's three planes.
uint64_t TableBytes(const DPHead& G) {
  return 3 * (static_cast<uint64_t>(G.lvl[G.nh + 1]) << (G.lb - 3));
}

// Bytes that a graph's table claims of the context's budget: one per subset,
// though only 3/8 are allocated, or (dp.packed with dp.class_bits) 17/32, so
// that a byte budget admits and refuses the same calls as with byte tables.
uint64_t ClaimedBytes(const DPHead& G, bool packed = false) {
  const uint64_t subsets = 1ull << G.n;
  return std::max(TableBytes(G), packed ? subsets / 2 + subsets / 32 : subsets);
}

// binomials, O_k, the 16-bit unrank table (2 entries per word), then the
// binomials by leading zeros of the vertex bit
std::vector<uint32_t> PascalTable() {
  std::vector<uint32_t> cb(kPascalWords, 0);
  for (int x = 0; x < 32; ++x)
    for (int j = 0; j < kCbStride; ++j) {
      cb[x * kCbStride + j] = static_cast<uint32_t>(Binom(x, j));
      cb[kRevWord + (31 - x) * kCbStride + j] = static_cast<uint32_t>(Binom(x, j));
    }
  uint16_t* tail = reinterpret_cast<uint16_t*>(cb.data() + kTailWord);
  uint32_t off = 0;
  for (int k = 0; k <= kTailBits; ++k) {
    cb[kCbOffs + k] = off;
    // the k-subsets of {0..15} in colex order = increasing integers
    for (uint32_t m = 0; m < (1u << kTailBits); ++m)
      if (__builtin_popcount(m) == k) tail[off++] = static_cast<uint16_t>(m);
  }
  return cb;
}

const uint32_t* PascalDevice(td_ctx* ctx) {
  auto it = ctx->bufs.find("dp.pascal");
  if (it != ctx->bufs.end() && it->second.p)
    return static_cast<const uint32_t*>(it->second.p);
  const std::vector<uint32_t> cb = PascalTable();
  void* d = ctx->Buffer("dp.pascal", cb.size() * 4);
  ctx->Copy(d, cb.data(), cb.size() * 4, hipMemcpyHostToDevice);
  return static_cast<const uint32_t*>(d);
}

int GridFor(td_ctx* ctx, uint64_t lanes_needed, int block) {
  const uint64_t blocks = (lanes_needed + block - 1) / block;
  const uint64_t cap = static_cast<uint64_t>(ctx->prop.multiProcessorCount) *
                       (2048 / block) * static_cast<uint64_t>(ctx->dp.grid_mult);
  // the same number of passes for every workgroup
  const uint64_t passes = std::max<uint64_t>(1, (blocks + cap - 1) / cap);
  return static_cast<int>(std::max<uint64_t>(1, (blocks + passes - 1) / passes));
}

// Runs of small levels at either end of a graph's level sequence go to one
// workgroup each (DPSmallLevelsKernel): levels [0, lo] and [hi, nh].
constexpr uint64_t kSmallTiles = 320;
void SmallLevelRuns(int nh, int* lo, int* hi) {
  int a = -1, b = nh + 1;
  while (a + 1 <= nh && Binom(nh, a + 1) <= kSmallTiles) ++a;
  while (b - 1 > a && Binom(nh, b - 1) <= kSmallTiles) --b;
  *lo = a;
  *hi = b;
}

// Part of level h when a graph's level sequence is cut into K parts of about
// equal subset counts: the level's first tile, as a fraction of the graph's
// 2^nh tiles, times K (for K = 2 and odd nh, levels 0 .. (nh - 1) / 2 hold
// exactly half).
int PartOf(const DPGraph& G, int h, int K) {
  const int nh = static_cast<int>(G.nh);
  uint64_t before = 0;
  for (int l = 0; l < h; ++l) before += Binom(nh, l);
  const int p = static_cast<int>((before * static_cast<uint64_t>(K)) >> nh);
  return std::min(p, K - 1);
}

// Level launches of one solve of G: all of them (part = -1), or those whose
// first level lies in part `part` of K.  Counts what LaunchLevels launches
// for the same part.
uint64_t PartLaunches(const DPGraph& G, int part, int K) {
  const int nh = static_cast<int>(G.nh);
  auto want = [&](int h0) { return part < 0 || PartOf(G, h0, K) == part; };
  uint64_t c = 0;
  int lo, hi;
  SmallLevelRuns(nh, &lo, &hi);
  if (lo >= 0 && want(0)) ++c;
  for (int h = lo + 1; h < hi; ++h) c += want(h) ? 1 : 0;
  if (hi <= nh && want(hi)) ++c;
  return c;
}

// level kernels one solve of G executes
uint64_t LevelKernelCount(const DPGraph& G) { return PartLaunches(G, -1, 1); }

// The level launches of one graph on stream `st`: all of them (part = -1),
// or the launches whose first level lies in part `part` of K (PartOf).
template <int WB>
void LaunchLevels(td_ctx* ctx, const DPGraph& G, const DPGraph* dG,
                  const uint32_t* cb, uint8_t* arena, uint64_t* launches,
                  hipStream_t st, int part, int K) {
  const int R = ctx->dp.tiles_per_lane, block = ctx->dp.block;
  auto want = [&](int h0) { return part < 0 || PartOf(G, h0, K) == part; };
  const int nh = static_cast<int>(G.nh);
  int lo, hi;
  SmallLevelRuns(nh, &lo, &hi);
  if (lo >= 0 && want(0)) {
    hipLaunchKernelGGL(DPSmallLevelsKernel<WB>, dim3(1), dim3(1024), 0, st, dG, cb,
                       arena, 0, lo);
    ++*launches;
  }
  for (int h = lo + 1; h < hi; ++h) {
    if (!want(h)) continue;
    const uint32_t ntiles = static_cast<uint32_t>(Binom(G.nh, h));
    int grid = GridFor(ctx, (ntiles + R - 1) / R, block);
    if (grid >= 64) grid = (grid + 7) / 8 * 8;  // slices, see DPLevelKernel
    hipLaunchKernelGGL(DPLevelKernel<WB>, dim3(grid), dim3(block), 0,
                       st, dG, cb, arena, h, ntiles, R);
    ++*launches;
  }
  if (hi <= nh && want(hi)) {
    hipLaunchKernelGGL(DPSmallLevelsKernel<WB>, dim3(1), dim3(1024), 0, st, dG, cb,
                       arena, hi, nh);
    ++*launches;
  }
  TD_HIP(hipGetLastError());
}

// Whether every one of K parts holds at least one launch.
bool SplitsInto(const DPGraph& G, int K) {
  for (int p = 0; p < K; ++p)
    if (PartLaunches(G, p, K) == 0) return false;
  return true;
}

void LaunchLevelsLB(td_ctx* ctx, const DPGraph& G, const DPGraph* dG,
                    const uint32_t* cb, uint8_t* arena, uint64_t* launches,
                    hipStream_t st, int part, int K) {
  switch (G.lb) {
    case 5: LaunchLevels<0>(ctx, G, dG, cb, arena, launches, st, part, K); break;
    case 6: LaunchLevels<1>(ctx, G, dG, cb, arena, launches, st, part, K); break;
    default: LaunchLevels<2>(ctx, G, dG, cb, arena, launches, st, part, K); break;
  }
}

// Level sequence of one graph (or part `part` of K of it, as in
// LaunchLevels) on stream `st`, replayed from a captured hipGraph when the
// same (n, launch shape, buffers, part) was seen before.  `slot` tells apart
// the table buffers of the large-graph pipeline, so each keeps its own
// graphs.
void RunLevels(td_ctx* ctx, const DPGraph& G, const DPGraph* dG,
               const uint32_t* cb, uint8_t* arena, uint64_t* launches, int slot = 0,
               hipStream_t st = nullptr, int part = -1, int K = 1) {
  if (!st) st = ctx->stream;
  if (!ctx->dp.use_graph) {
    LaunchLevelsLB(ctx, G, dG, cb, arena, launches, st, part, K);
    return;
  }
  // key includes the buffer addresses baked into the captured launches
  td_ctx::GraphKey key{static_cast<int>(G.n) | (slot << 16) | ((part + 1) << 24) | (K << 28),
                       static_cast<int>(G.lb), ctx->dp.tiles_per_lane, ctx->dp.block};
  auto& p = ctx->dp_graph_ptrs[key];
  auto it = ctx->dp_graphs.find(key);
  if (it != ctx->dp_graphs.end() &&
      (p.first != static_cast<const void*>(arena) ||
       p.second != static_cast<const void*>(dG))) {
    (void)hipGraphExecDestroy(it->second);
    ctx->dp_graphs.erase(it);
    it = ctx->dp_graphs.end();
  }
  if (it == ctx->dp_graphs.end()) {
    hipGraph_t graph;
    uint64_t dummy = 0;
    TD_HIP(hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
    try {
      LaunchLevelsLB(ctx, G, dG, cb, arena, &dummy, st, part, K);
    } catch (...) {
      (void)hipStreamEndCapture(st, &graph);
      throw;
    }
    TD_HIP(hipStreamEndCapture(st, &graph));
    hipGraphExec_t exec;
    TD_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    (void)hipGraphDestroy(graph);
    it = ctx->dp_graphs.emplace(key, exec).first;
    p = {arena, dG};
  }
  TD_HIP(hipGraphLaunch(it->second, st));
  ++*launches;
}

float Elapsed(hipEvent_t a, hipEvent_t b) {
  float ms = 0.f;
  TD_HIP(hipEventElapsedTime(&ms, a, b));
  return ms;
}

// Record of one graph for the single-graph level kernels.  Larger tiles cost
// fewer instructions and bytes per subset, but leave fewer lanes: tiles take
// the context's words only as far as 22 high vertices remain (705,432 tiles in
// the middle level).  Level kernels of one graph with 1 / 2 / 4 words, us:
// n = 23: 92 / 97 / 108; n = 27: 168 / 170 / 180; n = 28: 236 / 227 / 233;
// n = 29: 366 / 341 / 331; n = 30: 635 / 560 / 527.
int SingleWordBits(int n, int low_bits) {
  return std::min(WordBits(low_bits), std::max(0, n - 27));
}
DPGraph SingleGraph(td_ctx* ctx, int n, const uint64_t* adj, bool tables = true) {
  return MakeGraph(n, adj, SingleWordBits(n, ctx->dp.low_bits), tables);
}

// Whether the context claims a packed table's bytes for this graph.
bool ClaimsPacked(const td_ctx* ctx, int n) {
  const int lb = std::max(ctx->dp.low_bits, n - 28);  // of the byte tables
  return ctx->dp.packed && ctx->dp.class_bits > 0 && lb >= 4 && n - lb >= ctx->dp.class_min_nh;
}

// The descriptor goes up from page-locked staging in one copy; the tree (64
// parents, then the depth) comes back the same way.
constexpr size_t kInBytes = (sizeof(DPGraph) + 15) / 16 * 16 + 16;
constexpr size_t kTreeBytes = 64 + 16;

// What a single solve reports besides its answer.
void FillStats(td_dp_stats* stats, int n, uint64_t launches, uint64_t level_kernels,
               double level_ms, double tree_ms, std::chrono::steady_clock::time_point t0) {
  stats->graphs = 1;
  stats->level_kernels = level_kernels;
  stats->subsets = 1ull << n;
  stats->alg_bytes = (1ull << (n - 1)) * static_cast<uint64_t>(n + 2);
  stats->launches = launches;
  stats->level_ms = level_ms;
  stats->tree_ms = tree_ms;
  stats->total_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

// Results of DPLdsKernel in host-visible memory: 64 parents, the depth, three
// readings of the device's clock, and "done".
struct LdsOut {
  int8_t parent[64];
  int32_t td;
  int32_t status;
  unsigned long long clock[4];
};

// Waits until the last kernel of a single solve has published its results, its
// last act: tree and tables are written, and all that is left of the call on
// the device is the kernel's own end.
// Reading the flag it writes sees them 5 to 6 us before
// hipStreamSynchronize returns (n = 9: 27 to 21 us a call).  Should it not
// come within a few milliseconds (a busy device, or an error), and once in a
// while, for the runtime to take its launch resources back, the stream is
// synchronized.
void WaitDone(td_ctx* ctx, LdsOut* out) {
  const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(5);
  if (++ctx->unsynced < 64) {
    for (int i = 1;; ++i) {
      if (__atomic_load_n(&out->clock[3], __ATOMIC_ACQUIRE)) return;
      __builtin_ia32_pause();
      if (i % 256 == 0 && std::chrono::steady_clock::now() > until) break;
    }
  }
  ctx->unsynced = 0;
  TD_HIP(hipStreamSynchronize(ctx->stream));
}


// One launch for a graph of at most kLdsMaxN vertices: the graph goes up in
// the kernel's arguments and the kernel writes its results to `out` itself, so
// no copy and no event stands beside it.
void LaunchLds(td_ctx* ctx, const DPGraph& G, const uint32_t* cb, uint8_t* arena, LdsOut* out) {
  LdsGraph one;
  one.n = G.n;
  for (int v = 0; v < kLdsMaxN; ++v) one.adj[v] = G.adj[v];
  const int n = static_cast<int>(G.n);
  hipLaunchKernelGGL(DPLdsKernel, dim3(1), dim3(LdsThreads(n)), LdsBytes(n), ctx->stream,
                     static_cast<const LdsGraph*>(nullptr), one, cb,
                     reinterpret_cast<uint32_t*>(arena), out->parent, &out->td, out->clock);
  TD_HIP(hipGetLastError());
}

// DPFlowKernel's buffer with room for `words` bytes of published words behind
// the ticket counter: null where the byte budget or the device has no room for
// it (the other kernels do without).  It is cleared when it is new and
// (LaunchFlow) when the 16-bit tags have come round, so no word in it carries
// a tag that is still to come.  The tag is kFlowStale while it is not known
// what the buffer holds, an error included: the next call clears it.
constexpr size_t kFlowHead = 256;
constexpr uint32_t kFlowStale = 0xFFFFu;
void ClearFlow(td_ctx* ctx) {
  const auto& b = ctx->bufs["dp.flow"];
  ctx->flow_tag = kFlowStale;
  TD_HIP(hipMemsetAsync(b.p, 0, b.bytes, ctx->stream));
  ctx->flow_tag = 0;
  ctx->flow_tickets = 0;
}
uint8_t* FlowBuffer(td_ctx* ctx, size_t words) {
  const size_t bytes = kFlowHead + words;
  auto it = ctx->bufs.find("dp.flow");
  const bool fits = it != ctx->bufs.end() && it->second.p && it->second.bytes >= bytes;
  uint8_t* p = nullptr;
  try {
    p = static_cast<uint8_t*>(ctx->Buffer("dp.flow", bytes));
  } catch (const Error& e) {
    if (e.code != TD_E_NOMEM) throw;
    return nullptr;
  }
  if (!fits) ClearFlow(ctx);
  return p;
}

// The first of `count` graphs of kFlowMinN..kFlowMaxN vertices, largest first
// (sizes in ns), as many as fit one launch of a workgroup per CU
// (or one graph): the launch's classes.  *words and *planes receive the bytes
// of published words and planes, *groups the workgroups; returns the graphs.
int PlanFlow(const td_ctx* ctx, int count, const uint32_t* ns, FlowCall* f, size_t* words,
             size_t* planes, uint32_t* groups) {
  *words = *planes = 0;
  *groups = 0;
  f->classes = 0;
  int i = 0;
  for (; i < count; ++i) {
    const uint32_t n = ns[i];
    const uint32_t more = 1u << FlowTop(static_cast<int>(n));
    if (i && *groups + more > static_cast<uint32_t>(ctx->prop.multiProcessorCount)) break;
    if (!f->classes || f->c[f->classes - 1].n != n)
      f->c[f->classes++] = {n, *groups, static_cast<uint32_t>(i), *words / 8, *planes / 4};
    *groups += more;
    *words += FlowBytes(static_cast<int>(n));
    *planes += DirectBytes(static_cast<int>(n));
  }
  return i;
}

// The levels and decompositions of the planned graphs.
void LaunchFlow(td_ctx* ctx, FlowCall& f, int count, uint32_t groups, const FlowGraph* gs,
                const uint32_t* cb, uint8_t* planes, uint8_t* buf, int8_t* parents, int32_t* tds,
                int32_t* status, unsigned long long* clock) {
  if (ctx->flow_tag >= kFlowStale) ClearFlow(ctx);
  f.ticket0 = ctx->flow_tickets;
  f.tag = ctx->flow_tag + 1;
  // the kernel's indexes come from its tickets: a launch check that fails (for
  // an error of some earlier call of this thread, too, with the kernel on its
  // way) must not leave them out of step
  ctx->flow_tag = kFlowStale;
  f.spin = static_cast<uint32_t>(ctx->dp.flow_spin);
  uint32_t* ticket = reinterpret_cast<uint32_t*>(buf);
  auto* ex = reinterpret_cast<unsigned long long*>(buf + kFlowHead);
  uint32_t* table = reinterpret_cast<uint32_t*>(planes);
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(groups), dim3(512), 0, ctx->stream, f, gs, cb, ex, ticket,
                       table, status, clock);
  };
  switch (f.c[0].n) {  // the largest
    case 19: launch(DPFlowKernel<3>); break;
    case 20: launch(DPFlowKernel<4>); break;
    case 21: launch(DPFlowKernel<5>); break;
    case 22: launch(DPFlowKernel<6>); break;
    case 23: launch(DPFlowKernel<7>); break;
    default: launch(DPFlowKernel<8>); break;
  }
  TD_HIP(hipGetLastError());
  ctx->flow_tag = f.tag;
  ctx->flow_tickets += groups;
  hipLaunchKernelGGL(DPDirectTreeKernel, dim3(count), dim3(64), 0, ctx->stream, f, gs, table,
                     parents, tds, clock);
  TD_HIP(hipGetLastError());
}

void SolveOne(td_ctx* ctx, int n, const uint64_t* adj, uint8_t* td_out,
              int8_t* parent_out, td_dp_stats* stats) {
  const auto t0 = std::chrono::steady_clock::now();
  ValidateGraph(n, adj, kMaxDPN);
  // the buffers below may be reallocated: until this solve completes, the
  // queries have no tables to read
  ctx->have_dp = false;
  const bool lds = n <= kLdsMaxN, flow = !lds && n <= kFlowMaxN;
  DPGraph G = SingleGraph(ctx, n, adj, !lds && !flow);
  uint8_t* arena = static_cast<uint8_t*>(
      ctx->Buffer("dp.arena", TableBytes(G), ClaimedBytes(G, ClaimsPacked(ctx, n))));
  uint8_t* din = static_cast<uint8_t*>(ctx->Buffer("dp.graph", kInBytes));
  DPGraph* dG = reinterpret_cast<DPGraph*>(din);
  const uint32_t* cb = PascalDevice(ctx);
  (void)ctx->Buffer("dp.tree_out", kTreeBytes);  // asks the byte budget
  uint8_t* stage = static_cast<uint8_t*>(ctx->Pinned(kInBytes + std::max(sizeof(LdsOut), kTreeBytes)));
  uint8_t* fbuf = flow ? FlowBuffer(ctx, FlowBytes(n)) : nullptr;
  ctx->last_n = n;
  ctx->record_up = !lds && !fbuf;
  if (lds || fbuf) {
    LdsOut* out = reinterpret_cast<LdsOut*>(stage + kInBytes);
    out->clock[3] = 0;
    if (lds) {
      LaunchLds(ctx, G, cb, arena, out);
    } else {
      FlowCall f;
      size_t words, planes;
      uint32_t groups;
      PlanFlow(ctx, 1, &G.n, &f, &words, &planes, &groups);
      std::memcpy(f.one.adj, G.adj, sizeof(f.one.adj));
      out->status = 0;
      LaunchFlow(ctx, f, 1, groups, nullptr, cb, arena, fbuf, out->parent, &out->td, &out->status,
                 out->clock);
    }
    WaitDone(ctx, out);
    if (lds || !out->status) {
      if (td_out) *td_out = static_cast<uint8_t>(out->td);
      if (parent_out) std::memcpy(parent_out, out->parent, n);
      G.direct = 1;
      ctx->last_graph = G;
      ctx->have_dp = true;
      if (stats) {
        const double ms = 1.0 / ctx->clock_khz;
        FillStats(stats, n, lds ? 1 : 2, 1,
                  static_cast<double>(out->clock[1] - out->clock[0]) * ms,
                  static_cast<double>(out->clock[2] - out->clock[1]) * ms, t0);
      }
      return;
    }
    ctx->record_up = true;  // a wait was given up: the level kernels solve it
  }
  if (flow) G = SingleGraph(ctx, n, adj);
  ctx->last_graph = G;
  std::memcpy(stage, &G, sizeof(G));
  TD_HIP(hipMemcpyAsync(din, stage, kInBytes, hipMemcpyHostToDevice, ctx->stream));
  uint64_t launches = 0;
  TD_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
  RunLevels(ctx, G, dG, cb, arena, &launches);
  TD_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
  // the tree goes straight to page-locked memory
  uint8_t* staged = stage + kInBytes;
  hipLaunchKernelGGL(DPTreeKernel<DPGraph>, dim3(1), dim3(64), 0, ctx->stream, dG, cb, arena,
                     reinterpret_cast<int8_t*>(staged), reinterpret_cast<int32_t*>(staged + 64));
  TD_HIP(hipGetLastError());
  ++launches;
  TD_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
  TD_HIP(hipStreamSynchronize(ctx->stream));
  int32_t td = 0;
  std::memcpy(&td, staged + 64, 4);
  if (td_out) *td_out = static_cast<uint8_t>(td);
  if (parent_out) std::memcpy(parent_out, staged, n);
  ctx->have_dp = true;
  if (stats)
    FillStats(stats, n, launches, LevelKernelCount(G), Elapsed(ctx->ev[0], ctx->ev[1]),
              Elapsed(ctx->ev[1], ctx->ev[2]), t0);
}

// Where the codes that make up td(S) are in the last single solve's table (see
// DPReadKernel; the walk is LookupTd's).
ReadAt ReadOffsets(const DPHead& G, uint32_t S) {
  ReadAt r{};
  const int lb = static_cast<int>(G.lb);
  r.plane = G.direct ? uint64_t{4} << (G.n > 5 ? G.n - 5 : 0)
                     : static_cast<uint64_t>(G.lvl[G.nh + 1]) << (lb - 3);
  const uint32_t words = (1u << (lb - 5)) - 1u;
  uint64_t rank = 0;
  uint32_t T = 0;
  int h = 0, since = 0;
  while (S) {
    const int v = __builtin_ctz(S);
    S &= S - 1;
    T |= 1u << v;
    if (v >= lb && !G.direct) rank += Binom(v - lb, ++h);
    if (++since == 3 || !S) {
      since = 0;
      const uint64_t tile = G.direct ? T >> 5 : G.lvl[h] + rank;
      r.word[r.sets] = G.table + (tile << (lb - 3)) + 4 * ((T >> 5) & words);
      r.bit[r.sets++] = static_cast<uint8_t>(T & 31u);
    }
  }
  return r;
}

// The device record of the last single solve, which the queries read; a graph
// solved by DPLdsKernel has none until the first query.
const DPGraph* LastRecord(td_ctx* ctx) {
  void* d = ctx->bufs["dp.graph"].p;
  if (!ctx->record_up) {
    TD_HIP(hipMemcpyAsync(d, &ctx->last_graph, sizeof(DPHead), hipMemcpyHostToDevice,
                          ctx->stream));
    ctx->record_up = true;
  }
  return static_cast<const DPGraph*>(d);
}

// ---------------------------------------------------------------------------
// td_dp_solve_noalloc: the single-graph solve for callers that cannot
// allocate device memory.  Descriptor, tree output, Pascal tables and level
// tables live in one file-scope device array (`scratch`), loaded with the
// code object on each device the library runs on and held until the process
// ends.  Host code never passes `scratch` itself (its host-side name is not a
// device address): set-up takes each device's address once with
// hipGetSymbolAddress and every launch and copy uses that address.
// ---------------------------------------------------------------------------
constexpr int kNoAllocMaxN = 24;
constexpr size_t kNoAllocTreeOff = 8192;
constexpr size_t kNoAllocPascalOff = 16384;
constexpr size_t kNoAllocArenaOff = 256 * 1024;
// at most 2^n table bytes (3/8 of them used) plus padding
constexpr size_t kNoAllocArenaBytes = (size_t{1} << kNoAllocMaxN) + 64 * 1024;
constexpr size_t kNoAllocScratchBytes = kNoAllocArenaOff + kNoAllocArenaBytes;
static_assert(kInBytes <= kNoAllocTreeOff, "descriptor block overlaps the tree output");
static_assert(kNoAllocTreeOff + kTreeBytes <= kNoAllocPascalOff, "tree output too large");
static_assert(kNoAllocPascalOff + 4 * size_t{kPascalWords} <= kNoAllocArenaOff,
              "Pascal tables overlap the level tables");

static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

constexpr int kNoAllocMaxDevices = 64;
std::mutex g_noalloc_mu;
uint8_t* g_noalloc_ptr[kNoAllocMaxDevices] = {};

void SolveOneNoAlloc(td_ctx* ctx, int n, const uint64_t* adj, uint8_t* td_out,
                     int8_t* parent_out, td_dp_stats* stats) {
  const auto t0 = std::chrono::steady_clock::now();
  TD_REQUIRE(n >= 1 && n <= kNoAllocMaxN, TD_E_INVALID,
             "td_dp_solve_noalloc takes n in [1, " + std::to_string(kNoAllocMaxN) +
                 "] (its level tables live in a fixed " +
                 std::to_string(kNoAllocArenaBytes) + "-byte device array); use td_dp_solve");
  ValidateGraph(n, adj, kNoAllocMaxN);
  uint8_t* base = ctx->device >= 0 && ctx->device < kNoAllocMaxDevices
                      ? g_noalloc_ptr[ctx->device]
                      : nullptr;
  TD_REQUIRE(base != nullptr, TD_E_STATE, "no device scratch address for this device");
  // the queries read the context's own tables, which this call leaves alone,
  // but the last td_dp_solve's results are no longer the last solve's
  ctx->have_dp = false;
  const DPGraph G = SingleGraph(ctx, n, adj);
  TD_REQUIRE(TableBytes(G) <= kNoAllocArenaBytes, TD_E_INVALID,
             "level tables exceed the fixed device array");
  uint8_t* din = base;
  const DPGraph* dG = reinterpret_cast<const DPGraph*>(din);
  uint8_t* dtree = base + kNoAllocTreeOff;
  const uint32_t* cb = reinterpret_cast<const uint32_t*>(base + kNoAllocPascalOff);
  uint8_t* arena = base + kNoAllocArenaOff;
  // inputs from this frame (pageable host memory; the call synchronizes
  // before the frame ends), results back into it
  alignas(16) uint8_t in[kInBytes];
  alignas(16) uint8_t tree[kTreeBytes];
  std::memcpy(in, &G, sizeof(G));
  TD_HIP(hipMemcpyAsync(din, in, kInBytes, hipMemcpyHostToDevice, ctx->stream));
  uint64_t launches = 0;
  TD_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
  // direct launches: a captured graph would be instantiated (allocated) here
  LaunchLevelsLB(ctx, G, dG, cb, arena, &launches, ctx->stream, -1, 1);
  TD_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
  hipLaunchKernelGGL(DPTreeKernel<DPGraph>, dim3(1), dim3(64), 0, ctx->stream, dG, cb, arena,
                     reinterpret_cast<int8_t*>(dtree), reinterpret_cast<int32_t*>(dtree + 64));
  TD_HIP(hipGetLastError());
  ++launches;
  TD_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
  TD_HIP(hipMemcpyAsync(tree, dtree, 64 + 4, hipMemcpyDeviceToHost, ctx->stream));
  TD_HIP(hipStreamSynchronize(ctx->stream));
  int32_t td = 0;
  std::memcpy(&td, tree + 64, 4);
  if (td_out) *td_out = static_cast<uint8_t>(td);
  if (parent_out) std::memcpy(parent_out, tree, n);
  if (stats)
    FillStats(stats, n, launches, LevelKernelCount(G), Elapsed(ctx->ev[0], ctx->ev[1]),
              Elapsed(ctx->ev[1], ctx->ev[2]), t0);
}

// ---------------------------------------------------------------------------
// batch
// ---------------------------------------------------------------------------
constexpr int kMaxStreams = 3;
constexpr int kSlots = kMaxStreams;
static_assert(4 * kSlots + 1 <= static_cast<int>(sizeof(td_ctx::pev) / sizeof(hipEvent_t)),
              "pipeline events");
static_assert(kMaxStreams - 1 <= static_cast<int>(sizeof(td_ctx::lvl) / sizeof(hipStream_t)),
              "level streams");

// Graphs above kMaxBatchN vertices in a batch go through the single-graph
// level kernels, S = max(2, K) slots of (table, descriptor, tree output,
// staging) taken in turn, K = dp.streams; a slot is reused only after the
// host has waited for its previous tree (graph j - S, long done when graph
// j's turn comes).  With K > 1 consecutive graphs run their levels on K
// streams in turn, each sequence cut into K parts of about equal subset
// counts, and each graph's levels start when the previous graph (on another
// stream) has finished its first part: K graphs are in flight, one graph's
// small end levels and kernel tails, which fill a fraction of the device,
// run beside the others' large middle levels.  With K = 1 the levels run one
// graph after another on the context's stream.  Every graph's decomposition
// runs on a further stream while the next levels run.  Adds the level time
// (the union of the graphs' level intervals, so time in which graphs' levels
// overlap counts once), the tree time (end of levels to end of tree),
// launches and level-kernel count of these graphs to the outputs.
void SolveLarge(td_ctx* ctx, const std::vector<int>& idx, const int32_t* ns,
                const uint64_t* adj_concat, const std::vector<size_t>& row_off,
                uint8_t* td_out, int8_t* parent_concat, double* level_ms, double* tree_ms,
                uint64_t* launches, uint64_t* level_kernels) {
  if (idx.empty()) return;
  const int K = std::max(1, std::min(kMaxStreams, ctx->dp.streams));
  const int S = std::max(2, K);
  if (!ctx->side) TD_HIP(hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking));
  for (int k = 1; k < K; ++k)
    if (!ctx->lvl[k - 1]) TD_HIP(hipStreamCreateWithFlags(&ctx->lvl[k - 1], hipStreamNonBlocking));
  for (auto& e : ctx->pev)
    if (!e) TD_HIP(hipEventCreate(&e));
  // every buffer at its final size before the first launch
  uint64_t tmax = 0, cmax = 0;
  for (int i : idx) {
    const DPGraph G = SingleGraph(ctx, ns[i], adj_concat + row_off[i], false);
    tmax = std::max(tmax, TableBytes(G));
    cmax = std::max(cmax, ClaimedBytes(G, ClaimsPacked(ctx, ns[i])));
  }
  uint8_t *arena[kSlots], *din[kSlots], *dtree[kSlots];
  for (int s = 0; s < S; ++s) {
    const std::string sfx = s ? std::to_string(s) : std::string();
    arena[s] = static_cast<uint8_t*>(ctx->Buffer("dp.arena" + sfx, tmax, cmax));
    din[s] = static_cast<uint8_t*>(ctx->Buffer("dp.graph" + sfx, kInBytes));
    dtree[s] = static_cast<uint8_t*>(ctx->Buffer("dp.tree_out" + sfx, kTreeBytes));
  }
  const uint32_t* cb = PascalDevice(ctx);
  constexpr size_t kSlot = kInBytes + kTreeBytes;
  uint8_t* stage = static_cast<uint8_t*>(ctx->Pinned(S * kSlot));
  hipStream_t lvs[kMaxStreams] = {ctx->stream, ctx->stream, ctx->stream};
  for (int k = 1; k < K; ++k) lvs[k] = ctx->lvl[k - 1];
  hipEvent_t* lv_start = ctx->pev;                // [slot]
  hipEvent_t* lv_end = ctx->pev + kSlots;         // [slot]
  hipEvent_t* tree_end = ctx->pev + 2 * kSlots;   // [slot]
  hipEvent_t* first = ctx->pev + 3 * kSlots;      // [slot]: first part of the levels done
  hipEvent_t base = ctx->pev[4 * kSlots];         // time origin of the level intervals
  std::vector<std::pair<float, float>> span;
  span.reserve(idx.size());
  // results of the graph in slot s: its tree came back into the staging
  auto consume = [&](int j) {
    const int s = j % S, i = idx[j];
    TD_HIP(hipEventSynchronize(tree_end[s]));
    const uint8_t* staged = stage + s * kSlot + kInBytes;
    int32_t td = 0;
    std::memcpy(&td, staged + 64, 4);
    if (td_out) td_out[i] = static_cast<uint8_t>(td);
    if (parent_concat) std::memcpy(parent_concat + row_off[i], staged, ns[i]);
    span.emplace_back(Elapsed(base, lv_start[s]), Elapsed(base, lv_end[s]));
    *tree_ms += Elapsed(lv_end[s], tree_end[s]);
  };
  const int L = static_cast<int>(idx.size());
  try {
    TD_HIP(hipEventRecord(base, ctx->stream));
    for (int k = 1; k < K; ++k) TD_HIP(hipStreamWaitEvent(lvs[k], base, 0));
    bool prev_split = false;
    for (int j = 0; j < L; ++j) {
      const int s = j % S, i = idx[j];
      hipStream_t st = lvs[j % K];
      if (j >= S) consume(j - S);  // frees slot s: its tree, copies and levels are done
      const DPGraph G = SingleGraph(ctx, ns[i], adj_concat + row_off[i]);
      uint8_t* in = stage + s * kSlot;
      std::memcpy(in, &G, sizeof(G));
      TD_HIP(hipMemcpyAsync(din[s], in, kInBytes, hipMemcpyHostToDevice, st));
      const DPGraph* dG = reinterpret_cast<const DPGraph*>(din[s]);
      const bool split = K > 1 && SplitsInto(G, K);
      if (prev_split) TD_HIP(hipStreamWaitEvent(st, first[(j - 1) % S], 0));
      TD_HIP(hipEventRecord(lv_start[s], st));
      if (split) {
        for (int p = 0; p < K; ++p) {
          RunLevels(ctx, G, dG, cb, arena[s], launches, s, st, p, K);
          if (p == 0) TD_HIP(hipEventRecord(first[s], st));
        }
      } else {
        RunLevels(ctx, G, dG, cb, arena[s], launches, s, st, -1, 1);
      }
      TD_HIP(hipEventRecord(lv_end[s], st));
      prev_split = split;
      *level_kernels += LevelKernelCount(G);
      TD_HIP(hipStreamWaitEvent(ctx->side, lv_end[s], 0));
      hipLaunchKernelGGL(DPTreeKernel<DPGraph>, dim3(1), dim3(64), 0, ctx->side, dG, cb, arena[s],
                         reinterpret_cast<int8_t*>(dtree[s]),
                         reinterpret_cast<int32_t*>(dtree[s] + 64));
      TD_HIP(hipGetLastError());
      ++*launches;
      TD_HIP(hipMemcpyAsync(stage + s * kSlot + kInBytes, dtree[s], 64 + 4,
                            hipMemcpyDeviceToHost, ctx->side));
      TD_HIP(hipEventRecord(tree_end[s], ctx->side));
    }
    for (int j = std::max(0, L - S); j < L; ++j) consume(j);
  } catch (...) {
    // nothing queued may still use the slots when the error reaches the caller
    (void)hipStreamSynchronize(ctx->stream);
    for (hipStream_t q : ctx->lvl)
      if (q) (void)hipStreamSynchronize(q);
    (void)hipStreamSynchronize(ctx->side);
    throw;
  }
  // union of the level intervals
  std::sort(span.begin(), span.end());
  double lo = 0.0, hi = -1.0, total = 0.0;
  for (const auto& iv : span) {
    if (iv.first > hi) {
      if (hi > lo) total += hi - lo;
      lo = iv.first;
      hi = iv.second;
    } else {
      hi = std::max(hi, static_cast<double>(iv.second));
    }
  }
  if (hi > lo) total += hi - lo;
  *level_ms += total;
}

template <int WB>
void LaunchPersistent(td_ctx* ctx, int ngraphs, const DPHead* dGs, const uint32_t* cb,
                      uint8_t* arena, uint32_t* dqueue, uint64_t* launches) {
  const int R = ctx->dp.tiles_per_lane;
  // queue reset (a kernel, not a memset, so the pair can be captured) and
  // the persistent launch, replayed from a hipGraph cached per batch shape
  const int grid = ctx->prop.multiProcessorCount * ctx->dp.batch_wg_per_cu;
  const int bblock = ctx->dp.batch_block;
  auto launch = [&] {
    hipLaunchKernelGGL(ResetCounter, dim3(1), dim3(64), 0, ctx->stream, dqueue);
    hipLaunchKernelGGL(DPPersistentKernel<WB>, dim3(grid), dim3(bblock), 0,
                       ctx->stream, dGs, cb, arena, ngraphs, dqueue, R);
  };
  if (!ctx->dp.use_graph) {
    launch();
    *launches += 2;
  } else {
    const td_ctx::GraphKey key{-ngraphs, WB, R, bblock * 64 + ctx->dp.batch_wg_per_cu};
    const void* sig[3] = {arena, dGs, dqueue};
    auto it = ctx->dp_graphs.find(key);
    auto& p = ctx->dp_graph_ptrs[key];
    if (it != ctx->dp_graphs.end() && (p.first != sig[0] || p.second != sig[1])) {
      (void)hipGraphExecDestroy(it->second);
      ctx->dp_graphs.erase(it);
      it = ctx->dp_graphs.end();
    }
    if (it == ctx->dp_graphs.end()) {
      hipGraph_t graph;
      TD_HIP(hipStreamBeginCapture(ctx->stream, hipStreamCaptureModeThreadLocal));
      launch();
      TD_HIP(hipStreamEndCapture(ctx->stream, &graph));
      hipGraphExec_t exec;
      TD_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
      (void)hipGraphDestroy(graph);
      it = ctx->dp_graphs.emplace(key, exec).first;
      p = {sig[0], sig[1]};
    }
    TD_HIP(hipGraphLaunch(it->second, ctx->stream));
    *launches += 1;
  }
  TD_HIP(hipGetLastError());
}

// Modes 1 and 2 of a batch call.
template <int WB>
void LaunchBatch(td_ctx* ctx, int mode, int ngraphs,
                 const DPGraph* Gs, const DPGraph* dGs,
                 const uint32_t* cb, uint8_t* arena,
                 uint64_t* launches) {
  const int R = ctx->dp.tiles_per_lane, block = ctx->dp.block;
  if (mode == 1) {
    int maxnh = 0;
    for (int i = 0; i < ngraphs; ++i) maxnh = std::max(maxnh, static_cast<int>(Gs[i].nh));
    const uint32_t chunk_tiles = static_cast<uint32_t>(block) * R * 2;
    std::vector<std::vector<Chunk>> per_level(maxnh + 1);
    size_t total = 0;
    for (int h = 0; h <= maxnh; ++h) {
      for (int i = 0; i < ngraphs; ++i) {
        if (h > static_cast<int>(Gs[i].nh)) continue;
        const uint32_t nt = static_cast<uint32_t>(Binom(Gs[i].nh, h));
        for (uint32_t f = 0; f < nt; f += chunk_tiles)
          per_level[h].push_back(
              {static_cast<uint32_t>(i), f, std::min(nt, f + chunk_tiles), 0});
      }
      total += per_level[h].size();
    }
    Chunk* dch = static_cast<Chunk*>(
        ctx->Buffer("dp.batch_chunks", std::max<size_t>(1, total) * sizeof(Chunk)));
    std::vector<Chunk> flat;
    flat.reserve(total);
    for (auto& v : per_level) flat.insert(flat.end(), v.begin(), v.end());
    TD_HIP(hipMemcpyAsync(dch, flat.data(), flat.size() * sizeof(Chunk),
                          hipMemcpyHostToDevice, ctx->stream));
    size_t off = 0;
    for (int h = 0; h <= maxnh; ++h) {
      const size_t cnt = per_level[h].size();
      if (cnt) {
        hipLaunchKernelGGL(DPChunkKernel<WB>, dim3(cnt), dim3(block), 0,
                           ctx->stream, dGs, cb, arena, dch + off, h, R);
        ++*launches;
      }
      off += cnt;
    }
  } else {
    for (int i = 0; i < ngraphs; ++i)
      for (int h = 0; h <= static_cast<int>(Gs[i].nh); ++h) {
        const uint32_t ntiles = static_cast<uint32_t>(Binom(Gs[i].nh, h));
        const int grid = GridFor(ctx, (ntiles + R - 1) / R, block);
        hipLaunchKernelGGL(DPLevelKernel<WB>, dim3(grid), dim3(block), 0,
                           ctx->stream, dGs + i, cb, arena, h, ntiles, R);
        ++*launches;
      }
  }
  TD_HIP(hipGetLastError());
}

// Whether DPFlowKernel takes a batch's graphs of 19..24 vertices (the first
// `count` of perm, largest first) rather than the persistent kernel.  A launch
// of DPFlowKernel (one workgroup per CU) and its trees takes 70 us or less; the
// persistent kernel takes a workgroup's time for the largest graph, measured as 75 us +
// 1150 us 2^(n - 24) (n = 19: 103 us, 20: 135, 22: 345, 24: 1220), and then
// the others cost it little.  16 graphs of n = 19 / 20 / 22: 76 / 82 / 240 us
// a call against 134 / 173 / 398, four of n = 24 345 against 1283.
bool FlowPays(const td_ctx* ctx, int count, const int32_t* ns, const std::vector<int>& perm) {
  if (count == 0 || ns[perm[0]] > kFlowMaxN) return false;
  uint64_t groups = 0;
  for (int j = 0; j < count; ++j) groups += 1ull << FlowTop(ns[perm[j]]);
  const uint64_t cus = static_cast<uint64_t>(ctx->prop.multiProcessorCount);
  return (groups + cus - 1) / cus * 70 <= 75 + (1150u >> (24 - ns[perm[0]]));
}

// Graphs of at most kLdsMaxN vertices, largest first, one workgroup each.
// More graphs than CUs go in one launch per workgroup size, so that small
// graphs do not hold the LDS and threads of large ones; fewer fit in one
// launch, a CU each.
uint64_t LaunchLdsBatch(td_ctx* ctx, hipStream_t st, int count, const LdsGraph* Ls,
                        const uint32_t* cb, int8_t* parents, int32_t* tds) {
  uint64_t launches = 0;
  for (int at = 0; at < count;) {
    const int n = static_cast<int>(Ls[at].n), threads = LdsThreads(n);
    int end = at + 1;
    while (end < count && (count <= ctx->prop.multiProcessorCount ||
                           LdsThreads(static_cast<int>(Ls[end].n)) == threads))
      ++end;
    hipLaunchKernelGGL(DPLdsKernel, dim3(end - at), dim3(threads), LdsBytes(n), st,
                       Ls + at, LdsGraph{}, cb, static_cast<uint32_t*>(nullptr),
                       parents + 64ull * at, tds + at,
                       static_cast<unsigned long long*>(nullptr));
    TD_HIP(hipGetLastError());
    ++launches;
    at = end;
  }
  return launches;
}

void SolveBatch(td_ctx* ctx, int ngraphs, const int32_t* ns,
                const uint64_t* adj_concat, uint8_t* td_out,
                int8_t* parent_concat, int mode, td_dp_stats* stats,
                bool* persistent = nullptr) {
  const auto t0 = std::chrono::steady_clock::now();
  // queries refer to single-graph solves only, and the large-graph pipeline
  // below reuses the single-graph buffers: clear the query state before any
  // of them is touched, so that an error part-way leaves TD_E_STATE behind
  ctx->have_dp = false;
  TD_REQUIRE(ngraphs >= 1 && ns && adj_concat, TD_E_INVALID,
             "empty batch or null pointer");
  TD_REQUIRE(mode >= 0 && mode <= 2, TD_E_INVALID, "mode must be 0, 1 or 2");
  const int lb = ctx->dp.low_bits;
  TD_REQUIRE(lb >= 2 && lb <= 5, TD_E_INVALID, "low_bits must be in [2, 5]");
  std::vector<size_t> row_off(ngraphs + 1, 0);
  for (int i = 0; i < ngraphs; ++i) {
    TD_REQUIRE(ns[i] >= 1 && ns[i] <= kMaxDPN, TD_E_INVALID,
               "batch graphs need n in [1, 32]");
    row_off[i + 1] = row_off[i] + ns[i];
  }
  // graphs above kMaxBatchN vertices go through the single-graph kernels;
  // the rest run largest first, so the persistent queue ends with short work
  std::vector<int> large;
  int first[kMaxBatchN + 2] = {};  // first[n]: graphs of more than n vertices, <= kMaxBatchN
  for (int i = 0; i < ngraphs; ++i) {
    if (ns[i] > kMaxBatchN) large.push_back(i);
    else ++first[ns[i] - 1];
  }
  for (int n = kMaxBatchN - 1; n >= 0; --n) first[n] += first[n + 1];
  const int nsmall = first[0];
  std::vector<int> perm(nsmall);
  std::vector<uint32_t> sizes(nsmall);
  for (int i = 0; i < ngraphs; ++i)
    if (ns[i] <= kMaxBatchN) {
      const int at = first[ns[i]]++;
      perm[at] = i;
      sizes[at] = static_cast<uint32_t>(ns[i]);
    }
  // of these, mode 0 gives the last ones, of at most kLdsMaxN vertices, to
  // DPLdsKernel
  int nmid = nsmall;
  while (mode == 0 && nmid > 0 && ns[perm[nmid - 1]] <= kLdsMaxN) --nmid;
  // and, where that is faster, the others to DPFlowKernel
  int nbig = mode == 0 && FlowPays(ctx, nmid, ns, perm) ? 0 : nmid;
  // page-locked block of the small graphs' records and results; the kernels
  // write the results (and DPLdsKernel reads its graphs) there themselves
  const size_t record = mode == 0 ? sizeof(DPHead) : sizeof(DPGraph);
  const size_t o_lds = record * nsmall;
  const size_t o_flow = o_lds + sizeof(LdsGraph) * (nsmall - nmid);
  const size_t o_par = (o_flow + sizeof(FlowGraph) * (nmid - nbig) + 63) / 64 * 64;
  const size_t o_td = o_par + 64ull * nsmall;
  uint8_t* block = static_cast<uint8_t*>(ctx->Pinned(o_td + 4ull * nsmall + 16, 1));
  int32_t* flow_status = reinterpret_cast<int32_t*>(block + o_td + 4ull * nsmall);
  *flow_status = 0;
  DPGraph* Gs = reinterpret_cast<DPGraph*>(block);   // modes 1 and 2
  DPHead* heads = reinterpret_cast<DPHead*>(block);  // mode 0
  LdsGraph* Ls = reinterpret_cast<LdsGraph*>(block + o_lds);
  FlowGraph* Fs = reinterpret_cast<FlowGraph*>(block + o_flow);
  // every graph is checked, and the small graphs' records are built, on the
  // context's worker threads (about 0.3 us and 0.1 to 1 us a graph) before any GPU work;
  // a failure is reported for the lowest failing graph, as a serial check
  // would
  {
    std::atomic<int> bad{ngraphs};
    auto work = [&](int t, int T) {
      for (int i = t; i < ngraphs; i += T) {
        try {
          ValidateGraph(ns[i], adj_concat + row_off[i], kMaxDPN);
        } catch (const Error&) {
          int cur = bad.load();
          while (i < cur && !bad.compare_exchange_weak(cur, i)) {
          }
        }
      }
      for (int j = t; j < nsmall; j += T) {
        const int i = perm[j];
        const uint64_t* rows = adj_concat + row_off[i];
        if (mode != 0) {
          Gs[j] = MakeGraph(ns[i], rows, WordBits(lb));
        } else if (j < nmid) {
          heads[j] = MakeHead(ns[i], rows, WordBits(lb));
          if (j >= nbig)
            for (int v = 0; v < kFlowMaxN; ++v) Fs[j - nbig].adj[v] = heads[j].adj[v];
        } else {
          LdsGraph& L = Ls[j - nmid];
          L.n = sizes[j];
          for (int v = 0; v < kLdsMaxN; ++v)
            L.adj[v] = v < ns[i] ? static_cast<uint32_t>(rows[v]) : 0u;
        }
      }
    };
    if (ngraphs < 256) {
      work(0, 1);
    } else {
      ctx->workers.Start(static_cast<int>(
          std::min<unsigned>(16u, std::max(1u, std::thread::hardware_concurrency()))));
      ctx->workers.Run(work);
    }
    if (bad.load() < ngraphs) {
      const int i = bad.load();
      ValidateGraph(ns[i], adj_concat + row_off[i], kMaxDPN);  // throws its error
    }
  }
  uint64_t subsets = 0, alg = 0;
  for (int i = 0; i < ngraphs; ++i) {
    subsets += 1ull << ns[i];
    alg += (1ull << (ns[i] - 1)) * static_cast<uint64_t>(ns[i] + 2);
  }
  double level_ms = 0.0, tree_ms = 0.0;
  uint64_t launches = 0, level_kernels = 0;
  SolveLarge(ctx, large, ns, adj_concat, row_off, td_out, parent_concat, &level_ms, &tree_ms,
             &launches, &level_kernels);
  const int total_graphs = ngraphs;
  auto finish = [&] {
    if (!stats) return;
    stats->graphs = static_cast<uint64_t>(total_graphs);
    stats->level_kernels = level_kernels;
    stats->subsets = subsets;
    stats->alg_bytes = alg;
    stats->launches = launches;
    stats->level_ms = level_ms;
    stats->tree_ms = tree_ms;
    stats->total_ms = std::chrono::duration<double, std::milli>(
                          std::chrono::steady_clock::now() - t0)
                          .count();
  };
  if (nsmall == 0) {
    finish();
    return;
  }
  ngraphs = nsmall;
  // bytes used and claimed by a graph of n vertices
  uint64_t used[kMaxBatchN + 1], claims[kMaxBatchN + 1];
  const uint64_t none[kMaxBatchN] = {};
  for (int n = 1; n <= kMaxBatchN; ++n) {
    const DPHead H = MakeHead(n, none, WordBits(lb));
    used[n] = (TableBytes(H) + 255) / 256 * 256;
    claims[n] = (ClaimedBytes(H) + 255) / 256 * 256;
  }
  uint64_t off = 0, room = 0, claimed = 0;
  auto place = [&](int j) {
    (mode == 0 ? heads[j].table : Gs[j].table) = off;
    off += used[sizes[j]];
  };
  for (int j = 0; j < ngraphs; ++j) {
    if (j < nbig) place(j);
    if (j < nmid) room += used[sizes[j]];  // the persistent kernel may have to take any of them
    claimed += claims[sizes[j]];
  }
  uint8_t* arena = static_cast<uint8_t*>(ctx->Buffer("dp.batch_arena", room, claimed));
  void* drec = ctx->Buffer("dp.batch_graphs", record * ngraphs, sizeof(DPGraph) * ngraphs);
  const uint32_t* cb = PascalDevice(ctx);
  uint32_t* dq = static_cast<uint32_t*>(ctx->Buffer("dp.batch_queue", 256));
  int8_t* par = reinterpret_cast<int8_t*>(block + o_par);
  int32_t* tds = reinterpret_cast<int32_t*>(block + o_td);
  // without room for DPFlowKernel's words its graphs take the persistent launch
  FlowCall flow;
  size_t flow_words = 0, flow_planes = 0;
  uint32_t flow_groups = 0;
  uint8_t* fbuf = nullptr;
  if (nbig < nmid) {
    // the first launch holds the largest graphs, but later ones more of them
    size_t most = 0;
    for (int j = nbig; j < nmid;) {
      j += PlanFlow(ctx, nmid - j, &sizes[j], &flow, &flow_words, &flow_planes, &flow_groups);
      most = std::max(most, flow_words);
    }
    fbuf = FlowBuffer(ctx, most);
  }
  if (!fbuf) {
    for (int j = nbig; j < nmid; ++j) place(j);
    nbig = nmid;
  }
  if (nbig > 0)
    TD_HIP(hipMemcpyAsync(drec, block, record * nbig, hipMemcpyHostToDevice, ctx->stream));
  uint64_t small_launches = 0;
  TD_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
  // Beside a persistent launch the graphs in LDS run on a stream of their own,
  // started first: the persistent workgroups take what room they leave, and
  // share the rest out by their queue (4096 graphs of 12..24 vertices: 3.48 ms
  // instead of 3.61 one after the other).
  hipStream_t lds_stream = ctx->stream;
  struct Drain {  // the kernels write to the block: none may outlive an error
    hipStream_t a, b;
    ~Drain() {
      if (a) (void)hipStreamSynchronize(a);
      if (b) (void)hipStreamSynchronize(b);
    }
  } drain{ctx->stream, nullptr};
  if (nmid < nsmall) {
    if (nbig > 0) {
      if (!ctx->side) TD_HIP(hipStreamCreateWithFlags(&ctx->side, hipStreamNonBlocking));
      drain.b = lds_stream = ctx->side;
    }
    small_launches += LaunchLdsBatch(ctx, lds_stream, nsmall - nmid, Ls, cb, par + 64ull * nmid,
                                     tds + nmid);
    if (lds_stream != ctx->stream) TD_HIP(hipEventRecord(ctx->ev[3], lds_stream));
  }
  if (persistent) *persistent = mode == 0 && nbig > 0;
  auto launch_levels = [&] {
    auto launch = [&](auto wb) {
      constexpr int WB = decltype(wb)::value;
      if (mode == 0)
        LaunchPersistent<WB>(ctx, nbig, static_cast<const DPHead*>(drec), cb, arena, dq,
                             &small_launches);
      else
        LaunchBatch<WB>(ctx, mode, nbig, Gs, static_cast<const DPGraph*>(drec), cb, arena,
                        &small_launches);
    };
    switch (WordBits(lb)) {
      case 0: launch(std::integral_constant<int, 0>()); break;
      case 1: launch(std::integral_constant<int, 1>()); break;
      default: launch(std::integral_constant<int, 2>()); break;
    }
  };
  auto launch_trees = [&] {
    if (mode == 0)
      hipLaunchKernelGGL(DPTreeKernel<DPHead>, dim3(nbig), dim3(64), 0, ctx->stream,
                         static_cast<const DPHead*>(drec), cb, arena, par, tds);
    else
      hipLaunchKernelGGL(DPTreeKernel<DPGraph>, dim3(nbig), dim3(64), 0, ctx->stream,
                         static_cast<const DPGraph*>(drec), cb, arena, par, tds);
    TD_HIP(hipGetLastError());
    ++small_launches;
  };
  if (nbig > 0) launch_levels();
  for (int j = nbig; j < nmid;) {
    const int k = PlanFlow(ctx, nmid - j, &sizes[j], &flow, &flow_words, &flow_planes,
                           &flow_groups);
    LaunchFlow(ctx, flow, k, flow_groups, Fs + (j - nbig), cb, arena + off, fbuf, par + 64ull * j,
               tds + j, flow_status, nullptr);
    off += (flow_planes + 255) / 256 * 256;
    small_launches += 2;
    j += k;
  }
  if (lds_stream != ctx->stream) TD_HIP(hipStreamWaitEvent(ctx->stream, ctx->ev[3], 0));
  TD_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
  // mode 0 counts as one level kernel however its graphs were shared out;
  // else the launches
  level_kernels += mode == 0 ? 1 : small_launches;
  if (nbig > 0) launch_trees();
  TD_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
  TD_HIP(hipStreamSynchronize(ctx->stream));
  level_ms += Elapsed(ctx->ev[0], ctx->ev[1]);
  tree_ms += Elapsed(ctx->ev[1], ctx->ev[2]);
  if (*flow_status) {
    // a wait was given up: the persistent kernel takes those graphs instead,
    // as it does without room for the published words; the arena holds them
    nbig = nmid;
    off = 0;
    for (int j = 0; j < nbig; ++j) place(j);
    TD_HIP(hipMemcpyAsync(drec, block, record * nbig, hipMemcpyHostToDevice, ctx->stream));
    TD_HIP(hipEventRecord(ctx->ev[0], ctx->stream));
    launch_levels();
    ++level_kernels;
    TD_HIP(hipEventRecord(ctx->ev[1], ctx->stream));
    launch_trees();
    TD_HIP(hipEventRecord(ctx->ev[2], ctx->stream));
    TD_HIP(hipStreamSynchronize(ctx->stream));
    level_ms += Elapsed(ctx->ev[0], ctx->ev[1]);
    tree_ms += Elapsed(ctx->ev[1], ctx->ev[2]);
  }
  drain.a = drain.b = nullptr;
  launches += small_launches;
  for (int j = 0; j < ngraphs; ++j) {
    const int i = perm[j];
    if (td_out) td_out[i] = static_cast<uint8_t>(tds[j]);
    if (parent_concat) std::memcpy(parent_concat + row_off[i], par + 64ull * j, ns[i]);
  }
  finish();
}

// ---------------------------------------------------------------------------
// autotuner: a sweep over candidate configurations, timed by the level
// kernels' HIP events, with results kept as JSON lines in a cache file
// (one line per candidate, then one "best" line per key and device arch)
// ---------------------------------------------------------------------------
bool JsonInt(const std::string& line, const char* name, int* v) {
  const std::string k = std::string("\"") + name + "\":";
  const size_t p = line.find(k);
  return p != std::string::npos && std::sscanf(line.c_str() + p + k.size(), "%d", v) == 1;
}

bool JsonDouble(const std::string& line, const char* name, double* v) {
  const std::string k = std::string("\"") + name + "\":";
  const size_t p = line.find(k);
  return p != std::string::npos && std::sscanf(line.c_str() + p + k.size(), "%lf", v) == 1;
}

std::string JsonLine(const std::string& key, const DPConfig& c, double ms, bool best,
                     const char* arch) {
  char line[400];
  std::snprintf(line, sizeof(line),
                "{\"key\":\"%s\",\"best\":%s,\"low_bits\":%d,\"tiles_per_lane\":%d,"
                "\"block\":%d,\"class_bits\":%d,\"batch_block\":%d,"
                "\"batch_wg_per_cu\":%d,\"grid_mult\":%d,\"packed\":%d,\"level_ms\":%.4f,"
                "\"arch\":\"%s\"}\n",
                key.c_str(), best ? "true" : "false", c.low_bits, c.tiles_per_lane,
                c.block, c.class_bits, c.batch_block, c.batch_wg_per_cu, c.grid_mult, c.packed,
                ms, arch);
  return line;
}

// The last "best" line of the cache for this key and arch, if any.
bool CacheLookup(const char* path, const std::string& key, const char* arch,
                 DPConfig* cfg, double* ms) {
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
    DPConfig c = *cfg;
    double m = 0;
    (void)JsonInt(line, "grid_mult", &c.grid_mult);  // absent in older caches
    if (c.grid_mult < 1 || c.grid_mult > 64) continue;
    c.packed = 0;  // caches written before packed tiles timed byte tiles
    (void)JsonInt(line, "packed", &c.packed);
    c.packed = c.packed ? 1 : 0;
    if (JsonInt(line, "low_bits", &c.low_bits) && JsonInt(line, "tiles_per_lane", &c.tiles_per_lane) &&
        JsonInt(line, "block", &c.block) && JsonInt(line, "batch_block", &c.batch_block) &&
        JsonInt(line, "batch_wg_per_cu", &c.batch_wg_per_cu) && JsonDouble(line, "level_ms", &m) &&
        JsonInt(line, "class_bits", &c.class_bits) &&
        (c.class_bits == 0 || c.class_bits == 3 || c.class_bits == 4) &&
        c.low_bits >= 2 && c.low_bits <= 5 && c.tiles_per_lane >= 1 && c.tiles_per_lane <= 64 &&
        c.block >= 64 && c.block <= 1024 && c.block % 64 == 0 && c.batch_block >= 64 &&
        c.batch_block <= 1024 && c.batch_block % 64 == 0 && c.batch_wg_per_cu >= 1 &&
        c.batch_wg_per_cu <= 32) {
      *cfg = c;
      *ms = m;
      found = true;
    }
  }
  return found;
}

void ApplyTuned(td_ctx* ctx, const DPConfig& best) {
  const int use_graph = ctx->dp.use_graph;
  ctx->dp = best;
  ctx->dp.use_graph = use_graph;
  ctx->DropDPGraphs();
}

// Times run() (level-kernel ms) under each candidate: one warm-up, then the
// mean of three.  Candidates under which run() launches the same, by
// same(a, b), share the least of their times (a shape timed once can lose to a
// worse one by noise); where all do, the first is timed alone.  Returns the best
// time; *best receives its configuration: the present one where that launches
// the same, else the present one with adopt(&present, winner).
template <typename Run, typename Same, typename Adopt>
double Sweep(td_ctx* ctx, const std::string& key, const std::vector<DPConfig>& cands,
             const char* cache_path, DPConfig* best, Run run, Same same, Adopt adopt) {
  const DPConfig saved = ctx->dp;
  const bool alike = std::all_of(cands.begin(), cands.end(),
                                 [&](const DPConfig& c) { return same(cands.front(), c); });
  std::vector<std::pair<DPConfig, double>> timed;  // by launch
  auto at = [&](const DPConfig& c) {
    return std::find_if(timed.begin(), timed.end(),
                        [&](const auto& t) { return same(t.first, c); });
  };
  try {
    for (const DPConfig& c : cands) {
      auto it = at(c);
      if (alike && it != timed.end()) break;
      ctx->dp = c;
      run();
      double t = 0;
      for (int rep = 0; rep < 3; ++rep) t += run();
      t /= 3;
      if (it == timed.end()) timed.push_back({c, t});
      else it->second = std::min(it->second, t);
    }
  } catch (...) {
    ctx->dp = saved;
    throw;
  }
  double best_ms = 1e30;
  std::string log;
  DPConfig winner = saved;
  for (const DPConfig& c : cands) {
    const double t = at(c)->second;
    log += JsonLine(key, c, t, false, ctx->prop.gcnArchName);
    if (t < best_ms) {
      best_ms = t;
      winner = c;
    }
  }
  ctx->dp = saved;
  *best = saved;
  if (!same(saved, winner)) adopt(best, winner);
  if (cache_path) {
    std::ofstream f(cache_path, std::ios::app);
    f << log << JsonLine(key, *best, best_ms, true, ctx->prop.gcnArchName);
    TD_REQUIRE(f.good(), TD_E_INVALID, "cannot write the autotune cache file");
  }
  return best_ms;
}

}  // namespace

// Once per device, with that device current (td_ctx_create): the address of
// this device's copy of `scratch`, and the Pascal tables written into it.
void NoAllocSetup(td_ctx* ctx) {
  std::lock_guard<std::mutex> lk(g_noalloc_mu);
  TD_REQUIRE(ctx->device >= 0 && ctx->device < kNoAllocMaxDevices, TD_E_INVALID,
             "device index beyond the scratch table");
  if (g_noalloc_ptr[ctx->device]) return;
  // DPLdsKernel takes up to 96 KiB of words
  TD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&DPLdsKernel),
                             hipFuncAttributeMaxDynamicSharedMemorySize,
                             static_cast<int>(LdsBytes(kLdsMaxN))));
  void* p = nullptr;
  TD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
  TD_REQUIRE(p != nullptr, TD_E_HIP, "hipGetSymbolAddress returned no address");
  const std::vector<uint32_t> cb = PascalTable();
  // on the null stream: no context of this device can be capturing yet, and with
  // its hardware queue taken first, fewer contexts get their level streams on
  // one queue (8 graphs of n = 30 in turn on three contexts: 3.58 ms a call,
  // 3.93 with this copy on the context's stream)
  TD_HIP(hipMemcpy(static_cast<uint8_t*>(p) + kNoAllocPascalOff, cb.data(), cb.size() * 4,
                   hipMemcpyHostToDevice));
  g_noalloc_ptr[ctx->device] = static_cast<uint8_t*>(p);
}

}  // namespace tdhip

using namespace tdhip;  // NOLINT

extern "C" {

int td_dp_solve(td_ctx* ctx, int32_t n, const uint64_t* adj,
                uint8_t* treedepth_out, int8_t* parent_out,
                td_dp_stats* stats) {
  return Guard(ctx, [&] {
    SolveOne(ctx, n, adj, treedepth_out, parent_out, stats);
  });
}

int td_dp_solve_noalloc(td_ctx* ctx, int32_t n, const uint64_t* adj,
                        uint8_t* treedepth_out, int8_t* parent_out,
                        td_dp_stats* stats) {
  return Guard(ctx, [&] {
    SolveOneNoAlloc(ctx, n, adj, treedepth_out, parent_out, stats);
  });
}

int td_dp_get_treedepth(td_ctx* ctx, int32_t k, uint64_t code,
                        uint32_t* td_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_dp, TD_E_STATE, "no td_dp_solve result to query");
    TD_REQUIRE(td_out != nullptr, TD_E_INVALID, "td_out is null");
    const int n = ctx->last_n;
    TD_REQUIRE(k >= 0 && k <= n && code < Binom(n, k), TD_E_STATE,
               "subset code out of range");
    const ReadAt r = ReadOffsets(ctx->last_graph, static_cast<uint32_t>(UnrankColex(n, k, code)));
    LdsOut* out = static_cast<LdsOut*>(ctx->Pinned(sizeof(LdsOut)));
    out->clock[3] = 0;
    hipLaunchKernelGGL(DPReadKernel, dim3(1), dim3(64), 0, ctx->stream, r,
                       static_cast<const uint8_t*>(ctx->bufs["dp.arena"].p), &out->td, out->clock);
    TD_HIP(hipGetLastError());
    WaitDone(ctx, out);
    *td_out = static_cast<uint32_t>(out->td);
  });
}

int td_dp_get_level(td_ctx* ctx, int32_t k, uint8_t* out, uint64_t out_len) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_dp, TD_E_STATE, "no td_dp_solve result to query");
    const int n = ctx->last_n;
    TD_REQUIRE(k >= 0 && k <= n, TD_E_STATE, "level out of range");
    const uint64_t count = Binom(n, k);
    TD_REQUIRE(out && out_len >= count, TD_E_INVALID, "output too small");
    // The kernel writes to page-locked memory itself, kPart bytes at a time in
    // two halves by turns: the host copies one while the other is written.
    // Into a buffer in use C(20, 10) subsets take 27 us, C(23, 11) 90, C(26, 13)
    // 452 and C(30, 15) 5620 (102, 109, 675 and 10400 through device memory and
    // a copy to pageable memory).
    constexpr uint64_t kPart = 4u << 20;
    (void)ctx->Buffer("dp.export", 1, count);  // (the byte budget is asked for a read of any size)
    uint8_t* half[2] = {static_cast<uint8_t*>(ctx->Pinned(std::min(count, 2 * kPart)))};
    half[1] = half[0] + kPart;
    const DPHead& head = ctx->last_graph;
    const uint8_t* arena = static_cast<const uint8_t*>(ctx->bufs["dp.arena"].p);
    const uint64_t parts = (count + kPart - 1) / kPart;
    auto bytes = [&](uint64_t p) { return std::min(kPart, count - p * kPart); };
    for (uint64_t p = 0; p <= parts; ++p) {
      if (p < parts) {
        hipLaunchKernelGGL(DPExportLevelKernel, dim3(GridFor(ctx, (bytes(p) + 3) / 4, 256)),
                           dim3(256), 0, ctx->stream, head, PascalDevice(ctx), arena, k,
                           static_cast<uint32_t>(p * kPart), static_cast<uint32_t>(bytes(p)),
                           half[p % 2]);
        TD_HIP(hipGetLastError());
        TD_HIP(hipEventRecord(ctx->ev[p % 2], ctx->stream));
      }
      if (p > 0) {
        TD_HIP(hipEventSynchronize(ctx->ev[(p - 1) % 2]));
        std::memcpy(out + (p - 1) * kPart, half[(p - 1) % 2], bytes(p - 1));
      }
    }
  });
}

int td_dp_get_elimination(td_ctx* ctx, int32_t nverts, int32_t subset_size,
                          uint64_t subset_code, int32_t* order_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_dp, TD_E_STATE, "no td_dp_solve result to query");
    const int n = ctx->last_n;
    TD_REQUIRE(nverts == n, TD_E_INVALID, "nverts differs from the solved graph");
    TD_REQUIRE(subset_size >= 0 && subset_size <= n &&
                   subset_code < Binom(n, subset_size),
               TD_E_STATE, "subset code out of range");
    TD_REQUIRE(order_out != nullptr || subset_size == 0, TD_E_INVALID,
               "order_out is null");
    if (subset_size == 0) return;
    const uint32_t S = static_cast<uint32_t>(UnrankColex(n, subset_size, subset_code));
    int32_t* dorder = static_cast<int32_t*>(ctx->Buffer("dp.walk_order", 64 * 4));
    const DPGraph* dG = LastRecord(ctx);
    const uint8_t* arena = static_cast<const uint8_t*>(ctx->bufs["dp.arena"].p);
    hipLaunchKernelGGL(DPWalkKernel, dim3(1), dim3(64), 0, ctx->stream, dG,
                       PascalDevice(ctx), arena, S, subset_size, dorder);
    TD_HIP(hipGetLastError());
    TD_HIP(hipMemcpyAsync(order_out, dorder, 4 * subset_size,
                          hipMemcpyDeviceToHost, ctx->stream));
    TD_HIP(hipStreamSynchronize(ctx->stream));
  });
}

int td_dp_solve_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                      const uint64_t* adj_concat, uint8_t* treedepth_out,
                      int8_t* parent_concat, int32_t mode,
                      td_dp_stats* stats) {
  return Guard(ctx, [&] {
    SolveBatch(ctx, ngraphs, n, adj_concat, treedepth_out, parent_concat, mode,
               stats);
  });
}

int td_dp_autotune(td_ctx* ctx, int32_t n, const char* cache_path,
                   double* best_ms_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(n >= 8 && n <= kMaxDPN, TD_E_INVALID, "autotune n in [8, 32]");
    const std::string key = "single n=" + std::to_string(n);
    // graphs of at most kFlowMaxN vertices take one launch that reads none of
    // the shape: it is timed, and the context stays as it is
    const bool shaped = n > kFlowMaxN;
    DPConfig best = ctx->dp;
    double best_ms = 0;
    if (!CacheLookup(cache_path, key, ctx->prop.gcnArchName, &best, &best_ms)) {
      // seeded G(n, 0.25) (SplitMix64)
      std::vector<uint64_t> adj(n, 0);
      uint64_t s = 0x9E3779B97F4A7C15ull * (n + 1);
      auto next = [&]() {
        s += 0x9E3779B97F4A7C15ull;
        uint64_t z = s;
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
      };
      for (int i = 0; i < n; ++i)
        for (int j = i + 1; j < n; ++j)
          if ((next() >> 11) * (1.0 / (1ull << 53)) < 0.25) {
            adj[i] |= 1ull << j;
            adj[j] |= 1ull << i;
          }
      std::vector<DPConfig> cands;
      // (tiles per lane, grid multiple): one tile per lane at three grid
      // sizes, and two consecutive tiles per lane
      const int shapes[4][2] = {{1, 2}, {1, 4}, {1, 8}, {2, 4}};
      // (class_bits and packed no longer change a launch: the candidates are
      // still those that existing caches and their readers know, but these two,
      // which decide the bytes claimed, stay as the context has them)
      for (int cbits : {0, 4})
        for (int lb : {3, 4, 5})
          for (int pk : {0, 1}) {
            if (pk && (cbits == 0 || lb < 4)) continue;
            for (const auto& rg : shapes)
              for (int blk : {128, 256, 512}) {
                DPConfig c = ctx->dp;
                c.class_bits = cbits;
                c.low_bits = lb;
                c.packed = pk;
                c.tiles_per_lane = rg[0];
                c.grid_mult = rg[1];
                c.block = blk;
                c.use_graph = 0;
                cands.push_back(c);
              }
          }
      uint8_t td;
      int8_t par[64];
      // graphs above the batch kernel's 26 vertices also run through these
      // kernels in batch calls, where their tree kernel is hidden behind the
      // next graph's levels: time the levels alone.  Smaller graphs use this
      // shape only in single solves, which wait for the tree as well.
      best_ms = Sweep(ctx, key, cands, cache_path, &best, [&] {
        td_dp_stats st{};
        SolveOne(ctx, n, adj.data(), &td, par, &st);
        return n > kMaxBatchN ? st.level_ms : st.level_ms + st.tree_ms;
      }, [&](const DPConfig& a, const DPConfig& b) {
        return !shaped || (SingleWordBits(n, a.low_bits) == SingleWordBits(n, b.low_bits) &&
                           a.tiles_per_lane == b.tiles_per_lane && a.block == b.block &&
                           a.grid_mult == b.grid_mult);
      }, [&](DPConfig* to, const DPConfig& c) {
        if (SingleWordBits(n, to->low_bits) != SingleWordBits(n, c.low_bits))
          to->low_bits = c.low_bits;
        to->tiles_per_lane = c.tiles_per_lane;
        to->block = c.block;
        to->grid_mult = c.grid_mult;
      });
    }
    if (shaped) ApplyTuned(ctx, best);
    if (best_ms_out) *best_ms_out = best_ms;
  });
}

int td_dp_autotune_batch(td_ctx* ctx, int32_t ngraphs, const int32_t* n,
                         const uint64_t* adj_concat, const char* cache_path,
                         double* best_ms_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ngraphs >= 1 && n && adj_concat, TD_E_INVALID,
               "empty batch or null pointer");
    int nmax = 0;
    uint64_t nsum = 0;
    for (int i = 0; i < ngraphs; ++i) {
      TD_REQUIRE(n[i] >= 1 && n[i] <= kMaxBatchN, TD_E_INVALID,
                 "batch graphs need n in [1, 26]");
      nmax = std::max(nmax, static_cast<int>(n[i]));
      nsum += static_cast<uint64_t>(n[i]);
    }
    const std::string key = "batch graphs=" + std::to_string(ngraphs) +
                            " nmax=" + std::to_string(nmax) +
                            " nsum=" + std::to_string(nsum);
    DPConfig best = ctx->dp;
    double best_ms = 0;
    if (!CacheLookup(cache_path, key, ctx->prop.gcnArchName, &best, &best_ms)) {
      std::vector<DPConfig> cands;
      for (int lb : {4, 5})
        for (int r : {1, 2, 4})
          for (int blk : {256, 512, 1024})
            for (int wg : {1, 2, 4, 8}) {
              if (blk * wg > 4096) continue;  // at most 64 waves per CU in flight
              DPConfig c = ctx->dp;
              c.low_bits = lb;
              c.tiles_per_lane = r;
              c.batch_block = blk;
              c.batch_wg_per_cu = wg;
              c.use_graph = 0;
              cands.push_back(c);
            }
      // a batch without a persistent launch reads none of the shape
      bool persistent = false;
      SolveBatch(ctx, ngraphs, n, adj_concat, nullptr, nullptr, 0, nullptr, &persistent);
      best_ms = Sweep(ctx, key, cands, cache_path, &best, [&] {
        td_dp_stats st{};
        SolveBatch(ctx, ngraphs, n, adj_concat, nullptr, nullptr, 0, &st);
        return st.level_ms;
      }, [&](const DPConfig& a, const DPConfig& b) {
        return !persistent || (WordBits(a.low_bits) == WordBits(b.low_bits) &&
                               a.tiles_per_lane == b.tiles_per_lane &&
                               a.batch_block == b.batch_block &&
                               a.batch_wg_per_cu == b.batch_wg_per_cu);
      }, [&](DPConfig* to, const DPConfig& c) {
        to->low_bits = c.low_bits;
        to->tiles_per_lane = c.tiles_per_lane;
        to->batch_block = c.batch_block;
        to->batch_wg_per_cu = c.batch_wg_per_cu;
      });
    }
    ApplyTuned(ctx, best);
    if (best_ms_out) *best_ms_out = best_ms;
  });
}

}  // extern "C"
