// Runs the LDS kernel of the subset DP (gisbdw_amd/csrc/dplds.hpp) on the CPU,
// a coroutine per thread, waves in ascending order: wave 0 always gets as far
// as it can before any other wave moves.  At the moment the kernel publishes
// "done", the whole of a graph's three planes must have been written, and every
// thread must have passed a release fence after its last plane word.
// usage: lds_publish_check n.  Prints "ok" and the words found in the planes.
#include <ucontext.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <vector>

// ---- the kernel language, for the CPU --------------------------------------
#define __device__
#define __global__
#define __shared__
#define __forceinline__ inline
#define __launch_bounds__(...)
#define __restrict__
#define __HIP_MEMORY_SCOPE_AGENT 0
#define __HIP_MEMORY_SCOPE_SYSTEM 0

struct Dim {
  unsigned x = 0;
};
static Dim threadIdx, blockIdx, blockDim;

enum State { kRun, kBallot, kBarrier, kDone };
struct Lane {
  ucontext_t at;
  std::vector<char> stack;
  State state = kRun;
  bool vote = false, fenced = false;
  unsigned long long ballot = 0;
};
static std::vector<Lane> lanes;
static ucontext_t scheduler;
static bool published = false;
static void Published();

static Lane& Me() { return lanes[threadIdx.x]; }
static void Wait(State s) {
  Lane& me = Me();
  me.state = s;
  swapcontext(&me.at, &scheduler);
}
static void __syncthreads() { Wait(kBarrier); }
static unsigned long long __ballot(bool p) {
  Me().vote = p;
  Wait(kBallot);
  return Me().ballot;
}
static unsigned long long wall_clock64() { return 1; }
static void __threadfence_system() { Me().fenced = true; }
static void Fence() { Me().fenced = true; }
#define __builtin_amdgcn_fence(order, scope) Fence()
#define __builtin_amdgcn_s_sleep(x) (void)0
static unsigned atomicAdd(uint32_t* p, unsigned v) { return *p += v, *p - v; }
template <typename T>
static T Load(const T* p) {
  return *p;
}
static void Store(unsigned long long* p, unsigned long long v) {
  *p = v;
  if (v == 1) Published();
}
#define __hip_atomic_load(p, order, scope) Load(p)
#define __hip_atomic_store(p, v, order, scope) Store(p, v)

// ---- what the kernel takes from the rest of the library --------------------
namespace tdhip {
namespace {
constexpr int kCbStride = 33, kTailBits = 16, kCbOffs = 32 * kCbStride;
constexpr int kTailWord = (kCbOffs + kTailBits + 1 + 31) / 32 * 32;
struct AnyLane {
  bool operator()(uint32_t x) const { return __ballot(x != 0u) != 0ull; }
};
// the decomposition is not what is looked at; its ballots keep a wave together
template <typename Differ>
int DecomposeWave(uint32_t, uint32_t, int* depth, Differ) {
  *depth = __ballot(true) ? 1 : 0;
  return -1;
}
uint32_t s[64 * 1024];
}  // namespace
}  // namespace tdhip
#include "../gisbdw_amd/csrc/dplds.hpp"

using namespace tdhip;

static std::vector<uint32_t> table, cb;
static LdsGraph graph;
static int words = 0, early = 0, unfenced = 0;
constexpr uint32_t kUnset = 0xDEADBEEFu;

static void Published() {
  if (published) return;
  published = true;
  const uint32_t* w = s + kLdsHead;
  for (size_t i = 0; i < table.size(); ++i) {
    if (table[i] != w[i]) ++early;
    else ++words;
  }
  for (size_t t = 64; t < lanes.size(); ++t) unfenced += lanes[t].fenced ? 0 : 1;
}

static void Entry() {
  static int8_t parent[64];
  static int32_t td;
  static unsigned long long clock[4];
  DPLdsKernel(nullptr, graph, cb.data(), table.data(), parent, &td, clock);
  Wait(kDone);
}

int main(int argc, char** argv) {
  const int n = argc > 1 ? std::atoi(argv[1]) : 14, threads = LdsThreads(n);
  std::mt19937 rng(n);
  graph = LdsGraph{};
  graph.n = n;
  for (int i = 0; i < n; ++i)
    for (int j = i + 1; j < n; ++j)
      if (rng() % 4 == 0) {
        graph.adj[i] |= 1u << j;
        graph.adj[j] |= 1u << i;
      }
  // binomials, first entries and the 16-bit subsets by size
  cb.assign(kTailWord + (1 << kTailBits) / 2, 0);
  for (int x = 0; x < 32; ++x)
    for (int j = 0; j < kCbStride; ++j)
      cb[x * kCbStride + j] = j == 0 ? 1u
                              : x == 0 ? 0u
                                       : cb[(x - 1) * kCbStride + j - 1] + cb[(x - 1) * kCbStride + j];
  uint16_t* tail = reinterpret_cast<uint16_t*>(cb.data() + kTailWord);
  uint32_t off = 0;
  for (int k = 0; k <= kTailBits; ++k) {
    cb[kCbOffs + k] = off;
    for (uint32_t m = 0; m < (1u << kTailBits); ++m)
      if (__builtin_popcount(m) == k) tail[off++] = static_cast<uint16_t>(m);
  }
  table.assign(3u << (n - 5), kUnset);
  for (uint32_t& x : s) x = kUnset;
  blockDim.x = threads;
  lanes.resize(threads);
  for (int t = 0; t < threads; ++t) {
    Lane& l = lanes[t];
    l.stack.resize(64 * 1024);
    getcontext(&l.at);
    l.at.uc_stack.ss_sp = l.stack.data();
    l.at.uc_stack.ss_size = l.stack.size();
    l.at.uc_link = nullptr;
    makecontext(&l.at, Entry, 0);
  }
  for (bool going = true; going;) {
    for (int w = 0; w < threads; w += 64) {  // a wave as far as it can go
      for (bool moved = true; moved;) {
        moved = false;
        for (int t = w; t < w + 64; ++t)
          if (lanes[t].state == kRun) {
            threadIdx.x = t;
            swapcontext(&scheduler, &lanes[t].at);
            moved = true;
          }
        unsigned long long votes = 0;
        for (int t = w; t < w + 64; ++t)
          if (lanes[t].state == kBallot && lanes[t].vote) votes |= 1ull << (t - w);
        for (int t = w; t < w + 64; ++t)
          if (lanes[t].state == kBallot) {
            lanes[t].ballot = votes;
            lanes[t].state = kRun;
            moved = true;
          }
      }
    }
    going = false;  // every wave waits or has ended: the barrier opens
    for (Lane& l : lanes)
      if (l.state == kBarrier) {
        l.state = kRun;
        going = true;
      }
  }
  if (!published || early || unfenced) {
    std::printf("n = %d: published %d, plane words missing at that time %d, threads without a "
                "fence %d\n", n, published, early, unfenced);
    return 1;
  }
  std::printf("ok %d\n", words);
  return 0;
}
