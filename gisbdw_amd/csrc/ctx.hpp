// ctx.hpp -- the td_ctx object behind include/tdhip.h and shared helpers.
#pragma once
#include <hip/hip_runtime.h>

#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <exception>
#include <functional>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "../../include/tdhip.h"

namespace tdhip {

// Error reporting: every entry point returns a td_status and leaves a
// message in ctx->err.  HIP failures are turned into TD_E_HIP here.
struct Error {
  int code;
  std::string msg;
};

#define TD_HIP(call)                                                      \
  do {                                                                    \
    hipError_t e_ = (call);                                               \
    if (e_ != hipSuccess)                                                 \
      throw ::tdhip::Error{TD_E_HIP, std::string(#call) + ": " +          \
                                         hipGetErrorString(e_)};          \
  } while (0)

#define TD_REQUIRE(cond, code, msg)                  \
  do {                                               \
    if (!(cond)) throw ::tdhip::Error{(code), (msg)}; \
  } while (0)

// Per-graph DP descriptor, one per graph, read by the kernels with scalar
// loads.  Vertices 0..4 are the bits of a word of 32 subsets, vertices
// 5..lb-1 pick a word of a tile, and vertices lb..n-1 are the "high" vertices
// whose subset H selects the tile.  The head is all that the batch's
// persistent kernel and the tree kernel read.
struct DPHead {
  uint32_t n;        // vertices
  uint32_t nh;       // high vertices, max(n - lb, 0)
  uint32_t lb;       // 5 + log2(words per tile): 5, 6 or 7
  uint32_t direct;   // planes indexed by S >> 5 itself, 2^max(n-5, 0) words each
  uint64_t table;    // byte offset of this graph's tables in the arena
  uint32_t lvl[34];  // tile offset of high level h; lvl[nh+1] = 2^nh
  uint32_t adj[32];  // adjacency rows
};
// The head and the level kernels' tables: three consecutive arrays, which the
// kernels copy to LDS as one block.  Vertices above 4 come in 7-bit chunks,
// chunk c from vertex 5 + 7 c on.
struct DPGraph : DPHead {
  uint32_t nbh[512];  // neighbours of a set of them: nbh[128 c + chunk]
  uint32_t isoh[512]; // by a set X of them: the L that give every x in X a
                      // neighbour
  uint32_t isol[32];  // by set Y of vertices 0..4: the L in which every
                      // y in Y n L has a neighbour in L
};
constexpr int kTabNbh = 0, kTabIsoH = 512, kTabIsoL = 1024, kTabWords = 1056;
static_assert(sizeof(DPGraph) == sizeof(DPHead) + 4 * kTabWords,
              "nbh, isoh and isol must follow each other and the head");

// Whether row v of a graph of n vertices is one that ValidateGraph takes: no
// vertex n or above, no self loop, and (rows[u] for every neighbour u < 64)
// symmetric.  A row v >= n has to be empty.
__device__ __forceinline__ bool RowFine(const uint64_t* rows, uint64_t row, int n, int v) {
  if (v >= n) return row == 0ull;
  if ((n < 64 && row >> n) || (row >> v & 1ull)) return false;
  bool ok = true;
  for (uint64_t m = row; m; m &= m - 1) ok = ok && (rows[__builtin_ctzll(m)] >> v & 1ull);
  return ok;
}

// DP launch configuration (autotuned).
struct DPConfig {
  int low_bits = 4;        // 2..5: tiles of 1, 1, 2 or 4 words
  int tiles_per_lane = 1;  // consecutive tiles per lane (Gosper steps)
  int block = 512;         // threads per workgroup
  int batch_wg_per_cu = 4; // persistent batch kernel: workgroups per CU
  int batch_block = 1024;  // persistent batch kernel: threads per workgroup
  int use_graph = 1;       // capture the level sequence into a hipGraph
  int xcd_remap = 0;       // accepted, without effect (slices are always on)
  int class_bits = 0;      // accepted; with packed, only the bytes claimed
  int class_min_nh = 16;
  int grid_mult = 4;       // level launch: at most grid_mult x the resident workgroups
  int packed = 0;          // with class_bits and low_bits >= 4: claim 17/32 bytes a subset
  int flow_spin = 1 << 17; // reads of one published word before DPFlowKernel gives up
  int streams = 2;         // batch calls: large graphs' level sequences in flight (1-3)
};

struct DeviceBuffer {
  void* p = nullptr;
  size_t bytes = 0;
  size_t claimed = 0;  // of the byte budget, at least bytes
};

}  // namespace tdhip

namespace tdhip {
// Host worker threads kept for the context's lifetime: Run(f) calls f(t, T)
// on T threads (the caller is thread 0) and returns when all are done.
// Starting threads costs about 50 us each, more than the per-call work
// they share out.
class WorkerPool {
 public:
  ~WorkerPool() {
    {
      std::lock_guard<std::mutex> lk(mu_);
      stop_ = true;
      ++gen_;
    }
    cv_.notify_all();
    for (auto& th : threads_) th.join();
  }
  int Size() const { return static_cast<int>(threads_.size()) + 1; }
  void Start(int n) {
    if (!threads_.empty() || n <= 1) return;
    for (int t = 1; t < n; ++t) threads_.emplace_back([this, t] { Loop(t); });
  }
  // f must not throw on the worker threads; an exception on the caller's
  // share is rethrown after every worker has finished.
  void Run(const std::function<void(int, int)>& f) {
    const int T = Size();
    {
      std::lock_guard<std::mutex> lk(mu_);
      job_ = &f;
      pending_ = T - 1;
      ++gen_;
    }
    cv_.notify_all();
    std::exception_ptr err;
    try {
      f(0, T);
    } catch (...) {
      err = std::current_exception();
    }
    {
      std::unique_lock<std::mutex> lk(mu_);
      done_.wait(lk, [this] { return pending_ == 0; });
      job_ = nullptr;
    }
    if (err) std::rethrow_exception(err);
  }

 private:
  void Loop(int t) {
    uint64_t seen = 0;
    for (;;) {
      const std::function<void(int, int)>* job;
      {
        std::unique_lock<std::mutex> lk(mu_);
        cv_.wait(lk, [&] { return gen_ != seen; });
        seen = gen_;
        if (stop_) return;
        job = job_;
      }
      try {
        (*job)(t, Size());
      } catch (...) {
        // jobs catch their own errors; nothing may leave a worker thread
      }
      {
        std::lock_guard<std::mutex> lk(mu_);
        if (--pending_ == 0) done_.notify_one();
      }
    }
  }
  std::vector<std::thread> threads_;
  std::mutex mu_;
  std::condition_variable cv_, done_;
  const std::function<void(int, int)>* job_ = nullptr;
  uint64_t gen_ = 0;
  int pending_ = 0;
  bool stop_ = false;
};
}  // namespace tdhip

struct td_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  uint64_t budget = 0;
  uint64_t allocated = 0;  // bytes claimed of the budget
  std::string err;
  hipDeviceProp_t prop{};
  double clock_khz = 1e5;  // rate of the device's wall clock
  tdhip::DPConfig dp;
  std::map<std::string, int64_t> params;

  // named device buffers (grown on demand, freed with the context); a buffer
  // takes `claim` bytes of the budget if that is more than its own
  std::map<std::string, tdhip::DeviceBuffer> bufs;
  void* Buffer(const std::string& name, size_t bytes, size_t claim = 0);
  void Release(const std::string& name);
  size_t Held(const std::string& name) const;  // bytes that a buffer claims, 0 if there is none
  // page-locked host staging for the per-call copies, two independent
  // buffers (grown on demand): slot 0 for single-graph staging, slot 1 for the
  // batch records and results, which live across the large-graph pipeline.
  // They are reused because no call returns while the device may still access
  // them: it has synchronized, or (a single solve of at most 24 vertices) read
  // the flag that the last kernel writes after everything else
  void* pinned[2] = {nullptr, nullptr};
  size_t pinned_bytes[2] = {0, 0};
  void* Pinned(size_t bytes, int slot = 0);
  // waits for everything this context has launched
  void Settle();
  // hipMemcpy on the context's stream: one on the null stream fails while some
  // other thread captures a launch sequence, and ends that capture
  void Copy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind);

  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  tdhip::WorkerPool workers;  // host threads for per-graph setup work
  // streams and events of the pipeline of large graphs in a batch call
  // (created on first use): consecutive graphs' levels run on `stream` and
  // the dp.streams - 1 streams `lvl` in turn, every graph's decomposition on
  // `side`; events: level start, level end, tree end and first part of the
  // levels done per slot (up to 3 slots), and one time origin
  hipStream_t side = nullptr;
  hipStream_t lvl[2] = {nullptr, nullptr};
  hipEvent_t pev[13] = {};

  // branch-and-bound memo tables: entries are tagged per graph serial
  void* bnb_memo_ptr = nullptr;
  size_t bnb_memo_bytes = 0;
  uint32_t bnb_tag = 0;
  struct BnBDetail {
    uint32_t heur;
    int32_t lb;
    uint64_t nodes;
    int32_t last_k;       // last k the descent tried (-1: none)
    uint64_t last_nodes;  // nodes spent on that k
  };
  std::vector<BnBDetail> bnb_last;  // per graph, last td_bnb_* call
  // captured queue reset + search launch, and the launch shape and buffers
  // baked into it
  hipGraphExec_t bnb_graph = nullptr;
  std::vector<uint64_t> bnb_graph_key;

  // state of the last td_dp_solve (for the queries)
  int last_n = 0;
  bool have_dp = false;
  // DPFlowKernel's buffer: the words published in it carry the call's tag, and
  // its ticket counter has seen flow_tickets workgroups (see FlowBuffer)
  uint32_t flow_tag = 0, flow_tickets = 0;
  int unsynced = 0;  // single solves since their stream was last synchronized
  bool record_up = false;  // its record is in "dp.graph" (see LastRecord)
  tdhip::DPGraph last_graph{};

  // state of the last td_bottom_up (for its queries): vertex count, levels
  // run, and the offset of each level in the history arrays
  int bu_n = 0, bu_iters = 0;
  bool have_bu = false;
  std::vector<uint64_t> bu_off;

  // cached hipGraph per (n, config) for the single-graph level sequence
  struct GraphKey {
    int n, lb, r, block;
    bool operator<(const GraphKey& o) const {
      if (n != o.n) return n < o.n;
      if (lb != o.lb) return lb < o.lb;
      if (r != o.r) return r < o.r;
      return block < o.block;
    }
  };
  std::map<GraphKey, hipGraphExec_t> dp_graphs;
  // buffer addresses baked into each captured graph (arena, descriptor)
  std::map<GraphKey, std::pair<const void*, const void*>> dp_graph_ptrs;
  void DropDPGraphs();
};

namespace tdhip {
// binomial table C(i, j), i, j <= 64, host side
uint64_t Binom(int n, int k);
// colex unrank on the host (n vertices, k-subset)
uint64_t UnrankColex(int n, int k, uint64_t code);
uint64_t RankColex(uint64_t mask);
// The body of an entry point: f() with the context's device current, its errors
// as a td_status and a message.  An error can leave f() with kernels in flight
// that read and write the page-locked staging: they end before the caller has
// the context back, whose next call uses that memory again.
template <typename F>
int Guard(td_ctx* ctx, F&& f) {
  if (!ctx) return TD_E_INVALID;
  int code = TD_E_INVALID;
  try {
    TD_HIP(hipSetDevice(ctx->device));
    f();
    ctx->err.clear();
    return TD_OK;
  } catch (const Error& e) {
    ctx->err = e.msg;
    code = e.code;
  } catch (const std::exception& e) {
    ctx->err = e.what();
  }
  ctx->Settle();
  return code;
}
// validate a graph; returns the adjacency as 32-bit rows when n <= 32
void ValidateGraph(int n, const uint64_t* adj, int max_n);
// Runs call(), a td_dp_solve_batch of graphs of at most 26 vertices, without
// ending the last single solve's queries: such a batch has buffers of its own.
template <typename Call>
int KeepDP(td_ctx* ctx, Call&& call) {
  const bool had = ctx->have_dp;
  const int rc = call();
  ctx->have_dp = had;
  return rc;
}
// device address of td_dp_solve_noalloc's fixed scratch array for the
// context's device (once per device; the device must be current)
void NoAllocSetup(td_ctx* ctx);
}  // namespace tdhip
