// ctx.hip -- context lifetime, device buffers, parameters and host-side
// combinatorics shared by the DP and the branch-and-bound.
#include <algorithm>
#include <cstring>

#include "ctx.hpp"

namespace tdhip {

uint64_t Binom(int n, int k) {
  static uint64_t table[65][65];
  static bool init = false;
  if (!init) {
    for (int i = 0; i <= 64; ++i) {
      table[i][0] = 1;
      for (int j = 1; j <= 64; ++j)
        table[i][j] = (i == 0) ? 0 : table[i - 1][j - 1] + table[i - 1][j];
    }
    init = true;
  }
  if (n < 0 || k < 0 || k > n) return 0;
  return table[n][k];
}

// colex: rank(S) = sum_i C(s_i, i+1) over the sorted elements s_0 < s_1 < ...
uint64_t RankColex(uint64_t mask) {
  uint64_t r = 0;
  int i = 0;
  while (mask) {
    int v = __builtin_ctzll(mask);
    mask &= mask - 1;
    r += Binom(v, ++i);
  }
  return r;
}

uint64_t UnrankColex(int n, int k, uint64_t code) {
  uint64_t m = 0;
  for (int v = n - 1; v >= 0 && k > 0; --v) {
    uint64_t c = Binom(v, k);
    if (code >= c) {
      m |= 1ull << v;
      code -= c;
      --k;
    }
  }
  return m;
}

void ValidateGraph(int n, const uint64_t* adj, int max_n) {
  TD_REQUIRE(n >= 1 && n <= max_n, TD_E_INVALID,
             "n must be in [1, " + std::to_string(max_n) + "]");
  TD_REQUIRE(adj != nullptr, TD_E_INVALID, "adjacency is null");
  uint64_t full = n >= 64 ? ~0ull : ((1ull << n) - 1);
  for (int v = 0; v < n; ++v) {
    TD_REQUIRE(!(adj[v] & ~full), TD_E_INVALID,
               "row " + std::to_string(v) + " names a vertex >= n");
    TD_REQUIRE(!(adj[v] >> v & 1), TD_E_INVALID,
               "self loop at vertex " + std::to_string(v));
    for (uint64_t m = adj[v]; m; m &= m - 1) {
      int u = __builtin_ctzll(m);
      TD_REQUIRE(adj[u] >> v & 1, TD_E_INVALID,
                 "asymmetric edge " + std::to_string(v) + "-" +
                     std::to_string(u));
    }
  }
}

}  // namespace tdhip

void td_ctx::Settle() {
  (void)hipStreamSynchronize(stream);
  if (side) (void)hipStreamSynchronize(side);
  for (hipStream_t q : lvl)
    if (q) (void)hipStreamSynchronize(q);
}

void td_ctx::Copy(void* dst, const void* src, size_t bytes, hipMemcpyKind kind) {
  TD_HIP(hipMemcpyAsync(dst, src, bytes, kind, stream));
  TD_HIP(hipStreamSynchronize(stream));
}

void* td_ctx::Pinned(size_t bytes, int slot) {
  void*& p = pinned[slot];
  if (p && pinned_bytes[slot] >= bytes) return p;
  if (p) {
    TD_HIP(hipStreamSynchronize(stream));
    if (side) TD_HIP(hipStreamSynchronize(side));
    TD_HIP(hipHostFree(p));
    p = nullptr;
    pinned_bytes[slot] = 0;
  }
  TD_HIP(hipHostMalloc(&p, bytes, hipHostMallocDefault));
  pinned_bytes[slot] = bytes;
  return p;
}

void* td_ctx::Buffer(const std::string& name, size_t bytes, size_t claim) {
  claim = std::max(claim, bytes);
  auto& b = bufs[name];
  if (b.bytes >= bytes && b.claimed >= claim && b.p) return b.p;
  if (b.p) {
    Settle();
    TD_HIP(hipFree(b.p));
    allocated -= b.claimed;
    b = {};
  }
  // DPFlowKernel's buffer is a help, not a need: it makes room
  if (budget && allocated + claim > budget && name != "dp.flow") Release("dp.flow");
  if (budget && allocated + claim > budget)
    throw tdhip::Error{TD_E_NOMEM, "buffer '" + name + "' of " +
                                       std::to_string(claim) +
                                       " bytes exceeds the context budget"};
  hipError_t e = hipMalloc(&b.p, bytes ? bytes : 1);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    b.p = nullptr;
    throw tdhip::Error{TD_E_NOMEM, "hipMalloc of " + std::to_string(bytes) +
                                       " bytes for '" + name +
                                       "' failed: " + hipGetErrorString(e)};
  }
  b.bytes = bytes;
  b.claimed = claim;
  allocated += claim;
  return b.p;
}

size_t td_ctx::Held(const std::string& name) const {
  const auto it = bufs.find(name);
  return it != bufs.end() && it->second.p ? it->second.claimed : 0;
}

void td_ctx::DropDPGraphs() {
  for (auto& kv : dp_graphs) (void)hipGraphExecDestroy(kv.second);
  dp_graphs.clear();
  dp_graph_ptrs.clear();
}

void td_ctx::Release(const std::string& name) {
  auto it = bufs.find(name);
  if (it == bufs.end()) return;
  if (it->second.p) {
    Settle();
    (void)hipFree(it->second.p);
    allocated -= it->second.claimed;
  }
  bufs.erase(it);
}

namespace {
// A plain streaming copy, 16 bytes per lane per step: the reference point for
// HBM bandwidth and for scaling rocprof's FETCH_SIZE / WRITE_SIZE counters.
__global__ __launch_bounds__(256) void CopyKernel(const uint4* __restrict__ src,
                                                  uint4* __restrict__ dst, size_t n) {
  for (size_t i = blockIdx.x * static_cast<size_t>(blockDim.x) + threadIdx.x; i < n;
       i += static_cast<size_t>(gridDim.x) * blockDim.x)
    dst[i] = src[i];
}
}  // namespace

extern "C" {

int td_ctx_copy_bench(td_ctx* c, uint64_t bytes, int32_t reps, double* gbps_out) {
  if (!c || bytes < 16 || reps < 1) return TD_E_INVALID;
  try {
    TD_HIP(hipSetDevice(c->device));
    bytes &= ~15ull;
    void* a = c->Buffer("copy.src", bytes);
    void* b = c->Buffer("copy.dst", bytes);
    const size_t n = bytes / 16;
    const int grid = c->prop.multiProcessorCount * 8;
    hipLaunchKernelGGL(CopyKernel, dim3(grid), dim3(256), 0, c->stream,
                       static_cast<const uint4*>(a), static_cast<uint4*>(b), n);
    TD_HIP(hipEventRecord(c->ev[0], c->stream));
    for (int r = 0; r < reps; ++r)
      hipLaunchKernelGGL(CopyKernel, dim3(grid), dim3(256), 0, c->stream,
                         static_cast<const uint4*>(a), static_cast<uint4*>(b), n);
    TD_HIP(hipEventRecord(c->ev[1], c->stream));
    TD_HIP(hipEventSynchronize(c->ev[1]));
    float ms = 0.f;
    TD_HIP(hipEventElapsedTime(&ms, c->ev[0], c->ev[1]));
    if (gbps_out) *gbps_out = 2.0 * bytes * reps / (ms * 1e-3) / 1e9;
    c->Release("copy.src");
    c->Release("copy.dst");
    c->err.clear();
    return TD_OK;
  } catch (const tdhip::Error& e) {
    c->err = e.msg;
    return e.code;
  }
}

int td_ctx_create(td_ctx** out, int device, uint64_t mem_budget_bytes) {
  if (!out) return TD_E_INVALID;
  *out = nullptr;
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || count <= 0) {
    (void)hipGetLastError();
    return TD_E_HIP;
  }
  if (device < 0 || device >= count) return TD_E_INVALID;
  td_ctx* c = new td_ctx();
  c->device = device;
  c->budget = mem_budget_bytes;
  if (hipSetDevice(device) != hipSuccess ||
      hipGetDeviceProperties(&c->prop, device) != hipSuccess ||
      hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess) {
    delete c;
    return TD_E_HIP;
  }
  for (auto& e : c->ev)
    if (hipEventCreate(&e) != hipSuccess) {
      td_ctx_destroy(c);
      return TD_E_HIP;
    }
  int khz = 0;
  if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, device) == hipSuccess && khz > 0)
    c->clock_khz = khz;
  try {
    tdhip::NoAllocSetup(c);
  } catch (const tdhip::Error&) {
    (void)hipGetLastError();
    td_ctx_destroy(c);
    return TD_E_HIP;
  }
  *out = c;
  return TD_OK;
}

void td_ctx_destroy(td_ctx* c) {
  if (!c) return;
  (void)hipSetDevice(c->device);
  if (c->stream) c->Settle();
  c->DropDPGraphs();
  if (c->bnb_graph) (void)hipGraphExecDestroy(c->bnb_graph);
  for (auto& kv : c->bufs)
    if (kv.second.p) (void)hipFree(kv.second.p);
  for (void* p : c->pinned)
    if (p) (void)hipHostFree(p);
  for (auto& e : c->ev)
    if (e) (void)hipEventDestroy(e);
  for (auto& e : c->pev)
    if (e) (void)hipEventDestroy(e);
  if (c->side) (void)hipStreamDestroy(c->side);
  for (hipStream_t q : c->lvl)
    if (q) (void)hipStreamDestroy(q);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

const char* td_last_error(const td_ctx* c) {
  return c ? c->err.c_str() : "null context";
}

int td_ctx_set_param(td_ctx* c, const char* key, int64_t v) {
  if (!c || !key) return TD_E_INVALID;
  std::string k(key);
  auto bad = [&](const char* why) {
    c->err = k + ": " + why;
    return TD_E_INVALID;
  };
  if (k == "dp.low_bits") {
    if (v < 2 || v > 5) return bad("must be in [2, 5]");
    c->dp.low_bits = (int)v;
  } else if (k == "dp.tiles_per_lane") {
    if (v < 1 || v > 64) return bad("must be in [1, 64]");
    c->dp.tiles_per_lane = (int)v;
  } else if (k == "dp.block") {
    if (v < 64 || v > 1024 || v % 64) return bad("must be a multiple of 64 in [64, 1024]");
    c->dp.block = (int)v;
  } else if (k == "dp.batch_wg_per_cu") {
    if (v < 1 || v > 32) return bad("must be in [1, 32]");
    c->dp.batch_wg_per_cu = (int)v;
  } else if (k == "dp.batch_block") {
    if (v < 64 || v > 1024 || v % 64) return bad("must be a multiple of 64 in [64, 1024]");
    c->dp.batch_block = (int)v;
  } else if (k == "dp.use_graph") {
    c->dp.use_graph = v ? 1 : 0;
  } else if (k == "dp.xcd_remap") {
    c->dp.xcd_remap = v ? 1 : 0;
  } else if (k == "dp.class_bits") {
    if (v != 0 && v != 3 && v != 4) return bad("must be 0, 3 or 4");
    c->dp.class_bits = (int)v;
  } else if (k == "dp.class_min_nh") {
    if (v < 5 || v > 32) return bad("must be in [5, 32]");
    c->dp.class_min_nh = (int)v;
  } else if (k == "dp.grid_mult") {
    if (v < 1 || v > 64) return bad("must be in [1, 64]");
    c->dp.grid_mult = (int)v;
  } else if (k == "dp.packed") {
    c->dp.packed = v ? 1 : 0;
  } else if (k == "dp.flow_spin") {
    if (v < 0 || v > (1 << 30)) return bad("must be in [0, 2^30]");
    c->dp.flow_spin = (int)v;
  } else if (k == "dp.streams") {
    if (v < 1 || v > 3) return bad("must be 1, 2 or 3");
    c->dp.streams = (int)v;
  } else if (k.rfind("bnb.", 0) == 0 || k.rfind("mlp.", 0) == 0) {
    c->params[k] = v;
  } else {
    return bad("unknown parameter");
  }
  // a change of DP launch shape invalidates the captured level graphs
  c->DropDPGraphs();
  return TD_OK;
}

int td_ctx_get_param(const td_ctx* c, const char* key, int64_t* v) {
  if (!c || !key || !v) return TD_E_INVALID;
  std::string k(key);
  if (k == "dp.low_bits") *v = c->dp.low_bits;
  else if (k == "dp.tiles_per_lane") *v = c->dp.tiles_per_lane;
  else if (k == "dp.block") *v = c->dp.block;
  else if (k == "dp.batch_wg_per_cu") *v = c->dp.batch_wg_per_cu;
  else if (k == "dp.batch_block") *v = c->dp.batch_block;
  else if (k == "dp.use_graph") *v = c->dp.use_graph;
  else if (k == "dp.xcd_remap") *v = c->dp.xcd_remap;
  else if (k == "dp.class_bits") *v = c->dp.class_bits;
  else if (k == "dp.class_min_nh") *v = c->dp.class_min_nh;
  else if (k == "dp.grid_mult") *v = c->dp.grid_mult;
  else if (k == "dp.packed") *v = c->dp.packed;
  else if (k == "dp.flow_spin") *v = c->dp.flow_spin;
  else if (k == "dp.streams") *v = c->dp.streams;
  else {
    auto it = c->params.find(k);
    if (it == c->params.end()) return TD_E_INVALID;
    *v = it->second;
  }
  return TD_OK;
}

}  // extern "C"
