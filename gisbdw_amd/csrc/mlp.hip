// mlp.hip -- the learned proposal: a message-passing MLP that scores
// vertices as roots of an elimination tree.  BF16 weights and activations on
// MFMA (v_mfma_f32_16x16x32_bf16) with FP32 accumulation; hand-written
// forward and backward; Adam on FP32 master weights.
//
// It has no counterpart in the reference; it plugs into the reference's two
// extension points of BranchAndBound: LowerBound::LowerBoundInfo::attempt_order
// (Treedepth/src/branch_and_bound/branch_and_bound.hpp:21-24, used at
// branch_and_bound.cpp:81-87) and Heuristic::Get (branch_and_bound.hpp:38-42,
// used at :78).  It only orders the search and seeds its upper bound.
//
// Network (n <= 64 vertices, rows padded to 64, H = 64):
//   x_v   = [deg/4, core/4, twohop/16, ecc/8]
//   h0    = relu(W0 x + b0)                                   (4 -> 64)
//   m_r   = mean_{u in N(v)} h_{r-1,u}                        (r = 1, 2)
//   h_r   = relu(Ws_r h_{r-1} + Wn_r m_r + b_r)               (64+64 -> 64)
//   z1    = relu(W3 h2 + b3), z2 = relu(W4 z1 + b4)           (64 -> 64)
//   s_v   = w5 . z2 + b5                                      (64 -> 1)
// Loss per graph: cross-entropy of softmax(s) over its vertices against the
// uniform distribution on the optimal roots.  Values are rounded to bf16 at
// every MFMA input; the CPU reference in tests/ rounds at the same points.
#include <cmath>
#include <cstring>
#include <random>
#include <vector>

#include "ctx.hpp"

namespace tdhip {
namespace {

constexpr int kH = 64;
// parameter offsets in the FP32 master vector
constexpr int P_W0 = 0, P_B0 = 256, P_WS1 = 320, P_WN1 = 4416, P_B1 = 8512,
              P_WS2 = 8576, P_WN2 = 12672, P_B2 = 16768, P_W3 = 16832,
              P_B3 = 20928, P_W4 = 20992, P_B4 = 25088, P_W5 = 25152,
              P_B5 = 25216, kNParams = 25217;
// per-graph working set, in LDS: 7 activation matrices and, for training,
// one bf16 gradient matrix (64x64 each) and two fp32 matrices: 56 KiB for
// scoring, 96 KiB for training (gfx950 has 160 KiB of LDS per CU)
// LDS row strides: 72 bf16 (144 bytes: rows stay 16-byte aligned for the
// MFMA operand loads, and lane v walking row v meets at most 4-way bank
// conflicts) and 65 fp32 (conflict-free)
constexpr int kLd = kH + 8;
constexpr int kLdF = kH + 1;
constexpr int kMatLd = kH * kLd;
constexpr int kMatLdF = kH * kLdF;
enum { A_H0 = 0, A_M1, A_H1, A_M2, A_H2, A_Z1, A_Z2, G_A, kNBf16 };
constexpr int kScoreMats = A_Z2 + 1;

typedef __bf16 v8bf __attribute__((ext_vector_type(8)));
typedef short v8s __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));

__host__ __device__ inline uint16_t ToBf16(float f) {
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  u += 0x7FFFu + ((u >> 16) & 1u);  // round to nearest even
  return static_cast<uint16_t>(u >> 16);
}

__host__ __device__ inline float FromBf16(uint16_t h) {
  return __builtin_bit_cast(float, static_cast<uint32_t>(h) << 16);
}

__device__ __forceinline__ void Sync() { __syncthreads(); }

// A graph's 64x64 products are split over the workgroup's kWaves = 4 kSplit
// waves: wave w computes tile-row w / kSplit (rows 16 (w / kSplit) .. +15)
// and, of its four 16-column tiles, the kTN tiles of group w % kSplit.  The
// element-wise steps give each wave kCW = 64 / kWaves columns (or rows).
// One graph's working set fills most of a CU's LDS, so a workgroup is alone
// on its CU: 16 waves keep 4 per SIMD to hide LDS and MFMA latency.
constexpr int kSplit = 4;
constexpr int kWaves = 4 * kSplit;
constexpr int kTN = 4 / kSplit;
constexpr int kCW = 64 / kWaves;
constexpr int kBlock = 64 * kWaves;

__device__ __forceinline__ int Lane() { return threadIdx.x & 63; }
__device__ __forceinline__ int WaveId() { return threadIdx.x >> 6; }
__device__ __forceinline__ int TileRow() { return WaveId() / kSplit; }
__device__ __forceinline__ int TileCol0() { return (WaveId() % kSplit) * kTN; }

// acc.t[j][i] holds D[16 tm + 4 (lane/16) + i][16 (TileCol0() + j) + lane%16]
// of tile-row tm.
struct AccRow {
  v4f t[kTN];
};

__device__ __forceinline__ void Zero(AccRow& a) {
#pragma unroll
  for (int j = 0; j < kTN; ++j) a.t[j] = v4f{0.f, 0.f, 0.f, 0.f};
}

// acc += A (rows 16tm..16tm+15 of a 64x64 A) * B (this wave's column
// tiles of a 64x64 B); A(m,k) =
// A[m*am + k*ak], B(k,n) = B[k*bk + n*bn], bf16 bit patterns.  Lane l
// supplies row/col l%16 and the k-group l/16 (8 consecutive k) of each
// 16x16x32 step.  kAc / kBc: ak == 1 / bk == 1, so a lane's 8 k-values are
// 16 contiguous, 16-byte aligned bytes and come in one load.
template <bool kAc, bool kBc>
__device__ __forceinline__ void MatMulRow(AccRow& acc, int tm, const uint16_t* __restrict__ A,
                                          int am, int ak, const uint16_t* __restrict__ B,
                                          int bk, int bn) {
  const int lane = Lane();
  const int r = lane & 15, g = lane >> 4, t0 = TileCol0();
#pragma unroll
  for (int ks = 0; ks < 2; ++ks) {
    v8s a, b[kTN];
    const int k0 = 32 * ks + 8 * g;
    if constexpr (kAc) {
      a = __builtin_bit_cast(v8s, *reinterpret_cast<const uint4*>(A + (16 * tm + r) * am + k0));
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) a[j] = static_cast<short>(A[(16 * tm + r) * am + (k0 + j) * ak]);
    }
#pragma unroll
    for (int t = 0; t < kTN; ++t) {
      const int col = 16 * (t0 + t) + r;
      if constexpr (kBc) {
        b[t] = __builtin_bit_cast(v8s, *reinterpret_cast<const uint4*>(B + col * bn + k0));
      } else {
#pragma unroll
        for (int j = 0; j < 8; ++j)
          b[t][j] = static_cast<short>(B[(k0 + j) * bk + col * bn]);
      }
    }
#pragma unroll
    for (int tn = 0; tn < kTN; ++tn)
      acc.t[tn] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
          __builtin_bit_cast(v8bf, a), __builtin_bit_cast(v8bf, b[tn]), acc.t[tn], 0, 0, 0);
  }
}

// element (row, col) owned by this lane for tile (tm, tn), register i
__device__ __forceinline__ int AccRowIdx(int tm, int i) { return 16 * tm + 4 * (Lane() >> 4) + i; }
__device__ __forceinline__ int AccCol(int tn) { return 16 * (TileCol0() + tn) + (threadIdx.x & 15); }

// Y = relu(acc + bias[col]) -> bf16 at Y[row*kLd + col], tile-row tm
__device__ __forceinline__ void StoreReluBf16(const AccRow& acc, int tm, const float* bias,
                                              uint16_t* Y) {
#pragma unroll
  for (int tn = 0; tn < kTN; ++tn)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = AccRowIdx(tm, i), col = AccCol(tn);
      const float v = acc.t[tn][i] + bias[col];
      Y[row * kLd + col] = ToBf16(v > 0.f ? v : 0.f);
    }
}

__device__ __forceinline__ void StoreF32(const AccRow& acc, int tm, float* Y, int ym, int yn) {
#pragma unroll
  for (int tn = 0; tn < kTN; ++tn)
#pragma unroll
    for (int i = 0; i < 4; ++i) Y[AccRowIdx(tm, i) * ym + AccCol(tn) * yn] = acc.t[tn][i];
}

// m[v][c] = mean over neighbours u of h[u][c] (fp32 sum of bf16 values),
// rounded; lane v, this wave's kCW columns
__device__ __forceinline__ void Aggregate(const uint16_t* h, uint16_t* m, uint64_t myadj) {
  const int v = Lane(), c0 = kCW * WaveId();
  const int deg = __builtin_popcountll(myadj);
  const float inv = deg ? 1.0f / static_cast<float>(deg) : 0.f;
  // neighbours in ascending order for each column, one pass over them
  float s[kCW];
#pragma unroll
  for (int j = 0; j < kCW; ++j) s[j] = 0.f;
  for (uint64_t a = myadj; a; a &= a - 1) {
    const uint16_t* row = h + __builtin_ctzll(a) * kLd + c0;
#pragma unroll
    for (int j = 0; j < kCW; ++j) s[j] += FromBf16(row[j]);
  }
#pragma unroll
  for (int j = 0; j < kCW; ++j) m[v * kLd + c0 + j] = ToBf16(s[j] * inv);
}

struct Net {
  const float* w;      // fp32 master (biases, W0 and w5 are read as bf16 values)
  const uint16_t* wb;  // bf16 copy
  const uint16_t* wt;  // bf16 copy with each 64x64 matrix transposed
};

// index of parameter p in the copy with the 64x64 matrices transposed
__host__ __device__ inline int TransposedIndex(int p) {
  const int bases[6] = {P_WS1, P_WN1, P_WS2, P_WN2, P_W3, P_W4};
  for (int i = 0; i < 6; ++i) {
    const int q = p - bases[i];
    if (q >= 0 && q < kH * kH) return bases[i] + (q % kH) * kH + q / kH;
  }
  return p;
}

__device__ __forceinline__ float Wb(const Net& N, int p) { return FromBf16(N.wb[p]); }

// Sum of the kWaves partial values s_red[w * 64 + v], in wave order.
__device__ __forceinline__ float WaveOrderSum(const float* s_red, int v) {
  float a = s_red[v];
#pragma unroll
  for (int i = 1; i < kWaves; ++i) a += s_red[i * 64 + v];
  return a;
}

// Forward for one graph (this workgroup); activations to S (LDS); returns
// s_v in lane v of every wave.  s_red: kWaves x 64 floats of scratch.
__device__ float Forward(const Net& N, const float* __restrict__ x, uint64_t myadj,
                         uint16_t* S, float* s_red) {
  const int v = Lane(), w = WaveId(), c0 = kCW * w, tm = TileRow();
  uint16_t* h0 = S + A_H0 * kMatLd;
  uint16_t* m1 = S + A_M1 * kMatLd;
  uint16_t* h1 = S + A_H1 * kMatLd;
  uint16_t* m2 = S + A_M2 * kMatLd;
  uint16_t* h2 = S + A_H2 * kMatLd;
  uint16_t* z1 = S + A_Z1 * kMatLd;
  uint16_t* z2 = S + A_Z2 * kMatLd;
  const float xv[4] = {x[v * 4 + 0], x[v * 4 + 1], x[v * 4 + 2], x[v * 4 + 3]};
  for (int o = c0; o < c0 + kCW; ++o) {
    float a = N.w[P_B0 + o];
#pragma unroll
    for (int i = 0; i < 4; ++i) a += Wb(N, P_W0 + o * 4 + i) * xv[i];
    h0[v * kLd + o] = ToBf16(a > 0.f ? a : 0.f);
  }
  Sync();
  Aggregate(h0, m1, myadj);
  Sync();
  AccRow acc;
  Zero(acc);
  MatMulRow<true, true>(acc, tm, h0, kLd, 1, N.wb + P_WS1, 1, kH);
  MatMulRow<true, true>(acc, tm, m1, kLd, 1, N.wb + P_WN1, 1, kH);
  StoreReluBf16(acc, tm, N.w + P_B1, h1);
  Sync();
  Aggregate(h1, m2, myadj);
  Sync();
  Zero(acc);
  MatMulRow<true, true>(acc, tm, h1, kLd, 1, N.wb + P_WS2, 1, kH);
  MatMulRow<true, true>(acc, tm, m2, kLd, 1, N.wb + P_WN2, 1, kH);
  StoreReluBf16(acc, tm, N.w + P_B2, h2);
  Sync();
  Zero(acc);
  MatMulRow<true, true>(acc, tm, h2, kLd, 1, N.wb + P_W3, 1, kH);
  StoreReluBf16(acc, tm, N.w + P_B3, z1);
  Sync();
  Zero(acc);
  MatMulRow<true, true>(acc, tm, z1, kLd, 1, N.wb + P_W4, 1, kH);
  StoreReluBf16(acc, tm, N.w + P_B4, z2);
  Sync();
  // s_v = b5 + w5 . z2[v]: this wave's kCW terms, then the kWaves partial
  // sums in wave order
  float part = 0.f;
  for (int j = c0; j < c0 + kCW; ++j) part += FromBf16(z2[v * kLd + j]) * Wb(N, P_W5 + j);
  s_red[w * 64 + v] = part;
  Sync();
  const float s = N.w[P_B5] + WaveOrderSum(s_red, v);
  Sync();
  return s;
}

__device__ __forceinline__ float WaveMaxF(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off));
  return v;
}
__device__ __forceinline__ float WaveSumF(float v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
  return v;
}

// ---------------------------------------------------------------------------
// features: one wave per graph, lanes = vertices
// ---------------------------------------------------------------------------
__device__ void Features(const uint64_t* s_adj, uint64_t myadj, int n, float* x) {
  const int v = threadIdx.x & 63;
  const bool in = v < n;
  const uint64_t V = n >= 64 ? ~0ull : ((1ull << n) - 1ull);
  const int deg = __builtin_popcountll(myadj);
  // core number: largest k whose k-core holds v (parallel peeling)
  int core = 0;
  for (int k = 1; k < 64; ++k) {
    uint64_t X = V;
    for (;;) {
      const bool inx = (X >> v) & 1ull;
      const int d = inx ? __builtin_popcountll(myadj & X) : 0;
      const uint64_t keep = static_cast<uint64_t>(__ballot(inx && d >= k));
      if (keep == X) break;
      X = keep;
    }
    if (!X) break;
    if ((X >> v) & 1ull) core = k;
  }
  // vertices within distance 2, and BFS eccentricity inside v's component
  uint64_t n2 = myadj;
  for (uint64_t a = myadj; a; a &= a - 1) n2 |= s_adj[__builtin_ctzll(a)];
  n2 &= ~(1ull << v);
  int ecc = 0;
  if (in) {
    uint64_t seen = 1ull << v, front = seen;
    for (;;) {
      uint64_t nb = 0;
      for (uint64_t f = front; f; f &= f - 1) nb |= s_adj[__builtin_ctzll(f)];
      nb &= ~seen;
      if (!nb) break;
      seen |= nb;
      front = nb;
      ++ecc;
    }
  }
  x[v * 4 + 0] = in ? deg * 0.25f : 0.f;
  x[v * 4 + 1] = in ? core * 0.25f : 0.f;
  x[v * 4 + 2] = in ? __builtin_popcountll(n2) * 0.0625f : 0.f;
  x[v * 4 + 3] = in ? ecc * 0.125f : 0.f;
  Sync();
}

// A call's graphs from page-locked host memory, which each wave reads once:
// checked (status[i] = 1: graph i is not a valid one, and an empty graph takes
// its place), copied to the device arrays, and their features.  Against the
// checks and pageable copies on the host this takes 1024 graphs' scores from
// 360 to 92 us a call, the gradient of 512 graphs from 235 to 116.
__global__ __launch_bounds__(64) void MLPIntakeKernel(
    const int32_t* __restrict__ ns, const uint64_t* __restrict__ adj,
    const uint64_t* __restrict__ tgt, int32_t* __restrict__ ns_out,
    uint64_t* __restrict__ adj_out, uint64_t* __restrict__ tgt_out, float* __restrict__ feat,
    int32_t* __restrict__ status) {
  __shared__ uint64_t s_adj[64];
  const int gi = blockIdx.x, v = threadIdx.x;
  const int n = ns[gi];
  uint64_t myadj = adj[static_cast<size_t>(gi) * 64 + v];
  s_adj[v] = myadj;
  Sync();
  const bool bad = __ballot(!RowFine(s_adj, myadj, n, v)) != 0ull;
  Sync();
  if (bad) s_adj[v] = myadj = 0ull;
  Sync();
  adj_out[static_cast<size_t>(gi) * 64 + v] = myadj;
  if (v == 0) {
    ns_out[gi] = n;
    if (tgt) tgt_out[gi] = tgt[gi];
    status[gi] = bad ? 1 : 0;
  }
  Features(s_adj, myadj, n, feat + static_cast<size_t>(gi) * 256);
}

__global__ __launch_bounds__(kBlock) void MLPScoreKernel(Net N, const int32_t* __restrict__ ns,
                                                         const uint64_t* __restrict__ adj,
                                                         const float* __restrict__ feat,
                                                         float* __restrict__ scores) {
  __shared__ uint16_t s_act[kScoreMats * kMatLd];
  __shared__ float s_red[kWaves * 64];
  const int gi = blockIdx.x, v = Lane();
  const int n = ns[gi];
  const uint64_t myadj = v < n ? adj[static_cast<size_t>(gi) * 64 + v] : 0ull;
  const float s = Forward(N, feat + static_cast<size_t>(gi) * 256, myadj, s_act, s_red);
  if (WaveId() == 0) scores[static_cast<size_t>(gi) * 64 + v] = v < n ? s : 0.f;
}

// Forward + backward of one graph per workgroup (kWaves waves; wave w owns
// its tile-row and column tiles of every product and columns (or rows)
// kCW w .. kCW w + kCW - 1 of every element-wise step).  Gradient of scale * loss_i goes to part[i][*] (one row per graph,
// reduced later).  Sums split over the waves are combined in wave order.
__global__ __launch_bounds__(kBlock) void MLPTrainKernel(
    Net N, const int32_t* __restrict__ ns, const uint64_t* __restrict__ adj,
    const uint64_t* __restrict__ targets, const float* __restrict__ feat,
    const int32_t* __restrict__ index, float* __restrict__ part, float* __restrict__ loss,
    float scale) {
  const int bi = blockIdx.x;
  const int gi = index ? index[bi] : bi;
  const int v = Lane(), w = WaveId(), c0 = kCW * w, tm = TileRow();
  const int n = ns[gi];
  const bool in = v < n;
  const uint64_t myadj = in ? adj[static_cast<size_t>(gi) * 64 + v] : 0ull;
  __shared__ uint16_t s_act[kNBf16 * kMatLd];
  __shared__ float s_f[2 * kMatLdF];
  __shared__ float s_invdeg[64];  // 1 / deg(u), 0 for an isolated u
  __shared__ float s_red[kWaves * 64 * 5];
  if (w == 0) {  // read after Forward's syncs
    const int d = __builtin_popcountll(myadj);
    s_invdeg[v] = d ? 1.0f / static_cast<float>(d) : 0.f;
  }
  uint16_t* S = s_act;
  float* SF = s_f;
  float* G = part + static_cast<size_t>(bi) * kNParams;
  const float* x = feat + static_cast<size_t>(gi) * 256;
  const float s = Forward(N, x, myadj, S, s_red);
  // ---- loss: softmax over the graph's vertices vs uniform optimal roots
  // (every wave computes it; wave 0 writes it)
  const uint64_t tgt = targets[gi];
  const int npos = __builtin_popcountll(tgt);
  const float mx = WaveMaxF(in ? s : -INFINITY);
  const float e = in ? expf(s - mx) : 0.f;
  const float z = WaveSumF(e);
  const float p = e / z;
  const float t = ((tgt >> v) & 1ull) ? 1.0f / static_cast<float>(npos) : 0.f;
  const float li = (t > 0.f) ? -t * (s - mx - logf(z)) : 0.f;
  const float lsum = WaveSumF(li);
  if (w == 0 && v == 0) loss[bi] = lsum;
  const float ds = in ? (p - t) * scale : 0.f;  // dL/ds_v
  uint16_t* h0 = S + A_H0 * kMatLd;
  uint16_t* m1 = S + A_M1 * kMatLd;
  uint16_t* h1 = S + A_H1 * kMatLd;
  uint16_t* m2 = S + A_M2 * kMatLd;
  uint16_t* h2 = S + A_H2 * kMatLd;
  uint16_t* z1 = S + A_Z1 * kMatLd;
  uint16_t* z2 = S + A_Z2 * kMatLd;
  uint16_t* gA = S + G_A * kMatLd;  // bf16 gradient (pre-activation)
  float* F0 = SF;                   // fp32 gradient w.r.t. an activation
  float* F1 = SF + kMatLdF;
  // ---- head: s = w5 . z2 + b5
  // dw5[j] = sum_r ds_r z2[r][j] (lane j, rows of this wave); db5 = sum_r ds_r
  {
    float dw = 0.f;
    for (int r = c0; r < c0 + kCW; ++r) dw += __shfl(ds, r) * FromBf16(z2[r * kLd + v]);
    s_red[w * 64 + v] = dw;
    // da4[r][j] = ds_r w5[j] (z2 > 0)  (lane r, this wave's columns j)
    for (int j = c0; j < c0 + kCW; ++j) {
      const float zz = FromBf16(z2[v * kLd + j]);
      gA[v * kLd + j] = ToBf16(zz > 0.f ? ds * Wb(N, P_W5 + j) : 0.f);
    }
  }
  Sync();
  if (w == 0) {
    G[P_W5 + v] = WaveOrderSum(s_red, v);
    const float db = WaveSumF(ds);
    if (v == 0) G[P_B5] = db;
  }
  // dense layer backward: given gA = d pre-activation (bf16, [r][o]),
  // input X ([r][i]) and weight W ([o][i]): dW = gA^T X, db = colsum gA,
  // dX (fp32, [r][i]) = gA W into Fout.  Ends with a barrier.
  auto dense_back = [&](const uint16_t* Xin, int pW, int pB, float* Fout) {
    float db = 0.f;
    for (int r = c0; r < c0 + kCW; ++r) db += FromBf16(gA[r * kLd + v]);
    Sync();  // s_red is free again
    s_red[w * 64 + v] = db;
    AccRow acc;
    Zero(acc);
    MatMulRow<false, false>(acc, tm, gA, 1, kLd, Xin, kLd, 1);  // (o, r) x (r, i)
    StoreF32(acc, tm, G + pW, kH, 1);
    if (Fout) {
      Zero(acc);
      MatMulRow<true, true>(acc, tm, gA, kLd, 1, N.wt + pW, 1, kH);  // (r, o) x (o, i)
      StoreF32(acc, tm, Fout, kLdF, 1);
    }
    Sync();
    if (w == 0) G[pB + v] = WaveOrderSum(s_red, v);
  };
  // d pre-activation of a relu layer: gA = (y > 0) * F0, this wave's columns
  auto relu_grad = [&](const uint16_t* y) {
    for (int j = c0; j < c0 + kCW; ++j) {
      const float yy = FromBf16(y[v * kLd + j]);
      gA[v * kLd + j] = ToBf16(yy > 0.f ? F0[v * kLdF + j] : 0.f);
    }
    Sync();
  };
  // layer 4: z2 = relu(W4 z1 + b4)
  dense_back(z1, P_W4, P_B4, F0);
  relu_grad(z1);
  // layer 3: z1 = relu(W3 h2 + b3)
  dense_back(h2, P_W3, P_B3, F0);
  relu_grad(h2);
  // message-passing layer: h_out = relu(Ws h_in + Wn m + b), m = mean_N h_in
  auto mp_back = [&](const uint16_t* hin, const uint16_t* mag, int pWs, int pWn, int pB) {
    dense_back(hin, pWs, pB, F0);  // dWs, db, F0 = gA Ws
    AccRow acc;
    Zero(acc);
    MatMulRow<false, false>(acc, tm, gA, 1, kLd, mag, kLd, 1);
    StoreF32(acc, tm, G + pWn, kH, 1);
    Zero(acc);
    MatMulRow<true, true>(acc, tm, gA, kLd, 1, N.wt + pWn, 1, kH);
    StoreF32(acc, tm, F1, kLdF, 1);  // dL/dm
    Sync();
    // d h_in[u] += sum_{v in N(u)} dm[v] / deg_v   (lane u; inverse degrees
    // from LDS; neighbours in ascending order for each of the wave's columns)
    float a[kCW];
#pragma unroll
    for (int j = 0; j < kCW; ++j) a[j] = F0[v * kLdF + c0 + j];
    for (uint64_t nb = myadj; nb; nb &= nb - 1) {
      const int u = __builtin_ctzll(nb);
      const float iu = s_invdeg[u];
#pragma unroll
      for (int j = 0; j < kCW; ++j) a[j] += F1[u * kLdF + c0 + j] * iu;
    }
#pragma unroll
    for (int j = 0; j < kCW; ++j) F0[v * kLdF + c0 + j] = a[j];
    Sync();
  };
  mp_back(h1, m2, P_WS2, P_WN2, P_B2);
  relu_grad(h1);
  mp_back(h0, m1, P_WS1, P_WN1, P_B1);
  // layer 0: h0 = relu(W0 x + b0), computed in fp32 from the fp32 d h0.
  // Lane o accumulates dW0[o][0..3] and db0[o] over this wave's rows r.
  {
    float dw[4] = {0.f, 0.f, 0.f, 0.f}, db = 0.f;
    for (int r = c0; r < c0 + kCW; ++r) {
      const float y = FromBf16(h0[r * kLd + v]);
      const float da = y > 0.f ? F0[r * kLdF + v] : 0.f;
      db += da;
#pragma unroll
      for (int i = 0; i < 4; ++i) dw[i] += da * x[r * 4 + i];
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) s_red[(w * 5 + i) * 64 + v] = dw[i];
    s_red[(w * 5 + 4) * 64 + v] = db;
    Sync();
    if (w == 0) {
#pragma unroll
      for (int i = 0; i < 5; ++i) {
        float a = s_red[i * 64 + v];
#pragma unroll
        for (int j = 1; j < kWaves; ++j) a += s_red[(5 * j + i) * 64 + v];
        if (i < 4) G[P_W0 + v * 4 + i] = a;
        else G[P_B0 + v] = a;
      }
    }
  }
}

// grad[p] = sum over rows of part[*][p] in a fixed order (deterministic):
// a workgroup of kReduceWaves waves owns 64 parameters, wave w sums the rows
// r = w mod kReduceWaves (one coalesced 256-byte row slice per step, four
// loads in flight), then wave 0 adds the partial sums in wave order.
constexpr int kReduceParams = 64;
constexpr int kReduceWaves = 16;
__global__ __launch_bounds__(64 * kReduceWaves) void MLPReduceKernel(const float* __restrict__ part,
                                                                     int rows, float* __restrict__ grad) {
  __shared__ float s_part[kReduceWaves][kReduceParams];
  const int lane = threadIdx.x & 63;
  const int wid = threadIdx.x >> 6;
  const int p = blockIdx.x * kReduceParams + lane;
  constexpr int R = kReduceWaves;
  float s = 0.f;
  if (p < kNParams) {
    int r = wid;
    for (; r + 3 * R < rows; r += 4 * R) {
      const float a = part[static_cast<size_t>(r) * kNParams + p];
      const float b = part[static_cast<size_t>(r + R) * kNParams + p];
      const float c = part[static_cast<size_t>(r + 2 * R) * kNParams + p];
      const float d = part[static_cast<size_t>(r + 3 * R) * kNParams + p];
      s += a;
      s += b;
      s += c;
      s += d;
    }
    for (; r < rows; r += R) s += part[static_cast<size_t>(r) * kNParams + p];
  }
  s_part[wid][lane] = s;
  __syncthreads();
  if (wid == 0 && p < kNParams) {
    float a = s_part[0][lane];
#pragma unroll
    for (int i = 1; i < kReduceWaves; ++i) a += s_part[i][lane];
    grad[p] = a;
  }
}

__global__ void MLPAdamKernel(float* __restrict__ w, uint16_t* __restrict__ wb,
                              uint16_t* __restrict__ wt,
                              float* __restrict__ m1, float* __restrict__ m2,
                              const float* __restrict__ g, float lr, float b1,
                              float b2, float eps, float c1, float c2) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= kNParams) return;
  const float gp = g[p];
  const float a = b1 * m1[p] + (1.f - b1) * gp;
  const float b = b2 * m2[p] + (1.f - b2) * gp * gp;
  m1[p] = a;
  m2[p] = b;
  const float nw = w[p] - lr * (a / c1) / (sqrtf(b / c2) + eps);
  w[p] = nw;
  wb[p] = ToBf16(nw);
  wt[TransposedIndex(p)] = ToBf16(nw);
}

__global__ void MLPToBf16Kernel(const float* __restrict__ w, uint16_t* __restrict__ wb,
                                uint16_t* __restrict__ wt) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < kNParams) {
    wb[p] = ToBf16(w[p]);
    wt[TransposedIndex(p)] = ToBf16(w[p]);
  }
}

// Optimal-root labels from the last single-graph DP: for a connected vertex
// set S (one per wave), positives = {v in S : td(S \ v) = td(S) - 1}.
struct DPLookup {
  const uint8_t* table;
  uint32_t n, lb, nh, direct;  // as in DPGraph
  uint32_t lvl[34];
};

// Gray code of td(S) mod 4 from the tables (two bit planes; dpword.hpp)
__device__ __forceinline__ uint32_t LookupCode(const DPLookup& L, const uint32_t* cb, uint32_t S) {
  if (L.direct) {
    const size_t plane = static_cast<size_t>(1) << (L.n > 5 ? L.n - 5 : 0);
    const uint32_t* p = reinterpret_cast<const uint32_t*>(L.table) + (S >> 5);
    return (p[0] >> (S & 31u) & 1u) | (p[plane] >> (S & 31u) & 1u) << 1;
  }
  uint32_t H = S >> L.lb;
  size_t tile = L.lvl[__builtin_popcount(H)];
  for (int i = 1; H; ++i) {
    tile += cb[__builtin_ctz(H) * 33 + i];
    H &= H - 1;
  }
  const size_t plane = static_cast<size_t>(L.lvl[L.nh + 1]) << (L.lb - 3);
  const uint8_t* p = L.table + (tile << (L.lb - 3)) + 4 * ((S >> 5) & ((1u << (L.lb - 5)) - 1u));
  const uint32_t g0 = *reinterpret_cast<const uint32_t*>(p);
  const uint32_t g1 = *reinterpret_cast<const uint32_t*>(p + plane);
  return ((g0 >> (S & 31u)) & 1u) | (((g1 >> (S & 31u)) & 1u) << 1);
}

__global__ __launch_bounds__(64) void LabelKernel(DPLookup L, const uint32_t* __restrict__ g_cb,
                                                  const uint32_t* __restrict__ sets,
                                                  uint32_t* __restrict__ pos,
                                                  uint8_t* __restrict__ tdout) {
  __shared__ uint32_t s_cb[32 * 33];
  for (int i = threadIdx.x; i < 32 * 33; i += 64) s_cb[i] = g_cb[i];
  Sync();
  const uint32_t S = sets[blockIdx.x];
  const int v = threadIdx.x;
  const bool in = v < 32 && ((S >> v) & 1u);
  // td(S \ v) is td(S) or td(S) - 1: the codes mod 4 tell which
  const uint32_t all = LookupCode(L, s_cb, S);
  const uint32_t one = in ? LookupCode(L, s_cb, S & ~(1u << v)) : all;
  const uint64_t b = static_cast<uint64_t>(__ballot(in && one != all));
  // td(S): lane i reads the code of S's vertices 0..i; td is the number of
  // places where that code changes
  const uint32_t code = v < 32 ? LookupCode(L, s_cb, S & (v < 31 ? (2u << v) - 1u : ~0u)) : 0u;
  const uint32_t below = __shfl_up(code, 1);
  const uint64_t steps = static_cast<uint64_t>(__ballot(v < 32 && code != (v ? below : 0u)));
  if (v == 0) {
    pos[blockIdx.x] = static_cast<uint32_t>(b);
    tdout[blockIdx.x] = static_cast<uint8_t>(__builtin_popcountll(steps));
  }
}

// ---------------------------------------------------------------------------
// host
// ---------------------------------------------------------------------------
struct DevNet {
  float* w;
  uint16_t* wb;
  uint16_t* wt;
  float* m1;
  float* m2;
};

DevNet NetBuffers(td_ctx* ctx) {
  DevNet d;
  const bool fresh = ctx->bufs.find("mlp.w") == ctx->bufs.end();
  d.w = static_cast<float*>(ctx->Buffer("mlp.w", kNParams * 4));
  d.wb = static_cast<uint16_t*>(ctx->Buffer("mlp.wb", kNParams * 2));
  d.wt = static_cast<uint16_t*>(ctx->Buffer("mlp.wt", kNParams * 2));
  d.m1 = static_cast<float*>(ctx->Buffer("mlp.adam1", kNParams * 4));
  d.m2 = static_cast<float*>(ctx->Buffer("mlp.adam2", kNParams * 4));
  if (fresh) {
    TD_HIP(hipMemsetAsync(d.w, 0, kNParams * 4, ctx->stream));
    TD_HIP(hipMemsetAsync(d.wb, 0, kNParams * 2, ctx->stream));
    TD_HIP(hipMemsetAsync(d.wt, 0, kNParams * 2, ctx->stream));
    TD_HIP(hipMemsetAsync(d.m1, 0, kNParams * 4, ctx->stream));
    TD_HIP(hipMemsetAsync(d.m2, 0, kNParams * 4, ctx->stream));
  }
  return d;
}

void CheckGraphs(int ngraphs, const int32_t* ns, const uint64_t* adj64) {
  TD_REQUIRE(ngraphs >= 1 && ns && adj64, TD_E_INVALID, "empty batch or null pointer");
  for (int i = 0; i < ngraphs; ++i) {
    TD_REQUIRE(ns[i] >= 1 && ns[i] <= 64, TD_E_INVALID, "n must be in [1, 64]");
    ValidateGraph(ns[i], adj64 + static_cast<size_t>(i) * 64, 64);
    for (int v = ns[i]; v < 64; ++v)
      TD_REQUIRE(adj64[static_cast<size_t>(i) * 64 + v] == 0, TD_E_INVALID,
                 "rows beyond n must be zero");
  }
}

// Guard for a call whose graphs are checked on the device: where there is no
// memory to get them there, an invalid one is still the error that comes first.
template <typename F>
int GuardGraphs(td_ctx* ctx, int ngraphs, const int32_t* ns, const uint64_t* adj64, F&& f) {
  return Guard(ctx, [&] {
    try {
      f();
    } catch (const Error& e) {
      if (e.code == TD_E_NOMEM) CheckGraphs(ngraphs, ns, adj64);
      throw;
    }
  });
}

void CheckTargets(int ngraphs, const int32_t* ns, const uint64_t* targets) {
  for (int i = 0; i < ngraphs; ++i) {
    const uint64_t V = ns[i] >= 64 ? ~0ull : ((1ull << ns[i]) - 1ull);
    TD_REQUIRE(targets[i] && !(targets[i] & ~V), TD_E_INVALID,
               "each target must be a nonempty subset of the graph's vertices");
  }
}

// Page-locked staging of kChunk graphs: rows, vertex counts, targets, status
// and results.  A call of more graphs fills it several times.
constexpr int kChunk = 4096;
struct Staging {
  uint64_t *adj, *tgt;
  int32_t *ns, *status;
  float* out;  // kChunk graphs' rows of `floats`, or their losses and the gradient
};
Staging StagingBuffers(td_ctx* ctx, int ngraphs, size_t floats) {
  const size_t c = static_cast<size_t>(std::min(ngraphs, kChunk));
  const size_t out = std::max<size_t>(4 * floats * c, 4 * c + 4 * kNParams);
  uint8_t* p = static_cast<uint8_t*>(ctx->Pinned(528 * c + out));
  Staging s;
  s.adj = reinterpret_cast<uint64_t*>(p);
  s.tgt = s.adj + 64 * c;
  s.ns = reinterpret_cast<int32_t*>(s.tgt + c);
  s.status = s.ns + c;
  s.out = reinterpret_cast<float*>(s.status + c);
  return s;
}

struct Uploaded {
  int32_t* ns;
  uint64_t* adj;
  uint64_t* tgt;
  float* feat;
  Staging st;
  int last;  // graphs in the staging whose status is still to be read
};

// After the stream has been synchronized: the error of the first graph that
// is not a valid one, as CheckGraphs has it.
void CheckIntake(const Uploaded& u, int ngraphs, const int32_t* ns, const uint64_t* adj64) {
  for (int i = 0; i < u.last; ++i)
    if (u.st.status[i]) {
      CheckGraphs(ngraphs, ns, adj64);
      throw Error{TD_E_INVALID, "invalid graph"};
    }
}

// The graphs (and targets) of a call on their way to the device, checked
// there: the caller synchronizes and calls CheckIntake before it hands out any
// result.
Uploaded Intake(td_ctx* ctx, const char* tag, int ngraphs, const int32_t* ns,
                const uint64_t* adj64, const uint64_t* targets, size_t out_floats = 64) {
  TD_REQUIRE(ngraphs >= 1 && ns && adj64, TD_E_INVALID, "empty batch or null pointer");
  for (int i = 0; i < ngraphs; ++i)
    if (ns[i] < 1 || ns[i] > 64) CheckGraphs(ngraphs, ns, adj64);  // throws the first error
  Uploaded u;
  const std::string t(tag);
  u.ns = static_cast<int32_t*>(ctx->Buffer(t + ".n", 4ull * ngraphs));
  u.adj = static_cast<uint64_t*>(ctx->Buffer(t + ".adj", 512ull * ngraphs));
  u.feat = static_cast<float*>(ctx->Buffer(t + ".feat", 1024ull * ngraphs));
  u.tgt = targets ? static_cast<uint64_t*>(ctx->Buffer(t + ".tgt", 8ull * ngraphs)) : nullptr;
  u.st = StagingBuffers(ctx, ngraphs, out_floats);
  u.last = 0;
  for (int at = 0; at < ngraphs; at += kChunk) {
    const size_t c = static_cast<size_t>(std::min(ngraphs - at, kChunk));
    if (at) {
      TD_HIP(hipStreamSynchronize(ctx->stream));
      CheckIntake(u, ngraphs, ns, adj64);
    }
    std::memcpy(u.st.adj, adj64 + static_cast<size_t>(at) * 64, 512 * c);
    std::memcpy(u.st.ns, ns + at, 4 * c);
    if (targets) std::memcpy(u.st.tgt, targets + at, 8 * c);
    hipLaunchKernelGGL(MLPIntakeKernel, dim3(c), dim3(64), 0, ctx->stream, u.st.ns, u.st.adj,
                       targets ? u.st.tgt : nullptr, u.ns + at,
                       u.adj + static_cast<size_t>(at) * 64, u.tgt ? u.tgt + at : nullptr,
                       u.feat + static_cast<size_t>(at) * 256, u.st.status);
    TD_HIP(hipGetLastError());
    u.last = static_cast<int>(c);
  }
  return u;
}

}  // namespace
}  // namespace tdhip

using namespace tdhip;  // NOLINT

extern "C" {

int td_mlp_num_params(void) { return kNParams; }

int td_mlp_init(td_ctx* ctx, uint64_t seed) {
  return Guard(ctx, [&] {
    std::vector<float> w(kNParams, 0.f);
    std::mt19937_64 rng(seed);
    std::uniform_real_distribution<float> U(-1.f, 1.f);
    auto fill = [&](int off, int rows, int cols) {
      const float a = std::sqrt(6.0f / static_cast<float>(cols));
      for (int i = 0; i < rows * cols; ++i) w[off + i] = a * U(rng);
    };
    fill(P_W0, 64, 4);
    fill(P_WS1, 64, 64);
    fill(P_WN1, 64, 64);
    fill(P_WS2, 64, 64);
    fill(P_WN2, 64, 64);
    fill(P_W3, 64, 64);
    fill(P_W4, 64, 64);
    fill(P_W5, 1, 64);
    DevNet d = NetBuffers(ctx);
    TD_HIP(hipMemcpyAsync(d.w, w.data(), kNParams * 4, hipMemcpyHostToDevice, ctx->stream));
    TD_HIP(hipMemsetAsync(d.m1, 0, kNParams * 4, ctx->stream));
    TD_HIP(hipMemsetAsync(d.m2, 0, kNParams * 4, ctx->stream));
    hipLaunchKernelGGL(MLPToBf16Kernel, dim3((kNParams + 255) / 256), dim3(256), 0,
                       ctx->stream, d.w, d.wb, d.wt);
    TD_HIP(hipGetLastError());
    ctx->params["mlp.adam_t"] = 0;
    TD_HIP(hipStreamSynchronize(ctx->stream));
  });
}

int td_mlp_set_weights(td_ctx* ctx, const float* w, int64_t count) {
  return Guard(ctx, [&] {
    TD_REQUIRE(w && count == kNParams, TD_E_INVALID, "need td_mlp_num_params() floats");
    DevNet d = NetBuffers(ctx);
    TD_HIP(hipMemcpyAsync(d.w, w, kNParams * 4, hipMemcpyHostToDevice, ctx->stream));
    TD_HIP(hipMemsetAsync(d.m1, 0, kNParams * 4, ctx->stream));
    TD_HIP(hipMemsetAsync(d.m2, 0, kNParams * 4, ctx->stream));
    hipLaunchKernelGGL(MLPToBf16Kernel, dim3((kNParams + 255) / 256), dim3(256), 0,
                       ctx->stream, d.w, d.wb, d.wt);
    TD_HIP(hipGetLastError());
    ctx->params["mlp.adam_t"] = 0;
    TD_HIP(hipStreamSynchronize(ctx->stream));
  });
}

int td_mlp_get_weights(td_ctx* ctx, float* w, int64_t count) {
  return Guard(ctx, [&] {
    TD_REQUIRE(w && count == kNParams, TD_E_INVALID, "need td_mlp_num_params() floats");
    DevNet d = NetBuffers(ctx);
    TD_HIP(hipMemcpyAsync(w, d.w, kNParams * 4, hipMemcpyDeviceToHost, ctx->stream));
    TD_HIP(hipStreamSynchronize(ctx->stream));
  });
}

int td_mlp_features(td_ctx* ctx, int32_t ngraphs, const int32_t* ns, const uint64_t* adj64,
                    float* feat_out) {
  return GuardGraphs(ctx, ngraphs, ns, adj64, [&] {
    TD_REQUIRE(feat_out != nullptr, TD_E_INVALID, "features_out is null");
    // up to kChunk graphs' features wait in page-locked memory for the check,
    // so that one synchronization serves both
    const bool staged = ngraphs <= kChunk;
    const size_t bytes = 1024ull * ngraphs;
    Uploaded u = Intake(ctx, "mlp.in", ngraphs, ns, adj64, nullptr, 256);
    if (staged)
      TD_HIP(hipMemcpyAsync(u.st.out, u.feat, bytes, hipMemcpyDeviceToHost, ctx->stream));
    TD_HIP(hipStreamSynchronize(ctx->stream));
    CheckIntake(u, ngraphs, ns, adj64);
    if (staged) {
      std::memcpy(feat_out, u.st.out, bytes);
    } else {
      TD_HIP(hipMemcpyAsync(feat_out, u.feat, bytes, hipMemcpyDeviceToHost, ctx->stream));
      TD_HIP(hipStreamSynchronize(ctx->stream));
    }
  });
}

int td_mlp_scores(td_ctx* ctx, int32_t ngraphs, const int32_t* ns, const uint64_t* adj64,
                  float* scores_out) {
  return GuardGraphs(ctx, ngraphs, ns, adj64, [&] {
    TD_REQUIRE(scores_out != nullptr, TD_E_INVALID, "scores_out is null");
    DevNet d = NetBuffers(ctx);
    Uploaded u = Intake(ctx, "mlp.in", ngraphs, ns, adj64, nullptr);
    // up to kChunk graphs' scores go straight to host memory
    const bool direct = ngraphs <= kChunk;
    float* sc = direct ? u.st.out
                       : static_cast<float*>(ctx->Buffer("mlp.scores", 256ull * ngraphs));
    hipLaunchKernelGGL(MLPScoreKernel, dim3(ngraphs), dim3(kBlock), 0, ctx->stream,
                       Net{d.w, d.wb, d.wt}, u.ns, u.adj, u.feat, sc);
    TD_HIP(hipGetLastError());
    TD_HIP(hipStreamSynchronize(ctx->stream));
    CheckIntake(u, ngraphs, ns, adj64);
    if (direct) {
      std::memcpy(scores_out, sc, 256ull * ngraphs);
    } else {
      TD_HIP(hipMemcpyAsync(scores_out, sc, 256ull * ngraphs, hipMemcpyDeviceToHost,
                            ctx->stream));
      TD_HIP(hipStreamSynchronize(ctx->stream));
    }
  });
}

// Mean loss over the graphs and (grad_out non-null) its gradient.
int td_mlp_loss_grad(td_ctx* ctx, int32_t ngraphs, const int32_t* ns, const uint64_t* adj64,
                     const uint64_t* targets, float* loss_out, float* grad_out) {
  return GuardGraphs(ctx, ngraphs, ns, adj64, [&] {
    TD_REQUIRE(ngraphs >= 1 && ns && adj64, TD_E_INVALID, "empty batch or null pointer");
    if (!targets) CheckGraphs(ngraphs, ns, adj64);
    TD_REQUIRE(targets != nullptr, TD_E_INVALID, "targets is null");
    try {
      CheckTargets(ngraphs, ns, targets);
    } catch (const Error&) {
      CheckGraphs(ngraphs, ns, adj64);  // an invalid graph comes first
      throw;
    }
    DevNet d = NetBuffers(ctx);
    Uploaded u = Intake(ctx, "mlp.in", ngraphs, ns, adj64, targets);
    auto* part = static_cast<float*>(
        ctx->Buffer("mlp.part", 4ull * kNParams * static_cast<size_t>(ngraphs)));
    // up to kChunk graphs' losses, and the gradient, go straight to host memory
    const bool direct = ngraphs <= kChunk;
    auto* loss = direct ? u.st.out
                        : static_cast<float*>(ctx->Buffer("mlp.loss", 4ull * ngraphs));
    float* grad = u.st.out + std::min(ngraphs, kChunk);
    hipLaunchKernelGGL(MLPTrainKernel, dim3(ngraphs), dim3(kBlock), 0, ctx->stream,
                       Net{d.w, d.wb, d.wt}, u.ns, u.adj, u.tgt, u.feat, nullptr, part, loss,
                       1.0f / static_cast<float>(ngraphs));
    hipLaunchKernelGGL(MLPReduceKernel, dim3((kNParams + kReduceParams - 1) / kReduceParams),
                       dim3(64 * kReduceWaves), 0, ctx->stream, part, ngraphs, grad);
    TD_HIP(hipGetLastError());
    TD_HIP(hipStreamSynchronize(ctx->stream));
    CheckIntake(u, ngraphs, ns, adj64);
    std::vector<float> l(ngraphs);
    if (direct) {
      std::memcpy(l.data(), loss, 4ull * ngraphs);
    } else {
      TD_HIP(hipMemcpyAsync(l.data(), loss, 4ull * ngraphs, hipMemcpyDeviceToHost, ctx->stream));
      TD_HIP(hipStreamSynchronize(ctx->stream));
    }
    if (grad_out) std::memcpy(grad_out, grad, 4ull * kNParams);
    double s = 0;
    for (float x : l) s += x;
    if (loss_out) *loss_out = static_cast<float>(s / ngraphs);
  });
}

// Adam over shuffled minibatches, all on the device; epoch_loss_out[e] =
// mean training loss of epoch e.
int td_mlp_train(td_ctx* ctx, int32_t ngraphs, const int32_t* ns, const uint64_t* adj64,
                 const uint64_t* targets, int32_t epochs, int32_t batch, float lr,
                 uint64_t seed, float* epoch_loss_out) {
  return GuardGraphs(ctx, ngraphs, ns, adj64, [&] {
    TD_REQUIRE(ngraphs >= 1 && ns && adj64, TD_E_INVALID, "empty batch or null pointer");
    const bool args = targets && epochs >= 1 && batch >= 1 && lr > 0.f;
    if (!args) CheckGraphs(ngraphs, ns, adj64);  // an invalid graph comes first
    TD_REQUIRE(args, TD_E_INVALID, "bad training arguments");
    try {
      CheckTargets(ngraphs, ns, targets);
    } catch (const Error&) {
      CheckGraphs(ngraphs, ns, adj64);
      throw;
    }
    batch = std::min(batch, ngraphs);
    DevNet d = NetBuffers(ctx);
    Uploaded u = Intake(ctx, "mlp.train", ngraphs, ns, adj64, targets);
    TD_HIP(hipStreamSynchronize(ctx->stream));
    CheckIntake(u, ngraphs, ns, adj64);
    const uint64_t* tg = u.tgt;
    auto* part = static_cast<float*>(
        ctx->Buffer("mlp.part", 4ull * kNParams * static_cast<size_t>(batch)));
    auto* loss = static_cast<float*>(
        ctx->Buffer("mlp.trainloss", 4ull * static_cast<size_t>(ngraphs)));
    auto* grad = static_cast<float*>(ctx->Buffer("mlp.grad", 4ull * kNParams));
    auto* idx = static_cast<int32_t*>(ctx->Buffer("mlp.train.idx", 4ull * ngraphs));
    std::mt19937_64 rng(seed);
    std::vector<int32_t> perm(ngraphs);
    for (int i = 0; i < ngraphs; ++i) perm[i] = i;
    int64_t t = ctx->params["mlp.adam_t"];
    const float b1 = 0.9f, b2 = 0.999f, eps = 1e-8f;
    for (int e = 0; e < epochs; ++e) {
      std::shuffle(perm.begin(), perm.end(), rng);
      TD_HIP(hipMemcpyAsync(idx, perm.data(), 4ull * ngraphs, hipMemcpyHostToDevice,
                            ctx->stream));
      int nb = 0;
      for (int s0 = 0; s0 + batch <= ngraphs; s0 += batch, ++nb) {
        hipLaunchKernelGGL(MLPTrainKernel, dim3(batch), dim3(kBlock), 0, ctx->stream,
                           Net{d.w, d.wb, d.wt}, u.ns, u.adj, tg, u.feat, idx + s0, part, loss + s0,
                           1.0f / static_cast<float>(batch));
        hipLaunchKernelGGL(MLPReduceKernel,
                           dim3((kNParams + kReduceParams - 1) / kReduceParams),
                           dim3(64 * kReduceWaves), 0, ctx->stream, part, batch, grad);
        ++t;
        const float c1 = 1.f - std::pow(b1, static_cast<float>(t));
        const float c2 = 1.f - std::pow(b2, static_cast<float>(t));
        hipLaunchKernelGGL(MLPAdamKernel, dim3((kNParams + 255) / 256), dim3(256), 0,
                           ctx->stream, d.w, d.wb, d.wt, d.m1, d.m2, grad, lr, b1, b2, eps, c1, c2);
      }
      TD_HIP(hipGetLastError());
      std::vector<float> l(static_cast<size_t>(nb) * batch);
      TD_HIP(hipMemcpyAsync(l.data(), loss, 4ull * l.size(), hipMemcpyDeviceToHost,
                            ctx->stream));
      TD_HIP(hipStreamSynchronize(ctx->stream));
      double s = 0;
      for (float x : l) s += x;
      if (epoch_loss_out) epoch_loss_out[e] = l.empty() ? 0.f : static_cast<float>(s / l.size());
    }
    ctx->params["mlp.adam_t"] = t;
  });
}

// Labelled samples from the last td_dp_solve: random connected vertex sets
// (grown from a random vertex by random boundary vertices to a random size
// in [2, n]); outputs the induced graph relabelled to 0..|S|-1 (64 rows per
// sample), its optimal-root mask and td(S).
int td_mlp_make_samples(td_ctx* ctx, int32_t count, uint64_t seed, int32_t* n_out,
                        uint64_t* adj64_out, uint64_t* targets_out, uint8_t* td_out) {
  return Guard(ctx, [&] {
    TD_REQUIRE(ctx->have_dp, TD_E_STATE, "no td_dp_solve result to sample from");
    TD_REQUIRE(count >= 1 && n_out && adj64_out && targets_out, TD_E_INVALID,
               "bad arguments");
    const DPGraph& G = ctx->last_graph;
    const int n = static_cast<int>(G.n);
    TD_REQUIRE(n >= 2, TD_E_STATE, "graph too small to sample");
    std::mt19937_64 rng(seed);
    std::vector<uint32_t> sets(count);
    for (int i = 0; i < count; ++i) {
      uint32_t S = 0;
      for (int tries = 0; tries < 64 && __builtin_popcount(S) < 2; ++tries) {
        const int target = 2 + static_cast<int>(rng() % static_cast<uint64_t>(n - 1));
        const int start = static_cast<int>(rng() % static_cast<uint64_t>(n));
        S = 1u << start;
        while (__builtin_popcount(S) < target) {
          uint32_t bd = 0;
          for (uint32_t m = S; m; m &= m - 1) bd |= G.adj[__builtin_ctz(m)];
          bd &= ~S;
          if (!bd) break;
          int pick = static_cast<int>(rng() % static_cast<uint64_t>(__builtin_popcount(bd)));
          uint32_t b = bd;
          while (pick--) b &= b - 1;
          S |= b & (0u - b);
        }
      }
      sets[i] = S;
    }
    auto* dsets = static_cast<uint32_t*>(ctx->Buffer("mlp.lab.sets", 4ull * count));
    auto* dpos = static_cast<uint32_t*>(ctx->Buffer("mlp.lab.pos", 4ull * count));
    auto* dtd = static_cast<uint8_t*>(ctx->Buffer("mlp.lab.td", static_cast<size_t>(count)));
    TD_HIP(hipMemcpyAsync(dsets, sets.data(), 4ull * count, hipMemcpyHostToDevice, ctx->stream));
    DPLookup L;
    L.table = static_cast<const uint8_t*>(ctx->bufs["dp.arena"].p) + G.table;
    L.n = G.n;
    L.lb = G.lb;
    L.direct = G.direct;
    L.nh = G.nh;
    std::memcpy(L.lvl, G.lvl, sizeof(L.lvl));
    const uint32_t* cb = static_cast<const uint32_t*>(ctx->bufs["dp.pascal"].p);
    hipLaunchKernelGGL(LabelKernel, dim3(count), dim3(64), 0, ctx->stream, L, cb, dsets, dpos,
                       dtd);
    TD_HIP(hipGetLastError());
    std::vector<uint32_t> pos(count);
    std::vector<uint8_t> tds(count);
    TD_HIP(hipMemcpyAsync(pos.data(), dpos, 4ull * count, hipMemcpyDeviceToHost, ctx->stream));
    TD_HIP(hipMemcpyAsync(tds.data(), dtd, static_cast<size_t>(count), hipMemcpyDeviceToHost,
                          ctx->stream));
    TD_HIP(hipStreamSynchronize(ctx->stream));
    for (int i = 0; i < count; ++i) {
      const uint32_t S = sets[i];
      int map[32];
      int k = 0;
      for (int v = 0; v < 32; ++v) map[v] = (S >> v & 1u) ? k++ : -1;
      n_out[i] = k;
      uint64_t* rows = adj64_out + static_cast<size_t>(i) * 64;
      for (int r = 0; r < 64; ++r) rows[r] = 0;
      uint64_t tgt = 0;
      for (int v = 0; v < n; ++v) {
        if (map[v] < 0) continue;
        uint64_t row = 0;
        for (uint32_t m = G.adj[v] & S; m; m &= m - 1) row |= 1ull << map[__builtin_ctz(m)];
        rows[map[v]] = row;
        if (pos[i] >> v & 1u) tgt |= 1ull << map[v];
      }
      targets_out[i] = tgt;
      if (td_out) td_out[i] = tds[i];
    }
  });
}

}  // extern "C"
