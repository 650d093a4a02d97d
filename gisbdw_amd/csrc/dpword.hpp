// dpword.hpp -- the subset DP on words of 32 subsets (one bit per subset).
//
// Format.  td(S) and td(S \ v) differ by 0 or 1, so for a subset S all
// td(S \ v) lie in {m, m + 1}, and td modulo 4 is enough to order them.  A
// table holds three bits per subset: the 2-bit Gray code (g1 g0) of td mod 4
// (0 1 2 3 -> 00 01 11 10) and c = "S is connected".  Neighbouring codes
// differ in one bit, so the OR and the AND of the codes of the td(S \ v) tell
// both m and whether m + 1 occurs; neither needs a comparison.
//
// Word.  Vertices 0..4 are the word's: bit L of the words (g0, g1, c) of a
// set H of other vertices stands for S = H u L.  One bitwise instruction
// works on 32 subsets, where a byte per subset took four.
#pragma once
#include <cstdint>

#if defined(__HIPCC__)
#define TD_HD __host__ __device__ __forceinline__
#else
#define TD_HD inline
#endif

namespace tdhip {

struct DPWord {
  uint32_t g0, g1, c;
};

// OR and AND of the Gray planes and OR of the connectivity plane over the
// neighbours H \ x.  Any number of neighbours, none included.
struct DPFold {
  uint32_t o0 = 0u, a0 = ~0u, o1 = 0u, a1 = ~0u, oc = 0u;
  TD_HD void Add(uint32_t g0, uint32_t g1, uint32_t c) {
    o0 |= g0;
    a0 &= g0;
    o1 |= g1;
    a1 &= g1;
    oc |= c;
  }
  // two neighbours: three-input OR and AND
  TD_HD void Add2(const DPWord& p, const DPWord& q) {
    o0 = o0 | p.g0 | q.g0;
    a0 = a0 & p.g0 & q.g0;
    o1 = o1 | p.g1 | q.g1;
    a1 = a1 & p.g1 & q.g1;
    oc = oc | p.c | q.c;
  }
};

// OR over the word's vertices u of x at L \ u (for the L that hold u)
TD_HD uint32_t BelowAny(uint32_t x) {
  return (x << 16) | ((x & 0x00FF00FFu) << 8) | ((x & 0x0F0F0F0Fu) << 4) |
         ((x & 0x33333333u) << 2) | ((x & 0x55555555u) << 1);
}

// The word of H from the fold of the words of H \ x.
//   fine    bit L: no vertex of H u L is isolated in it (used for |S| >= 2)
//   single  bit L: H u L is a single vertex
//   empty   H is the empty set (no neighbours were folded)
//   any(x)  whether x != 0 in some lane (uniform); it only ends loops early
//
// Connectivity: S (|S| >= 2) is connected iff none of its vertices is
// isolated in S and some S \ v is connected: a least fixpoint over the word.
//
// Values, relative to b = the smallest td(H \ x), m' = (min over x of
// td(H \ x u L)) - b in [0, |L|]:  U_t = { L : td(H u L) - b <= t } for
// t = 0, 1, ...:
//   connected S:     some td(S \ v) <= t - 1: m' <= t - 1, or L \ u in U_{t-1};
//   disconnected S:  every td(S \ v) <= t: m' <= t - 1, or m' = t without
//                    t + 1 among the neighbours (d = 0), and L \ u in U_t for
//                    every u of L.  One pass over u in ascending order is
//                    enough for the last part: if it fails, a component K of S
//                    with td(K) > b + t keeps all of H, and from S down to K,
//                    the vertices of S \ K taken in descending order, every set
//                    before K is disconnected and so passes K's failure up.
// Each U_t takes about 25 instructions for 32 subsets, and the loop ends at
// the largest td(S) - b of the wave's words, 2 to 4 on the workloads' graphs.
template <typename Any>
TD_HD DPWord SolveWord(const DPFold& f, uint32_t fine, uint32_t single, bool empty, Any any) {
  uint32_t c = (f.oc & fine) | single;
  for (;;) {
    const uint32_t before = c;
    c |= ((c & 0x55555555u) << 1) & fine;
    c |= ((c & 0x33333333u) << 2) & fine;
    c |= ((c & 0x0F0F0F0Fu) << 4) & fine;
    c |= ((c & 0x00FF00FFu) << 8) & fine;
    c |= (c << 16) & fine;
    if (!any(c ^ before)) break;
  }
  const uint32_t d = (f.o0 ^ f.a0) | (f.o1 ^ f.a1);  // both m and m + 1 occur
  // Gray code of m mod 4
  const uint32_t m0 = empty ? 0u : f.a0 | (f.o0 & f.o1);
  const uint32_t m1 = empty ? 0u : f.a1 | (f.o1 & ~f.o0);
  // b = m at L = 0, as masks; subtracting b from a Gray code mod 4 swaps the
  // bits if b is odd and complements them by b's own bits
  const uint32_t s0 = 0u - (m0 & 1u), s1 = 0u - (m1 & 1u), odd = s0 ^ s1;
  const uint32_t r0 = ((m0 & ~odd) | (m1 & odd)) ^ s1;
  const uint32_t r1 = ((m1 & ~odd) | (m0 & odd)) ^ s0;
  // m' >= 4 (|L| >= 4 only): 0 mod 4 above an L \ u with 3, or above one
  // that is already past 4.  4-sets {0,1,2,3} from {0,1,2}, the others and
  // the full set from L \ 4.
  const uint32_t is0 = ~(r0 | r1), is3 = r1 & ~r0;
  uint32_t wrap = is0 & (((is3 << 16) & 0xE8800000u) | ((is3 << 8) & 0x8000u));
  wrap |= (wrap & 0x8000u) << 16;
  // m' <= 0, 1, 2, 3, 4
  uint32_t T[6] = {is0 & ~wrap, ~(r1 | wrap), (~r1 | r0) & ~wrap, ~wrap, ~(wrap & r0), ~0u};
  uint32_t okd = ~c & ~d;  // disconnected, all td(S \ x) equal
  if (empty) {  // no neighbours: the first condition never, the second always
#pragma unroll
    for (int t = 0; t < 6; ++t) T[t] = 0u;
    okd = 0u;
  }
  const uint32_t free_ = empty ? ~c : 0u;
  const uint32_t n0 = c | 0x55555555u, n1 = c | 0x33333333u, n2 = c | 0x0F0F0F0Fu,
                 n3 = c | 0x00FF00FFu, n4 = c | 0x0000FFFFu;
  uint32_t U = 0u, v0 = 0u, v1 = 0u;
#pragma unroll
  for (int t = 0; t < 6; ++t) {
    uint32_t X = (T[t] & okd) | free_;
    if (t > 0) X |= T[t - 1] | (c & BelowAny(U));
    X &= (X << 1) | n0;
    X &= (X << 2) | n1;
    X &= (X << 4) | n2;
    X &= (X << 8) | n3;
    X &= (X << 16) | n4;
    U = X;
    // past t: the code steps from t to t + 1
    if (t & 1) v1 ^= ~U;
    else v0 ^= ~U;
    if (!any(~U)) break;
  }
  // add b back
  const uint32_t g0 = ((v0 & ~odd) | (v1 & odd)) ^ s0;
  const uint32_t g1 = ((v1 & ~odd) | (v0 & odd)) ^ s1;
  return {g0, g1, c};
}

}  // namespace tdhip
