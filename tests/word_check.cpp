// Checks gisbdw_amd/csrc/dpword.hpp on the CPU: the word solver against the
// textbook recurrence, on every subset of random graphs, complete graphs and
// edgeless graphs with 1..14 vertices.  Prints "ok" and the word count.
#include <algorithm>
#include <cstdint>
#include <cstdio>
#include <random>
#include <vector>

#include "../gisbdw_amd/csrc/dpword.hpp"

int main() {
  std::mt19937 rng(7);
  long words = 0;
  for (int trial = 0; trial < 600; ++trial) {
    const int n = 1 + trial % 14, N = std::max(n, 5);
    const double p = trial % 5 == 0 ? 1.0 : trial % 7 == 0 ? 0.0 : (rng() % 1000) / 1000.0;
    std::vector<uint32_t> adj(N, 0);
    for (int i = 0; i < n; ++i)
      for (int j = i + 1; j < n; ++j)
        if ((rng() % 1000) / 1000.0 < p) {
          adj[i] |= 1u << j;
          adj[j] |= 1u << i;
        }
    std::vector<int> td(1u << N, 0);
    std::vector<char> conn(1u << N, 0);
    for (uint32_t S = 1; S < (1u << N); ++S) {
      uint32_t comp = S & (0u - S), front = comp;
      while (front) {
        uint32_t nb = 0;
        for (uint32_t m = front; m; m &= m - 1) nb |= adj[__builtin_ctz(m)];
        front = nb & S & ~comp;
        comp |= front;
      }
      conn[S] = comp == S;
      int lo = 99, hi = 0;
      for (uint32_t m = S; m; m &= m - 1) {
        lo = std::min(lo, td[S & ~(m & (0u - m))]);
        hi = std::max(hi, td[S & ~(m & (0u - m))]);
      }
      td[S] = conn[S] ? lo + 1 : hi;
    }
    std::vector<tdhip::DPWord> T(1u << (N - 5));
    for (uint32_t H = 0; H < (1u << (N - 5)); ++H) {
      tdhip::DPFold f;
      for (uint32_t m = H; m; m &= m - 1) {
        const tdhip::DPWord& w = T[H & ~(m & (0u - m))];
        f.Add(w.g0, w.g1, w.c);
      }
      uint32_t fine = 0, single = 0;
      for (uint32_t L = 0; L < 32; ++L) {
        const uint32_t S = (H << 5) | L;
        bool ok = true;
        for (uint32_t m = S; m; m &= m - 1) ok = ok && (adj[__builtin_ctz(m)] & S);
        if (ok) fine |= 1u << L;
        if (__builtin_popcount(S) == 1) single |= 1u << L;
      }
      T[H] = tdhip::SolveWord(f, fine, single, H == 0, [](uint32_t x) { return x != 0u; });
      ++words;
      for (uint32_t L = 0; L < 32; ++L) {
        const uint32_t S = (H << 5) | L;
        const uint32_t code = (T[H].g0 >> L & 1u) | (T[H].g1 >> L & 1u) << 1;
        if ((code ^ (code >> 1)) != (td[S] & 3u) || (T[H].c >> L & 1u) != (conn[S] ? 1u : 0u)) {
          std::printf("n = %d S = %x td = %d conn = %d: code %u c %u\n", n, S, td[S], conn[S],
                      code, T[H].c >> L & 1u);
          return 1;
        }
      }
    }
  }
  std::printf("ok %ld\n", words);
  return 0;
}
