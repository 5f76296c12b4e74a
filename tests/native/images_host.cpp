// The images of the products' entries stay words of the space: for terms on any of
// 64 bits, those of off_term, split as the products take them (mv_split), against
// the terms whose images have no bit past the words, in the order-free sense of
// equal lists.
#include <algorithm>
#include <cstdio>
#include <random>
#include <tuple>

#include "../../exactdiagonalization.jl_amd/csrc/host_logic.hpp"

using namespace edhip;

int main() {
  std::mt19937_64 rng(5);
  for (int nb : {1, 11, 12, 24, 25, 31, 32, 33, 36, 63, 64})
    for (int round = 0; round < 40; ++round) {
      const uint64_t full = nb >= 64 ? ~0ull : (1ull << nb) - 1;
      std::vector<OffTerm> all, kept;
      for (int k = 0; k < 90; ++k) {
        const int reach = std::min(64, nb + (k % 3 == 0 ? 0 : k % 3 == 1 ? 1 : 40));
        const uint64_t p = 1ull << (rng() % reach), q = 1ull << (rng() % reach), m = p | q;
        const uint64_t match = rng() & m, image = k % 2 ? match ^ m : rng() & m;
        if (match == image) continue;
        const double a = 1.0 + (double)(rng() % 2);
        all.push_back(OffTerm{m, match, image, a, 0.0});
        if (k % 2) all.push_back(OffTerm{m, image, match, a, 0.0});
      }
      for (const OffTerm& t : all) kept.push_back(off_term(t.mask, t.match, t.image, t.are, t.aim, nb));
      const MvSplit S = mv_split(kept, round % 2 == 0);
      for (int w = 0; w < 60; ++w) {
        const uint64_t b = w == 0 ? 0 : w == 1 ? full : rng() & full;
        std::vector<std::tuple<uint64_t, double>> want, got;
        for (const OffTerm& t : all) {
          const uint64_t s = (b & ~t.mask) | t.image;
          if ((b & t.mask) == t.match && (s & ~full) == 0) want.emplace_back(s, t.are);
        }
        for (size_t e = 0; e < S.lin.size(); ++e)
          if (((__builtin_popcountll(b & S.q[e]) & 1) ^ S.c[e]) == 1) got.emplace_back(b ^ S.lin[e].flip, S.lin[e].are);
        for (const OffTerm& t : S.rest)
          if ((b & t.mask) == t.match) got.emplace_back(b ^ (t.match ^ t.image), t.are);
        std::sort(want.begin(), want.end());
        std::sort(got.begin(), got.end());
        if (want != got) return std::printf("%d bits, word %llx: images differ\n", nb, (unsigned long long)b), 1;
      }
    }
  std::printf("ok\n");
  return 0;
}
