// The rank tables of a sector against counting, and the products' entries (mv_split, mv_tables of host_logic.hpp) against the
// terms they stand for: every word matches the same flips with the same
// amplitudes, counted with multiplicity, as when each term is tested by itself.
#include <algorithm>
#include <cstdio>
#include <random>
#include <tuple>

#include "../../exactdiagonalization.jl_amd/csrc/host_logic.hpp"

using Image = std::tuple<uint64_t, double, double>;

static int run(std::mt19937_64& rng, int nb, int n_masks) {
  const uint64_t full = nb == 64 ? ~0ull : (1ull << nb) - 1;
  std::vector<edhip::OffTerm> v;
  for (int k = 0; k < n_masks; ++k) {
    uint64_t m = 0;
    const int bits = 1 + (int)(rng() % 3);
    while (__builtin_popcountll(m) < std::min(bits, nb)) m |= 1ull << (rng() % nb);
    const int n_terms = 1 + (int)(rng() % 4);
    const bool same = rng() % 2;
    const double a = 1.0 + (double)(rng() % 3);
    for (int t = 0; t < n_terms; ++t) {
      const uint64_t match = rng() & m & full;
      uint64_t flip = same ? m : (rng() & m);
      if (!flip) flip = m;
      v.push_back({m, match, match ^ flip, same ? a : a + t, same ? 0.0 : 0.25 * t});
    }
    if (same && rng() % 2) {  // the complement of the first of them: a pair that merges
      const edhip::OffTerm o = v[v.size() - (size_t)n_terms];
      v.push_back({m, o.match ^ m, o.image ^ m, o.are, o.aim});
    }
  }
  const edhip::MvSplit S = edhip::mv_split(v, n_masks % 2 == 1);
  for (size_t e = 1; n_masks % 2 == 1 && e < S.lin.size(); ++e)
    if (__builtin_ctzll(S.lin[e].flip) > __builtin_ctzll(S.lin[e - 1].flip)) return std::printf("order\n"), 1;
  const std::vector<uint64_t> tab = edhip::mv_tables(S, nb);
  const int nc = edhip::mv_chunks(nb);
  if (nc % 3 || 4 * nc < nb) return std::printf("chunks\n"), 1;
  if (S.q.size() != S.lin.size() || S.c.size() != S.lin.size() || S.rest.size() % 2) return std::printf("sizes\n"), 1;
  for (size_t e = 0; e < S.rest.size(); e += 2)
    if (S.rest[e].mask != S.rest[e + 1].mask) return std::printf("pairs\n"), 1;
  for (int w = 0; w < 200; ++w) {
    const uint64_t b = w == 0 ? 0 : w == 1 ? full : rng() & full;
    std::vector<Image> want, got;
    for (const auto& t : v)
      if ((b & t.mask) == t.match) want.emplace_back((b & ~t.mask) | t.image, t.are, t.aim);
    for (size_t s = 0; s * 64 < S.lin.size(); ++s) {
      uint64_t bits = 0;
      for (int k = 0; k < nc; ++k) bits ^= tab[(s * nc + k) * 16 + (4 * k < 64 ? (b >> (4 * k)) & 15 : 0)];
      for (int j = 0; j < 64; ++j)
        if ((bits >> j) & 1) {
          if (s * 64 + j >= S.lin.size()) return std::printf("bit past the entries\n"), 1;
          const auto& e = S.lin[s * 64 + j];
          got.emplace_back(b ^ e.flip, e.are, e.aim);
        }
    }
    for (const auto& t : S.rest)
      if ((b & t.mask) == t.match) got.emplace_back(b ^ (t.match ^ t.image), t.are, t.aim);
    std::sort(want.begin(), want.end());
    std::sort(got.begin(), got.end());
    if (want != got) return std::printf("nb %d masks %d: word %llx differs\n", nb, n_masks, (unsigned long long)b), 1;
  }
  return 0;
}

// The rank tables against counting, word by word.
static int ranks(int n, int pop) {
  const edhip::RankTables T = edhip::rank_tables(n, pop);
  uint32_t rank = 0;
  for (uint64_t w = 0; w < (1ull << n); ++w)
    if (__builtin_popcountll(w) == pop) {
      const uint32_t got = T.base[w >> T.low_bits] + T.low[w & ((1ull << T.low_bits) - 1)];
      if (got != rank++) return std::printf("rank of %llx in (%d, %d): %u\n", (unsigned long long)w, n, pop, got), 1;
    }
  return T.base.size() % 4 ? 1 : 0;
}

int main() {
  for (int n : {1, 3, 11, 12, 13, 14, 20})
    for (int pop : {0, 1, 2, n / 2, n})
      if (pop <= n && ranks(n, pop)) return 1;
  for (int pop : {0, 2, 12, 13, 26})
    if (ranks(pop == 12 ? 24 : 26, pop == 12 ? 12 : std::min(pop, 26))) return 1;
  std::mt19937_64 rng(7);
  for (int nb : {1, 2, 5, 12, 13, 36, 37, 63, 64})
    for (int n_masks : {0, 1, 3, 63, 64, 65, 130, 300})
      if (run(rng, nb, n_masks)) return 1;
  std::printf("ok\n");
  return 0;
}
