// The diagonal elements by parities (diag_split and diag_value of host_logic.hpp)
// against the exact sum of the amplitudes of the terms that match (128-bit
// floating point), for operators with amplitudes that the rows do not share:
// exchange and fields beside penalties, projectors, densities, identities,
// repeated terms, masks past the words, infinities and NaN.  Sums of amplitudes
// within kDiagSpread of each other are plain ones.
#include <cmath>
#include <cstdio>
#include <limits>
#include <random>

#include "../../exactdiagonalization.jl_amd/csrc/host_logic.hpp"

using namespace edhip;

struct Terms {
  std::vector<uint64_t> mask, match;
  std::vector<double> amp;
  void add(uint64_t m, uint64_t c, double a) {
    mask.push_back(m);
    match.push_back(c);
    amp.push_back(a);
  }
  void bond(int i, int j, double h) {  // +h on parallel pairs, -h on antiparallel ones
    const uint64_t p = 1ull << i, q = 1ull << j;
    add(p | q, 0, h);
    add(p | q, p, -h);
    add(p | q, q, -h);
    add(p | q, p | q, h);
  }
};

static int check(const char* name, const Terms& T, int nb, std::mt19937_64& rng, size_t entries, bool carried) {
  const DiagSplit D = diag_split(T.mask, T.match, T.amp);
  if (D.entries.lin.size() != entries) return std::printf("%s: %zu entries\n", name, D.entries.lin.size()), 1;
  if (D.carried != carried) return std::printf("%s: carried %d\n", name, D.carried), 1;
  const std::vector<uint64_t> tab = mv_tables(D.entries, nb);
  std::vector<DiagSet> sets;
  for (size_t i = 0; i < D.sets.size(); ++i) sets.push_back(DiagSet{D.sets[i], D.coefs[i]});
  std::vector<DiagTerm> rest;
  for (size_t t : D.rest) rest.push_back(DiagTerm{T.mask[t], T.match[t], T.amp[t], 0.0});
  const uint64_t full = nb == 64 ? ~0ull : (1ull << nb) - 1;
  for (int k = 0; k < 2000; ++k) {
    const uint64_t b = k == 0 ? 0 : k == 1 ? full : k == 2 ? 0x5555555555555555ull & full : rng() & full;
    const auto value = carried ? diag_value<true, const uint64_t*> : diag_value<false, const uint64_t*>;
    const double got = value(tab.data(), sets.data(), D.first.data(), (int)D.first.size() - 1, mv_chunks(nb), rest.data(),
                             (int)rest.size(), b);
    __float128 want = 0;
    double plain = 0.0, sum = 0.0;
    for (size_t t = 0; t < T.mask.size(); ++t)
      if ((b & T.mask[t]) == T.match[t]) {
        want += T.amp[t];
        plain += T.amp[t];
        sum += std::fabs(T.amp[t]);
      }
    if (std::isnan(plain) || std::isinf(plain)) {
      if (std::isnan(plain) ? !std::isnan(got) : got != plain)
        return std::printf("%s: word %llx: %g, not %g\n", name, (unsigned long long)b, got, plain), 1;
      continue;
    }
    const double error = (double)(want - (__float128)got), exact = (double)want;
    // carried: half a unit of the result, and what the errors themselves round (200
    // values of at most 1e12, twice); plain: half a unit of the sum per addition
    const double bound = carried ? 1.2e-16 * std::fabs(exact) + 1e-16 : 1.2e-16 * sum * (double)T.mask.size();
    if (!(std::fabs(error) <= bound))
      return std::printf("%s: word %llx: %.17g, not %.17g (term by term %.17g)\n", name, (unsigned long long)b, got,
                         exact, plain), 1;
  }
  return 0;
}

int main() {
  std::mt19937_64 rng(11);
  const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
  for (int n : {16, 33, 64}) {
    Terms H;
    for (int i = 0; i < n; ++i) H.bond(i, (i + 1) % n, 0.25 + 0.37 * (i % 3));
    const size_t e = (size_t)n;
    if (check("exchange", H, n, rng, e, false)) return 1;
    for (double big : {1e3, 1e6, 1e8, 1e12, inf}) {
      Terms P = H;  // a penalty on parallel pairs two sites apart
      for (int i = 0; i < n; ++i) {
        const uint64_t p = 1ull << i, q = 1ull << ((i + 2) % n);
        P.add(p | q, 0, big);
        P.add(p | q, p | q, big);
      }
      if (check("penalty", P, n, rng, e, true)) return 1;
      Terms S = H;  // a projector on one site, a density on another, an identity that cancels it
      S.add(1ull << 3, 1ull << 3, -big);
      S.add(1ull << 5, 1ull << 5, 0.3);
      if (check("projector", S, n, rng, e, true)) return 1;
      S.add(0, 0, big);
      if (check("identity", S, n, rng, e, true)) return 1;
    }
    Terms F = H;  // fields: +h and -h on a site
    for (int i = 0; i < n; ++i) {
      F.add(1ull << i, 0, 0.1 * (1 + i % 2));
      F.add(1ull << i, 1ull << i, -0.1 * (1 + i % 2));
    }
    if (check("fields", F, n, rng, 2 * e, false)) return 1;
    Terms R = H;  // the same bonds again: sums that are exact, and sums that are not
    for (int i = 0; i < n; ++i) R.bond(i, (i + 1) % n, i % 2 ? 0.25 + 0.37 * (i % 3) : 1e12);
    size_t exact = 0;
    for (int i = 0; i < n; ++i) {
      const double a = 0.25 + 0.37 * (i % 3), b = i % 2 ? a : 1e12;
      exact += (__float128)(a + b) == (__float128)a + (__float128)b ? 1 : 0;
    }
    if (check("repeated", R, n, rng, exact, true)) return 1;
    Terms N = H;
    N.add(1ull << 2, 1ull << 2, nan);
    N.add(1ull << 4, 0, nan);
    N.add(1ull << 4, 1ull << 4, nan);
    if (check("nan", N, n, rng, e, true)) return 1;
    Terms V = H;  // infinite on both values of a site
    V.add(1ull << 2, 0, inf);
    V.add(1ull << 2, 1ull << 2, -inf);
    if (check("infinite field", V, n, rng, e, true)) return 1;
    if (n < 64) {  // masks with a bit past the words: never set
      Terms W = H;
      W.add(1ull << (n + 4), 1ull << (n + 4), 5.0);
      W.add((1ull << 63) | 1, 1, 0.5);
      if (check("past the words", W, n, rng, e, false)) return 1;
    }
  }
  std::printf("ok\n");
  return 0;
}
