// The window canonicaliser (window.hpp) against the smallest image by brute
// force over all translations, on every shape and chain length it covers.
#include <cstdio>
#include <random>

#include "../../exactdiagonalization.jl_amd/csrc/host_logic.hpp"

using namespace edhip;

static uint64_t translate(uint64_t b, int Lx, int Ly, int pos) {
  const int a = pos % Lx, s = pos / Lx;
  uint64_t out = 0;
  for (int y = 0; y < Ly; ++y)
    for (int x = 0; x < Lx; ++x)
      if ((b >> (x + Lx * y)) & 1) out |= 1ull << ((x + a) % Lx + Lx * ((y + s) % Ly));
  return out;
}

template <int KIND, int LX, int LY>
static int check(int Lx, int Ly, std::mt19937_64& rng) {
  using S = Win<KIND, LX, LY>;
  const int n = Lx * Ly;
  const std::vector<uint16_t> tab = win_table(Lx, Ly);
  const std::vector<int> pos = win_positions(Lx, Ly);
  if ((int)tab.size() != S::kTab) return std::printf("%d x %d: table size\n", Lx, Ly), 1;
  const uint64_t full = (1ull << n) - 1;
  for (int k = 0; k < 3000; ++k) {
    uint64_t b = rng() & full;
    if (k % 3 == 1) b &= rng();           // sparse
    if (k % 3 == 2) {                     // periodic in x or in y: several translations give the least image
      const uint64_t row = rng() & ((1ull << Lx) - 1);
      b = 0;
      for (int y = 0; y < Ly; ++y) b |= row << (Lx * y);
      if (k & 1) b = (rng() & 1) ? b : (0x5555555555555555ull & full);
    }
    if (k < 2) b = k ? full : 0;
    uint64_t want = ~0ull;
    for (int p = 0; p < n; ++p) want = std::min(want, translate(b, Lx, Ly, p));
    typename S::W s;
    int bit;
    S::canonical(tab.data(), (typename S::W)b, n, s, bit);
    if ((uint64_t)s != want || S::position(bit) != pos[bit] || translate(b, Lx, Ly, pos[bit]) != want)
      return std::printf("%d x %d: %llx -> %llx (bit %d), not %llx\n", Lx, Ly, (unsigned long long)b,
                         (unsigned long long)s, bit, (unsigned long long)want), 1;
  }
  return 0;
}

static uint64_t permuted(uint64_t b, const std::vector<int32_t>& perm) {
  uint64_t out = 0;
  for (size_t i = 0; i < perm.size(); ++i)
    if ((b >> i) & 1) out |= 1ull << perm[i];
  return out;
}

// Point operations: variants (bits) alone or with their transposes.
template <int L>
static int check_point(int variants, int swap, std::mt19937_64& rng) {
  using S = Win<kWinPoint, L, L>;
  using W = typename S::W;
  const int n = L * L;
  const std::vector<uint16_t> tab = win_point_table(L, variants);
  if (2 * tab.size() != S::kTabBytes) return std::printf("point %d: table size\n", L), 1;
  std::vector<std::vector<int32_t>> perms;
  for (int code = 0; code < 512; ++code)
    if ((code & 7) < L && ((code >> 3) & 7) < L && ((variants >> ((code >> 6) & 3)) & 1) && (swap || code < 256))
      perms.push_back(win_point_perm(L, code));
  const uint64_t full = (1ull << n) - 1;
  for (int k = 0; k < 1500; ++k) {
    uint64_t row = rng() & full;
    if (k % 4 == 1) row &= rng();
    if (k % 4 == 2) {  // symmetric: many candidates
      const uint64_t line = rng() & ((1ull << L) - 1);
      row = 0;
      for (int y = 0; y < L; ++y) row |= line << (L * y);
      row ^= (k & 4) ? 0 : S::transposed((W)row);
    }
    if (k < 2) row = k ? full : 0;
    const uint64_t flip = (k % 3) ? (1ull << (rng() % n)) ^ (1ull << (rng() % n)) : 0;
    uint64_t want = ~0ull;
    for (const auto& p : perms) want = std::min(want, permuted(row ^ flip, p));
    W s;
    int code;
    const W b = (W)(row ^ flip), bt = swap ? S::transposed((W)row) ^ S::transposed((W)flip) : b;
    S::template canonical<true>(tab.data(), b, bt, swap ? S::kWindows : S::kUpright, s, code);
    if ((uint64_t)s != want || permuted(row ^ flip, win_point_perm(L, code)) != want)
      return std::printf("point %d, variants %d, swap %d: %llx -> %llx (code %d), not %llx\n", L, variants, swap,
                         (unsigned long long)(row ^ flip), (unsigned long long)s, code, (unsigned long long)want), 1;
  }
  return 0;
}

int main() {
  std::mt19937_64 rng(3);
  for (int swap = 0; swap < 2; ++swap)
    for (int variants : {1, 3, 5, 9, 15})
      if (check_point<5>(variants, swap, rng) || check_point<6>(variants, swap, rng)) return 1;
#define EDHIP_X(K, X, Y) \
  if (check<K, X, Y>(X, Y, rng)) return 1;
  EDHIP_WIN_SHAPES(EDHIP_X)
#undef EDHIP_X
  for (int n = 12; n <= 32; ++n)
    if (check<kWinChain, 32, 1>(n, 1, rng)) return 1;
  for (int n = 12; n <= 48; ++n)
    if (check<kWinChain, 48, 1>(n, 1, rng)) return 1;
  std::printf("ok\n");
  return 0;
}
