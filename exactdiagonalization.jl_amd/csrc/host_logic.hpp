// Host-side logic with no device code, so that a host-only build (with
// sanitizers) can test it: the linear algebra of the eigensolver's small
// projected (tridiagonal or arrowhead) matrices, and the closure and
// inverses of a symmetry group given as bit permutations with XOR words, and
// the split of an operator's terms into the products' entries.
#pragma once

#include <stdint.h>

#include <algorithm>
#include <cmath>
#include <map>
#include <string>
#include <utility>
#include <vector>

#include "window.hpp"

namespace edhip {

// A launch of n_blocks blocks in two grid dimensions (numbered x first, the last
// row partly past n_blocks): a dimension holds fewer than 2^32 lanes, which one
// alone passes at 2^26 columns with a wave each.
struct BlockGrid {
  uint32_t x, y;
};
inline BlockGrid block_grid(uint64_t n_blocks) {
  const uint64_t x = std::min<uint64_t>(std::max<uint64_t>(n_blocks, 1), 1ull << 22);
  return BlockGrid{(uint32_t)x, (uint32_t)((n_blocks + x - 1) / x)};
}

// Rank tables of the n-bit words of popcount pop: rank(w) = base[w >> low_bits]
// + low[w & mask], low the rank of a low_bits-bit word among those of its
// popcount, base the number of words whose upper part is smaller.  base is
// padded to whole 16 bytes.
struct RankTables {
  int low_bits = 0;
  std::vector<uint16_t> low;
  std::vector<uint32_t> base;
};
inline RankTables rank_tables(int n, int pop) {
  RankTables T;
  T.low_bits = n <= 24 ? 12 : 13;
  T.low.resize((size_t)1 << T.low_bits);
  std::vector<uint32_t> of_pop((size_t)T.low_bits + 1, 0);
  for (size_t w = 0; w < T.low.size(); ++w) T.low[w] = (uint16_t)of_pop[(size_t)__builtin_popcountll(w)]++;
  const int hi = std::max(0, n - T.low_bits);
  uint32_t sum = 0;
  for (size_t w = 0; w < ((size_t)1 << hi); ++w) {
    T.base.push_back(sum);
    const int need = pop - __builtin_popcountll(w);
    // (a lower part wider than the word has its upper bits clear)
    if (need >= 0 && need <= T.low_bits && n >= T.low_bits) sum += of_pop[(size_t)need];
  }
  while (T.base.size() % 4) T.base.push_back(sum);
  return T;
}

// The values of n bits by popcount, ascending, and the offset of each popcount.
struct PopLists {
  std::vector<int32_t> list, off;
};
inline PopLists pop_lists(int n) {
  PopLists P;
  for (int p = 0; p <= n; ++p) {
    P.off.push_back((int32_t)P.list.size());
    for (int32_t w = 0; w < (1 << n); ++w)
      if (__builtin_popcount((unsigned)w) == p) P.list.push_back(w);
  }
  P.off.push_back((int32_t)P.list.size());
  return P;
}

// Window table of an Lx x Ly torus (window.hpp): entry = rank << mask bits | mask.
inline std::vector<uint16_t> win_table(int Lx, int Ly) {
  const int kind = win_kind(Lx, Ly);
  if (kind == kWinNone) return {};
  const int nv = 1 << win_index_bits(kind, Lx), mb = win_mask_bits(kind);
  const int na = kind == kWinChain ? 6 : Lx;
  const uint32_t rm = (1u << std::min(Lx, 12)) - 1u;
  auto rot = [&](uint32_t v, int a) { return ((v << a) | (v >> (Lx - a))) & rm; };
  auto beginning = [&](uint32_t v, int a) -> uint32_t {
    if (kind == kWinChain) return (v >> (5 - a)) & 127u;
    if (kind == kWinRows) return rot(v, a);
    return (rot(v >> Lx, a) << Lx) | rot(v & rm, a);
  };
  std::vector<uint32_t> least(nv, ~0u), mask(nv, 0);
  for (int v = 0; v < nv; ++v)
    for (int a = 0; a < na; ++a) {
      const uint32_t x = beginning((uint32_t)v, a);
      if (x < least[v]) least[v] = x, mask[v] = 0;
      if (x == least[v]) mask[v] |= 1u << a;
    }
  std::vector<uint32_t> order(least);
  std::sort(order.begin(), order.end());
  order.erase(std::unique(order.begin(), order.end()), order.end());
  std::vector<uint16_t> tab(nv);
  for (int v = 0; v < nv; ++v) {
    const size_t rank = (size_t)(std::lower_bound(order.begin(), order.end(), least[v]) - order.begin());
    tab[v] = (uint16_t)(rank << mb | mask[v]);
  }
  return tab;
}

// a + Lx b of the translation of every candidate bit 8 y + a (0 past the last).
inline std::vector<int> win_positions(int Lx, int Ly) {
  std::vector<int> pos(64, 0);
  const bool chain = win_kind(Lx, Ly) == kWinChain;
  for (int bit = 0; bit < 64; ++bit) {
    const int y = bit >> 3, a = bit & 7;
    if (chain ? (a < 6 && 6 * y + a < Lx) : (a < Lx && y < Ly)) pos[bit] = chain ? 6 * y + a : a + Lx * (Ly - 1 - y);
  }
  return pos;
}

// Tables of Win<kWinPoint, L, L> for the variants in the mask (bit 0 of a variant
// reverses the bits of the rows, bit 1 their order).
inline std::vector<uint16_t> win_point_table(int L, int variants) {
  const uint32_t nv = 1u << (2 * L), rm = (1u << L) - 1u;
  auto framed = [&](uint32_t v, int f) {  // frame f = 8 reversed + rotation
    uint32_t o = 0;
    for (int i = 0; i < L; ++i) o |= ((v >> i) & 1u) << (((f >> 3 ? L - 1 - i : i) + (f & 7)) % L);
    return o;
  };
  // sets of frames (bit f), numbered as they occur
  std::map<uint32_t, int> number{{0u, 0}};
  std::vector<uint32_t> sets{0u};
  auto class_of = [&](uint32_t set) {
    auto it = number.emplace(set, (int)sets.size());
    if (it.second) sets.push_back(set);
    return it.first->second;
  };
  std::vector<uint16_t> tab((size_t)nv * 2 + ((size_t)kPointClasses << L) + kPointClasses, 0);
  for (uint32_t w = 0; w < nv; ++w) {
    uint32_t least = ~0u, set[2] = {0, 0};
    for (int v = 0; v < 4; ++v)
      for (int a = 0; a < L; ++a) {
        if (!((variants >> v) & 1)) continue;
        const int f = 8 * (v & 1) + a;
        const uint32_t hi = framed(v & 2 ? w & rm : w >> L, f), lo = framed(v & 2 ? w >> L : w & rm, f);
        const uint32_t x = (hi << L) | lo;
        if (x < least) least = x, set[0] = set[1] = 0;
        if (x == least) set[v >> 1] |= 1u << f;
      }
    tab[w] = (uint16_t)least;
    tab[nv + w] = (uint16_t)(class_of(set[0]) | class_of(set[1]) << 8);
  }
  for (size_t c = 0; c < sets.size(); ++c) {  // (grows by the classes that the rows leave)
    if (c >= (size_t)kPointClasses) return {};
    const uint32_t set = sets[c];
    for (uint32_t r = 0; r <= rm && set; ++r) {
      uint32_t least = ~0u, left = 0;
      for (int f = 0; f < 16; ++f) {
        if (!((set >> f) & 1)) continue;
        const uint32_t x = framed(r, f);
        if (x < least) least = x, left = 0;
        if (x == least) left |= 1u << f;
      }
      tab[2 * nv + (c << L) + r] = (uint16_t)((uint32_t)class_of(left) << L | least);
    }
    tab[2 * nv + ((size_t)kPointClasses << L) + c] = (uint16_t)(set ? __builtin_ctz(set) : 0);
  }
  return tab;
}

// The bit permutation of a candidate code of Win<kWinPoint, L, L>.
inline std::vector<int32_t> win_point_perm(int L, int code) {
  const int v = (code >> 6) & 3, top = (code >> 3) & 7, a = code & 7;
  std::vector<int32_t> perm((size_t)(L * L));
  for (int y = 0; y < L; ++y)
    for (int x = 0; x < L; ++x) {
      int i = x, j = y;
      if (code >> 8) std::swap(i, j);
      if (v & 1) i = L - 1 - i;
      if (v & 2) j = L - 1 - j;
      perm[(size_t)(x + L * y)] = (i + a) % L + L * ((j + L - 1 - top) % L);
    }
  return perm;
}

// Off-diagonal term as the products see it: the row b matches iff
// (b & mask) == match; its image is (b & ~mask) | image.
struct OffTerm {
  uint64_t mask, match, image;
  double are, aim;
};

// A term as it acts on words of n_bits bits: one whose match or image has a bit
// past them takes no word to another, and is made to match none.  (The kernels that
// find an image by its position alone need every image to be such a word.)
inline OffTerm off_term(uint64_t mask, uint64_t match, uint64_t image, double are, double aim, int n_bits) {
  const uint64_t past = n_bits >= 64 ? 0ull : ~0ull << n_bits;
  if ((match | image) & past) return OffTerm{0, 1, 1, 0.0, 0.0};
  return OffTerm{mask, match, image, are, aim};
}

// One entry of the products: a matching row b has the image b ^ flip.
struct MvEntry {
  uint64_t flip;
  double are, aim;
};

// Parity entries of a list of terms (mv_split): entry e matches b iff
// parity(b & q[e]) ^ c[e] is 1.
struct MvSplit {
  std::vector<uint64_t> q;
  std::vector<int> c;
  std::vector<MvEntry> lin;   // the parity entries
  std::vector<OffTerm> rest;  // the other terms, runs of equal masks padded to even lengths
};

// Two terms on one mask of one or two bits with the same flip and amplitude
// whose matches are each other's complement match together wherever the parity
// of the masked bits has one value (two bits: 01 and 10, or 00 and 11), or
// everywhere (one bit: 0 and 1): S+S- + S-S+ bonds, transverse fields.  The
// padding terms of rest keep the mask, match nothing (a match outside the
// mask) and flip nothing.
// by_low_bit: the parity entries in descending order of the lowest bit they
// flip, else in the order of the terms.
inline MvSplit mv_split(const std::vector<OffTerm>& v, bool by_low_bit = false) {
  MvSplit S;
  std::vector<char> used(v.size(), 0);
  for (size_t i = 0; i < v.size();) {
    size_t j = i;
    while (j < v.size() && v[j].mask == v[i].mask) ++j;
    const uint64_t m = v[i].mask;
    const int bits = __builtin_popcountll(m);
    for (size_t a = i; a < j && (bits == 1 || bits == 2); ++a)
      for (size_t b = a + 1; b < j && !used[a]; ++b) {
        if (used[b] || (v[a].match ^ v[b].match) != m || (v[a].match ^ v[a].image) != (v[b].match ^ v[b].image) ||
            v[a].are != v[b].are || v[a].aim != v[b].aim)
          continue;
        used[a] = used[b] = 1;
        S.q.push_back(bits == 2 ? m : 0);
        S.c.push_back(bits == 2 ? 1 ^ (__builtin_popcountll(v[a].match) & 1) : 1);
        S.lin.push_back(MvEntry{v[a].match ^ v[a].image, v[a].are, v[a].aim});
      }
    size_t kept = 0;
    for (size_t a = i; a < j; ++a)
      if (!used[a]) {
        S.rest.push_back(v[a]);
        ++kept;
      }
    if (kept & 1) S.rest.push_back(OffTerm{m, ~m, ~m, 0.0, 0.0});
    i = j;
  }
  if (by_low_bit) {
    std::vector<size_t> at(S.lin.size());
    for (size_t e = 0; e < at.size(); ++e) at[e] = e;
    std::stable_sort(at.begin(), at.end(), [&](size_t a, size_t b) {
      return __builtin_ctzll(S.lin[a].flip) > __builtin_ctzll(S.lin[b].flip);
    });
    const MvSplit T = S;
    for (size_t e = 0; e < at.size(); ++e) {
      S.q[e] = T.q[at[e]];
      S.c[e] = T.c[at[e]];
      S.lin[e] = T.lin[at[e]];
    }
  }
  return S;
}

// 4-bit chunks of nb-bit words, rounded up to a multiple of 3 (the unroll of
// the kernels' loop over them).
inline int mv_chunks(int nb) { return ((nb + 3) / 4 + 2) / 3 * 3; }

// The parity tables: bit e of the XOR over the chunks k of entry
// [segment][k][k-th chunk of b] tells whether entry 64 segment + e matches b.
inline std::vector<uint64_t> mv_tables(const MvSplit& S, int nb) {
  const int nc = mv_chunks(nb);
  const size_t n_seg = (S.lin.size() + 63) / 64;
  std::vector<uint64_t> tab(n_seg * (size_t)nc * 16, 0);
  for (size_t e = 0; e < S.lin.size(); ++e)
    for (int k = 0; k < nc; ++k)
      for (int x = 0; x < 16; ++x) {
        const uint64_t part = 4 * k < 64 ? (uint64_t)x << (4 * k) : 0;
        const int bit = (__builtin_popcountll(part & S.q[e]) & 1) ^ (k == 0 ? S.c[e] : 0);
        if (bit) tab[((e / 64) * nc + (size_t)k) * 16 + (size_t)x] |= 1ull << (e % 64);
      }
  return tab;
}

// LDS offsets of the products' entries, from mv_lds.
struct MvLayout {
  uint32_t off_mm, off_fa, off_ai, total;
};
EDHIP_HD MvLayout mv_layout(int n_lin, int n_chunk, int n_rest, int paired) {
  MvLayout Y;
  Y.off_mm = (uint32_t)(((n_lin + 63) / 64) * n_chunk) * 128u;
  Y.off_fa = (Y.off_mm + (uint32_t)(paired ? n_rest / 2 * 24 : n_rest * 16) + 15u) & ~15u;
  Y.off_ai = Y.off_fa + (uint32_t)(n_lin + n_rest) * 16u;
  Y.total = Y.off_ai + (uint32_t)(n_lin + n_rest) * 8u;
  return Y;
}

// How an operator's terms find room in the 64 KiB of LDS beside its group's tables
// (group bytes, fewer without the row-pair table) and the rank table (rank bytes):
// plain, the list of the terms, always staged by the kernels that walk it, and full,
// the products' entries with their tables.  Entries, else the terms one by one, else
// the same without the row-pair table; what is accepted is decided by the plain list
// alone.
struct LdsPlan {
  bool one_by_one, drop_pairs;
};
inline LdsPlan lds_plan(uint32_t group, uint32_t group_without_pairs, uint32_t plain, uint32_t full, uint32_t rank) {
  const uint32_t most = std::max(plain, full);
  auto fits = [&](uint32_t g, uint32_t terms) { return g + terms + rank <= 64u * 1024u; };
  if (fits(group, most)) return {false, false};
  if (fits(group, plain)) return {true, false};
  return {!fits(group_without_pairs, most) && fits(group_without_pairs, plain), group_without_pairs != group};
}

// Diagonal term: adds its amplitude to the rows b with (b & mask) == match.
struct DiagTerm {
  uint64_t mask, match;
  double are, aim;
};

// A sum of doubles whose rounding errors are kept beside it: the result is the
// exact sum rounded about once.  An infinite or NaN sum is that of plain addition.
struct CarriedSum {
  double hi = 0.0, lo = 0.0;
  EDHIP_HD void add(double x) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
    const double s = hi + x, t = s - hi;
    lo += (hi - (s - t)) + (x - t);
    hi = s;
  }
  // coef * count
  EDHIP_HD void add_multiple(double coef, int count) {
#ifdef __clang__
#pragma clang fp contract(off)
#endif
    const double p = coef * (double)count;
    const double rest = __builtin_fma(coef, (double)count, -p);
    add(p);
    lo += rest;
  }
  EDHIP_HD double value() const {
    const double v = hi + lo;
    return v - v == 0.0 ? v : hi;
  }
};

// A diagonal operator with real amplitudes, sum of a_t [b & mask_t == match_t], by
// parities: masks of one or two sites whose amplitudes are +h where the parity of
// the masked bits is even and -h where it is odd (exchange, fields) become entries
// (parity mask, h); the entries of one h sum to h (even ones - odd ones), a product
// with an integer.  All other masks stay terms: split into a mean and +-h, a term
// would add its mean to rows that it does not touch and take it away again, and a
// row's element would carry the rounding of amplitudes that are not its own (a
// penalty of 1e8 on parallel pairs: 7e-8 on the rows without one).
//
// The sums run in an order of their own.  Where the amplitudes differ by more than
// kDiagSpread, what cancels in a row may be added apart, and they carry their
// rounding errors (4x6 XXZ, 48 coefficients, 2.7M rows: 86 us, 50 without).
constexpr double kDiagSpread = 64.0;
struct DiagSplit {
  MvSplit entries;            // q, c and one lin entry (are: h) each
  std::vector<size_t> rest;   // terms left
  std::vector<uint64_t> sets; // per segment and coefficient: the entries' bits
  std::vector<double> coefs;
  std::vector<int32_t> first; // offsets of the segments
  bool carried = false;       // the sums carry their rounding errors
};
inline DiagSplit diag_split(const std::vector<uint64_t>& mask, const std::vector<uint64_t>& match,
                            const std::vector<double>& amp) {
  DiagSplit D;
  std::map<uint64_t, std::vector<size_t>> by_mask;
  for (size_t t = 0; t < mask.size(); ++t) by_mask[mask[t]].push_back(t);
  std::vector<std::pair<double, uint64_t>> found;  // h, parity mask
  for (const auto& [m, ts] : by_mask) {
    const uint64_t lowest = m & (~m + 1);
    double f[4] = {0, 0, 0, 0};  // by (upper bit, lower bit)
    bool exact = true;           // several amplitudes of one pattern add up without rounding
    for (size_t t : ts) {
      double& s = f[((match[t] & lowest) ? 1 : 0) + ((match[t] & m & ~lowest) ? 2 : 0)];
      CarriedSum c;
      c.add(s);
      c.add(amp[t]);
      exact = exact && c.lo == 0.0;  // (false for infinities and NaN)
      s = c.hi;
    }
    const int n = __builtin_popcountll(m);
    if (exact && f[0] == -f[1] && (n == 1 || (n == 2 && f[0] == f[3] && f[1] == f[2]))) {
      if (f[0] != 0.0) found.emplace_back(f[0], m);
    } else {
      D.rest.insert(D.rest.end(), ts.begin(), ts.end());
    }
  }
  std::sort(D.rest.begin(), D.rest.end());
  std::sort(found.begin(), found.end());  // equal coefficients together
  for (size_t e = 0; e < found.size(); ++e) {
    if (e % 64 == 0) D.first.push_back((int32_t)D.sets.size());
    if (e % 64 == 0 || found[e].first != D.coefs.back()) {
      D.sets.push_back(0);
      D.coefs.push_back(found[e].first);
    }
    D.sets.back() |= 1ull << (e % 64);
    D.entries.q.push_back(found[e].second);
    D.entries.c.push_back(0);
    D.entries.lin.push_back(MvEntry{0, found[e].first, 0.0});
  }
  D.first.push_back((int32_t)D.sets.size());
  double least = INFINITY, most = 0.0;
  auto seen = [&](double a) {
    a = std::fabs(a);
    if (!std::isfinite(a)) D.carried = true;
    if (!(a > 0.0)) return;
    least = std::min(least, a);
    most = std::max(most, a);
  };
  for (double c : D.coefs) seen(c);
  for (size_t t : D.rest) seen(amp[t]);
  D.carried = D.carried || most > kDiagSpread * least;
  return D;
}

// Entries of one segment (bits of mask) that share a coefficient.
struct DiagSet {
  uint64_t mask;
  double coef;
};

// The diagonal element of the word b from the entries' tables (mv_tables, n_seg
// segments of n_chunk chunks), their sets by segment and the terms left.
template <bool CARRIED, typename P>
EDHIP_HD double diag_value(P tab, const DiagSet* sets, const int32_t* first, int n_seg, int n_chunk,
                           const DiagTerm* rest, int n_rest, uint64_t b) {
  CarriedSum v;
  double plain = 0.0;
  for (int seg = 0; seg < n_seg; ++seg) {
    uint64_t bits = 0;
    for (int k = 0; k < n_chunk; ++k)
      bits ^= tab[((seg * n_chunk + k) << 4) + (int)((b >> ((4 * k) & 63)) & 15ull)];
    for (int i = first[seg]; i < first[seg + 1]; ++i) {
      const int count = __builtin_popcountll(sets[i].mask) - 2 * __builtin_popcountll(bits & sets[i].mask);
      if (CARRIED)
        v.add_multiple(sets[i].coef, count);
      else
        plain += sets[i].coef * (double)count;
    }
  }
  for (int t = 0; t < n_rest; ++t)
    if ((b & rest[t].mask) == rest[t].match) {
      if (CARRIED)
        v.add(rest[t].are);
      else
        plain += rest[t].are;
    }
  return CARRIED ? v.value() : plain;
}

// Householder reduction of a dense symmetric matrix (row-major, n x n) to
// tridiagonal form A = Q T Q^T; returns d (diagonal), e (e[i] = T[i][i+1]).
inline void householder_tridiag(int n, std::vector<double>& A, std::vector<double>& Q, std::vector<double>& d,
                                std::vector<double>& e) {
  Q.assign((size_t)n * n, 0.0);
  for (int i = 0; i < n; ++i) Q[(size_t)i * n + i] = 1.0;
  std::vector<double> v(n), p(n), w(n);
  for (int k = 0; k + 2 < n; ++k) {
    double nx = 0.0;
    for (int i = k + 1; i < n; ++i) nx += A[(size_t)i * n + k] * A[(size_t)i * n + k];
    nx = std::sqrt(nx);
    if (nx == 0.0) continue;
    double x0 = A[(size_t)(k + 1) * n + k];
    double alpha = (x0 >= 0) ? -nx : nx;
    for (int i = 0; i < n; ++i) v[i] = 0.0;
    for (int i = k + 1; i < n; ++i) v[i] = A[(size_t)i * n + k];
    v[k + 1] -= alpha;
    double vn = 0.0;
    for (int i = k + 1; i < n; ++i) vn += v[i] * v[i];
    vn = std::sqrt(vn);
    if (vn == 0.0) continue;
    for (int i = k + 1; i < n; ++i) v[i] /= vn;
    // p = A v ; K = v^T p ; w = p - K v ; A -= 2 (v w^T + w v^T)
    for (int i = 0; i < n; ++i) {
      double s = 0.0;
      for (int j = k + 1; j < n; ++j) s += A[(size_t)i * n + j] * v[j];
      p[i] = s;
    }
    double K = 0.0;
    for (int i = k + 1; i < n; ++i) K += v[i] * p[i];
    for (int i = 0; i < n; ++i) w[i] = p[i] - K * v[i];
    for (int i = 0; i < n; ++i)
      for (int j = 0; j < n; ++j) A[(size_t)i * n + j] -= 2.0 * (v[i] * w[j] + w[i] * v[j]);
    // Q = Q H
    for (int i = 0; i < n; ++i) {
      double s = 0.0;
      for (int j = k + 1; j < n; ++j) s += Q[(size_t)i * n + j] * v[j];
      for (int j = k + 1; j < n; ++j) Q[(size_t)i * n + j] -= 2.0 * s * v[j];
    }
  }
  d.assign(n, 0.0);
  e.assign(n, 0.0);
  for (int i = 0; i < n; ++i) d[i] = A[(size_t)i * n + i];
  for (int i = 0; i + 1 < n; ++i) e[i] = A[(size_t)i * n + i + 1];
}

// Implicit QL with Wilkinson-type shifts on a symmetric tridiagonal matrix
// (d diagonal, e[i] coupling i and i+1): the published tql2 procedure of
// EISPACK (Bowdler, Martin, Reinsch and Wilkinson, "The QR and QL
// algorithms for symmetric matrices", Numer. Math. 11 (1968) 293-306).  Z (row-major n x n) accumulates the
// rotations: on entry the basis the tridiagonal matrix is expressed in, on
// exit the eigenvectors as columns.  Eigenvalues are sorted ascending.
inline bool tridiag_ql(int n, std::vector<double>& d, std::vector<double>& e, std::vector<double>& Z) {
  const double eps = 2.220446049250313e-16;
  for (int l = 0; l < n; ++l) {
    int iter = 0;
    while (true) {
      int m = l;
      for (; m < n - 1; ++m) {
        double dd = std::fabs(d[m]) + std::fabs(d[m + 1]);
        if (std::fabs(e[m]) <= eps * dd) break;
      }
      if (m == l) break;
      if (++iter > 200) return false;
      double g = (d[l + 1] - d[l]) / (2.0 * e[l]);
      double r = std::hypot(g, 1.0);
      g = d[m] - d[l] + e[l] / (g + (g >= 0 ? r : -r));
      double s = 1.0, c = 1.0, p = 0.0;
      int i = m - 1;
      bool early = false;
      for (; i >= l; --i) {
        double f = s * e[i];
        double b = c * e[i];
        r = std::hypot(f, g);
        e[i + 1] = r;
        if (r == 0.0) {
          d[i + 1] -= p;
          e[m] = 0.0;
          early = true;
          break;
        }
        s = f / r;
        c = g / r;
        g = d[i + 1] - p;
        r = (d[i] - g) * s + 2.0 * c * b;
        p = s * r;
        d[i + 1] = g + p;
        g = c * r - b;
        for (int k = 0; k < n; ++k) {
          double zf = Z[(size_t)k * n + i + 1];
          Z[(size_t)k * n + i + 1] = s * Z[(size_t)k * n + i] + c * zf;
          Z[(size_t)k * n + i] = c * Z[(size_t)k * n + i] - s * zf;
        }
      }
      if (early) continue;
      d[l] -= p;
      e[l] = g;
      e[m] = 0.0;
    }
  }
  // sort ascending
  std::vector<int> ord(n);
  for (int i = 0; i < n; ++i) ord[i] = i;
  std::sort(ord.begin(), ord.end(), [&](int a, int b) { return d[a] < d[b]; });
  std::vector<double> d2(n), Z2((size_t)n * n);
  for (int j = 0; j < n; ++j) {
    d2[j] = d[ord[j]];
    for (int k = 0; k < n; ++k) Z2[(size_t)k * n + j] = Z[(size_t)k * n + ord[j]];
  }
  d = d2;
  Z = Z2;
  return true;
}

// Closure of a group of G elements (bit permutation perm[g*nb + i]: bit i of
// b moves to bit perm[g*nb + i]; then XOR with xr[g]) and the index of each
// element's inverse.  An element (p, x) acts as b -> p(b) ^ x; (p1, x1)(p2, x2)
// = (p1 p2, p1(x2) ^ x1) = (p1 p2, x2 ^ x1) since every x is 0 or the full
// word, which every permutation fixes.  Returns an empty string, or the
// reason the elements are not a group: a repeated element, or a product
// outside the set.
inline std::string group_inverses(int G, int nb, const std::vector<int32_t>& perm, const std::vector<uint64_t>& xr,
                                  std::vector<int32_t>& inv) {
  std::map<std::pair<std::vector<int32_t>, uint64_t>, int> index;
  for (int g = 0; g < G; ++g) {
    std::vector<int32_t> p(perm.begin() + (size_t)g * nb, perm.begin() + (size_t)(g + 1) * nb);
    auto key = std::make_pair(p, xr[g]);
    if (index.count(key)) return "repeated symmetry operation";
    index[key] = g;
  }
  inv.assign(G, -1);
  std::vector<int32_t> comp(nb);
  for (int g1 = 0; g1 < G; ++g1)
    for (int g2 = 0; g2 < G; ++g2) {
      for (int i = 0; i < nb; ++i) comp[i] = perm[(size_t)g1 * nb + perm[(size_t)g2 * nb + i]];
      auto it = index.find(std::make_pair(comp, xr[g1] ^ xr[g2]));
      if (it == index.end()) return "symmetry operations must form a group";
      if (it->second == 0) inv[g1] = g2;
    }
  return std::string();
}

// Colex (combinatorial number system) rank of a 12-bit word among the 12-bit
// words of its popcount j, in [0, C(12, j)) with C(12, j) <= 924, from two
// 6-bit halves: rank(l) = lo[l & 63] + hi[(l >> 6) * 7 + popcount(l & 63)],
// lo[v] = sum_i C(p_i, i) over the set bits p_1 < p_2 < ... of v, and
// hi[v * 7 + m] = sum_i C(6 + q_i, m + i) over the set bits q_1 < ... of v.
// Returns the 64 + 64 * 7 entries (lo, then hi).
constexpr int kColexStride = 924;  // C(12, 6): room for every popcount class
// One step of the omega recurrence of partial reorthogonalisation (Simon,
// "The Lanczos algorithm with partial reorthogonalization", Math. Comp. 42
// (1984) 115-142).  Given the estimates om_cur[q] ~ <v_j, v_q> (q <= j) and
// om_prev[q] ~ <v_{j-1}, v_q> (q < j), the Lanczos coefficients alpha(q)
// (q <= j) and beta(q) (q < j: the coupling of v_q and v_{q+1}) and the new
// beta_j > 0, writes om_new[q] ~ <v_{j+1}, v_q> for q <= j + 1:
//   beta_j om_new[q] = beta(q) om_cur[q+1] + (alpha(q) - alpha(j)) om_cur[q]
//                      + beta(q-1) om_cur[q-1] - beta(j-1) om_prev[q]
// plus a rounding term eps (beta(q) + beta_j) of the sum's sign, with
// om_new[j] = eps and om_new[j+1] = 1.  Returns max |om_new[q]| over q < j.
template <typename Alpha, typename Beta>
inline double omega_step(int j, Alpha alpha, Beta beta, double beta_j, const std::vector<double>& om_cur,
                         const std::vector<double>& om_prev, double eps, std::vector<double>& om_new) {
  om_new.assign((size_t)j + 2, 0.0);
  const double a_j = alpha(j);
  const double b_jm1 = j > 0 ? beta(j - 1) : 0.0;
  double worst = 0.0;
  for (int q = 0; q < j; ++q) {
    const double b_q = beta(q);
    double v = b_q * om_cur[(size_t)q + 1] + (alpha(q) - a_j) * om_cur[(size_t)q] - b_jm1 * om_prev[(size_t)q];
    if (q > 0) v += beta(q - 1) * om_cur[(size_t)q - 1];
    v += std::copysign(eps * (b_q + beta_j), v);
    om_new[(size_t)q] = v / beta_j;
    worst = std::max(worst, std::fabs(om_new[(size_t)q]));
  }
  om_new[(size_t)j] = eps;
  om_new[(size_t)j + 1] = 1.0;
  return worst;
}

inline std::vector<uint16_t> colex12_tables() {
  auto binom = [](int n, int k) -> uint32_t {
    if (k < 0 || k > n) return 0;
    uint64_t r = 1;
    for (int i = 1; i <= k; ++i) r = r * (uint64_t)(n - k + i) / (uint64_t)i;
    return (uint32_t)r;
  };
  std::vector<uint16_t> t(64 + 64 * 7, 0);
  for (int v = 0; v < 64; ++v) {
    uint32_t r = 0;
    int i = 0;
    for (int p = 0; p < 6; ++p)
      if ((v >> p) & 1) r += binom(p, ++i);
    t[v] = (uint16_t)r;
    for (int m = 0; m <= 6; ++m) {
      uint32_t h = 0;
      int q = 0;
      for (int p = 0; p < 6; ++p)
        if ((v >> p) & 1) h += binom(6 + p, m + (++q));
      t[64 + v * 7 + m] = (uint16_t)h;
    }
  }
  return t;
}

// The rank of every 12-bit word (4096 entries) from the two halves above:
// one table read per word on the device.
inline std::vector<uint16_t> colex12_full() {
  const std::vector<uint16_t> t = colex12_tables();
  std::vector<uint16_t> f(4096);
  for (uint32_t l = 0; l < 4096; ++l)
    f[l] = (uint16_t)(t[l & 63u] + t[64u + (l >> 6) * 7u + (uint32_t)__builtin_popcount(l & 63u)]);
  return f;
}

}  // namespace edhip
