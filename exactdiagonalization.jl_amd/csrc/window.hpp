// The smallest translation image of a word, found through a table of windows.
//
// Every image of a word begins with the bits that the translation brings to
// the top, so only the translations whose beginning is the smallest can give
// the smallest image.  A table indexed by a window of the word holds, for the
// translations that start in that window, the rank of their smallest beginning
// and the mask of those that reach it, in 16 bits:
//   pairs (tori of rows of 3 to 6 bits): the window is a row y and the row
//     below it, the beginning both rows rotated by a (at most 700 ranks, 6 bits
//     of mask);
//   rows (rows of 7 or 8 bits): the window is the row y, the beginning the row
//     rotated by a (at most 36 ranks, 8 bits of mask);
//   chain (12 to 48 bits, one row): the window is 12 bits from the (6 y)-th
//     from the top down, the beginning the 7 bits from bit 6 y + a on, a < 6.
// The candidates (y, a) that reach the smallest rank are collected as bit
// 8 y + a of one mask and their images compared.
#pragma once

#include <stdint.h>

#ifndef __HIPCC__
#define EDHIP_HD inline
#else
#define EDHIP_HD __host__ __device__ __forceinline__
#endif

namespace edhip {

enum WinKind : int { kWinNone = 0, kWinPairs = 1, kWinRows = 2, kWinChain = 3, kWinPoint = 4 };

// Shapes compiled as their own kernels: tori of 16 to 36 sites with 3 to 8 rows of
// 3 to 8 bits, the most that a candidate mask holds (a byte per row, a bit per
// rotation) and the fewest that the windows pay for.  Longer and narrower ones (4x9,
// 2xN ladders) run the general kernels, as do smaller ones.
#define EDHIP_WIN_SHAPES(X)                                                                                       \
  X(kWinPairs, 3, 6) X(kWinPairs, 3, 7) X(kWinPairs, 3, 8) X(kWinPairs, 4, 4) X(kWinPairs, 4, 5) X(kWinPairs, 4, 6) \
  X(kWinPairs, 4, 7) X(kWinPairs, 4, 8) X(kWinPairs, 5, 4) X(kWinPairs, 5, 5) X(kWinPairs, 5, 6) X(kWinPairs, 5, 7) \
  X(kWinPairs, 6, 3) X(kWinPairs, 6, 4) X(kWinPairs, 6, 5) X(kWinPairs, 6, 6) X(kWinRows, 7, 3) X(kWinRows, 7, 4)   \
  X(kWinRows, 7, 5) X(kWinRows, 8, 3) X(kWinRows, 8, 4)

// The window kind of an Lx x Ly torus (a chain: Ly = 1).
inline int win_kind(int Lx, int Ly) {
#define EDHIP_X(K, X, Y) \
  if (Lx == X && Ly == Y) return K;
  EDHIP_WIN_SHAPES(EDHIP_X)
#undef EDHIP_X
  return (Ly == 1 && Lx >= 12 && Lx <= 48) ? kWinChain : kWinNone;
}

constexpr int win_mask_bits(int kind) { return kind == kWinRows ? 8 : 6; }
constexpr int win_index_bits(int kind, int Lx) { return kind == kWinPairs ? 2 * Lx : kind == kWinRows ? Lx : 12; }

template <bool WIDE>
struct WinWord {
  using T = uint64_t;
};
template <>
struct WinWord<false> {
  using T = uint32_t;
};

// KIND, LX, LY as above; a chain: LX = 32 for words of at most 32 bits, 48 else
// (its length n is a run-time value), LY = 1.
template <int KIND, int LX, int LY>
struct Win {
  static constexpr bool kChain = KIND == kWinChain;
  static constexpr bool kPoint = false;
  static constexpr int NB = LX * LY;  // (a chain: the longest)
  static constexpr int MB = win_mask_bits(KIND);
  static constexpr int NW = kChain ? (LX + 5) / 6 : LY;  // windows
  static constexpr int kTab = 1 << win_index_bits(KIND, LX);
  static constexpr uint32_t kTabBytes = 2u * kTab;
  static constexpr bool kWide = NB > 32;
  using W = typename WinWord<kWide>::T;
  using C = typename WinWord<(NW > 4)>::T;  // candidate mask
  static constexpr uint64_t kFull = NB >= 64 ? ~0ull : (1ull << (NB & 63)) - 1ull;

  EDHIP_HD static int ctz(uint64_t v) { return __builtin_ctzll(v); }
  EDHIP_HD static int ctz(uint32_t v) { return __builtin_ctz(v); }

  // Window y of b as a table index.
  EDHIP_HD static uint32_t window(W b, int n, int y) {
    if constexpr (KIND == kWinRows) {
      return (uint32_t)(b >> (y * LX)) & ((1u << LX) - 1u);
    } else if constexpr (KIND == kWinPairs) {
      constexpr uint32_t m2 = (1u << (2 * LX)) - 1u;
      if (y > 0) return (uint32_t)(b >> ((y - 1) * LX)) & m2;
      return (((uint32_t)b << LX) & m2) | (uint32_t)(b >> (NB - LX));
    } else {
      const uint64_t e = ((uint64_t)b << 12) | ((uint64_t)b >> (n - 12));
      return (uint32_t)(e >> (n - 6 * y)) & 0xfffu;
    }
  }

  // Candidates: bit 8 y + a for every (y, a) whose beginning is the smallest.
  template <typename P>
  EDHIP_HD static C candidates(P tab, W b, int n) {
    constexpr int NP = (NW + 1) / 2;
    constexpr uint32_t mask = (1u << MB) - 1u;
    C cand;
#ifdef __HIP_DEVICE_COMPILE__
    // two entries per register: packed 16-bit minima, differences to the
    // smallest rank (below 2^MB: the mask of a candidate, cut to 2^MB others),
    // then the low bytes of the halves gathered (v_perm_b32)
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 p[NP];
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      p[k].x = (!kChain || 12 * k < n) ? tab[window(b, n, 2 * k)] : (uint16_t)0xffffu;
      p[k].y = (2 * k + 1 < NW && (!kChain || 12 * k + 6 < n)) ? tab[window(b, n, 2 * k + 1)] : (uint16_t)0xffffu;
    }
    u16x2 m = p[0];
#pragma unroll
    for (int k = 1; k < NP; ++k) m = __builtin_elementwise_min(m, p[k]);
    const uint16_t lo = (uint16_t)((m.x < m.y ? m.x : m.y) & (uint16_t)~mask);
    uint32_t u[4] = {0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const u16x2 d = __builtin_elementwise_min((u16x2)(p[k] - (u16x2){lo, lo}),
                                                (u16x2){(uint16_t)(mask + 1u), (uint16_t)(mask + 1u)});
      u[k] = __builtin_bit_cast(uint32_t, d);
    }
    constexpr uint32_t keep = mask * 0x01010101u;  // (2^MB itself is not a mask; 256 has no low byte)
    const uint32_t lo32 = __builtin_amdgcn_perm(u[1], u[0], 0x06040200u) & keep;
    if constexpr (NW > 4)
      cand = ((C)(__builtin_amdgcn_perm(u[3], u[2], 0x06040200u) & keep) << 32) | lo32;
    else
      cand = lo32;
#else
    uint32_t e[2 * NP], lo = 0xffffu;
    for (int y = 0; y < 2 * NP; ++y) {
      e[y] = (y < NW && (!kChain || 6 * y < n)) ? tab[window(b, n, y)] : 0xffffu;
      lo = e[y] < lo ? e[y] : lo;
    }
    cand = 0;
    for (int y = 0; y < 2 * NP; ++y)
      if (e[y] - (lo & ~mask) <= mask) cand |= (C)(e[y] & mask) << (8 * y);
#endif
    if constexpr (kChain) {  // translations past the last are the first ones again
      const int last = (n - 1) / 6;
      cand &= (C)((1ull << (8 * last + n - 6 * last)) - 1ull);
    }
    return cand;
  }

  EDHIP_HD static W rotl_word(W b, int n, int back) {  // b rotated left by n - back of its n bits
    const uint64_t full = kChain ? (1ull << n) - 1ull : kFull;
    if constexpr (kWide)
      return ((b << (n - back)) | (b >> back)) & full;
    else
      return (W)((((uint64_t)b << n) | b) >> back) & (W)full;
  }

  // Image of b under the translation of candidate bit: row y to the top and
  // every row rotated left by a, or the chain rotated left by 6 y + a.
  EDHIP_HD static W image(W b, int n, int bit) {
    if constexpr (kChain) {
      return rotl_word(b, n, n - (6 * (bit >> 3) + (bit & 7)));
    } else {
      const int a = bit & 7;
      const W t = rotl_word(b, NB, ((bit >> 3) + 1) * LX);
      constexpr W ones = (W)(kFull / ((1u << LX) - 1u));  // bit 0 of every row
      const W low = (W)(ones << a) - ones;                // the low a bits of every row
      return (((W)(t << a) & ~low) | ((t >> (LX - a)) & low)) & (W)kFull;
    }
  }

  // The row below the beginning (pairs: the third, rows: the second) of the
  // image of candidate bit, and the same of an image: a candidate whose row is
  // larger than that of an image with the same beginning is larger.
  static constexpr int kNext = KIND == kWinPairs ? 2 : 1;
  static constexpr bool kScreen = !kChain && LY > kNext;
  EDHIP_HD static uint32_t next_row(W b, int bit) {
    constexpr uint32_t rm = (1u << LX) - 1u;
    const int a = bit & 7, y = bit >> 3;
    const int yn = y >= kNext ? y - kNext : y + LY - kNext;
    const uint32_t r = (uint32_t)(b >> (uint32_t)(yn * LX)) & rm;
    return ((r << a) | (r >> (LX - a))) & rm;
  }
  EDHIP_HD static uint32_t next_row_of(W s) { return (uint32_t)(s >> ((LY - 1 - kNext) * LX)) & ((1u << LX) - 1u); }

  // The smallest image s of b and the first candidate that gives it.
  template <typename P>
  EDHIP_HD static void canonical(P tab, W b, int n, W& s, int& bit) {
    C cand = candidates(tab, b, n);
    bit = ctz(cand);
    cand &= cand - 1;
    s = image(b, n, bit);
    while (cand) {
      const int q = ctz(cand);
      cand &= cand - 1;
      if constexpr (kScreen)
        if (next_row(b, q) > next_row_of(s)) continue;
      const W t = image(b, n, q);
      bit = t < s ? q : bit;
      s = t < s ? t : s;
    }
  }

  // a + Lx b of the translation T(a, b) of candidate bit.
  EDHIP_HD static int position(int bit) {
    if constexpr (kChain)
      return 6 * (bit >> 3) + (bit & 7);
    else
      return (bit & 7) + LX * (LY - 1 - (bit >> 3));
  }
};

// Translations and point operations of an L x L torus (L 5 or 6).  The images
// of the pair window (row y, the row below) under the rows' reversal, their
// exchange (the reflection in y shows the pair upside down) and both begin with
// permuted copies of the same two rows, so that one table read gives the least
// beginning over these four variants and all rotations.  The other four point
// operations are these after the transposition, whose windows are ranked
// beside.  Each of these maps commutes with XOR, so the transposed image is
// that of its row XORed with that of the flip, and nothing is permuted per
// image.  (Bounding eight cosets one by one, each permuted by 4-bit tables:
// 950 VALU instructions per image on the 6x6 A1 sector.)
//
// The frames (reversed or not, rotation) that reach a window's least beginning
// form one of few sets (cosets of subgroups of the dihedral group, at most 75),
// its class.  A table over (class, row) gives the least image of the next row
// over the frames of the class and the class of the frames that reach it: the
// least image of a window is read off row by row, ties and all, with no
// rotation (6x6 A1, FP64: 399 VALU instructions per image and 22.9 ms candidate
// by candidate, 313 and 20.8 ms this way, 239 with every table read at a
// compile-time LDS offset; what then bounds it is the L2 misses of its two
// gathers, 0.5 per image, 7.2 TB/s).
//
// Tables (u16): least beginning by window, classes by window (upright in the
// low byte, upside down in the high one, 0: none), next rows by class and row
// (class << L | row), a frame of each class (bit 3: reversed; rotation).
constexpr int kPointClasses = 80;
template <int L, int L2>
struct Win<kWinPoint, L, L2> {
  static constexpr bool kChain = false, kPoint = true;
  static constexpr int NB = L * L;
  static constexpr int kTab = 1 << (2 * L);
  static constexpr uint32_t kNext = 2 * kTab, kFrame = kNext + (kPointClasses << L);  // table offsets
  static constexpr uint32_t kTabBytes = 2u * (kFrame + kPointClasses);
  using W = typename WinWord<(NB > 32)>::T;
  using T = Win<kWinPairs, L, L>;

  EDHIP_HD static W transposed(W b) {
    W out = 0;
#pragma unroll
    for (int d = 1 - L; d < L; ++d) {  // the diagonal x - y = d moves by d (L - 1)
      W m = 0;
      for (int y = 0; y < L; ++y)
        if (y + d >= 0 && y + d < L) m |= (W)1 << (y + d + L * y);
      out |= d < 0 ? (b & m) >> (-d * (L - 1)) : (b & m) << (d * (L - 1));
    }
    return out;
  }

  // The smallest image s of the word b, whose transpose is bt, and (CODE) the
  // code of a candidate giving it: bit 8: transposed, bit 7: rows in reverse
  // order, bit 6: their bits reversed, then 8 y + a as for translations.
  // windows: the candidates to take, kWindows, or kUpright where the group
  // transposes nothing (and bt is b).
  static constexpr uint32_t kUpright = (1u << L) - 1u, kWindows = kUpright * 0x10001u;
  template <bool CODE, typename P>
  EDHIP_HD static void canonical(P tab, W b, W bt, uint32_t windows, W& s, int& code) {
    constexpr int kRest = L * (L - 2);  // bits after the beginning, fewer than 32
    uint32_t cand, lo;                  // bit y: window y of b, bit 16 + y: of bt
#ifdef __HIP_DEVICE_COMPILE__
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 p[L];
#pragma unroll
    for (int y = 0; y < L; ++y) p[y] = u16x2{tab[T::window(b, 0, y)], tab[T::window(bt, 0, y)]};
    u16x2 m = p[0];
#pragma unroll
    for (int y = 1; y < L; ++y) m = __builtin_elementwise_min(m, p[y]);
    lo = m.x < m.y ? m.x : m.y;
    // a half is above the least (by less than 2^12) iff its sum with 0x7fff - least has bit 15
    const uint32_t above = 0x7fff7fffu - lo * 0x10001u;
    uint32_t other = 0;
#pragma unroll
    for (int y = 0; y < L; ++y)
      other = (other >> 1) | ((__builtin_bit_cast(uint32_t, p[y]) + above) & 0x80008000u);
    cand = ~(other >> (16 - L)) & windows;
#else
    uint32_t p[2 * L];
    lo = 0xffffu;
    for (int y = 0; y < 2 * L; ++y) {
      p[y] = y < L ? tab[T::window(b, 0, y)] : tab[T::window(bt, 0, y - L)];
      lo = p[y] < lo ? p[y] : lo;
    }
    cand = 0;
    for (int y = 0; y < 2 * L; ++y)
      if (p[y] == lo) cand |= 1u << (y < L ? y : 16 + y - L);
    cand &= windows;
#endif
    uint32_t best = ~0u;
    uint32_t down = 0;  // class of the window's upside-down frames, to be taken next
    uint32_t rows = 0;
    int q = 0;
    code = 0;
    do {
      uint32_t c = down;
      int at = 0, step = L;  // upside down: the rows from y + 1 up
      if (!down) {
        q = T::ctz(cand);
        cand &= cand - 1;
        const W w = q >= 16 ? bt : b;
        const int n = ((q & 15) + 1) * L;  // row y to the top: the rows y - 2 down and y + 1 up are the low ones
        const W t = (W)(w >> n) | (W)(w << (NB - n));
        rows = (uint32_t)t;
        const uint32_t e = tab[kTab + ((uint32_t)(t >> kRest) & (uint32_t)(kTab - 1))];
        c = e & 255u;
        down = e >> 8;
        at = kRest - L;
        step = -L;
        if (c == 0) {
          c = down;
          at = 0;
          step = L;
          down = 0;
        }
      } else {
        down = 0;
      }
      uint32_t e = c << L, rest = 0;
      constexpr uint32_t rm = (1u << L) - 1u;
#pragma unroll
      for (int k = 0; k < L - 2; ++k) {
        e = tab[kNext + (e | ((rows >> at) & rm))];
        rest = (rest << L) | (e & rm);
        e &= ~rm;
        at += step;
      }
      if constexpr (CODE)
        if (rest < best) {
          const int y = q & 15, f = tab[kFrame + (e >> L)];
          code = (q >= 16 ? 256 : 0) + (step > 0 ? 128 + 8 * (y ? L - y : 0) : 8 * y) + 8 * (f & 8) + (f & 7);
        }
      best = rest < best ? rest : best;
    } while (down | cand);
    s = ((W)lo << kRest) | best;
  }
};

// The window tables exist for square tori of these sides with point operations.
inline bool win_point_side(int L) { return L == 5 || L == 6; }

// No group: every word is its own image (LX: bits of the widest word).
template <int LX, int LY>
struct Win<kWinNone, LX, LY> {
  static constexpr bool kChain = true;  // (the number of word bits is a run-time value)
  static constexpr bool kPoint = false;
  static constexpr int NB = LX;
  static constexpr uint32_t kTabBytes = 0;
  using W = typename WinWord<(LX > 32)>::T;
  template <typename P>
  EDHIP_HD static void canonical(P, W b, int, W& s, int& bit) {
    s = b;
    bit = 0;
  }
};

}  // namespace edhip
