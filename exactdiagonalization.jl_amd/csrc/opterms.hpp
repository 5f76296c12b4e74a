// Device code shared by the product kernels and the other kernels that walk an
// operator's terms: the canonicalisers by kernel specialisation, the staging of
// the tables in LDS, and the matching of a row against the terms.
#pragma once

#include <type_traits>

#include "kernels.hpp"

namespace edhip {

namespace {

constexpr int kBlock = 256;

// The products and the kernels that build assembled rows run 512-lane blocks
// over a grid that covers the rows in order (blocks that run together work on
// neighbouring rows, whose images share cache lines of the index and of x).
constexpr int kMvBlock = 512;

template <int MODE>
struct Canon {
  // NEED_H = false: h is left 0 where the canonicaliser can skip tracking it
  template <bool NEED_H = true>
  __device__ __forceinline__ static void run(const GroupDev& g, const GroupLds& L, uint64_t b, uint64_t& s, int& h,
                                             int& cnt) {
    if constexpr (MODE == kGroupNone) {
      s = b;
      h = 0;
      cnt = 1;
    } else if constexpr (MODE == kGroupTorusPairs) {
      canonicalize_torus_pairs<0, 0, NEED_H>(g, L, b, s, h, cnt);
    } else if constexpr (MODE == kTorusPairs6x6) {
      canonicalize_torus_pairs<6, 6, NEED_H>(g, L, b, s, h, cnt);
    } else if constexpr (MODE == kTorusPairs4x6) {
      canonicalize_torus_pairs<4, 6, NEED_H>(g, L, b, s, h, cnt);
    } else if constexpr (MODE == kTorusPairs6x4) {
      canonicalize_torus_pairs<6, 4, NEED_H>(g, L, b, s, h, cnt);
    } else if constexpr (MODE == kTorusPairs4x4) {
      canonicalize_torus_pairs<4, 4, NEED_H>(g, L, b, s, h, cnt);
    } else if constexpr (MODE >= kTransPairs6x6 && MODE <= kTransPairs4x4) {
      // translations only: the identity coset, whose element table maps the
      // translation found to the group element
      constexpr int LX = (MODE == kTransPairs6x6 || MODE == kTransPairs6x4) ? 6 : 4;
      constexpr int LY = (MODE == kTransPairs6x6 || MODE == kTransPairs4x6) ? 6 : 4;
      int pos;
      canonicalize_torus_pairs_t<LX, LY, NEED_H>(g, L, L.coset_inv, b, s, pos, cnt);
      h = NEED_H ? L.coset_elem[pos] : 0;
    } else {
      canonicalize(g, L, b, s, h, cnt);
    }
  }
};

struct Staged {
  GroupLds L;
  const OffTerm* off;
  const uint64_t* W;
};

template <int MODE>
__device__ __forceinline__ Staged stage_op(const OpDev& op, unsigned char* lds) {
  Staged S;
  if constexpr (MODE != kGroupNone) {
    S.L = stage_group(op.g, op.lay, lds);
  }
  lds_copy(lds + op.off_lds, op.off, (uint32_t)(op.n_off * sizeof(OffTerm)));
  S.off = (const OffTerm*)(lds + op.off_lds);
  lds_copy(lds + op.w_lds, op.ix.W, op.w_bytes);
  S.W = (const uint64_t*)(lds + op.w_lds);
  return S;
}

// The off-diagonal terms in LDS for the term pass, split by use: (mask, match)
// pairs read by every lane alike while matching a row, and (flip, amplitude)
// pairs read per matched term, where flip = match ^ image gives the image of a
// matching row b as b ^ flip.
struct PlainTerms {
  const uint64_t* mm;  // 2 per term: mask, match
  const uint64_t* fa;  // 2 per term: flip, bits of Re(amplitude)
};

__device__ __forceinline__ PlainTerms stage_plain_terms(const OpDev& op, unsigned char* lds) {
  const int n = op.n_off;
  uint64_t* mm = (uint64_t*)(lds + op.off_lds);  // at most 40 bytes per term, as reserved
  uint64_t* fa = mm + 2 * n;
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    const OffTerm o = op.off[t];
    mm[2 * t] = o.mask;
    mm[2 * t + 1] = o.match;
    fa[2 * t] = o.match ^ o.image;
    fa[2 * t + 1] = (uint64_t)__double_as_longlong(o.are);
  }
  return PlainTerms{mm, fa};
}

// The products' entries in LDS (layout mv_layout): the parity tables of the
// parity entries, the masks and matches of the others, and of every entry
// (parity entries first) flip, amplitude and, for complex vectors, Im(amplitude).
struct MvTerms {
  const uint64_t* tab;  // [segment][chunk][16]
  const uint64_t* mm;   // other entries: mask, match; paired: mask, match 2q, match 2q+1
  const uint64_t* fa;   // 2 per entry: flip, bits of Re(amplitude)
  const double* ai;     // Im(amplitude)
};

// amp32: the real amplitude is kept as an FP32 value in the low half of its
// slot.  with_im: imaginary parts are staged.  Amplitudes are staged times scale.
__device__ __forceinline__ MvTerms stage_mv_terms(const OpDev& op, unsigned char* lds, bool amp32, bool with_im,
                                                  double scale = 1.0) {
  const MvLayout Y = mv_layout(op.n_lin, op.n_chunk, op.n_rest, op.rest_paired);
  unsigned char* base = lds + op.mv_lds;
  uint64_t* mm = (uint64_t*)(base + Y.off_mm);
  uint64_t* fa = (uint64_t*)(base + Y.off_fa);
  double* ai = (double*)(base + Y.off_ai);
  lds_copy(base, op.lin_tab, Y.off_mm);
  for (int t = threadIdx.x; t < op.n_rest; t += blockDim.x) {
    const uint64_t mask = op.rest[t].mask, match = op.rest[t].match;
    if (!op.rest_paired) {
      mm[2 * t] = mask;
      mm[2 * t + 1] = match;
    } else if ((t & 1) == 0) {
      mm[3 * (t >> 1)] = mask;
      mm[3 * (t >> 1) + 1] = match;
    } else {
      mm[3 * (t >> 1) + 2] = match;
    }
  }
  for (int t = threadIdx.x; t < op.n_lin + op.n_rest; t += blockDim.x) {
    MvEntry e = op.ent[t];
    e.are *= scale;
    e.aim *= scale;
    fa[2 * t] = e.flip;
    fa[2 * t + 1] = amp32 ? (uint64_t)__float_as_uint((float)e.are) : (uint64_t)__double_as_longlong(e.are);
    if (with_im) ai[t] = e.aim;
  }
  return MvTerms{(const uint64_t*)base, mm, fa, ai};
}

// Number of segments of up to 64 entries (parity entries and the others apart).
__device__ __forceinline__ int mv_segments(const OpDev& op) { return (op.n_lin + 63) / 64 + (op.n_rest + 63) / 64; }

// Entries of segment seg that match the word b, as bits over the entries base,
// base + 1, ...  A parity entry matches when the parity of the bits of b it
// names is odd (even, with its constant): the XOR over b's 4-bit chunks of a
// table entry holding one bit per entry.  One table read and XOR per chunk
// tests 64 entries; the 16 entries of a chunk lie in 32 LDS banks, so that the
// lanes' reads do not conflict.  (Testing them one mask at a time took about
// 10 VALU instructions per pair of terms, 20 of the 162 per image at 6x6.)
__device__ __forceinline__ uint64_t mv_match(const OpDev& op, const MvTerms& T, uint64_t b, int seg, int& base) {
  const int n_ls = (op.n_lin + 63) / 64;
  uint64_t bits = 0;
  if (seg < n_ls) {
    base = 64 * seg;
    const uint64_t* tab = T.tab + seg * (op.n_chunk << 4);
    for (int k = 0; k < op.n_chunk; k += 3) {  // n_chunk is a multiple of 3; chunks past the word are zero
      uint64_t v[3];
#pragma unroll
      for (int q = 0; q < 3; ++q) v[q] = tab[((k + q) << 4) + (int)((b >> ((4 * (k + q)) & 63)) & 15ull)];
      bits ^= v[0] ^ v[1] ^ v[2];
    }
    return bits;
  }
  const int s0 = (seg - n_ls) * 64;
  base = op.n_lin + s0;
  const int n = op.n_rest - s0 < 64 ? op.n_rest - s0 : 64;
  if (op.rest_paired) {  // two terms with one mask per test (n is even)
#pragma unroll 2
    for (int j = 0; j < n; j += 2) {
      const uint64_t* m = T.mm + 3 * ((s0 + j) >> 1);
      const uint64_t xm = b & m[0];
      bits |= (uint64_t)((uint32_t)(xm == m[1]) | ((uint32_t)(xm == m[2]) << 1)) << j;
    }
  } else {
#pragma unroll 2
    for (int j = 0; j < n; ++j) {
      const uint64_t* m = T.mm + 2 * (s0 + j);
      bits |= (uint64_t)((b & m[0]) == m[1]) << j;
    }
  }
  return bits;
}

// Weight of an off-diagonal element without the row's own sqrt(N_r), which the
// products multiply into the finished sum: a * phase^(conj if TRANS) / sqrt(N_img)
// (SCALED: without 1 / sqrt(N_img), which the spread x sqrt(G / N) carries)
template <int MODE, bool TRANS, bool UNIT = false, bool SCALED = false>
__device__ __forceinline__ void element_weight_a(const OpDev& op, const GroupLds& L, double are, double aim, int h,
                                                 int cnt, double& wr, double& wi) {
  if constexpr (MODE == kGroupNone) {
    wr = are;
    wi = aim;
  } else {
    if (UNIT || op.g.unit_phases) {
      wr = are;
      wi = aim;
    } else {
      const double pr = L.ph_re[h];
      const double pi = TRANS ? -L.ph_im[h] : L.ph_im[h];
      wr = are * pr - aim * pi;
      wi = are * pi + aim * pr;
    }
    if constexpr (!SCALED) {
      wr *= L.sqcnt[cnt];
      wi *= L.sqcnt[cnt];
    }
  }
}

template <int MODE, bool TRANS>
__device__ __forceinline__ void element_weight(const OpDev& op, const Staged& S, const OffTerm& t, int h, int cnt,
                                               double sqrt_own, double& wr, double& wi) {
  if constexpr (MODE == kGroupNone) {
    wr = t.are;
    wi = t.aim;
  } else {
    double pr = S.L.ph_re[h];
    double pi = TRANS ? -S.L.ph_im[h] : S.L.ph_im[h];
    double sc = sqrt_own * S.L.sqcnt[cnt];
    wr = (t.are * pr - t.aim * pi) * sc;
    wi = (t.are * pi + t.aim * pr) * sc;
  }
}

__device__ __forceinline__ void diag_sum(const OpDev& op, uint64_t b, double& dre, double& dim_) {
  for (int t = 0; t < op.n_diag; ++t) {
    const DiagTerm d = op.diag[t];
    if ((b & d.mask) == d.match) {
      dre += d.are;
      dim_ += d.aim;
    }
  }
}
}  // namespace

}  // namespace edhip
