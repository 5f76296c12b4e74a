// Matrix-free application of an operator on a (possibly symmetry-reduced)
// basis, in gather form with no atomics: one lane owns one output entry.
//
// Row form (apply!(out, opr, state), abstract_operator_representation.jl:296-316):
//   y[r] += sum_t [ (b_r & m_t) == R_t ] w * x[s],  image b' = (b_r & ~m_t) | C_t
// Column form (apply!(out, state, opr), :327-347) swaps R_t and C_t and uses
// the column element of reduced_operator_representation.jl:88-116.
//
// For a reduced basis, b' is canonicalised to its representative s = h(b'),
// and the element is a * phase[h] * sqrt(N_r / N_s) (row form) with
// phase[h] = conj(chi(h^-1)); this equals a * U[b'] / U[b_r] of
// reduced_operator_representation.jl:57-85 with U[g(s)] = conj(chi(g))/sqrt(N_s).
#pragma once

#include "opterms.hpp"

namespace edhip {

namespace {

// Sum over the groups of 2^lg neighbouring lanes that share a row.
template <typename V>
__device__ __forceinline__ V row_lanes_sum(V acc, int lg) {
  for (int o = (1 << lg) >> 1; o > 0; o >>= 1) {
    if constexpr (VT<V>::cx) {
      acc.re += __shfl_xor(acc.re, o, 64);
      acc.im += __shfl_xor(acc.im, o, 64);
    } else {
      acc += __shfl_xor(acc, o, 64);
    }
  }
  return acc;
}

// UNIT: every character is 1 (op.g.unit_phases): the weight needs no phase,
// so the canonicaliser does not track the element reaching the image.
// SCALED: x is read from its spread holding x sqrt(G / N) (op.xm.scaled), so the
// weight needs no orbit size of the image and the stabiliser goes uncounted.
// 2^op.row_lanes lanes share a row and take its matched entries in turn
// (op.stripe): one lane per row on spaces that fill the chip by themselves,
// more on smaller ones (mv_row_lanes).
template <typename V, int MODE, bool TRANS, bool UNIT, bool SCALED>
__global__ __launch_bounds__(kMvBlock) void k_matvec(OpDev op, const V* __restrict__ x, V* __restrict__ y, int accumulate) {
  extern __shared__ unsigned char lds[];
  GroupLds L{};
  if constexpr (MODE != kGroupNone) L = stage_group(op.g, op.lay, lds);
  // FP32 weights: a real FP32 product whose images need no orbit size (scaled
  // spread) weighs each image in FP32, from FP32 amplitudes and phases of +-1
  // (no FP64 multiply and conversion per image)
  constexpr bool kW32 = SCALED && std::is_same<V, float>::value;
  // the weights of single precision carry sqrt(G) (row_result)
  constexpr bool kUnitScale = MODE != kGroupNone && (SCALED || std::is_same<typename VT<V>::R, float>::value);
  const MvTerms T = stage_mv_terms(op, lds, kW32, VT<V>::cx, kUnitScale && !SCALED ? sqrt((double)op.g.G) : 1.0);
  lds_copy(lds + op.mv_w_lds, op.ix.W, op.w_bytes);
  const uint64_t* W = (const uint64_t*)(lds + op.mv_w_lds);
  // code table of the spread x (the host sets xm only with room for it)
  uint16_t* codes = (uint16_t*)(lds + op.mv_codes_lds);
  if (op.xm.values) xmap_stage(op.xm, codes);
  __syncthreads();
  const int64_t lane = xcd_chunked_block(blockIdx.x, gridDim.x, op.xcd_chunk) * kMvBlock + threadIdx.x;
  const int64_t row = op.row_begin + (lane >> op.row_lanes);
  if (row >= op.dim) return;
  const int sub = (int)threadIdx.x & ((1 << op.row_lanes) - 1);
  using R = typename VT<V>::R;
  const uint64_t b = op.rows[row];

  // single precision sums the two images of a step apart (k_product_win); without
  // the spread the registers of a second sum would cost a wave (6x6, C64)
  constexpr bool kTwoSums = SCALED && std::is_same<R, float>::value;
  V sums[2] = {vzero<V>(), vzero<V>()};
  const int n_seg = mv_segments(op);
  for (int seg = 0; seg < n_seg; ++seg) {
    int base;
    uint64_t bits = mv_match(op, T, b, seg, base) & (op.stripe << sub);
    // two images per step: both canonical forms first, then both lookups and
    // both x gathers issued before either is used (twice the loads in flight;
    // measured 5% faster at 6x6 than one image per step, three or four per
    // step are slower: more steps end with an empty slot)
    constexpr int NW = 2;
    while (bits) {
      int t[NW];
      bool ok[NW];
      t[0] = base + __builtin_ctzll(bits);  // bits != 0 here
      ok[0] = true;
      bits &= bits - 1;
#pragma unroll
      for (int k = 1; k < NW; ++k) {  // an empty slot repeats the first image and is dropped
        ok[k] = bits != 0;
        t[k] = ok[k] ? base + __builtin_ctzll(bits) : t[0];
        bits &= ok[k] ? bits - 1 : bits;
      }
      ulonglong2 fa[NW];  // flip = match ^ image: a matching row b has the image b ^ flip
      uint64_t sk[NW];
      int hk[NW], ck[NW];
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        fa[k] = *(const ulonglong2*)(T.fa + 2 * t[k]);
        Canon<MODE>::template run<!UNIT>(op.g, L, b ^ fa[k].x, sk[k], hk[k], ck[k]);
      }
      int64_t ik[NW];
      V xv[NW];
      if (op.xm.values) {  // x of each image with one load at its word position
        xmap_fetch2(op.xm, codes, sk[0], sk[1], xv[0], xv[1]);
        ik[0] = 0;
        ik[1] = ok[1] ? 0 : -1;
      } else {
        index_of2(op.ix, W, sk[0], sk[1], ik[0], ik[1]);
#pragma unroll
        for (int k = 0; k < NW; ++k) {
          ik[k] = ok[k] ? ik[k] : -1;
          xv[k] = x[ik[k] >= 0 ? ik[k] : 0];
        }
      }
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        if (ik[k] >= 0) {
          if constexpr (kW32) {
            float w = __uint_as_float((uint32_t)fa[k].y);
            if constexpr (!UNIT) w *= (float)L.ph_re[hk[k]];
            vfma(sums[kTwoSums ? k : 0], w, 0.f, xv[k]);
          } else {
            double wr, wi;
            element_weight_a<MODE, TRANS, UNIT, SCALED>(op, L, __longlong_as_double((long long)fa[k].y),
                                                        VT<V>::cx ? T.ai[t[k]] : 0.0, hk[k], ck[k], wr, wi);
            vfma(sums[kTwoSums ? k : 0], (R)wr, (R)wi, xv[k]);
          }
        }
      }
    }
  }
  const V acc = row_lanes_sum(kTwoSums ? vadd(sums[0], sums[1]) : sums[0], op.row_lanes);
  if (sub != 0) return;
  // diagonal terms (C == R): the element is the summed amplitude (U[b]/U[b] = 1)
  double dre = 0.0, dim_ = 0.0;
  if (op.diag_re) {
    dre = op.diag_re[row];
    if (op.diag_im) dim_ = op.diag_im[row];
  } else {
    diag_sum(op, b, dre, dim_);
  }
  V out;
  if constexpr (MODE != kGroupNone) {
    const double n = kUnitScale ? (double)op.orbit[row] / (double)op.g.G : (double)op.orbit[row];
    out = row_result(dre, dim_, x[row], sqrt(n), acc);
  } else {
    out = vzero<V>();
    vfma(out, (R)dre, (R)dim_, x[row]);
    out = vadd(out, acc);
  }
  V* yr = y + (row - op.row_begin);
  *yr = accumulate ? vadd(*yr, out) : out;
}

// ---- translations alone on a shape of window.hpp, and sectors without a group ----
// Everything the kernel reads per image lies at LDS offsets known at compile
// time: the window table, the phases by candidate bit, the code table of the
// spread, the colex ranks, then the entries (by rank: the two rank tables, then
// the entries).
template <int KIND, int LX, int LY, bool UNIT>
struct WinLds {
  using S = Win<KIND, LX, LY>;
  static constexpr uint32_t n_codes = S::kPoint ? 512 : 64;  // candidates
  static constexpr uint32_t tab = 0;
  static constexpr uint32_t phase = tab + S::kTabBytes;
  static constexpr uint32_t codes = phase + (UNIT ? 0 : n_codes * 16);
  static constexpr uint32_t colex = codes + kXCodesBytesMax;
  static constexpr uint32_t entries = colex + 2 * 4096;
};

// One product entry in LDS, in 8 bytes where flip and amplitude fit (32-bit
// words, FP32 weights), else in 16.
template <typename W, typename A>
struct WinEntry {
  W flip;
  A amp;
};
// with point operations: the flip's transpose too
template <typename W, typename A>
struct PointEntry {
  W flip, turned;
  A amp;
};

// The product for translation groups on the shapes of window.hpp, x read from
// its colex spread x sqrt(G / N) (XMapDev: every image keeps the popcount, narrow).
// It is bound by instruction issue and by the line fills of the x gathers
// together, so what counts is the number of instructions per image: the shape,
// the word width (32 bits up to 32 sites) and the LDS offsets are fixed at
// compile time, the canonical form comes from 16-bit window entries (two per
// register), a position needs no test (XMapDev), and the phase is read by
// candidate bit.
//
// KIND = kWinNone: sectors of one popcount without a group.  RANK: of at most
// kRankBits bits, x is read itself, at the word's rank: the number of sector
// words with a smaller upper part plus the colex rank of the lower part, one
// read of each of two LDS tables (no spread to fill, and x is denser: 4x6 XXZ,
// 2.7e6 states, FP64: 174 us a call through the spread by the general kernel,
// 118 us by rank).
//
// KIND = kWinPoint: translations and point operations.  These spaces are 8
// times sparser in their words, so a spread would take a line per state (6x6
// A1, FP64: 8.2 GB for 31.6M states): the position of the spread is ranked
// through bits instead (RankBits, 258 MB beside x sqrt(G / N) itself).
template <typename V, int KIND, int LX, int LY, bool UNIT, bool TRANS, bool RANK = false>
__global__ __launch_bounds__(kMvBlock) void k_product_win(WinOp P, const V* __restrict__ x, V* __restrict__ y) {
  using S = Win<KIND, LX, LY>;
  using W = typename S::W;
  using R = typename VT<V>::R;
  using Lay = WinLds<KIND, LX, LY, UNIT>;
  constexpr bool CX = VT<V>::cx;
  // FP32 vectors without a complex phase weigh in FP32, from FP32 amplitudes and phases of +-1
  constexpr bool kW32 = std::is_same<R, float>::value && (!CX || UNIT);
  using A = typename std::conditional<kW32, float, double>::type;
  using E = typename std::conditional<S::kPoint, PointEntry<W, A>, WinEntry<W, A>>::type;
  extern __shared__ unsigned char lds[];
  lds_copy16(lds + Lay::tab, P.win_tab, S::kTabBytes);
  if constexpr (!UNIT) {
    double* ph = (double*)(lds + Lay::phase);
    if (threadIdx.x < Lay::n_codes) {
      const int h = P.win_elem[threadIdx.x];
      ph[2 * threadIdx.x] = P.ph_re[h];
      ph[2 * threadIdx.x + 1] = TRANS ? -P.ph_im[h] : P.ph_im[h];
    }
  }
  const uint32_t rank_low = 2u << P.low_bits;  // RANK: bytes of the lower table
  if constexpr (RANK) {
    lds_copy16(lds, P.rank_low, rank_low);
    lds_copy16(lds + rank_low, P.rank_base, P.base_bytes);
  } else {
    lds_copy16(lds + Lay::codes, P.topcode, xmap_codes_bytes(P.top_bits));
    lds_copy16(lds + Lay::colex, P.colex, 2u * 4096u);
  }
  constexpr int n_chunk = S::kChain ? 0 : (((S::NB + 3) / 4 + 2) / 3) * 3;
  const int nch = n_chunk ? n_chunk : P.n_chunk;
  const uint32_t tab_bytes = (uint32_t)(((P.n_lin + 63) / 64) * nch) * 128u;
  const uint32_t at_ptab = RANK ? rank_low + P.base_bytes : Lay::entries;
  lds_copy16(lds + at_ptab, P.lin_tab, tab_bytes);
  const int n_ent = P.n_lin + P.n_rest;
  const uint32_t at_ent = at_ptab + tab_bytes;
  const uint32_t at_aim = at_ent + (uint32_t)((n_ent + 1) & ~1) * (uint32_t)sizeof(E);
  const uint32_t at_mm = at_aim + (CX ? 8u * (uint32_t)n_ent : 0u);
  E* ent = (E*)(lds + at_ent);
  double* aim = (double*)(lds + at_aim);
  uint64_t* mm = (uint64_t*)(lds + at_mm);
#pragma unroll 1
  for (int t = threadIdx.x; t < n_ent; t += kMvBlock) {
    const MvEntry e = P.ent[t];
    if constexpr (S::kPoint) {
      ent[t] = E{(W)e.flip, P.point_swap ? S::transposed((W)e.flip) : (W)e.flip, (A)e.are};
    } else {
      ent[t] = E{(W)e.flip, (A)e.are};
    }
    if (CX) aim[t] = e.aim;
  }
#pragma unroll 1
  for (int t = threadIdx.x; t < P.n_rest; t += kMvBlock) {
    mm[2 * t] = P.rest[t].mask;
    mm[2 * t + 1] = P.rest[t].match;
  }
  __syncthreads();
  const int64_t lane = xcd_chunked_block(blockIdx.x, gridDim.x, P.xcd_chunk) * kMvBlock + threadIdx.x;
  const int64_t row = P.row_begin + (lane >> P.row_lanes);
  if (row >= P.dim) return;
  const int sub = (int)threadIdx.x & ((1 << P.row_lanes) - 1);
  const W b = (W)P.rows[row];

  const LdsPtr<uint16_t> tab = lds_at<uint16_t>(Lay::tab);
  const LdsPtr<uint16_t> codes = lds_at<uint16_t>(Lay::codes);
  const LdsPtr<uint16_t> colex = lds_at<uint16_t>(Lay::colex);
  const LdsPtr<double> phase = lds_at<double>(Lay::phase);
  const uint32_t top_max = 1u << P.top_bits;
  W turned = 0;  // (point operations: the row's transpose)
  if constexpr (S::kPoint) turned = P.point_swap ? S::transposed(b) : b;
  auto position = [&](W s) {  // of the canonical word s in the spread
    const uint32_t top = (uint32_t)(s >> P.top_shift);
    const uint32_t c = codes[top < top_max ? top : top_max];
    const uint32_t lo = (uint32_t)s;
    const uint32_t hc = (c << P.hbits) | __builtin_amdgcn_ubfe(lo, 12u, (uint32_t)P.hbits);
    return __umul24(hc, 924u) + (uint32_t)colex[lo & 0xfffu];
  };
  auto fetch = [&](W s) {  // x (sqrt(G / N)) of the canonical word s
    if constexpr (RANK) {
      const uint32_t lo = (uint32_t)s & ((1u << P.low_bits) - 1u);
      return x[lds_at<uint32_t>(rank_low)[s >> P.low_bits] + (uint32_t)lds_at<uint16_t>(0)[lo]];
    }
    return ((const V*)P.values)[(uint64_t)position(s)];
  };
  // single precision sums the two images of a step apart: half as many roundings in
  // either sum (5x6 (1,2), C64, x > 0: 1.44e-7 off in the norm with one sum, 9e-8
  // with two)
  constexpr bool kTwoSums = std::is_same<R, float>::value;
  V sums[2] = {vzero<V>(), vzero<V>()};
  auto add = [&](V& acc, const V& xv, int t, const E& e, int bit) {
    if constexpr (UNIT) {
      if (!CX || P.real_amp) {
        if constexpr (CX) {
          acc.re += (R)e.amp * xv.re;
          acc.im += (R)e.amp * xv.im;
        } else {
          acc += (R)e.amp * xv;
        }
      } else {
        vfma(acc, (R)e.amp, (R)lds_at<double>(at_aim)[t], xv);
      }
    } else if constexpr (!CX) {
      if constexpr (kW32)
        acc += e.amp * (float)phase[2 * bit] * xv;
      else
        acc += (R)(e.amp * phase[2 * bit]) * xv;
    } else {
      const double2 p{phase[2 * bit], phase[2 * bit + 1]};
      if (P.real_amp) {
        vfma(acc, (R)(e.amp * p.x), (R)(e.amp * p.y), xv);
      } else {
        const double ai = lds_at<double>(at_aim)[t];
        vfma(acc, (R)(e.amp * p.x - ai * p.y), (R)(e.amp * p.y + ai * p.x), xv);
      }
    }
  };
  const int n_ls = (P.n_lin + 63) / 64, n_seg = n_ls + (P.n_rest + 63) / 64;
  for (int seg = 0; seg < n_seg; ++seg) {
    uint64_t bits = 0;
    int base;
    if (seg < n_ls) {  // parity entries (mv_match)
      base = 64 * seg;
      const LdsPtr<uint64_t> pt = lds_at<uint64_t>(at_ptab) + seg * (nch << 4);
      if constexpr (n_chunk > 0) {
#pragma unroll
        for (int k = 0; k < n_chunk; ++k)
          if (4 * k < S::NB) bits ^= pt[(k << 4) + (int)((b >> (4 * k)) & 15)];
      } else {
        for (int k = 0; k < nch; k += 3) {
          uint64_t v[3];
#pragma unroll
          for (int q = 0; q < 3; ++q) v[q] = pt[((k + q) << 4) + (int)(((uint64_t)b >> (4 * (k + q))) & 15)];
          bits ^= v[0] ^ v[1] ^ v[2];
        }
      }
    } else {
      const int s0 = (seg - n_ls) * 64;
      base = P.n_lin + s0;
      const int n = P.n_rest - s0 < 64 ? P.n_rest - s0 : 64;
#pragma unroll 2
      for (int j = 0; j < n; ++j) bits |= (uint64_t)(((uint64_t)b & mm[2 * (s0 + j)]) == mm[2 * (s0 + j) + 1]) << j;
    }
    bits &= P.stripe << sub;
    // two images per step, as in k_matvec (three: 6x6 61.2 against 59.8 ms;
    // sectors without a group, six: 108 against 114 us on the 4x6 XXZ case)
    constexpr int NW = 2;
    while (bits) {
      int t[NW];
      bool ok[NW];
      t[0] = base + __builtin_ctzll(bits);
      bits &= bits - 1;
#pragma unroll
      for (int k = 1; k < NW; ++k) {
        ok[k] = bits != 0;
        t[k] = ok[k] ? base + __builtin_ctzll(bits) : t[0];
        bits &= ok[k] ? bits - 1 : bits;
      }
      E e[NW];
      W s[NW];
      int w[NW];
      V xv[NW];
#pragma unroll
      for (int k = 0; k < NW; ++k) {
        const uint32_t at = at_ent + __umul24((uint32_t)t[k], (uint32_t)sizeof(E));
        e[k].flip = *lds_at<W>(at);
        e[k].amp = *lds_at<A>(at + (uint32_t)offsetof(E, amp));
        if constexpr (S::kPoint)
          S::template canonical<!UNIT>(tab, b ^ e[k].flip, turned ^ *lds_at<W>(at + (uint32_t)sizeof(W)),
                                       P.point_swap ? S::kWindows : S::kUpright, s[k], w[k]);
        else
          S::canonical(tab, b ^ e[k].flip, P.n_bits, s[k], w[k]);
      }
      if constexpr (S::kPoint) {  // both blocks, then both elements
        uint32_t at[NW];
        RankBits r[NW];
#pragma unroll
        for (int k = 0; k < NW; ++k) r[k] = P.pos_bits[(at[k] = position(s[k])) >> 5];
#pragma unroll
        for (int k = 0; k < NW; ++k) xv[k] = ((const V*)P.values)[rank_of(r[k], at[k], P.none)];
      } else {
#pragma unroll
        for (int k = 0; k < NW; ++k) xv[k] = fetch(s[k]);
      }
      add(sums[0], xv[0], t[0], e[0], w[0]);
#pragma unroll
      for (int k = 1; k < NW; ++k)
        if (ok[k]) add(sums[kTwoSums ? k : 0], xv[k], t[k], e[k], w[k]);
    }
  }
  const V acc = row_lanes_sum(kTwoSums ? vadd(sums[0], sums[1]) : sums[0], P.row_lanes);
  if (sub != 0) return;
  V out = vzero<V>();
  if constexpr (KIND != kWinNone) {
    const bool diag = P.diag_re != nullptr;
    out = row_result(diag ? P.diag_re[row] : 0.0, diag && P.diag_im ? P.diag_im[row] : 0.0, diag ? x[row] : out,
                     sqrt((double)P.orbit[row] / (double)P.G), acc);
  } else {
    if (P.diag_re) vfma(out, (R)P.diag_re[row], (R)(P.diag_im ? P.diag_im[row] : 0.0), x[row]);
    out = vadd(out, acc);
  }
  V* yr = y + (row - P.row_begin);
  *yr = P.accumulate ? vadd(*yr, out) : out;
}

template <auto Kernel, typename V>
hipError_t launch_win_kernel(dim3 grid, uint32_t lds, hipStream_t st, const WinOp& P, const void* x, void* y) {
  const hipError_t e = lds_from_zero<Kernel>();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(Kernel, grid, dim3(kMvBlock), lds, st, P, (const V*)x, (V*)y);
  return hipGetLastError();
}

template <typename V, int KIND, int LX, int LY>
hipError_t launch_win_t(const WinOp& P, int unit, int transpose, const void* x, void* y, hipStream_t st) {
  const uint64_t lanes = (uint64_t)(P.dim - P.row_begin) << P.row_lanes;
  const dim3 grid((unsigned)((lanes + kMvBlock - 1) / kMvBlock));
  const uint32_t dyn =
      win_entries_bytes(P.n_lin, P.n_chunk, P.n_rest) + (KIND == kWinPoint ? 8u * (uint32_t)(P.n_lin + P.n_rest + 1) : 0u);
  // the column form only conjugates the phase
  constexpr bool kT = VT<V>::cx;
  constexpr uint32_t below_unit = WinLds<KIND, LX, LY, true>::entries, below = WinLds<KIND, LX, LY, false>::entries;
  if (unit) return launch_win_kernel<k_product_win<V, KIND, LX, LY, true, false>, V>(grid, below_unit + dyn, st, P, x, y);
  if (transpose) return launch_win_kernel<k_product_win<V, KIND, LX, LY, false, kT>, V>(grid, below + dyn, st, P, x, y);
  return launch_win_kernel<k_product_win<V, KIND, LX, LY, false, false>, V>(grid, below + dyn, st, P, x, y);
}

template <typename V>
hipError_t launch_win_v(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                        hipStream_t st) {
#define EDHIP_X(K, X, Y) \
  if (Lx == X && Ly == Y) return launch_win_t<V, K, X, Y>(P, unit, transpose, x, y, st);
  EDHIP_WIN_SHAPES(EDHIP_X)
#undef EDHIP_X
  return hipErrorInvalidValue;
}

template <typename V>
hipError_t launch_win_other(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                            hipStream_t st) {
  if (P.pos_bits) {
    if (Lx == 5 && Ly == 5) return launch_win_t<V, kWinPoint, 5, 5>(P, unit, transpose, x, y, st);
    if (Lx == 6 && Ly == 6) return launch_win_t<V, kWinPoint, 6, 6>(P, unit, transpose, x, y, st);
    return hipErrorInvalidValue;
  }
  if (Ly == 0) {  // no group
    const uint64_t lanes = (uint64_t)(P.dim - P.row_begin) << P.row_lanes;
    const dim3 grid((unsigned)((lanes + kMvBlock - 1) / kMvBlock));
    const uint32_t dyn = win_entries_bytes(P.n_lin, P.n_chunk, P.n_rest);
    constexpr uint32_t fixed = WinLds<kWinNone, 32, 1, true>::entries;
    if (P.rank_low)
      return launch_win_kernel<k_product_win<V, kWinNone, 32, 1, true, false, true>, V>(
          grid, (2u << P.low_bits) + P.base_bytes + dyn, st, P, x, y);
    if (P.n_bits <= 32)
      return launch_win_kernel<k_product_win<V, kWinNone, 32, 1, true, false>, V>(grid, fixed + dyn, st, P, x, y);
    return launch_win_kernel<k_product_win<V, kWinNone, 64, 1, true, false>, V>(grid, fixed + dyn, st, P, x, y);
  }
  if (Ly == 1 && Lx <= 32) return launch_win_t<V, kWinChain, 32, 1>(P, unit, transpose, x, y, st);
  if (Ly == 1 && Lx <= 48) return launch_win_t<V, kWinChain, 48, 1>(P, unit, transpose, x, y, st);
  return launch_win_v<V>(P, Lx, Ly, unit, transpose, x, y, st);
}

template <typename V, int MODE>
hipError_t launch_mv_t(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st) {
  const uint64_t lanes = (uint64_t)(op.dim - op.row_begin) << op.row_lanes;
  dim3 grid((unsigned)((lanes + kMvBlock - 1) / kMvBlock));
  // unit-phase kernels only where the canonicaliser can drop the element (row-pair tori)
  const bool unit = MODE >= kGroupTorusPairs && op.g.unit_phases;
  const uint32_t lds = op.xm.values ? op.mv_codes_lds + xmap_lds_bytes(op.xm) : op.mv_lds_total;
  // the column form only conjugates the phase: one kernel serves both for real vectors
  constexpr bool kT = VT<V>::cx;
#define EDHIP_MV(T, U, S)                                                                                              \
  hipLaunchKernelGGL((k_matvec<V, MODE, T, U, S>), grid, dim3(kMvBlock), lds, st, op, (const V*)x, (V*)y, accumulate)
  if constexpr (MODE != kGroupNone) {
    if (op.xm.values && op.xm.scaled) {
      if (transpose) {
        if (unit) EDHIP_MV(kT, MODE >= kGroupTorusPairs, true); else EDHIP_MV(kT, false, true);
      } else {
        if (unit) EDHIP_MV(false, MODE >= kGroupTorusPairs, true); else EDHIP_MV(false, false, true);
      }
      return hipGetLastError();
    }
  }
  if (transpose) {
    if (unit) EDHIP_MV(kT, MODE >= kGroupTorusPairs, false); else EDHIP_MV(kT, false, false);
  } else {
    if (unit) EDHIP_MV(false, MODE >= kGroupTorusPairs, false); else EDHIP_MV(false, false, false);
  }
#undef EDHIP_MV
  return hipGetLastError();
}

template <typename V>
hipError_t launch_mv_v(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st) {
  switch (op.g.mode) {
    case kGroupNone:
      return launch_mv_t<V, kGroupNone>(op, transpose, accumulate, x, y, st);
    case kGroupGeneric:
      return launch_mv_t<V, kGroupGeneric>(op, transpose, accumulate, x, y, st);
    default:
      if (op.g.pair_table) {
        const int Lx = op.g.Lx, Ly = op.g.Ly;
        if (Lx == 6 && Ly == 6) return launch_mv_t<V, kTorusPairs6x6>(op, transpose, accumulate, x, y, st);
        if (Lx == 4 && Ly == 6) return launch_mv_t<V, kTorusPairs4x6>(op, transpose, accumulate, x, y, st);
        if (Lx == 6 && Ly == 4) return launch_mv_t<V, kTorusPairs6x4>(op, transpose, accumulate, x, y, st);
        if (Lx == 4 && Ly == 4) return launch_mv_t<V, kTorusPairs4x4>(op, transpose, accumulate, x, y, st);
        return launch_mv_t<V, kGroupTorusPairs>(op, transpose, accumulate, x, y, st);
      }
      return launch_mv_t<V, kGroupTorus>(op, transpose, accumulate, x, y, st);
  }
}

}  // namespace

}  // namespace edhip
