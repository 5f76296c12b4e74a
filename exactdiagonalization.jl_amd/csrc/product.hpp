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
// SCALED: x is read from its spread holding x / sqrt(N) (op.xm.scaled), so the
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
  const MvTerms T = stage_mv_terms(op, lds, kW32, VT<V>::cx);
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

  V acc = vzero<V>();
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
        bool f0, f1;
        xmap_fetch2(op.xm, codes, sk[0], sk[1], xv[0], xv[1], f0, f1);
        ik[0] = f0 ? 0 : -1;
        ik[1] = (ok[1] && f1) ? 0 : -1;
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
            vfma(acc, w, 0.f, xv[k]);
          } else {
            double wr, wi;
            element_weight_a<MODE, TRANS, UNIT, SCALED>(op, L, __longlong_as_double((long long)fa[k].y),
                                                        VT<V>::cx ? T.ai[t[k]] : 0.0, hk[k], ck[k], wr, wi);
            vfma(acc, (R)wr, (R)wi, xv[k]);
          }
        }
      }
    }
  }
  acc = row_lanes_sum(acc, op.row_lanes);
  if (sub != 0) return;
  // diagonal terms (C == R): the element is the summed amplitude (U[b]/U[b] = 1)
  double dre = 0.0, dim_ = 0.0;
  if (op.diag_re) {
    dre = op.diag_re[row];
    if (op.diag_im) dim_ = op.diag_im[row];
  } else {
    diag_sum(op, b, dre, dim_);
  }
  V out = vzero<V>();
  vfma(out, (R)dre, (R)dim_, x[row]);
  if constexpr (MODE != kGroupNone)
    vfma(out, (R)sqrt((double)op.orbit[row]), (R)0, acc);
  else
    out = vadd(out, acc);
  V* yr = y + (row - op.row_begin);
  *yr = accumulate ? vadd(*yr, out) : out;
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
        if (op.g.n_cosets == 1) {
          if (Lx == 6 && Ly == 6) return launch_mv_t<V, kTransPairs6x6>(op, transpose, accumulate, x, y, st);
          if (Lx == 4 && Ly == 6) return launch_mv_t<V, kTransPairs4x6>(op, transpose, accumulate, x, y, st);
          if (Lx == 6 && Ly == 4) return launch_mv_t<V, kTransPairs6x4>(op, transpose, accumulate, x, y, st);
          if (Lx == 4 && Ly == 4) return launch_mv_t<V, kTransPairs4x4>(op, transpose, accumulate, x, y, st);
        }
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
