// The term pass (bilinear forms g_t = sum_r conj(phi_r) sum_{images of t} psi_s,
// unit amplitudes) on sectors of one popcount without a symmetry group, up to
// kRankBits bits, where a word's index is the sum of two table entries: the
// number of sector words with a smaller upper part, and the rank of its lower
// part (RankTables).
#include "opterms.hpp"

namespace edhip {

namespace {

template <typename V>
__device__ __forceinline__ void value_of(const V& v, double& re, double& im) {
  if constexpr (VT<V>::cx) {
    re = (double)v.re;
    im = (double)v.im;
  } else {
    re = (double)v;
    im = 0.0;
  }
}

__device__ __forceinline__ double wave_sum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// Off-diagonal terms: the lanes of a wave take the steps of a window (blockIdx.y)
// together, one row each, every step's sums in registers.  A step is a term, or
// two that share mask and flip (S+S- and S-S+), of which a row matches at most
// one: one test, one image and one gather for both, and psi read at its rank from
// two LDS tables, of which a step reads those of the parts that it flips.  Bound
// by instruction issue, about 26 VALU instructions per step and row.  4x6 XXZ, 96
// terms, FP64: 110 us; one term per step, psi from its spread: 236 us and 14 us to
// spread it.  (Windows of 8, 12 and 16 steps: 117, 139 and 236 us, their registers
// cost waves; loads under the lanes' own tests instead of a second choice of
// address: 152 us, each waits for the one before.)
template <typename V, int KT>
__global__ __launch_bounds__(kMvBlock) void k_expect_steps(ExpectRank E, int64_t dim, const V* __restrict__ phi,
                                                           const V* __restrict__ psi, double* __restrict__ partial) {
  constexpr bool CX = VT<V>::cx;
  extern __shared__ unsigned char lds[];
  const uint32_t at_base = 2u << E.low_bits;
  lds_copy16(lds, E.rank_low, at_base);
  lds_copy16(lds + at_base, E.rank_base, E.base_bytes);
  __syncthreads();
  const LdsPtr<uint16_t> low = lds_at<uint16_t>(0);
  const LdsPtr<uint32_t> base = lds_at<uint32_t>(at_base);
  const uint32_t lmask = (1u << E.low_bits) - 1u;
  const int j0 = (int)blockIdx.y * KT;
  double ar[2][KT], ai[2][KT];
#pragma unroll
  for (int q = 0; q < KT; ++q) ar[0][q] = ar[1][q] = ai[0][q] = ai[1][q] = 0.0;
  for (int64_t row = (int64_t)blockIdx.x * kMvBlock + threadIdx.x; row < dim; row += (int64_t)gridDim.x * kMvBlock) {
    const uint32_t b = (uint32_t)E.rows[row];
    double fr, fi;
    value_of(phi[row], fr, fi);
    // ranks of the parts, read where the step flips them (the same for all lanes)
    const uint32_t own_low = low[b & lmask], own_base = base[b >> E.low_bits];
    uint32_t rl[KT], rb[KT];
#pragma unroll
    for (int q = 0; q < KT; ++q) {
      const uint32_t f = E.steps[j0 + q].flip;  // (padded to whole windows with steps that match nothing)
      rl[q] = own_low;
      rb[q] = own_base;
      if (f & lmask) rl[q] = low[(b ^ f) & lmask];
      if (f >> E.low_bits) rb[q] = base[(b ^ f) >> E.low_bits];
    }
    V s[KT];
#pragma unroll
    for (int q = 0; q < KT; ++q) {  // a row that does not match reads its own element, and drops it
      const uint32_t m = b & E.steps[j0 + q].mask;
      const bool any = (m == E.steps[j0 + q].match[0]) | (m == E.steps[j0 + q].match[1]);
      s[q] = psi[any ? rb[q] + rl[q] : (uint32_t)row];
    }
#pragma unroll
    for (int q = 0; q < KT; ++q) {
      const uint32_t m = b & E.steps[j0 + q].mask;
      const bool hit[2] = {m == E.steps[j0 + q].match[0], m == E.steps[j0 + q].match[1]};
      double sr, si;
      value_of(s[q], sr, si);
      const double pr = fr * sr + fi * si, pi = fr * si - fi * sr;  // conj(phi_r) psi_s
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        ar[h][q] += hit[h] ? pr : 0.0;
        if constexpr (CX) ai[h][q] += hit[h] ? pi : 0.0;
      }
    }
  }
  __syncthreads();  // the tables are done with
  constexpr int kWaves = kMvBlock / 64;
  double* sums = (double*)lds;  // [wave][KT][2][2]
  const int wave = threadIdx.x >> 6;
#pragma unroll
  for (int q = 0; q < KT; ++q)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const double a = wave_sum(ar[h][q]), c = CX ? wave_sum(ai[h][q]) : 0.0;
      if ((threadIdx.x & 63) == 0) {
        sums[((wave * KT + q) * 2 + h) * 2] = a;
        sums[((wave * KT + q) * 2 + h) * 2 + 1] = c;
      }
    }
  __syncthreads();
  if (threadIdx.x < 4 * KT) {
    const int q = threadIdx.x >> 2, h = (threadIdx.x >> 1) & 1, c = threadIdx.x & 1;
    const int t = E.steps[j0 + q].term[h];
    double v = 0.0;
    for (int w = 0; w < kWaves; ++w) v += sums[w * KT * 4 + threadIdx.x];
    if (t >= 0) partial[(int64_t)blockIdx.x * 2 * E.n_off + 2 * t + c] = v;
      }
}

// Diagonal terms: sum_r [b_r & mask == match] p_r with p = conj(phi) psi.  The
// rows of one upper part are consecutive, so a term that looks at the upper part
// alone needs the sums of p by upper part, one that looks at the lower part alone
// those by lower part, and one that looks at the upper part and one lower bit
// the sums by upper part and lower bit value: two passes over phi and psi and no
// test per row and term (which took 119 us on the 4x6 XXZ pass, 192 terms; now 26 us
// by upper part, 16 by lower part and 12 for the terms).
//
// Sums by upper part: X[h][0] = sum of p, X[h][1 + 2 i + v] over lower bit i = v.
// One wave per upper part.
template <typename V, int LB>
__global__ __launch_bounds__(kBlock) void k_expect_upper(ExpectRank E, int64_t dim, const V* __restrict__ phi,
                                                         const V* __restrict__ psi, double* __restrict__ X) {
  constexpr int N = 1 + 2 * LB, NC = VT<V>::cx ? 2 : 1;
  const int h = (int)blockIdx.x * (kBlock / 64) + (int)(threadIdx.x >> 6), lane = (int)(threadIdx.x & 63);
  if (h >= E.n_upper) return;
  const int64_t r0 = E.rank_base[h], r1 = h + 1 < E.n_upper ? (int64_t)E.rank_base[h + 1] : dim;
  double a[NC][N];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int k = 0; k < N; ++k) a[c][k] = 0.0;
  for (int64_t r = r0 + lane; r < r1; r += 64) {
    const uint32_t b = (uint32_t)E.rows[r];
    double fr, fi, pr, pi;
    value_of(phi[r], fr, fi);
    value_of(psi[r], pr, pi);
    const double p[2] = {fr * pr + fi * pi, fr * pi - fi * pr};
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      a[c][0] += p[c];
#pragma unroll
      for (int i = 0; i < LB; ++i) {
        const bool one = (b >> i) & 1u;
        a[c][1 + 2 * i] += one ? 0.0 : p[c];
        a[c][2 + 2 * i] += one ? p[c] : 0.0;
      }
    }
  }
  double* out = X + (int64_t)h * N * 2;
#pragma unroll
  for (int k = 0; k < N; ++k) {
    const double re = wave_sum(a[0][k]), im = NC == 2 ? wave_sum(a[NC - 1][k]) : 0.0;
    if (lane == 0) {
      out[2 * k] = re;
      out[2 * k + 1] = im;
    }
  }
}

// Sums by lower part, over the upper parts hs[split], hs[split + n], ... of those
// with the popcount left: Q[blockIdx.y][lower part].  A block takes 64 lower
// parts of one popcount (their rows are neighbours), its four waves every fourth
// of the block's upper parts.
template <typename V>
__global__ __launch_bounds__(kBlock) void k_expect_lower(ExpectRank E, const V* __restrict__ phi,
                                                         const V* __restrict__ psi, double* __restrict__ Q) {
  __shared__ double part[kBlock / 64][64][2];
  const int pop = E.items[2 * blockIdx.x], k = E.items[2 * blockIdx.x + 1] + (int)(threadIdx.x & 63);
  const int wave = (int)threadIdx.x >> 6;
  const int n_lo = E.lo_off[pop + 1] - E.lo_off[pop];
  const int up = E.pop - pop;  // popcount of the upper part
  const int h0 = up >= 0 && up <= E.upper_bits ? E.up_off[up] : 0;
  const int h1 = up >= 0 && up <= E.upper_bits ? E.up_off[up + 1] : 0;
  double re = 0.0, im = 0.0;
  if (k < n_lo)
    for (int i = h0 + (int)blockIdx.y * 4 + wave; i < h1; i += 4 * kExpectSplits) {
      const int64_t r = (int64_t)E.rank_base[E.up_list[i]] + k;
      double fr, fi, pr, pi;
      value_of(phi[r], fr, fi);
      value_of(psi[r], pr, pi);
      re += fr * pr + fi * pi;
      im += fr * pi - fi * pr;
    }
  part[wave][threadIdx.x & 63][0] = re;
  part[wave][threadIdx.x & 63][1] = im;
  __syncthreads();
  if (wave == 0 && k < n_lo) {
    double s[2] = {0.0, 0.0};
    for (int w = 0; w < kBlock / 64; ++w) {
      s[0] += part[w][threadIdx.x][0];
      s[1] += part[w][threadIdx.x][1];
    }
    double* out = Q + (((int64_t)blockIdx.y << E.low_bits) + E.lo_list[E.lo_off[pop] + k]) * 2;
    out[0] = s[0];
    out[1] = s[1];
  }
}

// g of every diagonal term from the sums, one block per term.
__global__ __launch_bounds__(kBlock) void k_expect_diag(ExpectRank E, const DiagTerm* __restrict__ terms,
                                                        const double* __restrict__ X, const double* __restrict__ Q,
                                                        double* __restrict__ out) {
  __shared__ double part[kBlock / 64][2];
  const uint32_t mask = (uint32_t)terms[blockIdx.x].mask, match = (uint32_t)terms[blockIdx.x].match;
  const uint32_t lmask = (1u << E.low_bits) - 1u;
  const uint32_t ml = mask & lmask, cl = match & lmask, mh = mask >> E.low_bits, ch = match >> E.low_bits;
  double re = 0.0, im = 0.0;
  if (mh == 0) {
    for (uint32_t lo = threadIdx.x; lo <= lmask; lo += kBlock)
      if ((lo & ml) == cl)
        for (int s = 0; s < kExpectSplits; ++s) {
          const double2 v = ((const double2*)Q)[((int64_t)s << E.low_bits) + lo];
          re += v.x;
          im += v.y;
        }
  } else {
    const int n = 1 + 2 * E.low_bits, slot = ml ? 1 + 2 * (31 - __builtin_clz(ml)) + (cl ? 1 : 0) : 0;
    for (int h = (int)threadIdx.x; h < E.n_upper; h += kBlock)
      if (((uint32_t)h & mh) == ch) {
        const double2 v = ((const double2*)X)[(int64_t)h * n + slot];
        re += v.x;
        im += v.y;
      }
  }
  re = wave_sum(re);
  im = wave_sum(im);
  if ((threadIdx.x & 63) == 0) {
    part[threadIdx.x >> 6][0] = re;
    part[threadIdx.x >> 6][1] = im;
  }
  __syncthreads();
  if (threadIdx.x < 2) {
    double v = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) v += part[w][threadIdx.x];
    out[2 * blockIdx.x + threadIdx.x] = v;
  }
}

template <typename V>
hipError_t launch_rank_v(const ExpectRank& E, const OpDev& op, const void* phi, const void* psi, double* X, double* Q,
                         double* d_partial, double* d_out, hipStream_t st) {
  constexpr int KT = VT<V>::cx ? kExpectWindow / 2 : kExpectWindow;
  hipError_t e;
  if (op.n_diag > 0) {
    const dim3 up((unsigned)((E.n_upper + kBlock / 64 - 1) / (kBlock / 64)));
    if (E.low_bits == 12)
      hipLaunchKernelGGL((k_expect_upper<V, 12>), up, dim3(kBlock), 0, st, E, op.dim, (const V*)phi, (const V*)psi, X);
    else
      hipLaunchKernelGGL((k_expect_upper<V, 13>), up, dim3(kBlock), 0, st, E, op.dim, (const V*)phi, (const V*)psi, X);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_expect_lower<V>, dim3((unsigned)E.n_items, kExpectSplits), dim3(kBlock), 0, st, E,
                       (const V*)phi, (const V*)psi, Q);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    hipLaunchKernelGGL(k_expect_diag, dim3((unsigned)op.n_diag), dim3(kBlock), 0, st, E, op.diag, X, Q, d_out);
    if ((e = hipGetLastError()) != hipSuccess) return e;
  }
  if (E.n_steps > 0) {
    if ((e = lds_from_zero<k_expect_steps<V, KT>>()) != hipSuccess) return e;
    const int windows = E.n_steps / KT;
    const int64_t blocks = expect_rank_blocks(op.dim, windows);
    const uint32_t tables = (2u << E.low_bits) + E.base_bytes, sums = kMvBlock / 64 * KT * 4 * 8;
    hipLaunchKernelGGL((k_expect_steps<V, KT>), dim3((unsigned)blocks, (unsigned)windows), dim3(kMvBlock),
                       tables > sums ? tables : sums, st, E, op.dim, (const V*)phi, (const V*)psi, d_partial);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    return launch_expect_reduce(d_partial, blocks, 2 * op.n_off, d_out + 2 * (int64_t)op.n_diag, st);
  }
  return hipSuccess;
}

}  // namespace

hipError_t launch_term_expect_rank(const ExpectRank& E, const OpDev& op, int prec, const void* phi, const void* psi,
                                   double* X, double* Q, double* d_partial, double* d_out, hipStream_t st) {
  switch (prec) {
    case kF64:
      return launch_rank_v<double>(E, op, phi, psi, X, Q, d_partial, d_out, st);
    case kC128:
      return launch_rank_v<Cx<double>>(E, op, phi, psi, X, Q, d_partial, d_out, st);
    case kF32:
      return launch_rank_v<float>(E, op, phi, psi, X, Q, d_partial, d_out, st);
    case kC64:
      return launch_rank_v<Cx<float>>(E, op, phi, psi, X, Q, d_partial, d_out, st);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace edhip
