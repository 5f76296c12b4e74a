// Space kernels: sector enumeration, prefix table, symmetry reduction,
// mapping export and batched lookup.
#include <hipcub/hipcub.hpp>

#include "kernels.hpp"

namespace edhip {

namespace {

constexpr int kBlock = 256;

__global__ __launch_bounds__(kBlock) void k_enumerate_sector(uint64_t first, uint64_t count, int n_bits,
                                                             const uint64_t* __restrict__ W, uint64_t* __restrict__ out) {
  extern __shared__ unsigned char lds[];
  uint64_t* Wl = (uint64_t*)lds;
  const int nw = (n_bits + 1) * (n_bits + 1);
  for (int i = threadIdx.x; i < nw; i += blockDim.x) Wl[i] = W[i];
  __syncthreads();
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  out[i] = unrank_word(first + i, n_bits, Wl);
}

// Multi-quantum-number sectors (sites of any number of states, QN tuples):
// words[i] = the i-th word of the sector in ascending order.  The most
// significant site is the last one, so ascending words are the lexicographic
// order of (state of site n-1, ..., state of site 0); the walk fixes the sites
// from the top, skipping the counted completions of every smaller state.
// Table entry sites[j].off + u*sites[j].ns + s: the number of words whose sites
// above j sum to upper-sum u (an index into the sums reachable at that level)
// and whose site j is in state s, and the index of the new upper sum (-1 when
// no word has it; such an entry has count 0 and is never taken).
template <bool STAGE>
__global__ __launch_bounds__(kBlock) void k_enumerate_qn(uint64_t count, int n_sites, const QnSite* __restrict__ sites,
                                                         int n_entries, const uint64_t* __restrict__ cnt_g,
                                                         const int32_t* __restrict__ nxt_g, uint64_t* __restrict__ out) {
  extern __shared__ unsigned char lds[];
  const uint64_t* cnt = cnt_g;
  const int32_t* nxt = nxt_g;
  if (STAGE) {
    uint64_t* c = (uint64_t*)lds;
    int32_t* x = (int32_t*)(c + n_entries);
    for (int i = threadIdx.x; i < n_entries; i += blockDim.x) {
      c[i] = cnt_g[i];
      x[i] = nxt_g[i];
    }
    __syncthreads();
    cnt = c;
    nxt = x;
  }
  const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  uint64_t r = i, w = 0;
  int u = 0;
  for (int j = n_sites - 1; j >= 0; --j) {
    const QnSite st = sites[j];
    const int e = st.off + min(u, st.n_upper - 1) * st.ns;
    int pick = st.ns - 1;
    for (int s = 0; s < st.ns - 1; ++s) {
      const uint64_t c = cnt[e + s];
      if (r < c) {
        pick = s;
        break;
      }
      r -= c;
    }
    w |= (uint64_t)pick << st.shift;
    u = max(nxt[e + pick], 0);
  }
  out[i] = w;
}

__global__ __launch_bounds__(kBlock) void k_build_prefix(const uint64_t* __restrict__ keys, int64_t dim, int shift,
                                                         uint64_t n_buckets, uint32_t* __restrict__ prefix) {
  uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j > n_buckets) return;
  uint64_t key = j << shift;
  int64_t lo = 0, hi = dim;
  while (lo < hi) {
    int64_t mid = lo + ((hi - lo) >> 1);
    if (keys[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  prefix[j] = (uint32_t)lo;
}

// Walk the words of chunk [r0, r1) of the source in ascending order.
template <typename F>
__device__ __forceinline__ void for_chunk(const ReduceSource& src, const uint64_t* Wl, uint64_t r0, uint64_t r1, F&& f) {
  if (r0 >= r1) return;
  if (src.list) {
    for (uint64_t r = r0; r < r1; ++r) f(src.list[r]);
    return;
  }
  uint64_t w = unrank_word(r0, src.n_bits, Wl);
  for (uint64_t r = r0; r < r1; ++r) {
    if (r != r0) w = src.single_popcount ? next_same_popcount(w) : unrank_word(r, src.n_bits, Wl);
    f(w);
  }
}

__device__ __forceinline__ const uint64_t* stage_W(const ReduceSource& src, unsigned char* lds, uint32_t off) {
  uint64_t* Wl = (uint64_t*)(lds + off);
  if (!src.list) {
    const int nw = (src.n_bits + 1) * (src.n_bits + 1);
    for (int i = threadIdx.x; i < nw; i += blockDim.x) Wl[i] = src.W[i];
  }
  return Wl;
}

__global__ __launch_bounds__(kBlock) void k_reduce_count(ReduceSource src, uint64_t chunk, uint64_t n_threads, GroupDev g,
                                                         GroupLdsLayout lay, uint32_t* __restrict__ counts) {
  extern __shared__ unsigned char lds[];
  GroupLds L = stage_group(g, lay, lds);
  const uint64_t* Wl = stage_W(src, lds, lay.total);
  __syncthreads();
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_threads) return;
  uint64_t r0 = t * chunk;
  uint64_t r1 = r0 + chunk < src.n_words ? r0 + chunk : src.n_words;
  uint32_t c = 0;
  for_chunk(src, Wl, r0, r1, [&](uint64_t w) {
    int orbit;
    if (is_representative(g, L, w, orbit)) ++c;
  });
  counts[t] = c;
}

__global__ __launch_bounds__(kBlock) void k_reduce_write(ReduceSource src, uint64_t chunk, uint64_t n_threads, GroupDev g,
                                                         GroupLdsLayout lay, const uint64_t* __restrict__ offsets,
                                                         uint64_t* __restrict__ reps, uint16_t* __restrict__ orbits) {
  extern __shared__ unsigned char lds[];
  GroupLds L = stage_group(g, lay, lds);
  const uint64_t* Wl = stage_W(src, lds, lay.total);
  __syncthreads();
  uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_threads) return;
  uint64_t r0 = t * chunk;
  uint64_t r1 = r0 + chunk < src.n_words ? r0 + chunk : src.n_words;
  uint64_t pos = offsets[t];
  for_chunk(src, Wl, r0, r1, [&](uint64_t w) {
    int orbit;
    if (is_representative(g, L, w, orbit)) {
      reps[pos] = w;
      orbits[pos] = (uint16_t)orbit;
      ++pos;
    }
  });
}

// The same for the translations alone on a shape of window.hpp, from a sector of
// one popcount: a word whose own beginning is not among the least is dropped
// after its windows are read, as nearly all are; the images of the other
// candidates decide the rest.  Bound by instruction issue.  4x7 (0,0), 40M words:
// 92 us a pass, 225 us with the general test.
template <int KIND, int LX, int LY, bool WRITE>
__global__ __launch_bounds__(kBlock) void k_reduce_win(ReduceSource src, uint64_t chunk, uint64_t n_threads, GroupDev g,
                                                       uint32_t* __restrict__ counts,
                                                       const uint64_t* __restrict__ offsets,
                                                       uint64_t* __restrict__ reps, uint16_t* __restrict__ orbits) {
  using S = Win<KIND, LX, LY>;
  using W = typename S::W;
  using C = typename S::C;
  extern __shared__ unsigned char lds[];
  constexpr uint32_t at_trivial = S::kTabBytes, at_w = at_trivial + 64;
  lds_copy16(lds, g.win_tab, S::kTabBytes);
  if (threadIdx.x < 64) lds[at_trivial + threadIdx.x] = g.trivial[g.win_elem[threadIdx.x]];
  const uint64_t* Wl = stage_W(src, lds, at_w);
  __syncthreads();
  const uint64_t t = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n_threads) return;
  const uint64_t r0 = t * chunk, r1 = r0 + chunk < src.n_words ? r0 + chunk : src.n_words;
  const LdsPtr<uint16_t> tab = lds_at<uint16_t>(0);
  constexpr C own = S::kChain ? (C)1 : (C)1 << (8 * (LY - 1));  // the identity
  uint64_t pos = WRITE ? offsets[t] : 0;
  uint64_t w = unrank_word(r0, src.n_bits, Wl);
  for (uint64_t r = r0; r < r1; ++r) {
    if (r != r0) w = next_same_popcount(w);
    const W b = (W)w;
    C cand = S::candidates(tab, b, src.n_bits);
    bool rep = (cand & own) != 0;
    cand &= ~own;
    int stab = 1;
    while (rep && cand) {
      const int q = S::ctz(cand);
      cand &= cand - 1;
      const W img = S::image(b, src.n_bits, q);
      if (img == b) ++stab;
      rep = img > b || (img == b && lds[at_trivial + q]);
    }
    if (rep) {
      if constexpr (WRITE) {
        reps[pos] = w;
        orbits[pos] = (uint16_t)(g.G / stab);
      }
      ++pos;
    }
  }
  if constexpr (!WRITE) counts[t] = (uint32_t)pos;
}

template <bool WRITE>
hipError_t launch_reduce_win(const ReduceSource& src, uint64_t chunk, uint64_t n_threads, const GroupDev& g,
                             uint32_t* counts, const uint64_t* offsets, uint64_t* reps, uint16_t* orbits,
                             hipStream_t st) {
  const dim3 grid((unsigned)((n_threads + kBlock - 1) / kBlock));
  const uint32_t w = (uint32_t)((src.n_bits + 1) * (src.n_bits + 1) * 8);
#define EDHIP_REDUCE(K, X, Y)                                                                                        \
  const hipError_t e = lds_from_zero<k_reduce_win<K, X, Y, WRITE>>();                                                \
  if (e != hipSuccess) return e;                                                                                     \
  hipLaunchKernelGGL((k_reduce_win<K, X, Y, WRITE>), grid, dim3(kBlock), (Win<K, X, Y>::kTabBytes + 64 + w), st, src, \
                     chunk, n_threads, g, counts, offsets, reps, orbits);                                            \
  return hipGetLastError();
#define EDHIP_X(K, X, Y) \
  if (g.Lx == X && g.Ly == Y) { EDHIP_REDUCE(K, X, Y) }
  EDHIP_WIN_SHAPES(EDHIP_X)
#undef EDHIP_X
  if (src.n_bits <= 32) { EDHIP_REDUCE(kWinChain, 32, 1) }
  EDHIP_REDUCE(kWinChain, 48, 1)
#undef EDHIP_REDUCE
}

// Whether the reduction runs by windows.
bool reduce_by_windows(const ReduceSource& src, const GroupDev& g) {
  return g.win_tab && !src.list && src.single_popcount;
}

__global__ __launch_bounds__(kBlock) void k_export_mapping(ReduceSource src, GroupDev g, GroupLdsLayout lay, IndexDev ix,
                                                           const uint16_t* __restrict__ orbit,
                                                           int64_t* __restrict__ idx_out, double* __restrict__ re_out,
                                                           double* __restrict__ im_out) {
  extern __shared__ unsigned char lds[];
  GroupLds L = stage_group(g, lay, lds);
  const uint64_t* Wl = stage_W(src, lds, lay.total);
  __syncthreads();
  uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= src.n_words) return;
  uint64_t w = src.list ? src.list[p] : unrank_word(p, src.n_bits, Wl);
  uint64_t s;
  int h, cnt;
  canonicalize(g, L, w, s, h, cnt);
  int64_t r = search_sorted(ix.keys, ix.prefix, ix.n_buckets, ix.shift, s);
  if (r < 0) {
    idx_out[p] = -1;
    re_out[p] = 0.0;
    im_out[p] = 0.0;
    return;
  }
  double scale = g.invsqrt[orbit[r]];
  idx_out[p] = r;
  re_out[p] = g.ph_re[h] * scale;
  im_out[p] = g.ph_im[h] * scale;
}

// symmetry_unreduce (symmetry_reduce.jl:208-225): large[p] = U[p] * small[r(p)]
// for every parent word p, 0 where p lies outside the reduced space.  The
// mapping (r, U) is recomputed as in k_export_mapping; one lane per parent
// entry, coalesced writes.
template <typename V>
__global__ __launch_bounds__(kBlock) void k_vec_unreduce(ReduceSource src, GroupDev g, GroupLdsLayout lay, IndexDev ix,
                                                         const uint16_t* __restrict__ orbit, const V* __restrict__ small,
                                                         V* __restrict__ large) {
  extern __shared__ unsigned char lds[];
  GroupLds L = stage_group(g, lay, lds);
  const uint64_t* Wl = stage_W(src, lds, lay.total);
  __syncthreads();
  uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= src.n_words) return;
  uint64_t w = src.list ? src.list[p] : unrank_word(p, src.n_bits, Wl);
  uint64_t s;
  int h, cnt;
  canonicalize(g, L, w, s, h, cnt);
  int64_t r = search_sorted(ix.keys, ix.prefix, ix.n_buckets, ix.shift, s);
  V out = vzero<V>();
  if (r >= 0) {
    using R = typename VT<V>::R;
    const double scale = g.invsqrt[orbit[r]];
    vfma(out, (R)(L.ph_re[h] * scale), (R)(L.ph_im[h] * scale), small[r]);
  }
  large[p] = out;
}

// symmetry_reduce of a vector (symmetry_reduce.jl:38-56):
//   small[r] = sum_{p in orbit(r)} conj(U[p]) * large[p].
// Gather form, one lane per representative s: every element g gives the
// orbit member g(s) with conj(U[g(s)]) = chi(g) / sqrt(N_s); a member reached
// by |Stab(s)| elements (all with the same character, since s is compatible)
// is counted once by dividing by |Stab(s)| = G / N_s.
template <typename V>
__global__ __launch_bounds__(kBlock) void k_vec_reduce(const uint64_t* __restrict__ reps, const uint16_t* __restrict__ orbit,
                                                       int64_t dim, GroupDev g, GroupLdsLayout lay, IndexDev pix,
                                                       const V* __restrict__ large, V* __restrict__ small) {
  extern __shared__ unsigned char lds[];
  GroupLds L = stage_group(g, lay, lds);
  uint64_t* Wl = (uint64_t*)(lds + lay.total);
  if (pix.rank_mode) {
    const int nw = (pix.n_bits + 1) * (pix.n_bits + 1);
    for (int i = threadIdx.x; i < nw; i += blockDim.x) Wl[i] = pix.W[i];
  }
  __syncthreads();
  const int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= dim) return;
  using R = typename VT<V>::R;
  const uint64_t s = reps[r];
  const int n_orb = orbit[r];
  const double scale = g.invsqrt[n_orb] * (double)n_orb / (double)g.G;
  V acc = vzero<V>();
  auto add = [&](int e, uint64_t img) {
    const int64_t p = index_of(pix, Wl, img);
    if (p < 0) return;
    const int ie = L.inv[e];  // chi(e) = conj(phase[e^-1])
    vfma(acc, (R)(L.ph_re[ie] * scale), (R)(-L.ph_im[ie] * scale), large[p]);
  };
  if (g.mode == kGroupTorus) {
    const int nT = g.Lx * g.Ly;
    for (int p = 0; p < g.n_cosets; ++p) {  // elements T(pos) p
      const uint64_t sp = apply_coset(g, L, p, s);
      for (int bb = 0; bb < g.Ly; ++bb) {
        const uint64_t shifted = rows_shift(sp, bb, g.Lx, g.nb, g.full_mask);
        for (int a = 0; a < g.Lx; ++a)
          add(L.coset_elem[p * nT + a + g.Lx * bb], rows_rotl(shifted, a, g.Lx, L.rot_hi, L.rot_lo));
      }
    }
  } else {
    const int stride = g.n_nib << 4;
    with_nib_tables(g, L, [&](const uint64_t* nib) {
      for (int e = 0; e < g.G; ++e) add(e, perm_apply_nib(nib + e * stride, g.n_nib, s) ^ (g.has_xor ? L.xr[e] : 0ull));
    });
  }
  small[r] = acc;
}

__global__ __launch_bounds__(kBlock) void k_lookup(IndexDev ix, int64_t n, const uint64_t* __restrict__ keys,
                                                   int64_t* __restrict__ out) {
  extern __shared__ unsigned char lds[];
  uint64_t* Wl = (uint64_t*)lds;
  if (ix.rank_mode) {
    const int nw = (ix.n_bits + 1) * (ix.n_bits + 1);
    for (int i = threadIdx.x; i < nw; i += blockDim.x) Wl[i] = ix.W[i];
  }
  __syncthreads();
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  out[i] = index_of(ix, Wl, keys[i]);
}

// One block of the rank index: its first word is found through the prefix table,
// its words follow each other in the keys.  (Bits set by atomics, counted,
// scanned and written back by four more kernels over the blocks: 113 us on the
// 1.4M words of the 4x7 (0,0) sector, 44 us this way.)
__global__ __launch_bounds__(kBlock) void k_rank_blocks(const uint64_t* __restrict__ keys, int64_t dim,
                                                        const uint32_t* __restrict__ prefix, int shift,
                                                        uint64_t n_buckets, ulonglong2* __restrict__ blocks,
                                                        uint64_t n_blocks) {
  const uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= n_blocks) return;
  uint64_t key = j * kRankBlockWords;
  const uint64_t bucket = key >> shift;
  int64_t lo = dim, hi = dim;
  if (bucket < n_buckets) {
    lo = prefix[bucket];
    hi = prefix[bucket + 1];
  }
  while (lo < hi) {
    const int64_t mid = lo + ((hi - lo) >> 1);
    if (keys[mid] < key)
      lo = mid + 1;
    else
      hi = mid;
  }
  uint64_t word[8] = {0, 0, 0, 0, 0, 0, (uint64_t)lo, 0};
  uint32_t c = 0;
  uint64_t next = lo < dim ? keys[lo] : ~0ull;
#pragma unroll
  for (int w = 0; w < 6; ++w) {
    if (w > 0) word[7] |= (uint64_t)c << (9 * (w - 1));
    key += 64;
    while (next < key) {
      word[w] |= 1ull << (next & 63u);
      ++c;
      next = ++lo < dim ? keys[lo] : ~0ull;
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) blocks[4 * j + q] = ulonglong2{word[2 * q], word[2 * q + 1]};
}

// flags[key >> shift] = 1 for the top value of every key (idempotent stores)
__global__ __launch_bounds__(kBlock) void k_mark_tops(const uint64_t* __restrict__ keys, int64_t dim, int shift,
                                                      uint32_t* __restrict__ flags) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  flags[keys[i] >> shift] = 1u;
}

// Before a product: x spread over the word positions (XMapDev).
template <typename V>
__global__ __launch_bounds__(kBlock) void k_xmap_fill(XMapDev X, const uint64_t* __restrict__ keys, int64_t dim,
                                                      const V* __restrict__ x, const uint16_t* __restrict__ orbit, int G) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  const uint64_t k = keys[i];
  const uint64_t pos = xmap_pos(X, X.colex, X.topcode[k >> X.top_shift], k);
  V v = x[i];
  if (orbit) {  // x sqrt(G / N), scaled in double
    using R = typename VT<V>::R;
    const double sc = sqrt((double)G / (double)orbit[i]);
    if constexpr (VT<V>::cx) {
      v.re = (R)((double)v.re * sc);
      v.im = (R)((double)v.im * sc);
    } else {
      v = (R)((double)v * sc);
    }
  }
  ((V*)X.values)[pos] = v;
}

// Ranks of the positions: a word sets its bit, and the first word of a block,
// whose index is the rank below, the block's base.  (The bases of blocks without
// words are never read.)  One pass over the words, no scan.
__global__ __launch_bounds__(kBlock) void k_position_ranks(XMapDev X, const uint64_t* __restrict__ keys, int64_t dim,
                                                           RankBits* __restrict__ blocks) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= dim) return;
  const uint64_t k = keys[i];
  const uint32_t pos = (uint32_t)xmap_pos(X, X.colex, X.topcode[k >> X.top_shift], k);
  atomicOr(&blocks[pos >> 5].bits, 1u << (pos & 31u));
  bool first = i == 0;
  if (!first) {
    const uint64_t p = keys[i - 1];
    first = (uint32_t)xmap_pos(X, X.colex, X.topcode[p >> X.top_shift], p) >> 5 != pos >> 5;
  }
  if (first) blocks[pos >> 5].base = (uint32_t)i;
}

__global__ void k_u32_to_u64(const uint32_t* __restrict__ in, uint64_t* __restrict__ out, uint64_t n) {
  uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = in[i];
}

inline unsigned grid_for(uint64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }

inline uint32_t w_bytes(int n_bits) { return (uint32_t)((n_bits + 1) * (n_bits + 1) * sizeof(uint64_t)); }

}  // namespace

hipError_t launch_enumerate_sector(uint64_t first, uint64_t count, int n_bits, const uint64_t* d_W, uint64_t* d_out,
                                   hipStream_t st) {
  if (count == 0) return hipSuccess;
  hipLaunchKernelGGL(k_enumerate_sector, dim3(grid_for(count)), dim3(kBlock), w_bytes(n_bits), st, first, count, n_bits,
                     d_W, d_out);
  return hipGetLastError();
}

hipError_t launch_enumerate_qn(uint64_t count, int n_sites, const QnSite* d_sites, int n_entries, const uint64_t* d_cnt,
                               const int32_t* d_nxt, uint64_t* d_out, hipStream_t st) {
  if (count == 0) return hipSuccess;
  const size_t lds = (size_t)n_entries * (sizeof(uint64_t) + sizeof(int32_t));
  if (lds <= kQnStageBytes)
    hipLaunchKernelGGL(k_enumerate_qn<true>, dim3(grid_for(count)), dim3(kBlock), (uint32_t)lds, st, count, n_sites,
                       d_sites, n_entries, d_cnt, d_nxt, d_out);
  else
    hipLaunchKernelGGL(k_enumerate_qn<false>, dim3(grid_for(count)), dim3(kBlock), 0, st, count, n_sites, d_sites,
                       n_entries, d_cnt, d_nxt, d_out);
  return hipGetLastError();
}

hipError_t launch_build_prefix(const uint64_t* d_keys, int64_t dim, int shift, uint64_t n_buckets, uint32_t* d_prefix,
                               hipStream_t st) {
  hipLaunchKernelGGL(k_build_prefix, dim3(grid_for(n_buckets + 1)), dim3(kBlock), 0, st, d_keys, dim, shift, n_buckets,
                     d_prefix);
  return hipGetLastError();
}

hipError_t launch_reduce_count(const ReduceSource& src, uint64_t chunk, uint64_t n_threads, const GroupDev& g,
                               const GroupLdsLayout& lay, const uint64_t*, uint32_t* d_counts, hipStream_t st) {
  if (n_threads == 0) return hipSuccess;
  if (reduce_by_windows(src, g))
    return launch_reduce_win<false>(src, chunk, n_threads, g, d_counts, nullptr, nullptr, nullptr, st);
  uint32_t lds = lay.total + (src.list ? 0u : w_bytes(src.n_bits));
  hipLaunchKernelGGL(k_reduce_count, dim3(grid_for(n_threads)), dim3(kBlock), lds, st, src, chunk, n_threads, g, lay,
                     d_counts);
  return hipGetLastError();
}

hipError_t launch_reduce_write(const ReduceSource& src, uint64_t chunk, uint64_t n_threads, const GroupDev& g,
                               const GroupLdsLayout& lay, const uint64_t* d_offsets, uint64_t* d_reps,
                               uint16_t* d_orbit, hipStream_t st) {
  if (n_threads == 0) return hipSuccess;
  if (reduce_by_windows(src, g))
    return launch_reduce_win<true>(src, chunk, n_threads, g, nullptr, d_offsets, d_reps, d_orbit, st);
  uint32_t lds = lay.total + (src.list ? 0u : w_bytes(src.n_bits));
  hipLaunchKernelGGL(k_reduce_write, dim3(grid_for(n_threads)), dim3(kBlock), lds, st, src, chunk, n_threads, g, lay,
                     d_offsets, d_reps, d_orbit);
  return hipGetLastError();
}

hipError_t launch_export_mapping(const ReduceSource& src, const GroupDev& g, const GroupLdsLayout& lay,
                                 const IndexDev& reduced_index, const uint16_t* d_orbit, int64_t* d_idx, double* d_re,
                                 double* d_im, hipStream_t st) {
  if (src.n_words == 0) return hipSuccess;
  uint32_t lds = lay.total + (src.list ? 0u : w_bytes(src.n_bits));
  hipLaunchKernelGGL(k_export_mapping, dim3(grid_for(src.n_words)), dim3(kBlock), lds, st, src, g, lay, reduced_index,
                     d_orbit, d_idx, d_re, d_im);
  return hipGetLastError();
}

hipError_t launch_lookup(const IndexDev& ix, int64_t n, const uint64_t* d_keys, int64_t* d_idx, hipStream_t st) {
  if (n == 0) return hipSuccess;
  uint32_t lds = ix.rank_mode ? w_bytes(ix.n_bits) : 0u;
  hipLaunchKernelGGL(k_lookup, dim3(grid_for((uint64_t)n)), dim3(kBlock), lds, st, ix, n, d_keys, d_idx);
  return hipGetLastError();
}

hipError_t launch_rank_blocks(const uint64_t* d_keys, int64_t dim, const uint32_t* d_prefix, int shift,
                              uint64_t n_buckets, uint64_t* d_blocks, uint64_t n_blocks, hipStream_t st) {
  hipLaunchKernelGGL(k_rank_blocks, dim3(grid_for(n_blocks)), dim3(kBlock), 0, st, d_keys, dim, d_prefix, shift,
                     n_buckets, (ulonglong2*)d_blocks, n_blocks);
  return hipGetLastError();
}

hipError_t launch_mark_tops(const uint64_t* d_keys, int64_t dim, int shift, uint32_t* d_flags, hipStream_t st) {
  if (dim == 0) return hipSuccess;
  hipLaunchKernelGGL(k_mark_tops, dim3(grid_for((uint64_t)dim)), dim3(kBlock), 0, st, d_keys, dim, shift, d_flags);
  return hipGetLastError();
}

hipError_t launch_xmap_fill(int prec, const XMapDev& X, const uint64_t* d_keys, int64_t dim, const void* x,
                            const uint16_t* d_orbit, int G, hipStream_t st) {
  if (dim == 0) return hipSuccess;
  dim3 grid(grid_for((uint64_t)dim));
  switch (prec) {
    case kF64:
      hipLaunchKernelGGL(k_xmap_fill<double>, grid, dim3(kBlock), 0, st, X, d_keys, dim, (const double*)x, d_orbit, G);
      break;
    case kC128:
      hipLaunchKernelGGL(k_xmap_fill<Cx<double>>, grid, dim3(kBlock), 0, st, X, d_keys, dim, (const Cx<double>*)x,
                         d_orbit, G);
      break;
    case kF32:
      hipLaunchKernelGGL(k_xmap_fill<float>, grid, dim3(kBlock), 0, st, X, d_keys, dim, (const float*)x, d_orbit, G);
      break;
    case kC64:
      hipLaunchKernelGGL(k_xmap_fill<Cx<float>>, grid, dim3(kBlock), 0, st, X, d_keys, dim, (const Cx<float>*)x,
                         d_orbit, G);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_position_ranks(const XMapDev& X, const uint64_t* d_keys, int64_t dim, uint64_t n_blocks,
                                 RankBits* d_bits, hipStream_t st) {
  if (dim == 0) return hipSuccess;
  hipError_t e = hipMemsetAsync(d_bits, 0, n_blocks * sizeof(RankBits), st);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(k_position_ranks, dim3(grid_for((uint64_t)dim)), dim3(kBlock), 0, st, X, d_keys, dim, d_bits);
  return hipGetLastError();
}

hipError_t exclusive_scan_u32_to_u64(const uint32_t* d_in, uint64_t* d_out, uint64_t n, void* d_tmp, size_t& tmp_bytes,
                                     hipStream_t st) {
  // d_out doubles as the widened input; the scan runs in place.
  if (d_tmp == nullptr) {
    return hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, d_out, d_out, (int64_t)n, st);
  }
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_u32_to_u64, dim3(grid_for(n)), dim3(kBlock), 0, st, d_in, d_out, n);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  return hipcub::DeviceScan::ExclusiveSum(d_tmp, tmp_bytes, d_out, d_out, (int64_t)n, st);
}

hipError_t exclusive_scan_i64(const int64_t* d_in, int64_t* d_out, uint64_t n, void* d_tmp, size_t& tmp_bytes,
                              hipStream_t st) {
  if (d_tmp == nullptr) {
    return hipcub::DeviceScan::ExclusiveSum(nullptr, tmp_bytes, d_in, d_out, (int64_t)n, st);
  }
  if (n == 0) return hipSuccess;
  return hipcub::DeviceScan::ExclusiveSum(d_tmp, tmp_bytes, d_in, d_out, (int64_t)n, st);
}

namespace {
template <typename V>
hipError_t vec_unreduce_t(const ReduceSource& src, const GroupDev& g, const GroupLdsLayout& lay, const IndexDev& ix,
                          const uint16_t* d_orbit, const void* small, void* large, hipStream_t st) {
  uint32_t lds = lay.total + (src.list ? 0u : w_bytes(src.n_bits));
  hipLaunchKernelGGL(k_vec_unreduce<V>, dim3(grid_for(src.n_words)), dim3(kBlock), lds, st, src, g, lay, ix, d_orbit,
                     (const V*)small, (V*)large);
  return hipGetLastError();
}

template <typename V>
hipError_t vec_reduce_t(const uint64_t* d_reps, const uint16_t* d_orbit, int64_t dim, const GroupDev& g,
                        const GroupLdsLayout& lay, const IndexDev& pix, const void* large, void* small, hipStream_t st) {
  uint32_t lds = lay.total + (pix.rank_mode ? w_bytes(pix.n_bits) : 0u);
  hipLaunchKernelGGL(k_vec_reduce<V>, dim3(grid_for((uint64_t)dim)), dim3(kBlock), lds, st, d_reps, d_orbit, dim, g, lay,
                     pix, (const V*)large, (V*)small);
  return hipGetLastError();
}
}  // namespace

hipError_t launch_vec_unreduce(const ReduceSource& src, const GroupDev& g, const GroupLdsLayout& lay,
                               const IndexDev& reduced_index, const uint16_t* d_orbit, int prec, const void* d_small,
                               void* d_large, hipStream_t st) {
  if (src.n_words == 0) return hipSuccess;
  switch (prec) {
    case kF64:
      return vec_unreduce_t<double>(src, g, lay, reduced_index, d_orbit, d_small, d_large, st);
    case kC128:
      return vec_unreduce_t<Cx<double>>(src, g, lay, reduced_index, d_orbit, d_small, d_large, st);
    case kF32:
      return vec_unreduce_t<float>(src, g, lay, reduced_index, d_orbit, d_small, d_large, st);
    case kC64:
      return vec_unreduce_t<Cx<float>>(src, g, lay, reduced_index, d_orbit, d_small, d_large, st);
    default:
      return hipErrorInvalidValue;
  }
}

hipError_t launch_vec_reduce(const uint64_t* d_reps, const uint16_t* d_orbit, int64_t dim, const GroupDev& g,
                             const GroupLdsLayout& lay, const IndexDev& parent_index, int prec, const void* d_large,
                             void* d_small, hipStream_t st) {
  if (dim == 0) return hipSuccess;
  switch (prec) {
    case kF64:
      return vec_reduce_t<double>(d_reps, d_orbit, dim, g, lay, parent_index, d_large, d_small, st);
    case kC128:
      return vec_reduce_t<Cx<double>>(d_reps, d_orbit, dim, g, lay, parent_index, d_large, d_small, st);
    case kF32:
      return vec_reduce_t<float>(d_reps, d_orbit, dim, g, lay, parent_index, d_large, d_small, st);
    case kC64:
      return vec_reduce_t<Cx<float>>(d_reps, d_orbit, dim, g, lay, parent_index, d_large, d_small, st);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace edhip
