// Host-side launchers of the edhip kernels (implemented in the .hip files).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "device.hpp"
#include "host_logic.hpp"

namespace edhip {

// ---- space.hip -------------------------------------------------------------
// words[i] = unrank(first + i), i < count
hipError_t launch_enumerate_sector(uint64_t first, uint64_t count, int n_bits, const uint64_t* d_W, uint64_t* d_out,
                                   hipStream_t st);
// One site of a multi-quantum-number sector walk (k_enumerate_qn): its table
// entries start at off, ns states, bit offset shift, n_upper upper sums.
struct QnSite {
  int32_t off, ns, shift, n_upper;
};
// Tables up to this size are staged in LDS by the enumeration kernel.
constexpr size_t kQnStageBytes = 48 * 1024;
// words[i] = i-th word of a multi-QN sector in ascending order, i < count
hipError_t launch_enumerate_qn(uint64_t count, int n_sites, const QnSite* d_sites, int n_entries, const uint64_t* d_cnt,
                               const int32_t* d_nxt, uint64_t* d_out, hipStream_t st);
// flags[key >> shift] = 1 for every key
hipError_t launch_mark_tops(const uint64_t* d_keys, int64_t dim, int shift, uint32_t* d_flags, hipStream_t st);
// x spread over the word positions of X (before each product); with d_orbit,
// x sqrt(G / orbit) (the orbit factor of the images, X.scaled).
hipError_t launch_xmap_fill(int prec, const XMapDev& X, const uint64_t* d_keys, int64_t dim, const void* x,
                            const uint16_t* d_orbit, int G, hipStream_t st);
// Ranks of the words' positions in the spread X, which ascend with the words, in
// n_blocks blocks, which it clears first.
hipError_t launch_position_ranks(const XMapDev& X, const uint64_t* d_keys, int64_t dim, uint64_t n_blocks,
                                 RankBits* d_bits, hipStream_t st);
// prefix[j] = lower_bound(keys, j << shift), j <= n_buckets
hipError_t launch_build_prefix(const uint64_t* d_keys, int64_t dim, int shift, uint64_t n_buckets, uint32_t* d_prefix,
                               hipStream_t st);

struct ReduceSource {
  // either a popcount sector (unranked on the fly) or an explicit device list
  const uint64_t* list;  // nullptr for a sector
  uint64_t n_words;
  int n_bits;
  int single_popcount;   // 1: Gosper stepping is valid inside a chunk
  const uint64_t* W;     // completion counts (sector)
};

// pass 0: per-thread counts of representatives; pass 1: write them (ascending)
hipError_t launch_reduce_count(const ReduceSource& src, uint64_t chunk, uint64_t n_threads, const GroupDev& g,
                               const GroupLdsLayout& lay, const uint64_t* d_Wsrc, uint32_t* d_counts, hipStream_t st);
hipError_t launch_reduce_write(const ReduceSource& src, uint64_t chunk, uint64_t n_threads, const GroupDev& g,
                               const GroupLdsLayout& lay, const uint64_t* d_offsets, uint64_t* d_reps,
                               uint16_t* d_orbit, hipStream_t st);

// For every parent word p: mapping index (rep index or -1) and amplitude
// U[p] = phase[h] / sqrt(N_s) (0 when excluded).
hipError_t launch_export_mapping(const ReduceSource& src, const GroupDev& g, const GroupLdsLayout& lay,
                                 const IndexDev& reduced_index, const uint16_t* d_orbit, int64_t* d_idx, double* d_re,
                                 double* d_im, hipStream_t st);

hipError_t launch_lookup(const IndexDev& ix, int64_t n, const uint64_t* d_keys, int64_t* d_idx, hipStream_t st);

// Vector maps between a parent space and its reduction, in precision prec:
// large[p] = U[p] small[r(p)] (unreduce), small[r] = sum conj(U[p]) large[p]
// over the orbit of representative r (reduce).
hipError_t launch_vec_unreduce(const ReduceSource& src, const GroupDev& g, const GroupLdsLayout& lay,
                               const IndexDev& reduced_index, const uint16_t* d_orbit, int prec, const void* d_small,
                               void* d_large, hipStream_t st);
hipError_t launch_vec_reduce(const uint64_t* d_reps, const uint16_t* d_orbit, int64_t dim, const GroupDev& g,
                             const GroupLdsLayout& lay, const IndexDev& parent_index, int prec, const void* d_large,
                             void* d_small, hipStream_t st);

// Blocked rank index over the words [0, 384 n_blocks), layout as in IndexDev, from
// the sorted keys and their prefix table.
hipError_t launch_rank_blocks(const uint64_t* d_keys, int64_t dim, const uint32_t* d_prefix, int shift,
                              uint64_t n_buckets, uint64_t* d_blocks, uint64_t n_blocks, hipStream_t st);
hipError_t exclusive_scan_u32_to_u64(const uint32_t* d_in, uint64_t* d_out, uint64_t n, void* d_tmp, size_t& tmp_bytes,
                                     hipStream_t st);
hipError_t exclusive_scan_i64(const int64_t* d_in, int64_t* d_out, uint64_t n, void* d_tmp, size_t& tmp_bytes,
                              hipStream_t st);

// ---- matvec.hip, product_*.hip ---------------------------------------------
struct OpDev {
  IndexDev ix;           // lookup of canonical images
  GroupDev g;            // symmetry group
  GroupLdsLayout lay;    // LDS layout of the group tables
  const uint64_t* rows;  // basis words (the space's sorted keys)
  const uint16_t* orbit; // orbit sizes (reduced) or nullptr
  int64_t dim;           // rows of the space (products: the end of the rows computed)
  int64_t row_begin;     // products: first row computed; y holds rows row_begin .. dim - 1 from y[0]
  int n_off;             // number of off-diagonal terms (in the row or column sense)
  int n_diag;
  int word_bits;         // bits of the words and of every diagonal term's mask and match
  int xcd_chunk;         // products: consecutive blocks each XCD takes per window of 8 xcd_chunk (<= 1: plain order)
  const OffTerm* off;    // row form: match = R, image = C ; column form: match = C, image = R
  // The entries of the products (each an off-diagonal term, or two with one
  // flip and amplitude): n_lin parity entries, matched 64 at a time through
  // the tables lin_tab, then n_rest others matched by mask (rest).  Operators
  // without LDS room for them match off term by term (n_lin = 0, rest = off).
  const MvEntry* ent;       // n_lin + n_rest
  const uint64_t* lin_tab;  // [segment of 64 entries][chunk of 4 word bits][16]
  const OffTerm* rest;
  int n_lin;
  int n_chunk;              // chunks per segment (a multiple of 3; those past the word are zero)
  int n_rest;
  int rest_paired;          // rest comes in pairs that share a mask (runs of equal masks padded to even lengths
                            // with terms that match nothing and flip nothing)
  int row_lanes;            // products: log2 of the lanes that share a row
  uint64_t stripe;          // products: bits of a segment that the first of them takes
  const DiagTerm* diag;
  const double* diag_re; // per-row diagonal element (summed diagonal terms), or nullptr
  const double* diag_im; // its imaginary part, or nullptr when every diagonal amplitude is real
  uint32_t off_lds;      // LDS offset of the staged off-diagonal terms
  uint32_t w_lds;        // LDS offset of the staged rank table (rank mode)
  uint32_t w_bytes;
  XMapDev xm;            // matvec: x read from its spread over word positions (xm.values != null)
  uint32_t codes_lds;    // LDS offset of xm's code table, after lds_total (0: no room)
  uint32_t lds_total;    // LDS of the kernels (the term pass adds xm's code table)
  uint32_t mv_lds;       // the products' LDS: entries (mv_layout), rank table, xm's code table
  uint32_t mv_w_lds;
  uint32_t mv_codes_lds; // (0: no room for xm's code table)
  uint32_t mv_lds_total; // without xm's code table
};

// The products on the shapes of window.hpp (translations alone): what their
// kernels read.
struct WinOp {
  const uint64_t* rows;
  const uint16_t* orbit;
  const double* diag_re;  // null: no diagonal terms
  const double* diag_im;
  const uint16_t* win_tab;
  const int32_t* win_elem;
  const double* ph_re;
  const double* ph_im;
  const uint16_t* topcode;
  const uint16_t* colex;
  const void* values;     // the spread x sqrt(G / N)
  const uint64_t* lin_tab;
  const MvEntry* ent;
  const OffTerm* rest;
  uint64_t stripe;
  int64_t dim, row_begin;
  int n_bits, n_lin, n_chunk, n_rest, real_amp;
  int row_lanes, xcd_chunk, accumulate;
  int top_bits, top_shift, hbits;
  // sectors without a group, by rank (rank_low null: through the spread)
  const uint16_t* rank_low;   // colex rank of every low_bits-bit word among those of its popcount
  const uint32_t* rank_base;  // number of sector words with a smaller upper part
  int low_bits;
  uint32_t base_bytes;        // of rank_base, a multiple of 16
  // point operations (values: x sqrt(G / N) itself, 0 at the index none): ranks of the positions
  const RankBits* pos_bits;
  uint32_t none;
  int point_swap;
  int G;                  // order of the group (1: none)
};
// Sectors of up to this many bits are ranked by two LDS tables (13 + 13 bits: 48 KiB)
constexpr int kRankBits = 26;
// LDS bytes of the entries (at most: 16 per entry, 8 for Im(amplitude), 16 for mask and match)
inline uint32_t win_entries_bytes(int n_lin, int n_chunk, int n_rest) {
  return (uint32_t)(((n_lin + 63) / 64) * n_chunk) * 128u + (uint32_t)(n_lin + n_rest + 1) * 24u +
         (uint32_t)n_rest * 16u;
}
// LDS bytes below the entries (WinLds, at most)
inline uint32_t win_fixed_bytes(int kind, int Lx) {
  return (2u << win_index_bits(kind, Lx)) + 64u * 16u + kXCodesBytesMax + 2u * 4096u;
}

// The same with point operations of an L x L torus, phases by candidate code
// and the flips' transposes included
inline uint32_t win_point_bytes(int L, int n_lin, int n_chunk, int n_rest) {
  return 2u * ((2u << (2 * L)) + (kPointClasses << L) + kPointClasses) + 512u * 16u + kXCodesBytesMax + 2u * 4096u + win_entries_bytes(n_lin, n_chunk, n_rest) +
         8u * (uint32_t)(n_lin + n_rest + 1);
}

enum Prec : int { kF64 = 0, kC128 = 1, kF32 = 2, kC64 = 3 };

// y = (accumulate ? y : 0) + A x   (transpose=0: row form; 1: column form, y = x A)
hipError_t launch_matvec(const OpDev& op, int prec, int transpose, int accumulate, const void* x, void* y,
                         hipStream_t st);

// the same for one vector type (product_*.hip)
hipError_t launch_product_f32(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st);
hipError_t launch_product_f64(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st);
hipError_t launch_product_c64(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st);
hipError_t launch_product_c128(const OpDev& op, int transpose, int accumulate, const void* x, void* y, hipStream_t st);

// The same on a shape of window.hpp, x spread (P.values); Ly = 0: no group, x
// spread or ranked.
hipError_t launch_window_product(const WinOp& P, int Lx, int Ly, int unit, int prec, int transpose, const void* x,
                                 void* y, hipStream_t st);
hipError_t launch_window_product_f32(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                                    hipStream_t st);
hipError_t launch_window_product_f64(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                                    hipStream_t st);
hipError_t launch_window_product_c64(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                                    hipStream_t st);
hipError_t launch_window_product_c128(const WinOp& P, int Lx, int Ly, int unit, int transpose, const void* x, void* y,
                                    hipStream_t st);

// ---- assembled rows (row form): entries col | cls << col_bits per image ----
constexpr int kAsmMaxClasses = 256;
constexpr int kAsmBlock = 512;  // lanes per block of the assembled product
struct AsmFillDev {
  const uint64_t* rowptr;  // dim + 1 offsets of the rows' entries
  uint32_t* ent;
  const uint32_t* acls;    // per product entry: amplitude class, 1-based
  const uint32_t* pcls;    // per group element: phase class (nullptr: every phase 1)
  int n_ph;
  int col_bits;
};
struct AsmDev {
  const uint64_t* rowptr;
  const uint32_t* ent;
  const double* w_re;      // n_cls weights, class 0 = 0
  const double* w_im;
  int n_cls;
  int col_bits;
};
// counts[r] = entries of row r (terms matching it)
hipError_t launch_asm_count(const OpDev& op, uint32_t* d_counts, hipStream_t st);
hipError_t launch_asm_fill(const OpDev& op, const AsmFillDev& a, hipStream_t st);
// the same on a square torus with point operations (Win<kWinPoint>), the images
// ranked by position
hipError_t launch_asm_fill_point(const OpDev& op, const AsmFillDev& a, const XMapDev& X, const RankBits* pos_bits,
                                 uint32_t none, hipStream_t st);
// xt = x sqrt(G / orbit) (orbit != nullptr), in precision prec; xt[dim] = 0
hipError_t launch_asm_scale(int prec, int64_t dim, const uint16_t* d_orbit, int G, const void* x, void* xt,
                            hipStream_t st);
// y = (accumulate ? y : 0) + A x from the entries; xt = x scaled as above (x itself without orbits);
// lanes = lanes per row (4, 8, 16 or 32), batch = entries per lane loaded together (4, 8 or 16)
hipError_t launch_asm_spmv(const OpDev& op, const AsmDev& a, int prec, int lanes, int batch, int accumulate,
                           const void* x, const void* xt, void* y, hipStream_t st);

// Diagonal element of every row: re[r] (+ i im[r] when im != nullptr) = sum of
// the amplitudes of the diagonal terms that match row r.
hipError_t launch_diag_values(const OpDev& op, double* d_re, double* d_im, hipStream_t st);

// The same for real amplitudes by parities (DiagSplit): the coefficient of every
// set of entries (mask within its segment) times the number of them whose parity
// is even less that of those whose is odd, and the terms left (rest).
struct DiagParity {
  const uint64_t* tab;   // as OpDev::lin_tab, n_seg segments of n_chunk chunks
  const DiagSet* sets;   // by segment
  const int32_t* first;  // n_seg + 1 offsets into sets
  const DiagTerm* rest;
  int n_seg, n_chunk, n_rest;
  bool carried;
};
hipError_t launch_diag_parity(const DiagParity& P, const uint64_t* d_rows, int64_t dim, double* d_re, hipStream_t st);

// Total number of off-diagonal images the row form generates (atomic u64 add).
hipError_t launch_count_images(const OpDev& op, unsigned long long* d_total, hipStream_t st);

// Raw iterator elements (index or -1, value) in term order for the given rows.
hipError_t launch_iterate(const OpDev& op, const OffTerm* all_terms, int n_all, int transpose, int64_t n_rows,
                          const int64_t* d_rows, int64_t* d_idx, double* d_re, double* d_im, hipStream_t st);

// Merged, chopped, ascending entries of rows (row form, transpose = 0) or
// columns (column form, transpose = 1): entry k is vector d_sel[k] (k itself
// when d_sel is null), up to slot entries each, d_count[k] kept.
hipError_t launch_sparse_columns(const OpDev& op, int transpose, double tol, int slot, int64_t n_sel,
                                 const int64_t* d_sel, int64_t* d_scratch_idx, double* d_scratch_re,
                                 double* d_scratch_im, int64_t* d_count, hipStream_t st);
// Dense column-major matrix (column form operator) added into a cleared
// dim x dim buffer of doubles (complex_out: interleaved re, im pairs).
hipError_t launch_dense_columns(const OpDev& op, int complex_out, double* d_out, hipStream_t st);
// For the host: colptr then rowval in 4 bytes (idx32, where given), the values
// interleaved (cplx, where given).
hipError_t launch_sparse_pack(int64_t dim, int64_t nnz, const int64_t* d_colptr, const int64_t* d_rowval,
                              const double* d_re, const double* d_im, int32_t* d_idx32, double* d_cplx, hipStream_t st);
hipError_t launch_sparse_compact(int64_t dim, int slot, const int64_t* d_colptr, const int64_t* d_scratch_idx,
                                 const double* d_scratch_re, const double* d_scratch_im, int64_t* d_rowval,
                                 double* d_re, double* d_im, hipStream_t st);

// Per-term bilinear forms g_t = sum_r conj(phi_r) sum_{images of t} w psi_s,
// deterministic two-stage reduction.  n_terms = n_diag + n_off.
hipError_t launch_term_expect(const OpDev& op, int prec, const void* phi, const void* psi, double* d_partial,
                              int64_t n_blocks, double* d_out, hipStream_t st);
int64_t term_expect_blocks(const OpDev& op);
// rows of n_terms * 2 doubles the kernel needs in d_partial (per-block sums
// and the reduction's chunk sums); terms per pass for vectors of nc real
// components (0: the tables leave no LDS room)
int64_t term_expect_scratch_rows(const OpDev& op);

// The same on sectors that are ranked by two tables (expect.hip).  A step is one
// off-diagonal term, or two that share mask and flip (term[1] < 0: one; a match of
// all ones never occurs).
struct ExpectStep {
  uint32_t mask, match[2], flip;
  int32_t term[2];
};
struct ExpectRank {
  const uint64_t* rows;
  const uint16_t* rank_low;   // as in WinOp
  const uint32_t* rank_base;
  const ExpectStep* steps;    // whole windows
  // upper and lower parts by popcount: lists and their offsets; items: pairs
  // (popcount, first) of every 64 lower parts
  const int32_t *up_list, *up_off, *lo_list, *lo_off, *items;
  uint32_t base_bytes;
  int low_bits, upper_bits, n_upper, pop, n_off, n_steps, n_items;
};
constexpr int kExpectWindow = 6;  // steps per window (real vectors; half of it for complex ones)
constexpr int kExpectSplits = 16;
// Blocks of the steps' kernel per window, each with a row of 2 n_off partial sums:
// all windows together three blocks per CU, which the chip holds at once (4x6 XXZ,
// 8 windows: 110 us with 96 blocks, 124 with 64, 122 with 128, 140 with 384).
inline int64_t expect_rank_blocks(int64_t dim, int windows) {
  const int64_t n = (dim + 511) / 512, most = windows > 24 ? 32 : 768 / (windows < 1 ? 1 : windows);
  return n < 1 ? 1 : n > most ? most : n;
}
// X: n_upper (1 + 2 low_bits) sums, Q: kExpectSplits 2^low_bits, each 2 doubles;
// d_partial: expect_rank_blocks and their chunks (blocks / 64, rounded up) of 2 n_off doubles
hipError_t launch_term_expect_rank(const ExpectRank& E, const OpDev& op, int prec, const void* phi, const void* psi,
                                   double* X, double* Q, double* d_partial, double* d_out, hipStream_t st);
// sums of the rows of d_partial (n_blocks x width), in a fixed order, by way of
// the chunk sums behind them
hipError_t launch_expect_reduce(double* d_partial, int64_t n_blocks, int width, double* d_out, hipStream_t st);

// Fixed device scratch of the allocation-free term pass (one array per GPU,
// held until the process ends): room for the per-block partial sums and the
// result of at most kNoAllocMaxTerms terms.  term_expect_noalloc_setup runs
// once per device with that device current (the context's creation) and
// keeps the device address of the array; term_expect_noalloc_scratch returns
// it (nullptr before the setup).
constexpr int kNoAllocMaxTerms = 512;
hipError_t term_expect_noalloc_setup(int device);
double* term_expect_noalloc_scratch(int device);
size_t term_expect_noalloc_doubles();
int term_expect_window(const OpDev& op, int nc);

// ---- fast path: bond-pair term groups + register canonicaliser + hash lookup
// Terms grouped by bit mask (1 or 2 bits).  For a row b the group's pattern
// code = b[p] | b[q] << 1 (q = p for one-bit masks) selects the summed
// diagonal amplitude and at most one off-diagonal entry (new pattern code +
// amplitude).  meta[g] = p | q << 8 | offmask << 16 | newcode(4 x 2 bits) << 24.
struct PairGroupsDev {
  int n_groups;
  int pad_;
  const uint32_t* meta;
  const double* dre;  // 4 per group
  const double* dim;
  const double* ore;  // 4 per group
  const double* oim;
  double dconst_re, dconst_im;  // identity terms (empty mask)
};

struct FastOpDev {
  OpDev base;  // index, group, layout, rows, orbit, dim, rank table offsets (off terms unused)
  PairGroupsDev pg;
  HashDev hash;      // slots == nullptr: lookup through base.ix, x gathered separately
  uint32_t pg_lds;   // LDS offset of the staged groups
  uint32_t lds_total;
};

constexpr int kMaxPairGroups = 256;

hipError_t launch_matvec_pairs(const FastOpDev& op, int prec, int transpose, int accumulate, const void* x, void* y,
                               hipStream_t st);
hipError_t launch_hash_build(const uint64_t* d_keys, int64_t dim, const HashDev& h, uint32_t* d_slot_of,
                             hipStream_t st);
hipError_t launch_hash_scatter(int prec, int64_t dim, const void* x, const uint32_t* d_slot_of, const HashDev& h,
                               hipStream_t st);

// ---- vecops.hip ------------------------------------------------------------
// All reductions accumulate in double and are deterministic (fixed tree).
hipError_t vec_dot(int prec, int64_t n, const void* x, const void* y, double* d_partial, double* d_out2,
                   hipStream_t st);  // <x, y> (conjugated x), d_out2 = {re, im}
hipError_t vec_multi_dot(int prec, int64_t n, int k, const void* V, int64_t ldv, const void* w, double* d_partial,
                         double* d_out, hipStream_t st);  // d_out[2j..] = <V_j, w>
hipError_t vec_multi_axpy(int prec, int64_t n, int k, const void* V, int64_t ldv, const double* d_coef, void* w,
                          hipStream_t st);  // w -= sum_j coef_j V_j (complex coef)
hipError_t vec_axpby(int prec, int64_t n, double ar, double ai, const void* x, double br, double bi, void* y,
                     hipStream_t st);  // y = a x + b y
hipError_t vec_convert(int prec_in, int prec_out, int64_t n, const void* x, void* y, hipStream_t st);
hipError_t vec_gaussian(int prec, int64_t n, uint64_t seed, void* x, hipStream_t st);
hipError_t vec_fill_zero(int prec, int64_t n, void* x, hipStream_t st);
// out_l = sum_j coef[j*k + l] V_j for l < k (real coefficients, double accumulation)
hipError_t vec_combine(int prec_v, int prec_out, int64_t n, int m, const void* V, int64_t ldv, int k,
                       const double* d_coef, void* out, int64_t ldo, hipStream_t st);
int64_t vec_partial_blocks(int64_t n);

}  // namespace edhip
