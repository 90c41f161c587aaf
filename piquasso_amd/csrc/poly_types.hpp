// Device-side layout of one matrix-polynomial permanent problem
// (perm_poly.hip): coefficients [x^e] perm(B_0 + sum_m x_m B_m) by Ryser's
// formula over the column subsets, with each subset's polynomial kept on a
// downward-closed set of monomials stored level by level (total degree
// 0, 1, ..., L).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pqp {

constexpr int kPolyMaxN = 24;         // 2^24 - 1 column subsets at most
constexpr int kPolyMaxVars = 255;     // variable index in the low 8 bits of a link
constexpr int kPolyMaxMono = 1 << 23; // monomial index in the upper 23 bits of a link
constexpr int kPolyThreads = 256;          // polynomial in LDS
constexpr int kPolyThreadsGlobal = 1024;   // polynomial in global memory
constexpr int kPolyGroup = 2;              // subsets interleaved per workgroup (global memory)

struct PolyArgs {
  const double2 *b0;       // n x n, row-major
  const double2 *bm;       // M matrices n x n, one after another
  const int32_t *link_ptr; // n_mono + 1: links of monomial a are [link_ptr[a], link_ptr[a + 1])
  const int32_t *links;    // (index of a - e_m) << 8 | m, for every m with a_m > 0
  const int32_t *lvl_off;  // L + 2: monomials of total degree D are [lvl_off[D], lvl_off[D + 1])
  const int32_t *out_mono; // n_out: monomial of each requested coefficient
  double2 *scratch;        // global-memory polynomials, n_mono x group per workgroup (when not in LDS)
  double2 *acc;            // n_wg x n_out: each workgroup's signed subset sum
  double *out;             // 2 per requested coefficient
  int32_t n, M, L, n_mono, n_out, n_wg;
};

// The layer path (perm_poly.hip): rows 0..i-1 expanded over the column
// subsets S of i columns, f_i[e][S] = [x^e] of the sum over the ways to
// match those rows with S.
constexpr int kPolyLayerMaxN = 12;         // C(12, 6) = 924 subsets in the widest layer
constexpr int kPolyLayerThreads = 256;
constexpr int kPolyLayerLds = 40960;       // bytes of products a layer block keeps (four blocks per CU)
constexpr int kPolyMissFactor = 2;         // multiply only the missing columns from 2 (n - i) <= n on
constexpr int kPolyLayerAcc = 4;           // subsets per thread: ceil(924 / 256)

struct PolyLayerArgs {
  const double2 *b0, *bm;  // as in PolyArgs
  const int32_t *link_ptr, *links, *out_mono;
  const int16_t *sub;      // n_dst x n: place of S without column j in the source layer, -1 if j is not in S
  const uint16_t *src_bits, *dst_bits;  // each subset's columns
  const double2 *src;      // n_src_mono x n_src (null: the empty product 1)
  double2 *dst;            // n_dst_mono x n_dst
  double *out;             // last row: 2 per requested coefficient
  int32_t n, M, row;
  int32_t n_src, n_dst;            // subsets of `row` and of row + 1 columns
  int32_t n_src_mono, n_dst_mono;  // monomials of degree <= row and <= row + 1 (and <= L)
  int32_t n_out;
};

}  // namespace pqp
