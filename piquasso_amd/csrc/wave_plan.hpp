// A wave's own plan of one Glynn sweep, from the row multiplicities in its
// lanes (lane i: row i): the min-row prepend of src/permanent.cpp:54-95 and
// the split of the digits.  The lowest binary digits (rows of multiplicity
// 1) are inner: swept by all lanes in Gray order, at most kMaxInnerDigits of
// them.  The others, and the digits of larger radix, are the lane's, read
// off its index in row order (no Gray order is needed between lanes, since
// each starts from its own row sums).
#pragma once

#include <cstdint>

#include "sweep_common.hpp"

namespace pqp {

namespace {

constexpr int kMaxInnerDigits = 7;

template <typename I>  // the type of a top state's index
struct WavePlanOf {
  int rho;           // this lane's digit: its row's multiplicity, less the prepended one
  int i0;            // the prepended row
  uint64_t rows;     // rows that are digits
  uint64_t bin;      // binary digits that are not inner
  uint64_t inner;    // the inner rows, a byte each
  int k;             // inner digits
  I U;               // top states
};
using WavePlan = WavePlanOf<int>;

// occ: the lane's row multiplicity (n >= 1 in all).  At least `lanes` top
// states are kept where the digits allow it, at most k_max inner digits.
template <typename I = int>
__device__ __forceinline__ WavePlanOf<I> wave_plan(int occ, int n, int lanes, int k_max) {
  WavePlanOf<I> p;
  p.i0 = 0;
  for (int v = 1; v <= n; ++v) {
    const uint64_t at = __ballot(occ == v);
    if (at) {
      p.i0 = __builtin_ctzll(at);
      break;
    }
  }
  p.rho = occ - (lane_id() == p.i0 ? 1 : 0);
  p.bin = __ballot(p.rho == 1);
  const uint64_t multi = __ballot(p.rho > 1);
  p.rows = p.bin | multi;
  I states = 1;  // of the digits of larger radix
  for (uint64_t m = multi; m; m &= m - 1)
    states *= __builtin_amdgcn_readlane(p.rho, __builtin_ctzll(m)) + 1;
  const int nb = __builtin_popcountll(p.bin);
  p.k = 0;
  while (p.k < k_max && p.k < nb && ((states << (nb - p.k - 1)) >= lanes)) ++p.k;
  p.inner = 0;
  for (int q = 0; q < p.k; ++q) {
    p.inner |= static_cast<uint64_t>(__builtin_ctzll(p.bin)) << (8 * q);
    p.bin &= p.bin - 1;
  }
  p.U = states << (nb - p.k);
  return p;
}

// The row sums of top state u with the inner digits at 0, from rows of
// values `stride` doubles apart (W complex ones, or W doubles into cr alone
// when REAL), and its signed weight.  They start from row r0: the prepended
// row, or a copy of it.
template <int W, bool REAL = false, typename I>
__device__ __forceinline__ double wave_start(const WavePlanOf<I> &p, I u, cptr<double> rows, int stride,
                                             int r0, double (&cr)[W], double (&ci)[W]) {
  {
    // an opaque index: the row is the same for every chunk of top states,
    // and hoisting it would hold a second set of row sums in registers
    __asm__ volatile("" : "+s"(r0));
    const cptr<double> b = rows + r0 * stride;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      cr[j] = b[REAL ? j : 2 * j];
      if constexpr (!REAL) ci[j] = b[2 * j + 1];
    }
  }
  I rest = u;
  int parity = 0;
  double w = 1.0;
  for (uint64_t m = p.rows; m; m &= m - 1) {  // one loop for all digits: one block of row sums
    const int r = __builtin_ctzll(m);
    const int rr = __builtin_amdgcn_readlane(p.rho, r);
    double al = in_vgpr(1.0);  // inner digits start at 0
    if (rr > 1) {
      // u < 2^50: the quotient by a small radix is exact this way
      const I q = static_cast<I>((static_cast<double>(rest) + 0.5) * (1.0 / (rr + 1)));
      const int g = static_cast<int>(rest - q * (rr + 1));
      rest = q;
      parity ^= g & 1;
      w *= lane_binomial(rr, g);
      al = static_cast<double>(rr - 2 * g);
    } else if ((p.bin >> r) & 1) {
      al = (rest & 1) ? -1.0 : 1.0;
      parity ^= static_cast<int>(rest & 1);
      rest >>= 1;
    }
    const cptr<double> b = rows + r * stride;
#pragma unroll
    for (int j = 0; j < W; ++j) {
      cr[j] = fmaR(al, b[REAL ? j : 2 * j], cr[j]);
      if constexpr (!REAL) ci[j] = fmaR(al, b[2 * j + 1], ci[j]);
    }
  }
  return parity ? -w : w;
}

// The inner row that moves after inner state v (Gray order) and its factor
// +-2; after the last state (digit k) row 0, for an update that is not read.
template <typename I>
__device__ __forceinline__ int wave_step_row(const WavePlanOf<I> &p, int v) {
  return static_cast<int>((p.inner >> (8 * __builtin_ctz(v + 1))) & 255);
}
__device__ __forceinline__ double wave_step_factor(int v) {
  const int up = (v + 1) ^ ((v + 1) >> 1);
  return ((up >> __builtin_ctz(v + 1)) & 1) ? -2.0 : 2.0;
}

}  // namespace

}  // namespace pqp
