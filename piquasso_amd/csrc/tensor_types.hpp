// Kernel arguments of tensor permanents (uniformly partially distinguishable
// bosons), shared by capi.cpp and the kernels in tensor_perm.hip.
//
// T(A, x) = 4^-(n-1) sum over sign vectors delta, eps in {+1,-1}^n with
//           delta_0 = eps_0 = +1 of (prod delta)(prod eps)
//           prod_i ( x R_delta[i] conj(R_eps[i]) + (1 - x) Q_{delta eps}[i] ),
// the value piquasso sums over column subsets
// (piquasso/_simulators/passive/probabilities.py:193-237).
//
// Work split: sign vector delta is s (bit b set: delta_{b+1} = -1), one per
// lane, s = (s_hi << ls) | lane; a wave walks eps = t = (t_blk << kt) |
// gray(k), k = 0 .. 2^kt - 1, flipping one sign per step.  Term (t, s) is
// the conjugate of term (s, t), so only Re is summed, with weight 2 when
// t's lane block (t >> ls) is above s_hi, 1 when it is s_hi, and pairs
// below are not visited.  All items of a launch have the same order n,
// hence the same work units.
#pragma once

#include <cstdint>

namespace pqp {

constexpr int kTensorMaxN = 20;  // widest matrix the kernels are built for

struct TensorUnit {
  int32_t s_hi;       // s = (s_hi << ls) | lane
  int32_t t_blk;      // t = (t_blk << kt) | gray(k)
  int32_t mixed;      // 1: some steps have t >> ls <= s_hi (weight per step)
};

struct TensorArgs {
  const TensorUnit *units;  // n_units, by t_blk: neighbours walk the same eps
  const double *x;          // particle overlap per item
  double *cols;       // per item: n x n complex, column-major [c][i] (re, im)
  double *pw;         // per item: n x n real, (1 - x) |A[i, c]|^2 at [c][i]
  double *signs;      // per item: R_eps of every t: 2^(n-1) x n complex
  double *partials;   // per item and unit, 3 doubles: dd sum (hi, lo), sum of |terms|
  double *out;        // 2 doubles per item: T, sum over pairs of weight x |Re term|
  int32_t n, ls, kt;
  int32_t n_units, n_items;
  // tables: the interferometer's columns of the input particles (modes x n
  // complex) and each item's rows of them; prob[item] = T / norm[item]
  const double *u;
  const uint16_t *rows;  // n per item
  const double *norm;
  double *prob;          // null: no table
};

// The sign rows of items of several orders, one launch.
struct TensorSigns {
  struct Order {
    const double *cols;
    double *signs;
    int32_t n;
    uint32_t first, per_item;  // its first block, and blocks of an item
  } orders[kTensorMaxN];
  int32_t n_orders;
};

}  // namespace pqp
