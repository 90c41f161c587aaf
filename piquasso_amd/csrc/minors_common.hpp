// Device code shared by the column-minor kernels (perm_minors.hip,
// perm_minors_wave.hip).
#pragma once

#include "sweep_common.hpp"

namespace pqp {

namespace {

// Waves per SIMD the register budget is sized for: unit-multiplicity
// kernels keep m_c row sums, m_c - 1 prefix products and m_c + 1
// accumulators (about 12 m_c VGPRs); the general kernels also recompute
// column powers.
constexpr int minor_waves(int hi, bool ones) {
  return hi <= 8 ? 4 : (ones && hi <= 20) ? 2 : 1;
}

// One term of every column minor, columns of multiplicity 1: acc[l] += cf *
// prod_{k != l} cs_k, and where there are M = MCP + 1 accumulators acc[MCP]
// += cf * prod_k cs_k (the uncut product).
template <int MCP, int M>
__device__ __forceinline__ void minor_products(const double (&cr)[MCP], const double (&ci)[MCP], double cf,
                                               double (&acr)[M], double (&aci)[M]) {
  using R = double;
  // unit multiplicities: E_k = cs_k, F_k = 1.  Prefix products
  // P_k = prod_{k' < k} cs_k' are kept for even k only (P_0 = 1); an odd
  // P_{2m+1} = P_{2m} cs_{2m} is rebuilt in the backward pass, which
  // carries the running suffix Q: minor l = P_l Q_l, and the final Q is
  // the uncut product.  (Half the prefix registers for m_c / 2 extra
  // multiplies keeps the kernel within one register budget step.)
  constexpr int NP = (MCP + 1) / 2;  // P_0, P_2, ..., P_{2(NP-1)}
  R pr[NP], pi[NP];
  pr[0] = R(1);
  pi[0] = R(0);
  if constexpr (NP > 1) {
    pr[1] = cr[0];
    pi[1] = ci[0];
    cmul(pr[1], pi[1], cr[1], ci[1]);
#pragma unroll
    for (int m = 2; m < NP; ++m) {
      pr[m] = pr[m - 1];
      pi[m] = pi[m - 1];
      cmul(pr[m], pi[m], cr[2 * m - 2], ci[2 * m - 2]);
      cmul(pr[m], pi[m], cr[2 * m - 1], ci[2 * m - 1]);
    }
  }
  R qr = R(1), qi = R(0);
#pragma unroll
  for (int k = MCP - 1; k >= 0; --k) {
    R mr, mi;
    if (k % 2 == 0) {
      mr = pr[k / 2];
      mi = pi[k / 2];
    } else {
      mr = pr[k / 2];
      mi = pi[k / 2];
      if (k > 1) {
        cmul(mr, mi, cr[k - 1], ci[k - 1]);
      } else {
        mr = cr[0];
        mi = ci[0];
      }
    }
    if (k < MCP - 1) {
      if (k == 0) {
        mr = qr;
        mi = qi;
      } else {
        cmul(mr, mi, qr, qi);
      }
    }
    acr[k] = __builtin_fma(cf, mr, acr[k]);
    aci[k] = __builtin_fma(cf, mi, aci[k]);
    if (k == MCP - 1) {
      qr = cr[k];
      qi = ci[k];
    } else {
      cmul(qr, qi, cr[k], ci[k]);
    }
  }
  if constexpr (M > MCP) {
    acr[MCP] = __builtin_fma(cf, qr, acr[MCP]);
    aci[MCP] = __builtin_fma(cf, qi, aci[MCP]);
  }
}

}  // namespace

}  // namespace pqp
