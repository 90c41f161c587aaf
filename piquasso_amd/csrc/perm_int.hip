// Exact permanents of integer matrices on gfx950: the Glynn sweep
// (src/permanent.cpp:49-264, planned by the waves: wave_plan.hpp) with every
// product and sum taken modulo K <= 8 primes just below 2^49; the host
// recovers the integer from the residues by the Chinese remainder theorem.
//
// Row sums of an integer matrix are exact integers in FP64 (the host checks
// that they stay below 2^48), so the row updates are the ordinary ones, on
// real rows (columns of multiplicity c are laid out as c unit columns, the
// width padded to a multiple of 4, above 32 of 8, with columns that stay 1).  The product
// prod_j cs_j is formed in groups of G columns exactly in FP64 (the host
// picks the largest G with every group product below 2^49), and the group
// products are multiplied modulo each prime with a floating-point modular
// multiply:
//
//   h = x y, l = fma(x, y, -h)        (x y = h + l exactly)
//   q = rint(h * (1/p)), r = fma(-q, p, h) + l,
//
// exact for |x|, |y| <= 2p < 2^50: |h - q p| <= 1.5 p is an integer below
// 2^53 (the fma rounds nothing), |l| <= 2^46, so |r| <= 1.75 p stays a
// valid input.  Sums are reduced by r = fma(-rint(s / p), p, s) (exact for
// integers |s| < 2^53): every fourth term, |s| <= 7.5 p then.  The inner
// digits are binary, so a term's coefficient is its sign; each lane's sum is
// multiplied by its top weight, the wave reduces the residues with a
// butterfly, and the sum kernel adds the waves' residues, multiplies by
// 2^-(n-1) mod p and normalises to [0, p).
//
// Bound by FP64 issue in large sweeps.  Per term 2 W - NG operations and
// 6 (NG - 1) + 2 per prime, NG = ceil(W / G): wide groups take out most of
// the modular products (a 0/1 matrix of 24 columns has row sums below 16:
// G = 12 leaves one product per prime where G = 4 has five).  4096 waves (as
// 2048: the start of a wave costs a third of its 32 states, but twice the
// states leave half the waves to hide latency).  Measured, 0/1 matrices of
// density 0.3, two primes, a call and its sweep: n = 24 151 us (87) -> 65 us
// (38); n = 12 58 -> 30 us, copies, planning and two synchronisations gone.

#include <hip/hip_runtime.h>

#include <cstdint>

#include "int_types.hpp"
#include "perm_kernels.hpp"
#include "sweep_common.hpp"
#include "wave_plan.hpp"

namespace pqp {

namespace {

__device__ __forceinline__ double reduce_mod(double x, double p, double pinv) {
  const double q = __builtin_rint(x * pinv);
  return __builtin_fma(-q, p, x);
}

__device__ __forceinline__ double mul_mod(double x, double y, double p, double pinv) {
  const double h = x * y;
  const double l = __builtin_fma(x, y, -h);
  const double q = __builtin_rint(h * pinv);
  return __builtin_fma(-q, p, h) + l;
}

// Product of cs[LO .. HI) as a balanced tree (exact whatever the order; a
// chain of G multiplies would set the pace of a term).
template <int LO, int HI, int W>
__device__ __forceinline__ double group_product(const double (&cs)[W]) {
  if constexpr (HI - LO == 1) {
    return cs[LO];
  } else {
    constexpr int mid = LO + (HI - LO + 1) / 2;
    return group_product<LO, mid>(cs) * group_product<mid, HI>(cs);
  }
}

template <int G, int W, int NG, int g = 0>
__device__ __forceinline__ void group_products(const double (&cs)[W], double (&gp)[NG]) {
  if constexpr (g < NG) {
    gp[g] = group_product<g * G, (g + 1) * G < W ? (g + 1) * G : W>(cs);
    group_products<G, W, NG, g + 1>(cs, gp);
  }
}

// Sum of the lanes' residues (|r| <= p / 2), reduced at every step.
template <int STEP = 0>
__device__ __forceinline__ double wave_sum_mod(double r, double p, double pinv, int lane) {
  if constexpr (STEP < 6) {
    return wave_sum_mod<STEP + 1>(reduce_mod(r + wave_partner<STEP>(r, lane), p, pinv), p, pinv, lane);
  } else {
    return r;
  }
}

// One wave per block: top states 64 (wave + t waves).  K = 0: a.n_primes of
// them, else exactly K (their constants then stay in scalar registers and
// their chains interleave).
template <int W, int G, int K>
__global__ __launch_bounds__(kWave) void perm_int_kernel(IntArgs a) {
  constexpr int kMax = K ? K : kIntMaxPrimes;
  constexpr int NG = (W + G - 1) / G;
  const int lane = static_cast<int>(threadIdx.x);
  const int wave = static_cast<int>(blockIdx.x);
  const int occ = lane < a.modes ? a.occ[lane] : 0;
  const WavePlanOf<int64_t> p = wave_plan<int64_t>(occ, a.n, kWave, a.k_max);
  const int S = 1 << p.k;
  const cptr<double> rows = as_const<double>(a.rows);
  double mod[kMax], inv[kMax];
#pragma unroll
  for (int k = 0; k < kMax; ++k) {
    mod[k] = as_const<double>(a.mod)[k];
    inv[k] = as_const<double>(a.mod)[kIntMaxPrimes + k];
  }
  double total[kMax];
#pragma unroll
  for (int k = 0; k < kMax; ++k) total[k] = 0.0;
  for (int64_t u0 = static_cast<int64_t>(wave) * kWave; u0 < p.U; u0 += static_cast<int64_t>(a.waves) * kWave) {
    const bool active = u0 + lane < p.U;
    double cs[W], none[W];
    // row a.modes: the prepended row with 1 in the padding columns
    const double w_top = wave_start<W, true>(p, active ? u0 + lane : 0, rows, W, a.modes, cs, none);
    const double w = active ? w_top : 0.0;
    double acc[kMax];
#pragma unroll
    for (int k = 0; k < kMax; ++k) acc[k] = 0.0;
    for (int v = 0; v < S; ++v) {
      const cptr<double> row = rows + wave_step_row(p, v) * W;
      // exact group products (|product| <= 2^49); the first carries the sign
      double gp[NG];
      group_products<G>(cs, gp);
      gp[0] = (v & 1) ? -gp[0] : gp[0];
      const bool fold = (v & 3) == 3 || v == S - 1;
#pragma unroll
      for (int k = 0; k < kMax; ++k) {
        if (K || k < a.n_primes) {
          double x = gp[0];
#pragma unroll
          for (int g = 1; g < NG; ++g) x = mul_mod(x, gp[g], mod[k], inv[k]);
          acc[k] += x;
          if (fold) acc[k] = reduce_mod(acc[k], mod[k], inv[k]);
        }
      }
      const double s2 = in_vgpr(wave_step_factor(v));
#pragma unroll
      for (int j = 0; j < W; ++j) cs[j] = __builtin_fma(s2, row[j], cs[j]);
    }
#pragma unroll
    for (int k = 0; k < kMax; ++k)
      if (K || k < a.n_primes)
        total[k] = reduce_mod(total[k] + mul_mod(acc[k], reduce_mod(w, mod[k], inv[k]), mod[k], inv[k]),
                              mod[k], inv[k]);
  }
#pragma unroll
  for (int k = 0; k < kMax; ++k) {
    if (K || k < a.n_primes) {
      const double r = wave_sum_mod(total[k], mod[k], inv[k], lane);
      if (lane == 0) a.partials[static_cast<int64_t>(k) * a.waves + wave] = r;
    }
  }
}

// One block, a wave per prime: the waves' residues added (modular sums are
// exact, so the order does not matter), times 2^-(n-1) mod p, in [0, p); then
// the sequence number the host polls for.
__global__ __launch_bounds__(kIntMaxPrimes * kWave) void perm_int_sum_kernel(IntArgs a) {
  const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
  const int k = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  if (k < a.n_primes) {
    const cptr<double> mod = as_const<double>(a.mod);
    const double p = mod[k], pinv = mod[kIntMaxPrimes + k], inv2 = mod[2 * kIntMaxPrimes + k];
    double s = 0.0;
    const double *part = a.partials + static_cast<int64_t>(k) * a.waves;
    int u = lane;
    for (; u + 7 * kWave < a.waves; u += 8 * kWave) {  // eight loads in flight; |sum| <= 4.5 p
      double t[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) t[q] = part[u + q * kWave];
      s = reduce_mod(s + (((t[0] + t[1]) + (t[2] + t[3])) + ((t[4] + t[5]) + (t[6] + t[7]))), p, pinv);
    }
    for (; u < a.waves; u += kWave) s = reduce_mod(s + part[u], p, pinv);
    s = wave_sum_mod(s, p, pinv, lane);
    if (lane == 0) {
      double r = reduce_mod(mul_mod(s, inv2, p, pinv), p, pinv);
      if (r < 0.0) r += p;
      a.out[k] = r;
      __threadfence_system();
    }
  }
  __syncthreads();
  if (threadIdx.x == 0) __hip_atomic_store(a.done, a.seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int W, int G>
static void int_launch(const IntArgs &a, hipStream_t stream) {
#define PQP_INT_K(K) \
  hipLaunchKernelGGL((perm_int_kernel<W, G, K>), dim3(a.waves), dim3(kWave), 0, stream, a)
  if constexpr (W <= 32 && G >= 4) {
    switch (a.n_primes) {
      case 1: PQP_INT_K(1); return;
      case 2: PQP_INT_K(2); return;
      case 3: PQP_INT_K(3); return;
      case 4: PQP_INT_K(4); return;
      default: break;
    }
  }
  PQP_INT_K(0);
#undef PQP_INT_K
}

}  // namespace

// Compiled once per padded width (-DPQP_INT_WIDTH=4, 8, .. 32, 40, .. 64);
// the sum kernel with 8.
#ifndef PQP_INT_WIDTH
#error "compile with -DPQP_INT_WIDTH=<4, 8, .. 32, 40, .. 64>"
#endif
#define PQP_PASTE_(base, w) base##w
#define PQP_PASTE(base, w) PQP_PASTE_(base, w)

hipError_t PQP_PASTE(launch_int_w, PQP_INT_WIDTH)(const IntArgs &a, hipStream_t stream) {
  switch (a.group) {
    case 12: int_launch<PQP_INT_WIDTH, 12>(a, stream); break;
    case 8: int_launch<PQP_INT_WIDTH, 8>(a, stream); break;
    case 4: int_launch<PQP_INT_WIDTH, 4>(a, stream); break;
    case 2: int_launch<PQP_INT_WIDTH, 2>(a, stream); break;
    default: int_launch<PQP_INT_WIDTH, 1>(a, stream); break;
  }
  return hipGetLastError();
}

#if PQP_INT_WIDTH == 8
hipError_t launch_int_sum(const IntArgs &a, hipStream_t stream) {
  hipLaunchKernelGGL(perm_int_sum_kernel, dim3(1), dim3(kIntMaxPrimes * kWave), 0, stream, a);
  return hipGetLastError();
}
#endif

}  // namespace pqp
