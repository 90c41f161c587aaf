// Probability tables on gfx950: the amplitudes
//
//   <t| U |s> = perm(U; rows = t, cols = s) / sqrt(prod t! prod s!)
//
// (or their squared moduli) of many output occupations t for one
// interferometer U and input s (piquasso/_simulators/passive/
// probabilities.py:26-54, one permanent after another there), n <= 16
// particles.  Such permanents are small (at most 2^(n-1) Gray terms), and
// planning each on the host costs far more than its sum: 1.4 us against
// 2 ns for 7 particles.  So the kernel gets the occupations, a byte per
// mode, and every wave plans its own item (wave_plan.hpp).  U's occupied
// columns (at most 16 KB for every item alike) are read with scalar loads,
// a row at a time, so no table is built or loaded per item.
//
// Sums as in perm_fwd.hip: FP64 row sums and products, FP64 runs of at most
// 64 terms folded into double-double, the lanes' and waves' sums added in
// double-double in a fixed order, exact integer weights.
//
// Bound by the per-item work of one wave (the plan, D row updates, a product
// or a few, the double-double reduction), eight waves per SIMD hiding each
// other's latency: 77 520 outputs of 7 particles in 14 modes take 126 us of
// kernels, 1.6 ns an item, and 457 us a call, most of it the host packing
// the occupations to bytes (the planned batch: 110 ms).  One wave per item
// up to n = 9 (at most 256 terms, four per lane); 4 up to n = 12, 16 beyond,
// so that a lane sweeps at most 32 states and a table of few items still
// spreads (10 outputs of 16 particles: 49 us for 465 us planned; 1000: 128
// us for 4.1 ms).
//
// Inputs with several particles in a mode may have fewer digits than an
// output: such outputs are summed over the input's digits, whose row sums are
// the same for every output and are laid out once (table_states_kernel).  40
// outputs of 12 particles from one mode: 6.4e-15 of error (norm) for 2.1e-14
// by the output's digits, 44 us a call for 43; 5000 of 16 from two modes 138
// us for 292; 2000 from [2, 1 x 14], whose 24576 states few outputs use, 300
// for 280.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "dd.hpp"
#include "perm_kernels.hpp"
#include "sweep_common.hpp"
#include "table_types.hpp"
#include "wave_plan.hpp"

namespace pqp {

namespace {

__constant__ double kFactorial[kTableMaxN + 1] = {
    1.0,       1.0,        2.0,         6.0,          24.0,          120.0,
    720.0,     5040.0,     40320.0,     362880.0,     3628800.0,     39916800.0,
    479001600.0, 6227020800.0, 87178291200.0, 1307674368000.0, 20922789888000.0};

// The product over the columns of one state's row sums.
template <int W, bool ONES>
__device__ __forceinline__ void table_product(const double (&cr)[W], const double (&ci)[W],
                                              cptr<int32_t> mult, double &pr, double &pi) {
  double ar = cr[0], ai = ci[0];
  if constexpr (W > 1) {
    double br = cr[1], bi = ci[1];
#pragma unroll
    for (int j = 2; j + 1 < W; j += 2) {
      cmul(ar, ai, cr[j], ci[j]);
      cmul(br, bi, cr[j + 1], ci[j + 1]);
    }
    if constexpr (W % 2 == 1 && W > 2) cmul(ar, ai, cr[W - 1], ci[W - 1]);
    cmul(ar, ai, br, bi);
  }
  if constexpr (!ONES) {
#pragma unroll
    for (int j = 0; j < W; ++j)
      for (int q = mult[j]; q > 1; --q) cmul(ar, ai, cr[j], ci[j]);
  }
  pr = ar;
  pi = ai;
}

// Whether the sweep over the input's digits is the cheaper one for an output
// of mc occupied modes, `most` in one, and `terms` terms of its own digits:
// the planner's rule and cost of a term (plan.cpp, sweep_cost).  It is also
// the more accurate one there.  Its terms carry the row sums to the powers of
// the output, so an output mode of small amplitude scales every term, where
// the other sweep's terms add it to the larger ones and cancel.
__device__ __forceinline__ bool sweep_flips(int mc, int most, const TableArgs &a, double terms) {
  const double mult = mc <= kPowGroupedMaxCols && most <= 4 ? mc + most - 2 : a.n - 1;
  const double per = most <= 1 ? 8.0 * mc - 2.0 : (2.0 * mc + 6.0 * mult + 4.0) * 1.25;
  return a.states * per < 0.9 * (terms * a.per_given);
}

// The lane's share of that sweep: states at, at + step, ... of the input.
__device__ __forceinline__ cdd flipped_sum(const TableArgs &a, int occ, int at, int step) {
  cdd sum = cdd_zero();
  const uint64_t used = __ballot(occ > 0);
  const int lane = lane_id();
  for (int v0 = at - lane; v0 < a.states; v0 += step) {
    const bool active = v0 + lane < a.states;
    const int v = active ? v0 + lane : 0;
    const double w = active ? a.weights[v] : 0.0;
    double pr = 1.0, pi = 0.0;
    for (uint64_t m = used; m;) {
      // the loads of four modes together: a load waits longer than it multiplies
      double2 z[4];
      int power[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = __builtin_ctzll(m ? m : used);
        power[k] = m ? __builtin_amdgcn_readlane(occ, i) : 0;
        z[k] = a.sums[static_cast<int64_t>(i) * a.states + v];
        m &= m - 1;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        for (int q = power[k]; q > 0; --q) cmul(pr, pi, z[k].x, z[k].y);
    }
    sum = cdd_add(sum, cdd{dd_mul_d(dd{pr, 0.0}, w), dd_mul_d(dd{pi, 0.0}, w)});
  }
  return sum;
}

// The row sums sum_j (rho_j - 2 g_j) U[i, j] (the prepended column with 1) of
// every mode i at every state g of the input's digits, and the states' signed
// weights.  Grid (states / 256, modes), a thread each.
__global__ __launch_bounds__(256) void table_states_kernel(TableArgs a) {
  const int v = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  const int i = static_cast<int>(blockIdx.y);
  if (v >= a.states) return;
  const cptr<double> row = as_const<double>(a.rows, int64_t{16} * i * a.width);
  const cptr<int32_t> mult = as_const<int32_t>(a.mult);
  double2 s = make_double2(row[2 * a.first], row[2 * a.first + 1]);
  double w = 1.0;
  int rest = v;
  for (int j = 0; j < a.width; ++j) {
    const int rho = mult[j] - (j == a.first ? 1 : 0);
    // the quotient by a small radix is exact this way
    const int q = static_cast<int>((static_cast<double>(rest) + 0.5) * kInvSmall[rho + 1]);
    const int g = rest - q * (rho + 1);
    rest = q;
    const double al = rho - 2 * g;
    s.x = fmaR(al, row[2 * j], s.x);
    s.y = fmaR(al, row[2 * j + 1], s.y);
    if (i == 0) {
      w *= lane_binomial(rho, g);
      if (g & 1) w = -w;
    }
  }
  a.sums[static_cast<int64_t>(i) * a.states + v] = s;
  if (i == 0) a.weights[v] = w;
}

// NW waves per item, 4 / NW items per block (NW <= 4) or one.
template <int W, bool ONES, int NW>
__global__ __launch_bounds__(NW > 4 ? NW * kWave : 4 * kWave)
__attribute__((amdgpu_waves_per_eu(W <= 8 ? 7 : W <= 12 ? 5 : 4, 8))) void perm_table_kernel(TableArgs a) {
  constexpr int kPerBlock = NW < 4 ? 4 / NW : 1;
  __shared__ double part[NW > 1 ? NW : 1][4];
  const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
  const int bw = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int wave = NW > 1 ? bw % NW : 0;
  const int64_t item = static_cast<int64_t>(blockIdx.x) * kPerBlock + bw / NW;
  if (item >= a.count) return;  // whole blocks where NW > 1
  const int occ = lane < a.modes ? a.outs[item * a.modes + lane] : 0;

  int total = 0, most = 0;
  for (int v = 1; v <= a.n; ++v) {
    const uint64_t at = __ballot(occ == v);
    total += v * __builtin_popcountll(at);
    if (at) most = v;
  }
  const bool match = total == a.n && !__ballot(occ > a.n);
  double *out = a.out + (a.prob ? 1 : 2) * item;
  if (!match) {  // another particle number: amplitude 0
    if (lane == 0 && wave == 0) {
      out[0] = 0.0;
      if (!a.prob) out[1] = 0.0;
    }
    return;
  }
  const WavePlan p = wave_plan(occ, a.n, NW * kWave, 6);
  const int S = 1 << p.k;
  const cptr<double> rows = as_const<double>(a.rows);
  const cptr<int32_t> mult = as_const<int32_t>(a.mult);

  cdd sum = cdd_zero();
  bool flipped = false;
  if constexpr (!ONES) {
    flipped = sweep_flips(__builtin_popcountll(__ballot(occ > 0)), most, a, static_cast<double>(p.U) * S);
    if (flipped) sum = flipped_sum(a, occ, wave * kWave + lane, NW * kWave);
  }
  for (int u0 = flipped ? p.U : wave * kWave; u0 < p.U; u0 += NW * kWave) {
    const bool active = u0 + lane < p.U;
    double cr[W], ci[W];
    const double w_top = wave_start<W>(p, active ? u0 + lane : 0, rows, 2 * W, p.i0, cr, ci);
    const double w = active ? w_top : 0.0;
    // the inner states in Gray order
    double sr = 0.0, si = 0.0;
    for (int v = 0; v < S; ++v) {
      double pr, pi;
      table_product<W, ONES>(cr, ci, mult, pr, pi);
      sr += (v & 1) ? -pr : pr;
      si += (v & 1) ? -pi : pi;
      const cptr<double> b = rows + wave_step_row(p, v) * (2 * W);
      const double s2 = in_vgpr(wave_step_factor(v));
#pragma unroll
      for (int j = 0; j < W; ++j) {
        cr[j] = fmaR(s2, b[2 * j], cr[j]);
        ci[j] = fmaR(s2, b[2 * j + 1], ci[j]);
      }
    }
    sum = cdd_add(sum, cdd{dd_mul_d(dd{sr, 0.0}, w), dd_mul_d(dd{si, 0.0}, w)});
  }
  sum = wave_reduce<0>(sum, lane);
  if constexpr (NW > 1) {
    if (lane == 0) {
      part[wave][0] = sum.re.hi;
      part[wave][1] = sum.re.lo;
      part[wave][2] = sum.im.hi;
      part[wave][3] = sum.im.lo;
    }
    __syncthreads();
    if (wave != 0) return;
    // fixed order: lane l holds wave l's sum, then a butterfly over 16 lanes
    static_assert(NW <= 16, "one lane per wave of a 16-lane group");
    sum = lane < NW ? cdd{{part[lane][0], part[lane][1]}, {part[lane][2], part[lane][3]}} : cdd_zero();
    sum = wave_reduce<0, 4>(sum, lane);
  }
  double norm = 1.0;
  for (uint64_t m = __ballot(occ > 1); m; m &= m - 1)
    norm *= kFactorial[__builtin_amdgcn_readlane(occ, __builtin_ctzll(m))];
  norm = sqrt(norm * a.in_norm);
  if (lane == 0) {
    const int e = -(a.n - 1);
    const double re = (ldexp(sum.re.hi, e) + ldexp(sum.re.lo, e)) / norm;
    const double im = (ldexp(sum.im.hi, e) + ldexp(sum.im.lo, e)) / norm;
    if (a.prob) {
      out[0] = fmaR(re, re, im * im);
    } else {
      out[0] = re;
      out[1] = im;
    }
  }
}

template <int W, bool ONES>
hipError_t table_launch(const TableArgs &a, hipStream_t stream) {
  const unsigned n = static_cast<unsigned>(a.count);
  if (a.n <= 9)
    hipLaunchKernelGGL((perm_table_kernel<W, ONES, 1>), dim3((n + 3) / 4), dim3(4 * kWave), 0, stream, a);
  else if (a.n <= 12)
    hipLaunchKernelGGL((perm_table_kernel<W, ONES, 4>), dim3(n), dim3(4 * kWave), 0, stream, a);
  else
    hipLaunchKernelGGL((perm_table_kernel<W, ONES, 16>), dim3(n), dim3(16 * kWave), 0, stream, a);
  return hipGetLastError();
}

}  // namespace

hipError_t launch_table_states(const TableArgs &a, hipStream_t stream) {
  if (a.states < 1 || a.modes > kTableMaxModes || a.width < 1 || a.width > kTableMaxN) return hipErrorInvalidValue;
  hipLaunchKernelGGL(table_states_kernel, dim3((a.states + 255) / 256, a.modes), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_table(int width, bool ones, const TableArgs &a, hipStream_t stream) {
  if (a.count <= 0) return hipSuccess;
  if (a.count > INT32_MAX || a.n < 1 || a.n > kTableMaxN || a.modes > kTableMaxModes) return hipErrorInvalidValue;
  switch (width) {
#define PQP_TABLE_CASE(W) \
  case W:                 \
    return ones ? table_launch<W, true>(a, stream) : table_launch<W, false>(a, stream);
    PQP_TABLE_CASE(1)
    PQP_TABLE_CASE(2)
    PQP_TABLE_CASE(3)
    PQP_TABLE_CASE(4)
    PQP_TABLE_CASE(5)
    PQP_TABLE_CASE(6)
    PQP_TABLE_CASE(7)
    PQP_TABLE_CASE(8)
    PQP_TABLE_CASE(9)
    PQP_TABLE_CASE(10)
    PQP_TABLE_CASE(11)
    PQP_TABLE_CASE(12)
    PQP_TABLE_CASE(13)
    PQP_TABLE_CASE(14)
    PQP_TABLE_CASE(15)
    PQP_TABLE_CASE(16)
#undef PQP_TABLE_CASE
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace pqp
