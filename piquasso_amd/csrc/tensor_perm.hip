// Tensor permanent of uniformly partially distinguishable bosons on gfx950,
// the quantity behind piquasso's detection probability of such inputs
// (piquasso/_simulators/passive/probabilities.py:156-237; Tichy,
// arXiv:1410.7687 Sec. III).  The reference sums over pairs of column
// subsets (s, t); here the same value is summed over pairs of sign vectors
// (delta, eps) in {+1, -1}^n with delta_0 = eps_0 = +1, the form Glynn's
// formula gives the permanent:
//
//   T = 4^-(n-1) sum_{delta, eps} (prod delta)(prod eps)
//       prod_i ( x R_delta[i] conj(R_eps[i]) + (1 - x) Q_{delta eps}[i] ),
//   R_delta[i] = sum_c delta_c A[i, c],
//   Q_{delta eps}[i] = sum_c delta_c eps_c |A[i, c]|^2.
//
// Averaging prod delta prod_i delta_{sigma(i)} over the signs keeps exactly
// the maps sigma that are permutations, as for the subsets, so both sums
// expand to sum_{sigma, tau} prod_i A[i, sigma(i)] conj(A[i, tau(i)])
// x^#{i: sigma(i) != tau(i)}.  The sign form has 4^(n-1) pairs instead of
// 4^n and far less cancellation (sum |term| / |T| ~ 10 instead of ~1e5 at
// n = 8).
//
// One wave per work unit (tensor_types.hpp: delta's bits as s, eps's as t).
// Each lane owns one delta and keeps x R_delta (2n doubles) and Q (n) in
// registers; the wave walks 2^kt eps in Gray order.  R_eps is the same in
// every lane, so it is not kept: tensor_signs_kernel writes it for every t
// once (2^(n-1) rows, 1.8 MB at n = 14), a step reads its row with scalar
// loads, as operands, and a lane its R_delta when it starts.  A step costs 9
// VALU per row: the flip Q -+= 2 delta_c (1 - x)|A[:, c]|^2, the factor (4)
// and the product (4); only the term's real part is accumulated (the
// (delta, eps) and (eps, delta) terms are conjugate).  FP64 runs of 64 steps
// are folded into a double-double lane sum; the wave and then the item's
// units are reduced in double-double in a fixed order.  Each unit also sums
// |term| for a forward-error bound of the result.
//
// Bound by FP64 issue: 114 VALU a step at n = 14, which the sweep issues at
// about 0.8 of the rate of the card's clock under FP64 load.  With R_eps
// updated in every lane a step cost 11 per row and 10 n VGPRs held the chip
// to two or three waves per SIMD: 8 outputs of 14 particles 1650 -> 1195 us
// a call, one of 16 particles 3570 -> 2780, of 18 55.6 -> 46 ms.
//
// Tables of many outputs (pqp_overlap_table_c128) send each output's rows
// of the interferometer instead of its matrix, and tensor_gather_kernel lays
// the matrices out: 500 outputs of 6 particles 4640 -> 50 us, 2000 of 3
// 22 ms -> 59 us (the host laid out and sent every matrix).
//
// A lone small permanent is bound by latency: the matrices of all orders come
// in one copy, short walks touch their lines first, an only unit writes its
// item's result, and results of few items go to host memory.  One of 9
// particles, with R_eps in every lane 38.1 us a call, by sign rows at first
// 49.8, now 38; of 3 31, 36, 30; 30 of 7 particles 92, 107, 91; 60 of
// 2 to 6 particles 167, 257, 174.
//
// Compiled twice: -DPQP_TENSOR_PART=0 instantiates n = 1..12 and the other
// kernels, =1 instantiates n = 13..20.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "dd.hpp"
#include "sweep_common.hpp"
#include "tensor_types.hpp"

namespace pqp {

namespace {

constexpr int kTensorFinal = 512;  // threads of a finalize block
constexpr int kWaitScalar = 0xC07F;  // s_waitcnt lgkmcnt(0)

__device__ __forceinline__ dd wave_reduce_dd(dd v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    dd o;
    o.hi = __shfl_xor(v.hi, off);
    o.lo = __shfl_xor(v.lo, off);
    v = dd_add(v, o);
  }
  return v;
}

// An item's result from its units' sum and their |term| sum: T = hi + lo by
// Glynn's scale 4^-(n-1) (exact), for a table the probability.
__device__ __forceinline__ void tensor_result(const TensorArgs &a, int item, dd s, double sa) {
  const int e = -2 * (a.n - 1);
  const double t = ldexp(s.hi + s.lo, e);
  if (a.prob) {
    a.prob[item] = t / a.norm[item];
  } else {
    a.out[2 * item] = t;
    a.out[2 * item + 1] = ldexp(sa, e);
  }
}

// Every line of `bytes` bytes read as scalars, sixteen loads in flight.
__device__ __forceinline__ void touch(cptr<uint32_t> lines, int bytes) {
  const int end = (bytes - 1) / 64;
  auto line = [&](int l) { return lines[16 * (l < end ? l : end)]; };
  for (int l = 0; l <= end; l += 16) {
    const uint32_t v0 = line(l), v1 = line(l + 1), v2 = line(l + 2), v3 = line(l + 3), v4 = line(l + 4);
    const uint32_t v5 = line(l + 5), v6 = line(l + 6), v7 = line(l + 7), v8 = line(l + 8), v9 = line(l + 9);
    const uint32_t v10 = line(l + 10), v11 = line(l + 11), v12 = line(l + 12), v13 = line(l + 13);
    const uint32_t v14 = line(l + 14), v15 = line(l + 15);
    __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7), "s"(v8), "s"(v9),
                     "s"(v10), "s"(v11), "s"(v12), "s"(v13), "s"(v14), "s"(v15));
  }
}

// Grid (units, items).
template <int N>
__global__ __launch_bounds__(kWave) void tensor_perm_kernel(TensorArgs a) {
  const cptr<TensorUnit> up = as_const<TensorUnit>(a.units) + blockIdx.x;
  const int item = static_cast<int>(blockIdx.y);
  const uint32_t s_hi = static_cast<uint32_t>(up->s_hi);
  const uint32_t t_blk = static_cast<uint32_t>(up->t_blk);
  const int mixed = up->mixed;
  const int ls = a.ls;
  const int kt = a.kt;
  const double x = as_const<double>(a.x)[item];
  constexpr int64_t kStates = int64_t{1} << (N - 1);
  const cptr<double> col = as_const<double>(a.cols, int64_t{16} * N * N * item);  // [c][i] (re, im)
  const cptr<double> pw = as_const<double>(a.pw, int64_t{8} * N * N * item);      // [c][i]
  const cptr<double> signs = as_const<double>(a.signs, 16 * N * kStates * item);  // [t][i] (re, im)

  const int lane = static_cast<int>(threadIdx.x);
  const bool active = lane < (1 << ls);
  // sign vectors: column 0 fixed at +1, column b + 1 is -1 where bit b is set
  const uint32_t s = (s_hi << ls) | static_cast<uint32_t>(active ? lane : 0);
  const uint32_t t0 = t_blk << kt;

  // A short walk first touches the lines of its rows of `signs` and of the
  // columns, all in flight together (a lane each, then as scalars): in a
  // launch of few waves every step would wait for its own.
  if ((2 * N << kt) <= 8 * kWave) {
    const int64_t from = 2 * N * (kStates * item + t0);
    const int rows = 2 * N << kt, most = N * N;
    const double v = a.signs[from + min(8 * lane, rows - 1)];
    const double c = a.pw[static_cast<int64_t>(most) * item + min(8 * lane, most - 1)];
    __asm__ volatile("" ::"v"(v), "v"(c));
    touch(as_const<uint32_t>(a.pw, int64_t{8} * most * item), 8 * most);
    touch(as_const<uint32_t>(a.signs, 8 * from), 8 * rows);
  }

  // x R_delta and (1 - x) Q_{delta eps} at the walk's first eps
  double xr[N], xi[N], q[N];
  {
    const double2 *own = reinterpret_cast<const double2 *>(a.signs) + N * (kStates * item + s);
#pragma unroll
    for (int i = 0; i < N; ++i) {
      const double2 z = own[i];
      xr[i] = x * z.x;
      xi[i] = x * z.y;
      q[i] = 0.0;
    }
  }
#pragma unroll 1
  for (int c = 0; c < N; ++c) {
    const bool dneg = c > 0 && ((s >> (c - 1)) & 1u);
    const bool eneg = c > 0 && ((t0 >> (c - 1)) & 1u);  // wave-uniform
    const double de = (dneg != eneg) ? -1.0 : 1.0;
#pragma unroll
    for (int i = 0; i < N; ++i) q[i] = fmaR(de, pw[c * N + i], q[i]);
  }
  double sign = ((__builtin_popcount(s) ^ __builtin_popcount(t0)) & 1) ? -1.0 : 1.0;

  // The scalar operands of a step, its row of `signs` and the column it
  // flips, are loaded in groups of four rows (one 64-byte load; a single row
  // left over joins the last group): the next group's loads are issued
  // when the current group's have arrived and wait out its products.
  constexpr int kParts = N <= 4 ? 1 : N == 5 ? 2 : (N + 2) / 4;
  double r[2 * N], flip[N];
  auto request = [&](auto part, uint32_t t, int c) {
    constexpr int kFrom = 4 * part, kTo = part + 1 < kParts ? kFrom + 4 : N;
    const cptr<double> row = signs + static_cast<int64_t>(t) * (2 * N);
    const cptr<double> column = pw + c * N;
#pragma unroll
    for (int i = 2 * kFrom; i < 2 * kTo; ++i) r[i] = row[i];
#pragma unroll
    for (int i = kFrom; i < kTo; ++i) flip[i] = column[i];
  };

  dd acc_dd{0.0, 0.0};
  double acc = 0.0;
  double aabs = 0.0;  // sum of |term| as counted (forward-error scale)
  const int steps = 1 << kt;
  request(std::integral_constant<int, 0>{}, t0, steps > 1 ? 1 : 0);
  uint32_t t = t0;
  for (int k = 0; k < steps; ++k) {
    // the step to state k + 1 flips eps at column ctz(k + 1) + 1; after the
    // last state column 0, for a Q that is not read
    const int b = __builtin_ctz(static_cast<unsigned>(k + 1));
    const int c = k + 1 < steps ? b + 1 : 0;
    const uint32_t g = static_cast<uint32_t>((k + 1) ^ ((k + 1) >> 1));
    const int b_next = __builtin_ctz(static_cast<unsigned>(k + 2));
    const int c_next = k + 2 < steps ? b_next + 1 : 0;
    const uint32_t t_next = k + 1 < steps ? (t0 | g) : t0;
    const double sd2 = in_vgpr(((g >> b) & 1u) ? -2.0 : 2.0);
    const double sq2 = ((s >> b) & 1u) ? -sd2 : sd2;
    double pr = 0.0, pi = 0.0;
    auto part_of_step = [&](auto part) {
      constexpr int kFrom = 4 * part, kTo = part + 1 < kParts ? kFrom + 4 : N;
      __builtin_amdgcn_s_waitcnt(kWaitScalar);
      __builtin_amdgcn_sched_barrier(0);
      double mr[2 * (kTo - kFrom)], mf[kTo - kFrom];
#pragma unroll
      for (int i = kFrom; i < kTo; ++i) {
        mr[2 * (i - kFrom)] = r[2 * i];
        mr[2 * (i - kFrom) + 1] = r[2 * i + 1];
        mf[i - kFrom] = flip[i];
      }
      if constexpr (part + 1 < kParts)
        request(std::integral_constant<int, part + 1>{}, t, c);
      else
        request(std::integral_constant<int, 0>{}, t_next, c_next);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = kFrom; i < kTo; ++i) {
        // factor i: x R_delta[i] conj(R_eps[i]) + Q[i]
        const double rr = mr[2 * (i - kFrom)], ri = mr[2 * (i - kFrom) + 1];
        const double fr = fmaR(xi[i], ri, fmaR(xr[i], rr, q[i]));
        const double fi = fmaR(xi[i], rr, -(xr[i] * ri));
        if (i == 0) {
          pr = fr;
          pi = fi;
        } else if (i < N - 1) {
          cmul(pr, pi, fr, fi);
        } else {
          pr = fmaR(pr, fr, -(pi * fi));  // real part of the product
        }
        q[i] = fmaR(sq2, mf[i - kFrom], q[i]);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    part_of_step(std::integral_constant<int, 0>{});
    if constexpr (kParts > 1) part_of_step(std::integral_constant<int, 1>{});
    if constexpr (kParts > 2) part_of_step(std::integral_constant<int, 2>{});
    if constexpr (kParts > 3) part_of_step(std::integral_constant<int, 3>{});
    if constexpr (kParts > 4) part_of_step(std::integral_constant<int, 4>{});
    static_assert(kParts <= 5, "parts of a step");
    // pairs below the diagonal block are not counted, pairs in it half
    if (!mixed || (t >> ls) > s_hi) {
      acc = fmaR(sign, pr, acc);
      aabs += __builtin_fabs(pr);
    } else if ((t >> ls) == s_hi) {
      acc = fmaR(0.5 * sign, pr, acc);
      aabs = fmaR(0.5, __builtin_fabs(pr), aabs);
    }
    if ((k & (kDdFold - 1)) == kDdFold - 1) {
      acc_dd = dd_add_d(acc_dd, acc);
      acc = 0.0;
    }
    t = t_next;
    sign = -sign;
  }
  acc_dd = dd_add_d(acc_dd, acc);
  if (!active) {
    acc_dd = dd{0.0, 0.0};
    aabs = 0.0;
  }
  acc_dd = wave_reduce_dd(acc_dd);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) aabs += __shfl_xor(aabs, off);
  if (lane == 0) {
    // twice: the sum counts each pair with its conjugate
    acc_dd = dd{2.0 * acc_dd.hi, 2.0 * acc_dd.lo};
    aabs *= 2.0;
    if (a.n_units == 1) {  // the item's only unit
      tensor_result(a, item, acc_dd, aabs);
      return;
    }
    double *p = a.partials + 3 * (static_cast<int64_t>(item) * a.n_units + blockIdx.x);
    p[0] = acc_dd.hi;
    p[1] = acc_dd.lo;
    p[2] = aabs;
  }
}

#if PQP_TENSOR_PART == 0
// Tables: item's matrix A[i, c] = u[rows[i], c], with (1 - x) |A|^2 rounded
// as the host rounds it for single matrices.
__global__ __launch_bounds__(256) void tensor_gather_kernel(TensorArgs a) {
#pragma clang fp contract(off)
  const int item = static_cast<int>(blockIdx.x);
  const int n = a.n, nn = n * n;
  const double y = 1.0 - a.x[item];
  const double2 *u = reinterpret_cast<const double2 *>(a.u);
  for (int t = static_cast<int>(threadIdx.x); t < nn; t += 256) {
    const int c = t / n, i = t - c * n;
    const double2 z = u[static_cast<int64_t>(a.rows[static_cast<int64_t>(item) * n + i]) * n + c];
    reinterpret_cast<double2 *>(a.cols)[static_cast<int64_t>(item) * nn + t] = z;
    a.pw[static_cast<int64_t>(item) * nn + t] = y * (z.x * z.x + z.y * z.y);
  }
}

// R_eps[i] = sum_c eps_c A[i, c] for every t and row i: a thread each.  The
// items of all orders in one launch, since a launch costs small ones more than
// its work: five orders of 1 to 5 particles 80 -> 69 us a call.
__global__ __launch_bounds__(256) void tensor_signs_kernel(TensorSigns g) {
  int o = 0;
  while (o + 1 < g.n_orders && blockIdx.x >= g.orders[o + 1].first) ++o;
  const TensorSigns::Order a = g.orders[o];
  const uint32_t b = blockIdx.x - a.first, item = b / a.per_item;
  const int n = a.n;
  const int64_t all = static_cast<int64_t>(n) << (n - 1);
  const int64_t at = static_cast<int64_t>(b - item * a.per_item) * 256 + threadIdx.x;
  if (at >= all) return;
  const uint32_t t = static_cast<uint32_t>(at / n);
  const int i = static_cast<int>(at - static_cast<int64_t>(t) * n);
  const double2 *col = reinterpret_cast<const double2 *>(a.cols) + static_cast<int64_t>(item) * n * n;
  double2 r = col[i];
#pragma unroll 4
  for (int c = 1; c < n; ++c) {
    const double2 z = col[c * n + i];
    const bool neg = (t >> (c - 1)) & 1u;
    r.x += neg ? -z.x : z.x;
    r.y += neg ? -z.y : z.y;
  }
  reinterpret_cast<double2 *>(a.signs)[static_cast<int64_t>(item) * all + at] = r;
}

// One block per item: the dd sum of the item's unit partials (strided over
// the threads, a fixed butterfly in each wave, then the waves in order), and
// its result; items of one unit have written theirs.  Bound by the chain of
// loads and dd additions of one thread: one wave took 21 us over the 4160
// units of n = 14.
__global__ __launch_bounds__(kTensorFinal) void tensor_finalize_kernel(TensorArgs a) {
  const int threads = static_cast<int>(blockDim.x), waves = threads / kWave;
  __shared__ double part[kTensorFinal / kWave][3];
  const int item = static_cast<int>(blockIdx.x);
  dd s{0.0, 0.0};
  double sa = 0.0;
#pragma unroll 4
  for (int u = static_cast<int>(threadIdx.x); u < a.n_units; u += threads) {
    const double *p = a.partials + 3 * (static_cast<int64_t>(item) * a.n_units + u);
    s = dd_add(s, dd{p[0], p[1]});
    sa += p[2];
  }
  s = wave_reduce_dd(s);
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) sa += __shfl_xor(sa, off);
  if ((threadIdx.x & (kWave - 1)) == 0) {
    double *p = part[threadIdx.x / kWave];
    p[0] = s.hi;
    p[1] = s.lo;
    p[2] = sa;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < waves; ++w) {
      s = dd_add(s, dd{part[w][0], part[w][1]});
      sa += part[w][2];
    }
    tensor_result(a, item, s, sa);
  }
}
#endif

}  // namespace

#if PQP_TENSOR_PART == 0
#define PQP_TENSOR_CASES X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
hipError_t launch_tensor_p0(const TensorArgs &a, hipStream_t stream) {
#else
#define PQP_TENSOR_CASES X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20)
hipError_t launch_tensor_p1(const TensorArgs &a, hipStream_t stream) {
#endif
  switch (a.n) {
#define X(k)                                                                                       \
  case k:                                                                                          \
    hipLaunchKernelGGL(tensor_perm_kernel<k>, dim3(a.n_units, a.n_items), dim3(kWave), 0, stream, a); \
    return hipGetLastError();
    PQP_TENSOR_CASES
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

#if PQP_TENSOR_PART == 0
hipError_t launch_tensor_gather(const TensorArgs &a, hipStream_t stream) {
  hipLaunchKernelGGL(tensor_gather_kernel, dim3(a.n_items), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_tensor_signs(const TensorArgs *passes, int n, hipStream_t stream) {
  while (n > 0) {
    TensorSigns g{};
    uint64_t blocks = 0;
    for (; g.n_orders < kTensorMaxN && g.n_orders < n; ++g.n_orders) {
      const TensorArgs &a = passes[g.n_orders];
      const uint64_t per_item = ((static_cast<uint64_t>(a.n) << (a.n - 1)) + 255) / 256;
      if (g.n_orders > 0 && blocks + per_item * static_cast<uint64_t>(a.n_items) > INT32_MAX) break;
      g.orders[g.n_orders] = {a.cols, a.signs, a.n, static_cast<uint32_t>(blocks), static_cast<uint32_t>(per_item)};
      blocks += per_item * static_cast<uint64_t>(a.n_items);
    }
    hipLaunchKernelGGL(tensor_signs_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, stream, g);
    const hipError_t st = hipGetLastError();
    if (st != hipSuccess) return st;
    passes += g.n_orders;
    n -= g.n_orders;
  }
  return hipSuccess;
}

hipError_t launch_tensor_finalize(const TensorArgs &a, hipStream_t stream) {
  if (a.n_units == 1) return hipSuccess;
  const int waves = std::min((a.n_units + kWave - 1) / kWave, kTensorFinal / kWave);  // no idle ones to wait for
  hipLaunchKernelGGL(tensor_finalize_kernel, dim3(a.n_items), dim3(kWave * waves), 0, stream, a);
  return hipGetLastError();
}
#endif

}  // namespace pqp
