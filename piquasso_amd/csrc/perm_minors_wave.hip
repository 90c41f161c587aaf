// Column minors planned on the device, for gfx950: the sums of
// perm_minors.hip (unit column multiplicities, width - 1 particles in the
// rows) where every wave plans its item from the row multiplicities
// (wave_plan.hpp), and Clifford & Clifford sampling on top of them: all
// steps of all shots without the host.
//
// The minors of one sampling step have their own rows, hence their own Gray
// code, in every shot; planned on the host, that is 1 us per problem
// and a synchronisation per step, 20 of them for 20 photons, against 3.4 ms
// of kernels for 1024 shots.  The columns are the input modes in the order
// they join, known before the first step, so each shot's columns are laid
// out side by side once (sample_columns_kernel) and step k reads the first
// k + 1 of them.
//
// The minors kernel is bound by FP64 issue in the long items and by the
// fixed part of a wave in the short ones: the start state (one dependent
// row update per occupied row) and the sum of 2 (W + 1) double-double
// components over the lanes.  That sum is a reduce-scatter: two permlane
// stages halve the components a lane keeps, then the 16 lanes of a row
// exchange the rest through LDS, 44 double-double additions in all where a
// butterfly per component takes 252 (W = 20).  Measured, 20 photons in 40
// modes: one permanent_laplace call 136 -> 49 us (the minors 38 -> 23 us of
// kernel, their sum 58 -> 9 us with a block per column instead of one for
// all); 1024 samples 41 -> 11 ms, 2.1 ms of them kernels, 7 ms the host
// seeding a generator per shot.
#include <hip/hip_runtime.h>

#include <cstdint>

#include "dd.hpp"
#include "minors_common.hpp"
#include "minors_wave_types.hpp"
#include "perm_kernels.hpp"
#include "sweep_common.hpp"
#include "wave_plan.hpp"

namespace pqp {

namespace {

struct Pair {
  double a, b;  // lower half of the wave (or row): a of both partners; upper: b of both
};

// The partners l and l ^ (1 << B) trade one value: lanes with bit B clear
// get (x of this lane, x of the partner), lanes with it set (y of the
// partner, y of this lane).
template <int B>
__device__ __forceinline__ Pair trade(double x, double y) {
  const uint64_t xv = __builtin_bit_cast(uint64_t, x), yv = __builtin_bit_cast(uint64_t, y);
  const uint32_t xl = static_cast<uint32_t>(xv), xh = static_cast<uint32_t>(xv >> 32);
  const uint32_t yl = static_cast<uint32_t>(yv), yh = static_cast<uint32_t>(yv >> 32);
  const auto lo = B == 5 ? __builtin_amdgcn_permlane32_swap(xl, yl, false, false)
                         : __builtin_amdgcn_permlane16_swap(xl, yl, false, false);
  const auto hi = B == 5 ? __builtin_amdgcn_permlane32_swap(xh, yh, false, false)
                         : __builtin_amdgcn_permlane16_swap(xh, yh, false, false);
  return Pair{__builtin_bit_cast(double, (static_cast<uint64_t>(hi[0]) << 32) | lo[0]),
              __builtin_bit_cast(double, (static_cast<uint64_t>(hi[1]) << 32) | lo[1])};
}

constexpr int kSumStride = kWave + 1;  // LDS row stride in double2: rows fall on different banks

// The sums over the 64 lanes of M complex values, in double-double: lane l
// returns real component (l & 32 ? imaginary : real) of value 2 (l & 15) +
// (l & 16 ? 1 : 0), where that is below M.
template <int M>
__device__ __forceinline__ dd wave_sums(const double (&re)[M], const double (&im)[M], double2 *T, int lane) {
  constexpr int H = (M + 1) / 2;
  static_assert(H <= 16, "a 16-lane row holds at most 16 values");
  auto half = [&](int k) {  // lower lanes: real parts, upper: imaginary
    const Pair p = trade<5>(re[k], im[k]);
    return dd_two_sum(p.a, p.b);
  };
#pragma unroll
  for (int c = 0; c < H; ++c) {
    const dd even = half(2 * c);
    dd odd{0.0, 0.0};
    if (2 * c + 1 < M) odd = half(2 * c + 1);
    const Pair h = trade<4>(even.hi, odd.hi), l = trade<4>(even.lo, odd.lo);
    const dd s = dd_add(dd{h.a, l.a}, dd{h.b, l.b});
    T[c * kSumStride + lane] = make_double2(s.hi, s.lo);
  }
  __syncthreads();
  const int c = lane & 15;
  dd s{0.0, 0.0};
  if (c < H) {
    const double2 *row = T + c * kSumStride + (lane & ~15);
    s = dd{row[0].x, row[0].y};
#pragma unroll
    for (int i = 1; i < 16; ++i) s = dd_add(s, dd{row[i].x, row[i].y});
  }
  __syncthreads();
  return s;
}

}  // namespace

// Grid (waves, items), one wave per block.
template <int W>
__global__ __launch_bounds__(kWave)
__attribute__((amdgpu_waves_per_eu(minor_waves(W, true), 8))) void minors_wave_kernel(MinorsWaveArgs a) {
  __shared__ double2 T[((W + 1) / 2) * kSumStride];
  const int item = static_cast<int>(blockIdx.y);
  // Blocks go round the XCDs in turn; an item's working waves are its first
  // ones, so the turn starts elsewhere for each item (all items starting on
  // one XCD: 1283 us for the last step of 1024 shots of 20 photons, the
  // CUs busy for 545 of them).
  const int wave = (static_cast<int>(blockIdx.x) + item) % a.waves;
  if (a.units && wave >= as_const<int32_t>(a.units)[item]) return;
  const int lane = static_cast<int>(threadIdx.x);
  const int occ = lane < a.modes ? a.occ[static_cast<int64_t>(item) * a.modes + lane] : 0;
  const WavePlan p = wave_plan(occ, W - 1, kWave, a.k_max);
  const int S = 1 << p.k;
  const cptr<double> rows = as_const<double>(a.rows, static_cast<int64_t>(item) * a.item_stride * 8);
  const int stride = 2 * a.ld;

  double acr[W], aci[W];
#pragma unroll
  for (int k = 0; k < W; ++k) acr[k] = aci[k] = 0.0;
  constexpr int PF = W < 8 ? W : 8;  // row columns fetched ahead of the products
  for (int u0 = wave * kWave; u0 < p.U; u0 += a.waves * kWave) {
    const bool active = u0 + lane < p.U;
    double cr[W], ci[W];
    const double w_top = wave_start<W>(p, active ? u0 + lane : 0, rows, stride, p.i0, cr, ci);
    const double w = active ? w_top : 0.0;
    for (int v = 0; v < S; ++v) {
      const cptr<double> row = rows + wave_step_row(p, v) * stride;
      double ur[PF], ui[PF];
#pragma unroll
      for (int j = 0; j < PF; ++j) {
        ur[j] = row[2 * j];
        ui[j] = row[2 * j + 1];
      }
      // the sign and the lane's integer weight ride on the accumulation
      minor_products(cr, ci, (v & 1) ? -w : w, acr, aci);
      const double s2 = in_vgpr(wave_step_factor(v));
#pragma unroll
      for (int j = 0; j < PF; ++j) {
        cr[j] = fmaR(s2, ur[j], cr[j]);
        ci[j] = fmaR(s2, ui[j], ci[j]);
      }
#pragma unroll
      for (int j = PF; j < W; ++j) {
        cr[j] = fmaR(s2, row[2 * j], cr[j]);
        ci[j] = fmaR(s2, row[2 * j + 1], ci[j]);
      }
    }
  }
  const dd s = wave_sums<W>(acr, aci, T, lane);
  const int value = 2 * (lane & 15) + ((lane & 16) ? 1 : 0);
  if (value < W) {
    const int comp = ((lane & 32) ? W : 0) + value;
    double *out = a.partials + 2 * ((static_cast<int64_t>(item) * a.waves + wave) * (2 * W) + comp);
    out[0] = s.hi;
    out[1] = s.lo;
  }
}

// The minors of one item (item 0) from its waves' partials, a block per
// complex value: thread t adds partials t, t + NT, ... in double-double, the
// block its threads' sums in a fixed order; scaled by 2^-(width - 2).  The
// block that ends last publishes a.seq.
constexpr int kMinorsSumThreads = 256;

__global__ __launch_bounds__(kMinorsSumThreads) void minors_sum_kernel(MinorsWaveArgs a, int width) {
  __shared__ double part[kMinorsSumThreads / kWave][4];
  const int value = static_cast<int>(blockIdx.x);
  const int tid = static_cast<int>(threadIdx.x), lane = tid & (kWave - 1), wave = tid / kWave;
  const int comps = 2 * width;
  cdd s = cdd_zero();
  for (int k = tid; k < a.waves; k += kMinorsSumThreads) {
    const double *re = a.partials + 2 * (static_cast<int64_t>(k) * comps + value);
    const double *im = re + 2 * width;
    s = cdd_add(s, cdd{{re[0], re[1]}, {im[0], im[1]}});
  }
  s = wave_reduce<0>(s, lane);
  if (lane == 0) {
    part[wave][0] = s.re.hi;
    part[wave][1] = s.re.lo;
    part[wave][2] = s.im.hi;
    part[wave][3] = s.im.lo;
  }
  __syncthreads();
  if (tid != 0) return;
  for (int w = 1; w < kMinorsSumThreads / kWave; ++w)
    s = cdd_add(s, cdd{{part[w][0], part[w][1]}, {part[w][2], part[w][3]}});
  const int e = -(width - 2);
  a.out[2 * value] = ldexp(s.re.hi, e) + ldexp(s.re.lo, e);
  a.out[2 * value + 1] = ldexp(s.im.hi, e) + ldexp(s.im.lo, e);
  __threadfence_system();
  if (atomicAdd(a.last_counter, 1) == static_cast<int>(gridDim.x) - 1) {
    *a.last_counter = 0;
    __threadfence_system();
    __hip_atomic_store(a.done, a.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// Each shot's columns of the interferometer in the order its photons join,
// and empty outputs.  One block per shot.
__global__ __launch_bounds__(256) void sample_columns_kernel(SampleArgs a) {
  const int shot = static_cast<int>(blockIdx.x);
  const uint8_t *cols = a.cols + static_cast<int64_t>(shot) * a.photons;
  const int steps = a.steps[shot];
  const double2 *u = reinterpret_cast<const double2 *>(a.u_t);
  double2 *v = reinterpret_cast<double2 *>(a.v) + static_cast<int64_t>(shot) * a.modes * a.photons;
  for (int t = static_cast<int>(threadIdx.x); t < a.modes * a.photons; t += 256) {
    const int i = t / a.photons, p = t - i * a.photons;
    if (p < steps) v[t] = u[i * a.modes + cols[p]];
  }
  for (int t = static_cast<int>(threadIdx.x); t < a.modes; t += 256)
    a.occ[static_cast<int64_t>(shot) * a.modes + t] = 0;
  if (threadIdx.x == 0) a.units[shot] = 0;
  if (shot == 0 && threadIdx.x == 0) *a.failed = 0;
}

// Photon step + 1 of every shot: the minors from the waves' partials, the
// amplitudes sum_l U[j, col_l] M_l of the modes j (a lane each), the
// distribution's running sum, and the mode the shot's uniform number falls
// in (piquasso/_simulators/passive/sampling.py:711-749); then the waves the
// shot's next minors need.  One wave per shot.
__global__ __launch_bounds__(kWave) void sample_step_kernel(SampleArgs a) {
  const int shot = static_cast<int>(blockIdx.x);
  const int lane = static_cast<int>(threadIdx.x);
  const int steps = as_const<int32_t>(a.steps)[shot];
  if (steps <= a.step) return;
  const int W = a.step + 1;
  double mr = 1.0, mi = 0.0;  // the minor of an empty output
  if (a.step > 0) {
    const int used = as_const<int32_t>(a.units)[shot];
    cdd s = cdd_zero();
    if (lane < W) {
      const double *p = a.partials + static_cast<int64_t>(shot) * a.waves * (4 * W) + 2 * lane;
      for (int k = 0; k < used; ++k, p += 4 * W)
        s = cdd_add(s, cdd{{p[0], p[1]}, {p[2 * W], p[2 * W + 1]}});
    }
    const int e = -(W - 2);
    mr = ldexp(s.re.hi, e) + ldexp(s.re.lo, e);
    mi = ldexp(s.im.hi, e) + ldexp(s.im.lo, e);
  }
  const bool mode = lane < a.modes;
  const double2 *v = reinterpret_cast<const double2 *>(a.v) +
                     (static_cast<int64_t>(shot) * a.modes + (mode ? lane : 0)) * a.photons;
  double ar = 0.0, ai = 0.0;
  for (int l = 0; l < W; ++l) {
    const double xr = __shfl(mr, l), xi = __shfl(mi, l);
    const double2 z = v[l];
    ar = fmaR(z.x, xr, fmaR(-z.y, xi, ar));
    ai = fmaR(z.x, xi, fmaR(z.y, xr, ai));
  }
  double sum = mode ? fmaR(ar, ar, ai * ai) : 0.0;
  for (int off = 1; off < kWave; off *= 2) {  // running sum over the lanes
    const double below = __shfl_up(sum, off);
    if (lane >= off) sum += below;
  }
  const double total = __shfl(sum, kWave - 1);
  if (!(total > 0.0) || !(total < __builtin_inf())) {
    if (lane == 0) {
      atomicOr(a.failed, 1);
      a.units[shot] = 0;
    }
    return;
  }
  const double u = a.draws[static_cast<int64_t>(a.step) * a.shots + shot];
  const int at = min(__builtin_popcountll(__ballot(mode && sum / total <= u)), a.modes - 1);
  uint8_t *out = a.occ + static_cast<int64_t>(shot) * a.modes;
  int occ = mode ? out[lane] : 0;
  occ += lane == at ? 1 : 0;
  if (lane == at) out[lane] = static_cast<uint8_t>(occ);
  if (steps > W) {
    const WavePlan p = wave_plan(occ, W, kWave, a.next_k_max);
    if (lane == 0) a.units[shot] = min((p.U + kWave - 1) / kWave, a.next_waves);
  } else if (lane == 0) {
    a.units[shot] = 0;
  }
}

hipError_t launch_minors_wave(int width, const MinorsWaveArgs &a, int items, hipStream_t stream) {
  if (items <= 0) return hipSuccess;
  if (a.modes > kMinorsWaveMaxModes || a.waves < 1 || a.k_max > kMaxInnerDigits || items > 65535)
    return hipErrorInvalidValue;
  switch (width) {
#define PQP_WAVE_CASE(W)                                                                         \
  case W:                                                                                        \
    hipLaunchKernelGGL(minors_wave_kernel<W>, dim3(a.waves, items), dim3(kWave), 0, stream, a);  \
    break;
    PQP_WAVE_CASE(2)
    PQP_WAVE_CASE(3)
    PQP_WAVE_CASE(4)
    PQP_WAVE_CASE(5)
    PQP_WAVE_CASE(6)
    PQP_WAVE_CASE(7)
    PQP_WAVE_CASE(8)
    PQP_WAVE_CASE(9)
    PQP_WAVE_CASE(10)
    PQP_WAVE_CASE(11)
    PQP_WAVE_CASE(12)
    PQP_WAVE_CASE(13)
    PQP_WAVE_CASE(14)
    PQP_WAVE_CASE(15)
    PQP_WAVE_CASE(16)
    PQP_WAVE_CASE(17)
    PQP_WAVE_CASE(18)
    PQP_WAVE_CASE(19)
    PQP_WAVE_CASE(20)
    PQP_WAVE_CASE(21)
    PQP_WAVE_CASE(22)
    PQP_WAVE_CASE(23)
    PQP_WAVE_CASE(24)
#undef PQP_WAVE_CASE
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_minors_sum(int width, const MinorsWaveArgs &a, hipStream_t stream) {
  hipLaunchKernelGGL(minors_sum_kernel, dim3(width), dim3(kMinorsSumThreads), 0, stream, a, width);
  return hipGetLastError();
}

hipError_t launch_sample_columns(const SampleArgs &a, hipStream_t stream) {
  hipLaunchKernelGGL(sample_columns_kernel, dim3(a.shots), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_sample_step(const SampleArgs &a, hipStream_t stream) {
  if (a.modes > kWave || a.step >= kMinorsWaveMaxCols) return hipErrorInvalidValue;
  hipLaunchKernelGGL(sample_step_kernel, dim3(a.shots), dim3(kWave), 0, stream, a);
  return hipGetLastError();
}

}  // namespace pqp
