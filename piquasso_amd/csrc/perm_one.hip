// One permanent of up to 2^24 Gray terms in one launch on gfx950, for the
// single-call entry points (src/permanent.cpp:49-264 is the sum).  Nothing
// is planned into tables, copied and loaded: the kernel arguments hold the
// distinct rows, in the order of their digits, and the multiplicities.
//
// Sums as in perm_fwd.hip: row sums and products in Real (FP64, or FP32
// where the caller chose it), FP64 runs of at most 64 terms folded into
// double-double, exact integer weights, the lanes' and waves' sums added in
// double-double in a fixed order (a value does not depend on scheduling).
//
// Bound by latency: 2^19 terms of 20 columns are 3 us of FP64 issue for the
// whole chip.  What counts is the chain of one wave: its start, its inner
// states, the double-double reductions, and the way to the host.  So
//  * the lanes of a wave differ in a few digits only: six binary ones, or
//    those whose states fill sets of 64 lanes best (one_fill).  The rows of
//    all other digits are summed once per wave, a lane per component (their
//    loads are in flight together), and broadcast through the LDS; a lane
//    then adds a few rows instead of all;
//  * these rows and the inner ones are scalar operands, and the waves of
//    a block touch their lines, and the digits', together first;
//  * permanents of few terms stay in one block (no block waits for another),
//    others take up to one wave per SIMD with few inner states.  Their
//    blocks count themselves; the last one sums the partials and publishes
//    the result to mapped host memory;
//  * permanents of one particle in each row and column have kernels of their
//    own: all digits are binary, and no code of other digits is fetched.
//
// A call, against the planned sweep with occupations not seen before and with
// its plan kept: 8 particles 15.0 and 11.2 -> 10.3 us, 12 18.1 and 13.5 ->
// 12.5, 16 35.6 and 30 -> 16.3, 24 98 and 95 -> 61 (of it 55 us of FP64
// issue); 20 in 15 of 40 modes 49 and 43 -> 20.  Bunched on both sides, plan
// kept: [20, 20] in both 15.7 -> 13.0 us, [8, 8, 8] 18.3 -> 13.4, 36 in 9 and
// 18 modes 57 -> 42.  (With lanes of at most 64 states of whole digits, inner
// digits that left waves idle, powers by a masked pass for every multiplicity
// and binomials by a loop these took 47, 38 and 70.)  The kernel takes 4.7 us
// at 8 particles (one wave) and 12 at 18, of it about 3 for the blocks'
// meeting.
//
// Compiled once per type of the rows: -DPQP_ONE_FP32=0, 1.
#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>
#include <type_traits>

#include "dd.hpp"
#include "one_types.hpp"
#include "perm_kernels.hpp"
#include "sweep_common.hpp"

namespace pqp {

namespace {

constexpr int kOneChunk = 8;  // common rows of a wave loaded at once

#if PQP_ONE_FP32
using Real = float;
#else
using Real = double;
#endif

// The product over the columns of one state's row sums, in two chains of
// multiplies (even and odd columns).  more: the columns' further powers, a
// byte each.
template <int W, OneKind KIND>
__device__ __forceinline__ void one_product(const Real (&cr)[W], const Real (&ci)[W],
                                            const uint32_t (&more)[kOneMaxWidth / 4], Real &pr, Real &pi) {
  Real ar = cr[0], ai = ci[0];
  if constexpr (W > 1) {
    Real br = cr[1], bi = ci[1];
#pragma unroll
    for (int j = 2; j + 1 < W; j += 2) {
      cmul(ar, ai, cr[j], ci[j]);
      cmul(br, bi, cr[j + 1], ci[j + 1]);
    }
    if constexpr (W % 2 == 1 && W > 2) cmul(ar, ai, cr[W - 1], ci[W - 1]);
    if constexpr (KIND == kOneAny) {
#pragma unroll
      for (int j = 0; j < W; j += 2) {
        int qa = (more[j / 4] >> (8 * (j % 4))) & 255;
        int qb = 0;
        if (j + 1 < W) qb = (more[(j + 1) / 4] >> (8 * ((j + 1) % 4))) & 255;
        const int jb = j + 1 < W ? j + 1 : j;
        for (; qa > 0 && qb > 0; --qa, --qb) {
          cmul(ar, ai, cr[j], ci[j]);
          cmul(br, bi, cr[jb], ci[jb]);
        }
        for (; qa > 0; --qa) cmul(ar, ai, cr[j], ci[j]);
        for (; qb > 0; --qb) cmul(br, bi, cr[jb], ci[jb]);
      }
    }
    cmul(ar, ai, br, bi);
  } else if constexpr (KIND == kOneAny) {
    for (int q = more[0] & 255; q > 0; --q) cmul(ar, ai, cr[0], ci[0]);
  }
  pr = ar;
  pi = ai;
}

// u's lowest digit of radix r (inv: 1 / r), taken off u (u < 2^50: the
// quotient is exact this way).
__device__ __forceinline__ int one_digit(int &u, int r, double inv) {
  const int q = static_cast<int>((static_cast<double>(u) + 0.5) * inv);
  const int g = u - q * r;
  u = q;
  return g;
}

// C(rho, g), g <= rho <= 64, rounded once (exact up to 2^53), at rho (rho +
// 1) / 2 + g: read where a loop of rho rounded quotients took 2 us for a digit
// of 20 particles.
struct Binomials {
  double c[65 * 66 / 2];
};
constexpr Binomials binomials() {
  Binomials t{};
  uint64_t row[66] = {1};
  for (int rho = 0; rho <= 64; ++rho) {
    for (int g = 0; g <= rho; ++g) t.c[rho * (rho + 1) / 2 + g] = static_cast<double>(row[g]);
    for (int g = rho + 1; g >= 1; --g) row[g] += row[g - 1];
  }
  return t;
}
__constant__ Binomials kBinomials = binomials();

// The digit's C(rho, g), the small ones from its packed bytes.
__device__ __forceinline__ double one_binomial(uint64_t choose, int rho, int g) {
  if (choose) return static_cast<double>(static_cast<uint32_t>(choose >> (8 * min(g, rho - g))) & 255u);
  return kBinomials.c[rho * (rho + 1) / 2 + g];
}

// The sum over a block of nw waves, in the lanes 0..7 of wave 0.
__device__ __forceinline__ void block_sum(cdd &s, double &mag, double (&part)[kOneWaves][5], int nw, int wave, int lane) {
  s = wave_reduce<0>(s, lane);
  mag = wave_sum(mag, lane);
  if (nw == 1) return;
  if (lane == 0) {
    part[wave][0] = s.re.hi;
    part[wave][1] = s.re.lo;
    part[wave][2] = s.im.hi;
    part[wave][3] = s.im.lo;
    part[wave][4] = mag;
  }
  __syncthreads();
  const int w = lane < nw ? lane : 0;
  s = lane < nw ? cdd{{part[w][0], part[w][1]}, {part[w][2], part[w][3]}} : cdd_zero();
  mag = lane < nw ? part[w][4] : 0.0;
  static_assert(kOneWaves <= 8, "three butterfly steps");
  s = wave_reduce<0, 3>(s, lane);
  mag = wave_sum<0, 3>(mag, lane);
}

using OneRowsHost = decltype(OneArgs::rows);

// The kernel's part of the arguments.
template <int W, OneKind KIND>
using Rows = OneRows<one_row_bytes(KIND == kOneUnit ? W : kOneMaxRows, W, sizeof(Real))>;
template <int W, OneKind KIND>
using Args = std::conditional_t<KIND == kOneUnit, Rows<W, KIND>, OneArgsOf<sizeof(Rows<W, KIND>::b)>>;

template <int W, OneKind KIND>
__global__ __launch_bounds__(kWave * kOneWaves) void perm_one_kernel(Args<W, KIND> given) {
  constexpr bool kUnit = KIND == kOneUnit;
  const int nw = static_cast<int>(blockDim.x) / kWave;
  __shared__ double part[kOneWaves][5];
  __shared__ Real base[kOneWaves][2 * W];
  const int lane = static_cast<int>(threadIdx.x) & (kWave - 1);
  const int bw = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / kWave);
  const int waves = nw * static_cast<int>(gridDim.x);
  const int wave = nw * static_cast<int>(blockIdx.x) + bw;
  const uintptr_t all = reinterpret_cast<uintptr_t>(__builtin_amdgcn_kernarg_segment_ptr());
  uintptr_t self = all;  // the rows and their head
  const OneHead *head;
  if constexpr (kUnit) {
    head = &given.h;
  } else {
    head = &given.rows.h;
    self += offsetof(OneArgs, rows);
  }
  const OneHead &args = *head;
  const cptr<Real> rows = reinterpret_cast<cptr<Real>>(self + offsetof(OneRowsHost, b));
  const Real *vrows = reinterpret_cast<const Real *>(self + offsetof(OneRowsHost, b));
  // (of kind kOneUnit, not read)
  const cptr<OneTables> tables = reinterpret_cast<cptr<OneTables>>(all);
  const cptr<OneDigit> lane_digit = tables->lane, digit = tables->digit;
  uint32_t more[kOneMaxWidth / 4] = {};
  if constexpr (KIND == kOneAny) {
#pragma unroll
    for (int k = 0; k < (W + 3) / 4; ++k) more[k] = tables->more[k];
  }
  const int n = args.n, k = args.inner, rest = args.rest;
  const int L = args.lane_digits, P = args.lanes, S = args.S, chunks = args.chunks;
  bool binary = true, lane_binary = true;
  int lane_chunks = 1;
  if constexpr (!kUnit) {
    binary = tables->binary;
    lane_binary = tables->lane_binary;
    lane_chunks = tables->lane_chunks;
  }
  // The first rows common to a wave's lanes, a component per lane: requested
  // before the wave waits for anything else (a first touch costs about a
  // microsecond, and one after another these were most of the start).
  const int common = 1 + k + rest;
  const int at = lane < 2 * W ? lane : 0;
  Real first[kOneChunk];
#pragma unroll
  for (int i = 0; i < kOneChunk; ++i) first[i] = vrows[(L + min(i, common - 1)) * (2 * W) + at];
  {
    // every line of the rows read as scalars, eight loads of a wave in
    // flight, and of the digits
    const cptr<uint32_t> lines = reinterpret_cast<cptr<uint32_t>>(self + offsetof(OneRowsHost, b));
    const int end = ((L + 1 + k) * 2 * W * static_cast<int>(sizeof(Real)) - 1) / 64;
    auto line = [&](int l) { return lines[16 * min(l, end)]; };
    const uint32_t v0 = line(bw), v1 = line(bw + nw), v2 = line(bw + 2 * nw), v3 = line(bw + 3 * nw);
    const uint32_t v4 = line(bw + 4 * nw), v5 = line(bw + 5 * nw), v6 = line(bw + 6 * nw), v7 = line(bw + 7 * nw);
    if constexpr (!kUnit) {
      const cptr<uint32_t> d = reinterpret_cast<cptr<uint32_t>>(tables);
      const uint32_t d0 = d[0], d1 = d[16], d2 = d[32], d3 = d[48], d4 = d[64], d5 = d[80], d6 = d[96], d7 = d[112];
      const uint32_t d8 = d[128], d9 = d[144], d10 = d[160], d11 = d[176], d12 = d[192];
      static_assert(offsetof(OneTables, step) <= 13 * 64);
      __asm__ volatile("" ::"s"(d0), "s"(d1), "s"(d2), "s"(d3), "s"(d4), "s"(d5), "s"(d6), "s"(d7), "s"(d8), "s"(d9),
                       "s"(d10), "s"(d11), "s"(d12));
    }
    __asm__ volatile("" ::"s"(v0), "s"(v1), "s"(v2), "s"(v3), "s"(v4), "s"(v5), "s"(v6), "s"(v7));
    for (int l = bw + 8 * nw; l <= end; l += 8 * nw) {
      const uint32_t w0 = line(l), w1 = line(l + nw), w2 = line(l + 2 * nw), w3 = line(l + 3 * nw);
      const uint32_t w4 = line(l + 4 * nw), w5 = line(l + 5 * nw), w6 = line(l + 6 * nw), w7 = line(l + 7 * nw);
      __asm__ volatile("" ::"s"(w0), "s"(w1), "s"(w2), "s"(w3), "s"(w4), "s"(w5), "s"(w6), "s"(w7));
    }
  }
  if (nw > 1) __syncthreads();

  cdd sum = cdd_zero();
  double mag = 0.0;  // of the terms: |Re| + |Im| each
  // the lane's signed weight in a set of lane states
  auto lane_weight = [&](int at) {
    if (lane_binary) return __builtin_popcount(at) & 1 ? -1.0 : 1.0;
    double w = 1.0;
    int u = at, parity = 0;
    for (int t = 0; t < L; ++t) {
      const int rr = lane_digit[t].rho;
      const int g = one_digit(u, rr + 1, lane_digit[t].inv);
      parity ^= g & 1;
      w *= one_binomial(lane_digit[t].choose, rr, g);
    }
    return parity ? -w : w;
  };
  int held = 0;  // the set that lane_w belongs to
  double lane_w = lane < P ? lane_weight(lane) : 0.0;
  for (int chunk = wave; chunk < chunks; chunk += waves) {
    Real cr[W], ci[W];
    int u = chunk, set = 0;
    if (lane_chunks > 1) {
      set = __builtin_amdgcn_readfirstlane(one_digit(u, lane_chunks, tables->lane_inv));
      if (set != held) {
        const int v = kWave * set + lane;
        lane_w = v < P ? lane_weight(v) : 0.0;
        held = set;
      }
    }
    double w = lane_w;
    int parity = 0;
    // the rows common to the lanes: the prepended one, the inner ones at
    // their first state, then the rest digits
    double b = 0.0;
    for (int c0 = 0; c0 < common; c0 += kOneChunk) {
      Real v[kOneChunk];
#pragma unroll
      for (int i = 0; i < kOneChunk; ++i)
        v[i] = c0 == 0 ? first[i] : vrows[(L + min(c0 + i, common - 1)) * (2 * W) + at];
#pragma unroll
      for (int i = 0; i < kOneChunk; ++i) {
        const int t = c0 + i - 1;
        if (t < k + rest) {
          double al = 1.0;
          if constexpr (kUnit) {
            if (t >= k) {
              al = (u & 1) ? -1.0 : 1.0;
              parity ^= u & 1;
              u >>= 1;
            }
          } else if (t >= k) {
            const int rr = digit[t].rho;
            const int g = one_digit(u, rr + 1, digit[t].inv);
            parity ^= g & 1;
            w *= one_binomial(digit[t].choose, rr, g);
            al = static_cast<double>(rr - 2 * g);
          } else if (t >= 0) {
            al = digit[t].rho;
          }
          b = fmaR(al, static_cast<double>(v[i]), b);
        }
      }
    }
    if (lane < 2 * W) base[bw][lane] = static_cast<Real>(b);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int j = 0; j < W; ++j) {
      cr[j] = base[bw][2 * j];
      ci[j] = base[bw][2 * j + 1];
    }
    __builtin_amdgcn_wave_barrier();
    u = kWave * set + lane;
#pragma unroll 1
    for (int t = 0; t < L; ++t) {
      Real al;
      int rr = 1;
      if constexpr (!kUnit) rr = lane_digit[t].rho;
      if (rr == 1) {
        al = (u & 1) ? Real(-1) : Real(1);
        u >>= 1;
      } else {
        al = static_cast<Real>(rr - 2 * one_digit(u, rr + 1, lane_digit[t].inv));
      }
      const cptr<Real> row = rows + t * (2 * W);
#pragma unroll
      for (int j = 0; j < W; ++j) {
        cr[j] = fmaR(al, row[2 * j], cr[j]);
        ci[j] = fmaR(al, row[2 * j + 1], ci[j]);
      }
    }
    if (parity) w = -w;
    // the inner states in Gray order
    double sr = 0.0, si = 0.0, sa = 0.0;
    for (int v = 0; v < S; ++v) {
      // the digit that moves after state v (after the last one any: an
      // update that is not read)
      const int move = __builtin_ctz(v + 1);
      const int up = (v + 1) ^ ((v + 1) >> 1);
      int row = move < k ? 1 + move : 0;
      Real s2 = in_vgpr(((up >> move) & 1) ? Real(-2) : Real(2));
      double coef = in_vgpr((v & 1) ? -1.0 : 1.0);
      if (!binary) {
        row = tables->step[v].row;
        s2 = in_vgpr(static_cast<Real>(tables->step[v].factor));
        coef = in_vgpr(tables->step[v].coef);
      }
      const cptr<Real> b = rows + (L + row) * (2 * W);
      Real pr, pi;
      one_product<W, KIND>(cr, ci, more, pr, pi);
      const double dr = static_cast<double>(pr), di = static_cast<double>(pi);
      sr = fmaR(coef, dr, sr);
      si = fmaR(coef, di, si);
      sa = fmaR(__builtin_fabs(coef), __builtin_fabs(dr), sa);
      sa = fmaR(__builtin_fabs(coef), __builtin_fabs(di), sa);
#pragma unroll
      for (int j = 0; j < W; ++j) {
        cr[j] = fmaR(s2, b[2 * j], cr[j]);
        ci[j] = fmaR(s2, b[2 * j + 1], ci[j]);
      }
    }
    sum = cdd_add(sum, cdd{dd_mul_d(dd{sr, 0.0}, w), dd_mul_d(dd{si, 0.0}, w)});
    mag = fmaR(sa, __builtin_fabs(w), mag);
  }
  block_sum(sum, mag, part, nw, bw, lane);
  if (bw != 0) return;
  if (gridDim.x > 1) {
    // The block that counts last sums the blocks' partials.  They are
    // written and read at device scope, past the XCDs' own L2s, so that the
    // count needs to wait for the block's own writes only (a device-wide
    // fence writes a whole L2 back).
    const int blocks = static_cast<int>(gridDim.x);
    if (lane < 5) {
      const double x = lane == 0   ? sum.re.hi
                       : lane == 1 ? sum.re.lo
                       : lane == 2 ? sum.im.hi
                       : lane == 3 ? sum.im.lo
                                   : mag;
      __hip_atomic_store(args.partials + 5 * static_cast<int>(blockIdx.x) + lane, x, __ATOMIC_RELAXED,
                         __HIP_MEMORY_SCOPE_AGENT);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __builtin_amdgcn_s_waitcnt(0);
    int old = 0;
    if (lane == 0) old = __hip_atomic_fetch_add(args.counter, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(old) != blocks - 1) return;
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    sum = cdd_zero();
    mag = 0.0;
    for (int q0 = lane; q0 < blocks; q0 += kWave) {
      double q[5];
#pragma unroll
      for (int i = 0; i < 5; ++i)
        q[i] = __hip_atomic_load(args.partials + 5 * q0 + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      sum = cdd_add(sum, cdd{{q[0], q[1]}, {q[2], q[3]}});
      mag += q[4];
    }
    sum = wave_reduce<0>(sum, lane);
    mag = wave_sum(mag, lane);
    if (lane == 0) __hip_atomic_store(args.counter, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  if (lane == 0) {
    const int e = -(n - 1);
    const double re_hi = ldexp(sum.re.hi, e), re_lo = ldexp(sum.re.lo, e);
    const double im_hi = ldexp(sum.im.hi, e), im_lo = ldexp(sum.im.lo, e);
    args.out[0] = re_hi + re_lo;
    args.out[1] = im_hi + im_lo;
    args.out[2] = re_hi;
    args.out[3] = re_lo;
    args.out[4] = im_hi;
    args.out[5] = im_lo;
    args.out[6] = ldexp(mag, e);
    __threadfence_system();
    __hip_atomic_store(args.done, args.seq, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

// The kernel copies its own length of the arguments: they begin alike for
// every width.
template <int W, OneKind KIND>
static hipError_t one_launch(const OneArgs &a, dim3 grid, dim3 block, hipStream_t stream) {
  using R = Rows<W, KIND>;
  static_assert(offsetof(R, b) == offsetof(OneRowsHost, b) && sizeof(Args<W, KIND>) <= sizeof(OneArgs));
  const void *given = KIND == kOneUnit ? static_cast<const void *>(&a.rows) : static_cast<const void *>(&a);
  void *p[] = {const_cast<void *>(given)};
  return hipLaunchKernel(reinterpret_cast<const void *>(perm_one_kernel<W, KIND>), grid, block, p, 0, stream);
}

template <int W>
static hipError_t one_launch(OneKind kind, const OneArgs &a, dim3 grid, dim3 block, hipStream_t stream) {
  if (kind == kOneUnit) return one_launch<W, kOneUnit>(a, grid, block, stream);
  if (kind == kOneOnes) return one_launch<W, kOneOnes>(a, grid, block, stream);
  return one_launch<W, kOneAny>(a, grid, block, stream);
}

#if PQP_ONE_FP32
hipError_t launch_one_f(int width, OneKind kind, const OneArgs &a, int blocks, int waves, hipStream_t stream) {
#else
hipError_t launch_one_d(int width, OneKind kind, const OneArgs &a, int blocks, int waves, hipStream_t stream) {
#endif
  const OneHead &h = a.rows.h;
  if (blocks < 1 || blocks > kOneMaxBlocks || waves < 1 || waves > kOneWaves || h.n < 1 || h.chunks < 1)
    return hipErrorInvalidValue;
  if (kind == kOneUnit && (width != h.n || 1 + h.lane_digits + h.inner + h.rest != width)) return hipErrorInvalidValue;
  const dim3 grid(blocks), block(kWave * waves);
  switch (width) {
#define X(W) \
  case W:    \
    return one_launch<W>(kind, a, grid, block, stream);
    X(1) X(2) X(3) X(4) X(5) X(6) X(7) X(8) X(9) X(10) X(11) X(12)
    X(13) X(14) X(15) X(16) X(17) X(18) X(19) X(20) X(21) X(22) X(23) X(24)
#undef X
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace pqp
