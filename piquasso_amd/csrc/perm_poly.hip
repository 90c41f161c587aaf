// Coefficients of the permanent of a matrix polynomial on gfx950,
//
//   c_e = [x^e] perm(B_0 + sum_m x_m B_m),
//
// the quantity behind piquasso's lossy, partially distinguishable detection
// probabilities (B_0 = G o (I - T^dag T), B_m = G o t_m t_m^dag;
// piquasso/_simulators/passive/probabilities.py:244-384).  The reference
// keeps the polynomials on the box 0 <= a_m <= max e_m; here they are kept
// on the downward closure of the requested exponents (every monomial that
// divides one of them), which is all either path below ever reads and, for a
// table of all outputs with at most n photons, the simplex instead of the
// box ((n + M choose M) instead of (n + 1)^M coefficients).  The monomials
// are stored by total degree; each has "links" a - e_m to the degree below.
//
// Layer path (orders up to kPolyLayerMaxN; poly_layer_kernel): the permanent
// expanded row by row over the column subsets, f_i[e][S] for the subsets S
// of i columns.  It needs sum_i C(n, i) i times the monomials of degree <= i
// times M + 1 products where the subset sum below needs 2^n - 1 times those
// of every degree: 2.6e8 against 1.9e9 complex FMAs for 10 photons in 10
// modes, since the wide layers have few subsets.  It has no alternating sum.
// Bound by the reads of a layer through L2 and the Infinity Cache (31 MB for
// the largest) and, in the middle layers, by the FMAs.  Measured, 10 photons
// in 10 modes: ten launches, 0.32 ms, for 5.40 + 0.35 ms of the subset sum
// and its reduction; 9 photons in 8 modes: the whole call 235 us for 615 us,
// 6 in 7 104 for 103.
//
// Subset sum (larger orders, or coefficients or layers too large):
//
//   c_e = sum_S (-1)^(n - |S|) [x^e] prod_i ( c_i(S) + sum_m l_{m,i}(S) x_m ),
//   c_i(S) = sum_{j in S} B_0[i, j],   l_{m,i}(S) = sum_{j in S} B_m[i, j],
//
// Ryser's formula over the non-empty column subsets S, as the reference has
// it; the product is built row by row as a truncated polynomial.
// Multiplying by a factor updates degree D from degree D - 1 and itself, so
// the levels are updated from the top down with a workgroup barrier between
// levels, in place.
//
// One workgroup per group of K subsets at a time (groups strided over the
// grid).  The polynomial lives in LDS when it fits (kLds, K = 1; 256
// threads, several workgroups per CU), else in a per-workgroup global-memory
// slice (1024 threads, two workgroups per CU, so the slices and
// accumulators stay few; K = 2 subsets interleaved coefficient by
// coefficient, so a gather fetches 32 contiguous bytes for two lanes; each
// lane issues four links' loads and gathers before its first FMA waits).
// Each workgroup adds its subsets' signed coefficients into its own FP64
// accumulator; perm_poly_reduce_kernel then sums the workgroups'
// accumulators in double-double in workgroup order, so results do not
// depend on timing.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

#include "dd.hpp"
#include "perm_kernels.hpp"
#include "poly_types.hpp"
#include "sweep_common.hpp"

namespace pqp {

namespace {

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
  return make_double2(__builtin_fma(a.x, b.x, __builtin_fma(-a.y, b.y, c.x)),
                      __builtin_fma(a.x, b.y, __builtin_fma(a.y, b.x, c.y)));
}

template <bool kLds, int kThreads, int K>
__global__ __launch_bounds__(kThreads) void perm_poly_kernel(PolyArgs a) {
  extern __shared__ double2 smem[];
  const int n = a.n, M = a.M, L = a.L;
  const int tid = static_cast<int>(threadIdx.x);
  const int wg = static_cast<int>(blockIdx.x);
  const int per = n * (M + 1);  // row sums of one subset
  // LDS: row sums rs[(k * n + i) * (M + 1) + m] of the group's K subsets
  // (m = M: the constant term), then the polynomial when it is kept in LDS.
  // Coefficient a of subset k is poly[a * K + k]: the K subsets of a group
  // share each link and read K adjacent coefficients per gather.
  double2 *rs = smem;
  double2 *poly = kLds ? smem + K * per
                       : a.scratch + static_cast<int64_t>(wg) * a.n_mono * K;
  double2 *acc = a.acc + static_cast<int64_t>(wg) * a.n_out;
  const uint32_t n_subsets = (1u << n) - 1u;
  const uint32_t n_groups = (n_subsets + K - 1) / K;
  bool first = true;
  for (uint32_t g = static_cast<uint32_t>(wg); g < n_groups; g += static_cast<uint32_t>(a.n_wg)) {
    // the previous group's accumulation has read the polynomials
    __syncthreads();
    for (int t = tid; t < K * per; t += kThreads) {
      const int k = t / per, r = t - k * per;
      const int i = r / (M + 1), m = r - i * (M + 1);
      // a subset index past 2^n - 1 (the last group's tail) is computed like
      // the others and added with sign 0
      const uint32_t s = 1u + g * K + static_cast<uint32_t>(k);
      const double2 *B = (m == M) ? a.b0 : a.bm + static_cast<int64_t>(m) * n * n;
      double2 v = make_double2(0.0, 0.0);
      for (int j = 0; j < n; ++j)
        if (s >> j & 1u) {
          const double2 b = B[i * n + j];
          v.x += b.x;
          v.y += b.y;
        }
      rs[t] = v;
    }
    if (tid < K) poly[tid] = make_double2(1.0, 0.0);
    __syncthreads();
    for (int i = 0; i < n; ++i) {
      const int top = (i + 1 < L) ? i + 1 : L;
      for (int D = top; D >= 0; --D) {
        // degree i + 1 is new in this row: it has no old value to scale
        const bool fresh = (D == i + 1);
        const int lo = a.lvl_off[D], hi = a.lvl_off[D + 1];
        for (int t = tid; t < (hi - lo) * K; t += kThreads) {
          const int m_idx = lo + t / K, k = t % K;
          const double2 *r = rs + (k * n + i) * (M + 1);
          double2 v = fresh ? make_double2(0.0, 0.0) : cmul(r[M], poly[m_idx * K + k]);
          const int q1 = a.link_ptr[m_idx + 1];
          int q = a.link_ptr[m_idx];
          // four links at a time: their loads, then the four gathers, are
          // issued before the first FMA waits
          for (; q + 4 <= q1; q += 4) {
            const int e0 = a.links[q], e1 = a.links[q + 1], e2 = a.links[q + 2], e3 = a.links[q + 3];
            const double2 p0 = poly[(e0 >> 8) * K + k], p1 = poly[(e1 >> 8) * K + k];
            const double2 p2 = poly[(e2 >> 8) * K + k], p3 = poly[(e3 >> 8) * K + k];
            v = cfma(r[e0 & 0xff], p0, v);
            v = cfma(r[e1 & 0xff], p1, v);
            v = cfma(r[e2 & 0xff], p2, v);
            v = cfma(r[e3 & 0xff], p3, v);
          }
          for (; q < q1; ++q) {
            const int e = a.links[q];
            v = cfma(r[e & 0xff], poly[(e >> 8) * K + k], v);
          }
          poly[m_idx * K + k] = v;
        }
        __syncthreads();
      }
    }
    double sign[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      const uint32_t s = 1u + g * K + static_cast<uint32_t>(k);
      sign[k] = (s > n_subsets) ? 0.0 : (((n - __builtin_popcount(s)) & 1) ? -1.0 : 1.0);
    }
    for (int p = tid; p < a.n_out; p += kThreads) {
      const int64_t base = static_cast<int64_t>(a.out_mono[p]) * K;
      double2 v = make_double2(0.0, 0.0);
#pragma unroll
      for (int k = 0; k < K; ++k) {
        const double2 c = poly[base + k];
        v.x += sign[k] * c.x;
        v.y += sign[k] * c.y;
      }
      if (first) {
        acc[p] = v;
      } else {
        double2 w = acc[p];
        w.x += v.x;
        w.y += v.y;
        acc[p] = w;
      }
    }
    first = false;
  }
}

__global__ __launch_bounds__(256) void perm_poly_reduce_kernel(PolyArgs a) {
  const int p = static_cast<int>(blockIdx.x) * 256 + static_cast<int>(threadIdx.x);
  if (p >= a.n_out) return;
  dd re{0.0, 0.0}, im{0.0, 0.0};
  for (int w = 0; w < a.n_wg; ++w) {
    const double2 v = a.acc[static_cast<int64_t>(w) * a.n_out + p];
    re = dd_add_d(re, v.x);
    im = dd_add_d(im, v.y);
  }
  a.out[2 * p] = re.hi + re.lo;
  a.out[2 * p + 1] = im.hi + im.lo;
}

// acc[j] += f * (row of B for variable m, columns j0 .. j0 + JC - 1)
template <int JC, typename P>
__device__ __forceinline__ void layer_fma(double2 (&h)[JC], double2 f, P b, int last) {
#pragma unroll
  for (int j = 0; j < JC; ++j) {
    const int c = j <= last ? j : last;  // columns past n repeat the last one; never read
    const double br = b[2 * c], bi = b[2 * c + 1];
    h[j].x = __builtin_fma(br, f.x, h[j].x);
    h[j].y = __builtin_fma(br, f.y, h[j].y);
    h[j].x = __builtin_fma(-bi, f.y, h[j].x);
    h[j].y = __builtin_fma(bi, f.x, h[j].y);
  }
}

// One layer of the row expansion,
//
//   f_{i+1}[e][S] = sum_{j in S} ( B_0[i, j] f_i[e][S - j] + sum_m B_m[i, j] f_i[e - e_m][S - j] ),
//
// for every monomial e of degree <= i + 1 and every column subset S of
// i + 1 columns; f_i[e] holds the subsets side by side, so the reads and
// writes of a monomial are contiguous and only the subset step is a gather,
// within LDS.  A group of gs threads takes one monomial: each thread holds
// a source subset S', reads f_i[e - e_m][S'] once per link and adds it to
// the JC products h_j (coefficients B_m[i, j0 .. j0 + JC - 1]); the products
// go to LDS and each destination subset adds the h_j of its own columns.
// JC < n (the products of all n columns exceed kPolyLayerLds) repeats this
// over the columns in blocks.  WAVE: a group is whole waves, so the links
// and coefficients are scalar loads; narrower groups take the coefficients
// from LDS.  MISS: only the JC = n - i columns S' lacks are multiplied, each
// lane with its own columns' coefficients from LDS, for the last layers,
// where S' holds most columns and the products with those are thrown away:
// from 2 (n - i) <= n on (10 modes, 10 photons: layers 5 to 8 take 35, 64, 71
// and 73 us instead of 56, 128, 151 and 150).
template <int JC, bool WAVE, bool MISS>
__global__ __launch_bounds__(kPolyLayerThreads) void poly_layer_kernel(PolyLayerArgs a, int gs) {
  extern __shared__ double2 lds[];
  const int n = a.n, M = a.M, row = a.row, n_src = a.n_src, n_dst = a.n_dst;
  const int tid = static_cast<int>(threadIdx.x);
  const int groups = kPolyLayerThreads / gs;
  int g = tid / gs;
  if (WAVE) g = __builtin_amdgcn_readfirstlane(g);
  const int s0 = tid - g * gs;
  const int e = static_cast<int>(blockIdx.x) * groups + g;
  const bool live = e < a.n_dst_mono;
  double2 *h = lds + static_cast<int64_t>(g) * JC * n_src;
  double2 *lds_coef = lds + static_cast<int64_t>(groups) * JC * n_src;
  const double *coef = reinterpret_cast<const double *>(lds_coef);
  if (!WAVE || MISS) {
    // row `row` of every B_m, then of B_0
    for (int t = tid; t < (M + 1) * n; t += kPolyLayerThreads) {
      const int m = t / n, j = t - m * n;
      lds_coef[t] = (m == M) ? a.b0[row * n + j] : a.bm[(static_cast<int64_t>(m) * n + row) * n + j];
    }
    __syncthreads();
  }
  double2 acc[kPolyLayerAcc];
#pragma unroll
  for (int k = 0; k < kPolyLayerAcc; ++k) acc[k] = make_double2(0.0, 0.0);
  for (int j0 = 0; j0 < (MISS ? 1 : n); j0 += JC) {
    const int last = n - 1 - j0;  // the block's last column, if below JC
    if (live) {
      int q0, q1;
      if (WAVE) {
        const cptr<int32_t> lp = as_const<int32_t>(a.link_ptr);
        q0 = lp[e];
        q1 = lp[e + 1];
      } else {
        q0 = a.link_ptr[e];
        q1 = a.link_ptr[e + 1];
      }
      for (int s = s0; s < n_src; s += gs) {
        double2 p[JC];
#pragma unroll
        for (int j = 0; j < JC; ++j) p[j] = make_double2(0.0, 0.0);
        int col[MISS ? JC : 1];  // the columns S' lacks, ascending
        if constexpr (MISS) {
          int lacks = ~a.src_bits[s];
#pragma unroll
          for (int j = 0; j < JC; ++j) {
            col[j] = __builtin_ctz(lacks);
            lacks &= lacks - 1;
          }
        }
        auto value = [&](int mono) {
          return a.src ? a.src[static_cast<int64_t>(mono) * n_src + s] : make_double2(1.0, 0.0);
        };
        auto add = [&](int m, double2 f) {
          if constexpr (MISS) {
#pragma unroll
            for (int j = 0; j < JC; ++j) {
              const double2 b = lds_coef[m * n + col[j]];
              p[j] = cfma(b, f, p[j]);
            }
          } else if constexpr (WAVE) {
            const cptr<double> b = m == M ? as_const<double>(a.b0, int64_t(row * n + j0) * 16)
                                          : as_const<double>(a.bm, ((int64_t(m) * n + row) * n + j0) * 16);
            layer_fma<JC>(p, f, b, last);
          } else {
            layer_fma<JC>(p, f, coef + 2 * (m * n + j0), last);
          }
        };
        if (e < a.n_src_mono) add(M, value(e));
        if constexpr (WAVE) {
          const cptr<int32_t> links = as_const<int32_t>(a.links);
          int q = q0;
          for (; q + 4 <= q1; q += 4) {
            const int e0 = links[q], e1 = links[q + 1], e2 = links[q + 2], e3 = links[q + 3];
            const double2 f0 = value(e0 >> 8), f1 = value(e1 >> 8), f2 = value(e2 >> 8), f3 = value(e3 >> 8);
            add(e0 & 0xff, f0);
            add(e1 & 0xff, f1);
            add(e2 & 0xff, f2);
            add(e3 & 0xff, f3);
          }
          for (; q < q1; ++q) add(links[q] & 0xff, value(links[q] >> 8));
        } else {
          for (int q = q0; q < q1; ++q) {
            const int l = a.links[q];
            add(l & 0xff, value(l >> 8));
          }
        }
#pragma unroll
        for (int j = 0; j < JC; ++j) h[j * n_src + s] = p[j];
      }
    }
    __syncthreads();
    if (live) {
#pragma unroll
      for (int k = 0; k < kPolyLayerAcc; ++k) {
        const int S = s0 + k * gs;
        if (MISS && S < n_dst) {
          const int have = a.dst_bits[S];
          for (int j = 0; j < n; ++j) {
            const int r = a.sub[S * n + j];
            if (r >= 0) {
              // j is the t-th column S - j lacks: t columns below it are outside S
              const int t = __builtin_popcount(~have & ((1 << j) - 1));
              const double2 v = h[t * n_src + r];
              acc[k].x += v.x;
              acc[k].y += v.y;
            }
          }
        } else if (S < n_dst) {
          for (int j = 0; j < JC && j <= last; ++j) {
            const int r = a.sub[S * n + j0 + j];
            if (r >= 0) {
              const double2 v = h[j * n_src + r];
              acc[k].x += v.x;
              acc[k].y += v.y;
            }
          }
        }
      }
    }
    __syncthreads();
  }
  if (live) {
#pragma unroll
    for (int k = 0; k < kPolyLayerAcc; ++k) {
      const int S = s0 + k * gs;
      if (S < n_dst) a.dst[static_cast<int64_t>(e) * n_dst + S] = acc[k];
    }
  }
}

// The last row: S is all n columns, S - j (place n - 1 - j of the source
// layer) for every j, only the requested monomials.  One thread each.  The n
// products of a link are an FP64 run and the links' sums are folded in
// double-double, as the subset sum's workgroups are: bound by its gathers,
// the kernel takes the same 26 us for 184756 outputs (10 photons in 10
// modes) as in FP64 throughout, and the error of that table, the norm
// against 64 bits, is 1.4e-16 for 3.4e-16 (the subset sum's: 3.5e-16).
__global__ __launch_bounds__(kPolyLayerThreads) void poly_last_kernel(PolyLayerArgs a) {
  extern __shared__ double2 coef[];  // row n - 1 of every B_m, then of B_0
  const int n = a.n, M = a.M, row = a.row;
  for (int t = static_cast<int>(threadIdx.x); t < (M + 1) * n; t += kPolyLayerThreads) {
    const int m = t / n, j = t - m * n;
    coef[t] = (m == M) ? a.b0[row * n + j] : a.bm[(static_cast<int64_t>(m) * n + row) * n + j];
  }
  __syncthreads();
  const int p = static_cast<int>(blockIdx.x) * kPolyLayerThreads + static_cast<int>(threadIdx.x);
  if (p >= a.n_out) return;
  const int e = a.out_mono[p];
  cdd v = cdd_zero();
  auto add = [&](int m, int mono) {
    const double2 *c = coef + m * n;
    double2 t = c[0];  // n = 1: times the empty product
    if (a.src) {
      const double2 *f = a.src + static_cast<int64_t>(mono) * n;
      t = make_double2(0.0, 0.0);
      for (int j = 0; j < n; ++j) t = cfma(c[j], f[n - 1 - j], t);
    }
    const dd re = dd_two_sum(v.re.hi, t.x), im = dd_two_sum(v.im.hi, t.y);
    v.re = dd{re.hi, v.re.lo + re.lo};
    v.im = dd{im.hi, v.im.lo + im.lo};
  };
  if (e < a.n_src_mono) add(M, e);
  for (int q = a.link_ptr[e]; q < a.link_ptr[e + 1]; ++q) add(a.links[q] & 0xff, a.links[q] >> 8);
  a.out[2 * p] = v.re.hi + v.re.lo;
  a.out[2 * p + 1] = v.im.hi + v.im.lo;
}

}  // namespace

hipError_t launch_perm_poly(const PolyArgs &a, bool lds, int group, size_t lds_bytes,
                            hipStream_t stream) {
  if (lds)
    hipLaunchKernelGGL((perm_poly_kernel<true, kPolyThreads, 1>), dim3(a.n_wg), dim3(kPolyThreads),
                       lds_bytes, stream, a);
  else if (group == kPolyGroup)
    hipLaunchKernelGGL((perm_poly_kernel<false, kPolyThreadsGlobal, kPolyGroup>), dim3(a.n_wg),
                       dim3(kPolyThreadsGlobal), lds_bytes, stream, a);
  else
    hipLaunchKernelGGL((perm_poly_kernel<false, kPolyThreadsGlobal, 1>), dim3(a.n_wg),
                       dim3(kPolyThreadsGlobal), lds_bytes, stream, a);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(perm_poly_reduce_kernel, dim3((a.n_out + 255) / 256), dim3(256), 0, stream, a);
  return hipGetLastError();
}

template <int JC>
static void layer_launch(const PolyLayerArgs &a, int gs, bool miss, int blocks, size_t lds, hipStream_t stream) {
  if constexpr (JC <= kPolyLayerMaxN / 2) {
    if (miss) {
      if (gs >= kWave)
        hipLaunchKernelGGL((poly_layer_kernel<JC, true, true>), dim3(blocks), dim3(kPolyLayerThreads), lds,
                           stream, a, gs);
      else
        hipLaunchKernelGGL((poly_layer_kernel<JC, false, true>), dim3(blocks), dim3(kPolyLayerThreads), lds,
                           stream, a, gs);
      return;
    }
  }
  if (gs >= kWave)
    hipLaunchKernelGGL((poly_layer_kernel<JC, true, false>), dim3(blocks), dim3(kPolyLayerThreads), lds,
                       stream, a, gs);
  else
    hipLaunchKernelGGL((poly_layer_kernel<JC, false, false>), dim3(blocks), dim3(kPolyLayerThreads), lds,
                       stream, a, gs);
}

hipError_t launch_poly_layer(const PolyLayerArgs &a, hipStream_t stream) {
  const size_t row_bytes = static_cast<size_t>(a.M + 1) * a.n * sizeof(double2);
  if (a.row == a.n - 1) {
    hipLaunchKernelGGL(poly_last_kernel, dim3((a.n_out + kPolyLayerThreads - 1) / kPolyLayerThreads),
                       dim3(kPolyLayerThreads), row_bytes, stream, a);
    return hipGetLastError();
  }
  // threads per monomial: the subsets of both layers, up to the block
  const int wide = a.n_src > a.n_dst ? a.n_src : a.n_dst;
  int gs = 1;
  while (gs < wide && gs < kPolyLayerThreads) gs *= 2;
  const int groups = kPolyLayerThreads / gs;
  // columns per pass: all n where their products fit, else equal blocks
  const int fit = std::max(1, kPolyLayerLds / static_cast<int>(sizeof(double2) * groups * a.n_src));
  const int passes = (a.n + fit - 1) / fit;
  const int lacks = a.n - a.row;
  const bool miss = kPolyMissFactor * lacks <= a.n && lacks <= fit;
  const int jc = miss ? lacks : (a.n + passes - 1) / passes;
  const size_t lds =
      sizeof(double2) * static_cast<size_t>(groups) * jc * a.n_src + (gs >= kWave && !miss ? 0 : row_bytes);
  const int blocks = (a.n_dst_mono + groups - 1) / groups;
  switch (jc) {
#define PQP_LAYER_CASE(JC)                    \
  case JC:                                    \
    layer_launch<JC>(a, gs, miss, blocks, lds, stream); \
    break;
    PQP_LAYER_CASE(1)
    PQP_LAYER_CASE(2)
    PQP_LAYER_CASE(3)
    PQP_LAYER_CASE(4)
    PQP_LAYER_CASE(5)
    PQP_LAYER_CASE(6)
    PQP_LAYER_CASE(7)
    PQP_LAYER_CASE(8)
    PQP_LAYER_CASE(9)
    PQP_LAYER_CASE(10)
    PQP_LAYER_CASE(11)
    PQP_LAYER_CASE(12)
#undef PQP_LAYER_CASE
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace pqp
