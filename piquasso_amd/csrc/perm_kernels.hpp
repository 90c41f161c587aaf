// Host-side launch interface of the permanent kernels.  The kernel
// templates are instantiated once per column-width bucket and arithmetic
// variant (perm_fwd.hip is compiled once per pair); launch_fwd() in
// dispatch.cpp routes a launch to the right translation unit.
#pragma once

#include <hip/hip_runtime.h>

#include "int_types.hpp"
#include "pqp_types.hpp"
#include "tensor_types.hpp"
#include "poly_types.hpp"
#include "table_types.hpp"
#include "minors_wave_types.hpp"
#include "one_types.hpp"

namespace pqp {

struct FwdLaunch {
  LaunchArgs args;
  int first_unit = 0;   // first unit of this bucket's range in args.units
  int n_units = 0;      // units in the range
  int head_slot = 0;    // queue head used by a persistent launch
  int grid = 0;         // persistent launches: number of blocks
  bool persistent = true;
  bool fp32 = false;    // FP32 row sums and products
  bool comp = true;     // double-double accumulation (false: plain FP64)
  hipStream_t stream = nullptr;
};

// Per (bucket, variant) entry points, defined in perm_fwd.hip builds;
// variant suffix d = FP64 + dd, p = plain FP64, f = FP32 products + dd.
#define PQP_DECLARE(k, v)                                         \
  hipError_t launch_fwd_b##k##_##v(const FwdLaunch &l);           \
  hipError_t occupancy_fwd_b##k##_##v(bool persistent, int *blocks_per_cu);
#define PQP_DECLARE_BUCKET(k) PQP_DECLARE(k, d) PQP_DECLARE(k, p) PQP_DECLARE(k, f)
PQP_DECLARE_BUCKET(0)
PQP_DECLARE_BUCKET(1)
PQP_DECLARE_BUCKET(2)
PQP_DECLARE_BUCKET(3)
PQP_DECLARE_BUCKET(4)
PQP_DECLARE_BUCKET(5)
PQP_DECLARE_BUCKET(6)
PQP_DECLARE_BUCKET(7)
#undef PQP_DECLARE_BUCKET
#undef PQP_DECLARE

// Single permanents planned by their own waves (perm_one.hip): one launch
// of `blocks` blocks of `waves` waves for a permanent of `width` distinct columns (all of
// multiplicity 1: ones).
hipError_t launch_one_d(int width, OneKind kind, const OneArgs &a, int blocks, int waves, hipStream_t stream);
hipError_t launch_one_f(int width, OneKind kind, const OneArgs &a, int blocks, int waves, hipStream_t stream);

constexpr int kBuckets = 8;        // forward kernel width buckets
constexpr int kMinorBuckets = 9;   // column-minor kernel buckets
constexpr int kMaxRanges = 9;      // concurrent launches of one plan (one per bucket)

// Column-minor kernels (perm_minors.hip), buckets 0..3 (widths up to 32).
hipError_t launch_minors_b0(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b1(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b2(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b3(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b4(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b5(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b6(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b7(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors_b8(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_minors(int bucket, const LaunchArgs &a, int first_unit, int n_units,
                         hipStream_t stream);
hipError_t launch_minors_finalize(const LaunchArgs &a, int n_items, int max_units,
                                  hipStream_t stream);

// Column minors planned on the device (perm_minors_wave.hip): one launch for
// the items of one width, the sum of a lone item's partials, and the two
// kernels of the sampler around them.
hipError_t launch_minors_wave(int width, const MinorsWaveArgs &a, int items, hipStream_t stream);
hipError_t launch_minors_sum(int width, const MinorsWaveArgs &a, hipStream_t stream);
hipError_t launch_sample_columns(const SampleArgs &a, hipStream_t stream);
hipError_t launch_sample_step(const SampleArgs &a, hipStream_t stream);

// Gradient kernels (perm_grad.hip), unit column multiplicities: buckets for
// widths 1-8, 9-16, 17-19, 20, 21-32.
constexpr int kGradBuckets = 5;
hipError_t launch_grad_b0(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_grad_b1(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_grad_b2(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_grad_b3(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_grad_b4(const LaunchArgs &a, int first_unit, int n_units, hipStream_t s);
hipError_t launch_grad(int bucket, const LaunchArgs &a, int first_unit, int n_units,
                       hipStream_t stream);
// max_values: the largest 1 + rows of B x m_c over the items (the
// permanent and its gradient entries)
hipError_t launch_grad_finalize(const LaunchArgs &a, int n_items, int max_values,
                                hipStream_t stream);

// Exact integer permanents (perm_int.hip): the sweep of one padded width,
// then the sum of its waves' residues.
#define PQP_DECLARE_INT(w) hipError_t launch_int_w##w(const IntArgs &a, hipStream_t stream);
PQP_DECLARE_INT(4)
PQP_DECLARE_INT(8)
PQP_DECLARE_INT(12)
PQP_DECLARE_INT(16)
PQP_DECLARE_INT(20)
PQP_DECLARE_INT(24)
PQP_DECLARE_INT(28)
PQP_DECLARE_INT(32)
PQP_DECLARE_INT(40)
PQP_DECLARE_INT(48)
PQP_DECLARE_INT(56)
PQP_DECLARE_INT(64)
#undef PQP_DECLARE_INT
hipError_t launch_int(int width, const IntArgs &a, hipStream_t stream);
hipError_t launch_int_sum(const IntArgs &a, hipStream_t stream);

// Tensor permanents (tensor_perm.hip) of items of one order: the matrices
// of a table, the rows R_eps of every sign vector (of n such passes), the
// sweep, and the items' sums.
hipError_t launch_tensor_gather(const TensorArgs &a, hipStream_t stream);
hipError_t launch_tensor_signs(const TensorArgs *passes, int n, hipStream_t stream);
hipError_t launch_tensor_p0(const TensorArgs &a, hipStream_t stream);
hipError_t launch_tensor_p1(const TensorArgs &a, hipStream_t stream);
hipError_t launch_tensor(const TensorArgs &a, hipStream_t stream);
hipError_t launch_tensor_finalize(const TensorArgs &a, hipStream_t stream);

// Probability tables (perm_table.hip): `width` occupied input modes, `ones`:
// one particle in each.
hipError_t launch_table_states(const TableArgs &a, hipStream_t stream);
hipError_t launch_table(int width, bool ones, const TableArgs &a, hipStream_t stream);

// One row of the layer path of a matrix-polynomial permanent
// (perm_poly.hip): layer a.row + 1 from layer a.row, or for the last row the
// requested coefficients.
hipError_t launch_poly_layer(const PolyLayerArgs &a, hipStream_t stream);

// Matrix-polynomial permanent (perm_poly.hip): the subset sweep over
// a.n_wg workgroups (the polynomial in LDS when `lds`; else in global memory
// with `group` (1 or kPolyGroup) subsets interleaved; dynamic LDS of
// lds_bytes), then the reduction of the workgroups' accumulators.
hipError_t launch_perm_poly(const PolyArgs &a, bool lds, int group, size_t lds_bytes,
                            hipStream_t stream);

hipError_t launch_fwd(int bucket, const FwdLaunch &l);
hipError_t occupancy_fwd(int bucket, bool persistent, bool fp32, bool comp, int *blocks_per_cu);
// Finalize items [item0, item0 + n_items); block 0 also rewinds n_heads
// queue heads (pass 0 when a persistent launch may still be running).
hipError_t launch_finalize(bool comp, const LaunchArgs &a, int item0, int n_items,
                           int n_heads, int max_units, hipStream_t stream);

}  // namespace pqp
