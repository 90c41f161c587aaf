// Routes kernel launches and occupancy queries to the translation unit that
// instantiates the requested (column-width bucket, arithmetic variant).
#include "perm_kernels.hpp"

namespace pqp {

#define PQP_CASE(k)                                        \
  case k:                                                  \
    if (l.fp32) return launch_fwd_b##k##_f(l);             \
    return l.comp ? launch_fwd_b##k##_d(l) : launch_fwd_b##k##_p(l);

hipError_t launch_fwd(int bucket, const FwdLaunch &l) {
  if (l.fp32 && !l.comp) return hipErrorInvalidValue;  // FP32 products always use dd
  switch (bucket) {
    PQP_CASE(0)
    PQP_CASE(1)
    PQP_CASE(2)
    PQP_CASE(3)
    PQP_CASE(4)
    PQP_CASE(5)
    PQP_CASE(6)
    PQP_CASE(7)
    default:
      return hipErrorInvalidValue;
  }
}
#undef PQP_CASE

#define PQP_CASE(k)                                                        \
  case k:                                                                  \
    if (fp32) return occupancy_fwd_b##k##_f(persistent, blocks);           \
    return comp ? occupancy_fwd_b##k##_d(persistent, blocks)               \
                : occupancy_fwd_b##k##_p(persistent, blocks);

hipError_t occupancy_fwd(int bucket, bool persistent, bool fp32, bool comp, int *blocks) {
  switch (bucket) {
    PQP_CASE(0)
    PQP_CASE(1)
    PQP_CASE(2)
    PQP_CASE(3)
    PQP_CASE(4)
    PQP_CASE(5)
    PQP_CASE(6)
    PQP_CASE(7)
    default:
      return hipErrorInvalidValue;
  }
}
#undef PQP_CASE

hipError_t launch_grad(int bucket, const LaunchArgs &a, int first_unit, int n_units,
                       hipStream_t stream) {
  switch (bucket) {
    case 0: return launch_grad_b0(a, first_unit, n_units, stream);
    case 1: return launch_grad_b1(a, first_unit, n_units, stream);
    case 2: return launch_grad_b2(a, first_unit, n_units, stream);
    case 3: return launch_grad_b3(a, first_unit, n_units, stream);
    case 4: return launch_grad_b4(a, first_unit, n_units, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_minors(int bucket, const LaunchArgs &a, int first_unit, int n_units,
                         hipStream_t stream) {
  switch (bucket) {
    case 0: return launch_minors_b0(a, first_unit, n_units, stream);
    case 1: return launch_minors_b1(a, first_unit, n_units, stream);
    case 2: return launch_minors_b2(a, first_unit, n_units, stream);
    case 3: return launch_minors_b3(a, first_unit, n_units, stream);
    case 4: return launch_minors_b4(a, first_unit, n_units, stream);
    case 5: return launch_minors_b5(a, first_unit, n_units, stream);
    case 6: return launch_minors_b6(a, first_unit, n_units, stream);
    case 7: return launch_minors_b7(a, first_unit, n_units, stream);
    case 8: return launch_minors_b8(a, first_unit, n_units, stream);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_tensor(const TensorArgs &a, hipStream_t s) {
  if (a.n >= 1 && a.n <= 12) return launch_tensor_p0(a, s);
  if (a.n >= 13 && a.n <= kTensorMaxN) return launch_tensor_p1(a, s);
  return hipErrorInvalidValue;
}

hipError_t launch_int(int width, const IntArgs &a, hipStream_t stream) {
  if (a.waves < 1) return hipSuccess;
  switch (width) {
    case 4: return launch_int_w4(a, stream);
    case 8: return launch_int_w8(a, stream);
    case 12: return launch_int_w12(a, stream);
    case 20: return launch_int_w20(a, stream);
    case 28: return launch_int_w28(a, stream);
    case 16: return launch_int_w16(a, stream);
    case 24: return launch_int_w24(a, stream);
    case 32: return launch_int_w32(a, stream);
    case 40: return launch_int_w40(a, stream);
    case 48: return launch_int_w48(a, stream);
    case 56: return launch_int_w56(a, stream);
    case 64: return launch_int_w64(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace pqp
