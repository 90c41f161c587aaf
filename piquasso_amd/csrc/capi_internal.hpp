// Helpers of the C ABI shared between capi.cpp and the translation units
// that define further entry points (noalloc.hip): the thread-local error
// message, the device check, and the planning options of single-permanent
// calls, so that every single-permanent entry plans the same way.
#pragma once

#include <cstdint>
#include <string>

#include "one_types.hpp"
#include "plan.hpp"
#include "pqp_types.hpp"

namespace pqp {

// Record `msg` as the calling thread's pqp_last_error() and return `code`.
int capi_fail(int code, const std::string &msg);

// PQP_OK when a HIP device is usable, else PQP_ERR_DEVICE with the message.
int capi_require_device();

// Gray terms of one permanent, prod (rho_i + 1) after the prepend (the
// first minimal non-zero row loses one), as the planner counts them;
// `in.rows` must be valid (negative entries count as 0).
double gray_terms(const PermInput &in);

// Planned single permanents of at most this many Gray terms are planned for
// at most kSingleFewUnits waves, kSingleFewestUnits up to kSingleFewestTerms
// terms: each lane's start state costs about as much as a few Gray steps, so
// fewer, longer units finish sooner.
constexpr double kSingleFewTerms = 16384.0;
constexpr int kSingleFewUnits = 8;
constexpr double kSingleFewestTerms = 2048.0;
constexpr int kSingleFewestUnits = 4;

// Planning options of a single-permanent call of `in` with these
// PQP_FLAG_* flags: about 1.4 sqrt(T) waves, capped for few terms and per
// compute unit otherwise; one-wave permanents write their result from the
// sweep kernel.
PlanOptions single_plan_options(uint32_t flags, const PermInput &in);

// A single permanent without tables (perm_one.hip).
struct OnePlan {
  PermInput in;       // transposed where that sweep is clearly cheaper
  int n, width;       // particles, distinct columns
  OneKind kind;
  bool fp32;
  int blocks, waves;  // waves of a block
  double terms;       // Gray terms
};

// Whether a single-permanent call runs on perm_one.hip: 1 <= n <= 64
// particles, at most kOneMaxWidth distinct columns and kOneMaxTerms Gray
// terms, and not the plain baseline.  Arguments that are not valid are left
// to the planner.
bool one_plan(const PermInput &in, uint32_t flags, OnePlan &p);

// The launch's arguments but for its buffers; fits the blocks to the digits.
void one_fill(OnePlan &p, OneArgs &a);

// Bound on |computed - perm| of a floating-point sweep from its term
// magnitudes m = sum_t |term_t| / 2^(n-1) (as the kernels accumulate them):
// 4 (n + 2) u m, u the unit roundoff of the row sums and products (2^-53,
// or 2^-24 with FP32 products), plus the rounding of the double-double
// value (re, im) to FP64.  NaN when m is NaN (the plain kernel keeps none).
double sweep_error_bound(int n, bool fp32, double m, double re, double im);

// The calling thread's pqp_last_error_bound().
void capi_set_last_bound(double bound);

}  // namespace pqp
