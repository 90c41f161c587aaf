// Kernel arguments of the probability tables (perm_table.hip): one
// interferometer and input occupation, many output occupations.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

namespace pqp {

constexpr int kTableMaxN = 16;      // particles (and columns) of a table on the fused kernel
constexpr int kTableMaxModes = 64;  // one lane per mode

struct TableArgs {
  const double *rows;   // modes x width complex: the columns of occupied input modes
  const int32_t *mult;  // their occupations (width)
  const uint8_t *outs;  // count x modes output occupations
  double *out;          // 2 doubles per output (amplitude) or 1 (probability)
  double in_norm;       // prod of the input occupations' factorials
  int64_t count;
  int32_t modes, n;
  int32_t prob;         // 1: probabilities
  // Inputs with more than one particle in a mode: the sweep over the input's
  // digits (table_states_kernel), taken for the outputs where it is cheaper.
  int32_t states, width;  // prod (rho_j + 1) after the prepend, and occupied columns
  int32_t first;        // the prepended column: the first of the smallest occupation
  double per_given;     // cost of a state of the sweep over the output's digits
  double2 *sums;        // modes x states: the row sums of every output mode
  double *weights;      // states: signed binomial weights
};

}  // namespace pqp
