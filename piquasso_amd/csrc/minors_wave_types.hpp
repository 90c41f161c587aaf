// Kernel arguments of the column minors planned on the device
// (perm_minors_wave.hip).
#pragma once

#include <cstdint>

namespace pqp {

constexpr int kMinorsWaveMaxCols = 24;   // columns (one kernel per width)
constexpr int kMinorsWaveMaxModes = 64;  // rows: one lane each

// Items x waves: item i's waves share its top states; each leaves one
// double-double partial per real component, 2 width of them.
struct MinorsWaveArgs {
  const double *rows;    // per item (item_stride doubles apart): modes x ld complex
  const uint8_t *occ;    // items x modes: row multiplicities, width - 1 particles each
  const int32_t *units;  // waves each item needs (null: all that are launched)
  double *partials;      // [item][wave][component] (hi, lo)
  double *out;           // minors_sum: 2 doubles per column
  int64_t item_stride;
  int32_t ld, modes;
  int32_t waves;         // per item
  int32_t k_max;         // inner digits at most
  // the block that ends last publishes seq (see LaunchArgs)
  int *last_counter;
  uint64_t *done;
  uint64_t seq;
};

// Clifford & Clifford sampling, one photon a step (sample_step_kernel).
struct SampleArgs {
  const double *u_t;      // the interferometer, modes x modes complex, row-major
  const uint8_t *cols;    // shots x photons: the input mode of each photon, in the order they join
  const int32_t *steps;   // shots: photons each shot places
  const double *draws;    // photons x shots: uniform numbers
  double *v;              // shots x modes x photons complex: the interferometer's columns in joining order
  uint8_t *occ;           // shots x modes: output so far
  int32_t *units;         // shots: waves of the next step
  const double *partials; // as in MinorsWaveArgs
  int32_t *failed;        // set when a distribution has no finite positive sum
  int32_t shots, modes, photons;
  int32_t step;           // photons placed before this step
  int32_t waves;          // per item, of this step's minors
  int32_t next_waves, next_k_max;  // of the next step's
};

}  // namespace pqp
