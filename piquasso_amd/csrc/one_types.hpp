// Kernel arguments of single permanents without tables (perm_one.hip),
// shared with capi.cpp and noalloc.hip.
#pragma once

#include <cstddef>
#include <cstdint>

namespace pqp {

constexpr int kOneMaxWidth = 24;         // distinct columns
constexpr int kOneMaxRows = 25;          // the row the sums start from and the digits' rows (2^24 terms)
constexpr int kOneFew = 12;              // rows and columns of the kernels for few of them
constexpr int kOneMaxStates = 64;        // inner states of a lane: one FP64 run (kDdFold terms)
constexpr int kOneLaneDigits = 6;        // binary digits that the 64 lanes of a wave differ in
constexpr int kOneMaxMult = 64;          // largest multiplicity
constexpr int kOneMaxBlocks = 512;

constexpr int kOneWaves = 4;             // waves of a block at most: one per SIMD

// Inner state v of a mixed-radix sweep: its signed weight, and the row that
// is added, times factor, after it.
struct OneStep {
  double coef;
  int32_t factor, row;
};

// What only bunched rows or columns read.
struct OneTables {
  uint32_t over[kOneMaxMult];  // over[r - 2], r = 2 .. cmax: the columns of multiplicity >= r
  OneStep step[kOneMaxStates];
};

struct alignas(64) OneHead {
  double *partials;     // 5 doubles a block
  int *counter;         // finished blocks; 0 between launches
  double *out;          // 2 doubles, 4 (double-double), 1 (term magnitudes)
  uint64_t *done;       // receives seq
  uint64_t seq;
  int32_t n;            // particles
  int32_t lane_digits, lanes;  // their states
  int32_t inner, rest;  // inner digits, and the others
  int32_t S, chunks;    // states of the inner digits and of the others
  int32_t binary;       // the inner digits are binary: `step` is not used
  int32_t cmax;         // largest column multiplicity
  int32_t lane_rho[kOneLaneDigits];  // largest values of the lanes' digits
  int32_t rho[kOneMaxRows];          // and of the inner and the other ones
};

// The rows are in the order of their digits: the lanes' digits (six binary
// ones, or as many states in at most 64 as the digits allow), the prepended
// row, the inner digits, then the others.
template <size_t BYTES>
struct OneRows {
  OneHead h;
  char b[BYTES];
};

// The arguments are written for every launch (about 0.1 us a KB), so a
// kernel takes as many bytes of the host's OneArgs as its widths need: W
// columns of kOneMaxRows rows, or, where rows and columns hold one particle
// each and are few, of kOneFew rows without the tables, from `rows` on.
// 12 particles: 11 KB 14.1 us a call, 6 KB 13.7, 2.5 KB 13.5.
template <size_t BYTES>
struct OneArgsOf {
  OneTables tables;
  OneRows<BYTES> rows;
};
constexpr size_t one_row_bytes(int rows, int width, size_t real) {
  return 2 * static_cast<size_t>(rows) * static_cast<size_t>(width) * real;
}
using OneArgs = OneArgsOf<one_row_bytes(kOneMaxRows, kOneMaxWidth, sizeof(double))>;

}  // namespace pqp
