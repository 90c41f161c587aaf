// Kernel arguments of single permanents without tables (perm_one.hip),
// shared with capi.cpp and noalloc.hip.
#pragma once

#include <cstddef>
#include <cstdint>

namespace pqp {

constexpr int kOneMaxWidth = 24;         // distinct columns
constexpr int kOneMaxRows = 25;          // the row the sums start from and the digits' rows (2^24 terms)
constexpr int kOneMaxStates = 64;        // inner states of a lane: one FP64 run (kDdFold terms)
constexpr int kOneLaneDigits = 6;        // digits that the lanes of a wave differ in
constexpr int kOneLaneStates = 4096;     // and their states: 64 chunks of lanes
constexpr int kOneMaxBlocks = 512;
constexpr int kOneWaves = 8;             // waves of a block at most

// What the kernel is compiled for.
enum OneKind {
  kOneUnit,  // one particle in each row and column: binary digits, as many rows as columns
  kOneOnes,  // one particle in each column
  kOneAny,
};

// Inner state v of a mixed-radix sweep: its signed weight, and the row that
// is added, times factor, after it.
struct OneStep {
  double coef;
  int32_t factor, row;
};

// A digit of values 0 .. rho: 1 / (rho + 1), and its binomials C(rho, g) for g
// <= rho / 2, a byte each where the largest fits one (rho <= 10), else 0.
struct OneDigit {
  double inv;
  uint64_t choose;
  int32_t rho, pad;
};

// What a kOneUnit kernel has no use for.
struct OneTables {
  uint32_t more[kOneMaxWidth / 4];  // a byte a column: its multiplicity less one
  OneDigit lane[kOneLaneDigits];    // the lanes' digits
  OneDigit digit[kOneMaxRows];      // the inner and the other ones
  double lane_inv;      // 1 / lane_chunks
  int32_t lane_chunks;  // sets of 64 of the lanes' states
  int32_t lane_binary;  // the lanes' digits are binary
  int32_t binary;       // the inner digits are: `step` is not used
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
  int32_t S, chunks;    // states of the inner digits; of the others, times the lane chunks
};

// The rows are in the order of their digits: the lanes', the prepended row,
// the inner digits, then the others.
template <size_t BYTES>
struct OneRows {
  OneHead h;
  char b[BYTES];
};

// The arguments are written for every launch (about 0.1 us a KB), so a
// kernel takes as many bytes of the host's OneArgs as it reads: W columns of
// kOneMaxRows rows, or, of kind kOneUnit, of W rows without the tables, from
// `rows` on.  12 particles: 11 KB 14.1 us a call, 6 KB 13.7, 2.5 KB 13.5 (12.5
// with the kernel of this kind).
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
