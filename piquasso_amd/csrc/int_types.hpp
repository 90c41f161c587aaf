// Kernel arguments of exact integer permanents (perm_int.hip).
#pragma once

#include <cstdint>

namespace pqp {

constexpr int kIntMaxPrimes = 8;  // moduli at most

struct IntArgs {
  const double *rows;    // the occupied rows, `modes` x width, then the prepended row (padding columns 1)
  const uint8_t *occ;    // modes: row multiplicities, n particles
  const double *mod;     // the primes, their reciprocals, 2^-(n-1) modulo each (kIntMaxPrimes of each)
  double *partials;      // n_primes x waves residues
  double *out;           // n_primes residues of the permanent
  int32_t modes, n;
  int32_t n_primes;
  int32_t group;         // columns multiplied exactly: 12, 8, 4, 2 or 1
  int32_t waves;
  int32_t k_max;         // inner digits at most
  uint64_t *done;
  uint64_t seq;
};

}  // namespace pqp
