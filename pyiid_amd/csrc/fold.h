// A distance's place in the folded grids of fq_grid.h and gradspread.hip.  Plain
// C++, so that the host can check where a place lies.
#pragma once

#include <cmath>

namespace pyiid {
namespace {

// From this t = r / h on a pair is left out: its weight, at most 1.2 2^48 / t units
// of the fixed point, rounds to zero, and u below would not hold t's place in the
// period (its error is of the order of t's last bit, 0.1 here).
constexpr double kFarthest = 1e15;

// Brings t, which is not negative, into [0, n_f / 2]: u; neg: the reflected half
// (sin changes sign).  False from kFarthest on, and for a t that is not a number.
__host__ __device__ inline bool fold(double t, double nf, double& u, bool& neg) {
  if (!(t < kFarthest)) return false;
  // (below 2^50 the product and the difference are exact, so u < nf; t / nf may
  // round up to a whole number, which leaves u just below 0)
  u = fmax(t - nf * floor(t / nf), 0.0);
  neg = u > 0.5 * nf;
  if (neg) u = nf - u;
  return true;
}

}  // namespace
}  // namespace pyiid
