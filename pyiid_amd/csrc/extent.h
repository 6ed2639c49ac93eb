// How far the distances within the chains of a batch reach.  Plain C++.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstdint>
#include <limits>
#include <vector>

namespace pyiid {

// A bound of the distances within every chain [off[b], off[b + 1]) of the positions
// p (x, y, z at p[stride a]): the diagonal of its box or the diameter of the sphere
// about the box's middle, whichever is less.  Infinite where a position of a chain
// is not finite: then nothing may be left out on account of it.
template <typename T>
double chain_extent(const T* p, int stride, const std::vector<int64_t>& off) {
  double r_max = 0.0;
  for (size_t b = 0; b + 1 < off.size(); ++b) {
    if (off[b + 1] - off[b] < 2) continue;
    double lo[3], hi[3], mid[3];
    bool finite = true;
    for (int k = 0; k < 3; ++k) lo[k] = hi[k] = p[off[b] * stride + k];
    for (int64_t a = off[b]; a < off[b + 1]; ++a)
      for (int k = 0; k < 3; ++k) {
        const double x = p[a * stride + k];
        finite = finite && std::fabs(x) < 1e150;
        lo[k] = std::min(lo[k], x);
        hi[k] = std::max(hi[k], x);
      }
    if (!finite) return std::numeric_limits<double>::infinity();
    double diag = 0.0, rad = 0.0;
    for (int k = 0; k < 3; ++k) {
      mid[k] = 0.5 * (lo[k] + hi[k]);
      diag += (hi[k] - lo[k]) * (hi[k] - lo[k]);
    }
    for (int64_t a = off[b]; a < off[b + 1]; ++a) {
      double d = 0.0;
      for (int k = 0; k < 3; ++k) d += (p[a * stride + k] - mid[k]) * (p[a * stride + k] - mid[k]);
      rad = std::max(rad, d);
    }
    r_max = std::max(r_max, std::min(std::sqrt(diag), 2.0 * std::sqrt(rad)));
  }
  return r_max;
}

}  // namespace pyiid
