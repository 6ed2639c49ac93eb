"""CPU checks of the spreading kernels' constants and of the code that they
share with the host."""
import os
import re
import subprocess

import numpy as np

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "pyiid_amd", "csrc")


def constants(header, name):
    text = open(os.path.join(CSRC, header)).read()
    body = re.search(r"constexpr float %s\[\d\]\[\d\] = \{(.*?)\n\};" % name, text, re.S).group(1)
    rows = re.findall(r"\{([^{}]*)\}", body)
    return np.array([[np.float32(v.strip().rstrip("f")) for v in r.split(",")] for r in rows])


def test_window_has_no_common_factor():
    """The F grid's window, averaged over a pair's place between the grid points,
    against its transform phihat: what is left multiplies F as a whole, where the
    errors at single places average out.  v_rcp_f32, which the weight 1/r comes
    from, is 6.8e-9 short on average.  Allowed: 4e-9, the least squares residue
    of the window (3.6e-9 r.m.s.)."""
    v = constants("fq_grid.h", "kFqVal").astype(np.float64)
    assert v.shape == (3, 6)
    y = (np.arange(4000) + 0.5) / 4000 - 0.5
    powers = y[None] ** np.arange(6)[:, None]
    mirror = (-y)[None] ** np.arange(6)[:, None]
    taps = np.concatenate([v @ powers, (v @ mirror)[::-1]])
    beta = 15.160
    for q in np.linspace(0.0, np.pi / 6, 33):
        a = np.sqrt(beta ** 2 - 9.0 * q * q)
        phihat = np.sinh(a) / a / (np.sinh(beta) / beta)
        z = (taps * np.exp(1j * q * (np.arange(6)[:, None] - 2.5 - y[None]))).sum(0) / phihat
        assert abs(z.mean() * (1.0 - 6.755e-9) - 1.0) < 4e-9, q
        assert np.sqrt((np.abs(z - 1.0) ** 2).mean()) < 1.2e-8, q


FOLD = r"""
#define __host__
#define __device__
#include "fold.h"
#include <cstdint>
#include <initializer_list>
#include <cstdio>
using namespace pyiid;
int main() {
  uint64_t x = 88172645463325252ull, seen = 0, left_out = 0;
  for (int nf : {12, 13, 90, 1126, 3000, 13500, 40800})
    for (int k = 0; k < 400000; ++k) {
      x ^= x << 13; x ^= x >> 7; x ^= x << 17;
      // magnitudes 1 to 1e300, every eighth next to a multiple of the period
      double t = std::pow(10.0, (x >> 11) * 0x1p-53 * (k % 3 ? 300.0 : 20.0));
      if (k % 8 == 0) t = std::nextafter(std::floor(t / nf) * nf, k % 16 ? 0.0 : 1e301);
      double u = -1.0;
      bool neg;
      if (!fold(t, nf, u, neg)) {
        if (t < 1e15) return std::printf("left out: %.17g\n", t), 1;
        ++left_out;
        continue;
      }
      if (!(t < 1e15) || !(u >= 0.0 && u <= 0.5 * nf)) return std::printf("%d %.17g -> %.17g\n", nf, t, u), 1;
      // the place in the period, against the remainder (which is exact)
      const double r = std::remainder(t, nf);
      if (std::fabs(std::fabs(r) - u) > 4e-16 * t) return std::printf("%d %.17g -> %.17g not %.17g\n", nf, t, u, r), 1;
      if (u > 1e-9 * t && u < 0.5 * nf - 1e-9 * t && neg != (r < 0.0)) return std::printf("sign %d %.17g\n", nf, t), 1;
      ++seen;
    }
  double u;
  bool neg;
  if (fold(INFINITY, 90, u, neg) || fold(NAN, 90, u, neg)) return 1;
  return seen > 100000 && left_out > 100000 ? 0 : 2;
}
"""


def test_folded_place_lies_in_the_grid(tmp_path):
    """Distances of any finite size, also just beside a multiple of the period:
    the folded place lies in [0, n_f / 2], which the grids cover, or the pair is
    left out (from 1e15 on)."""
    src, exe = tmp_path / "fold.cpp", tmp_path / "fold"
    src.write_text(FOLD)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout


EXTENT = r"""
#include "extent.h"
#include <cstdio>
#include <limits>
using namespace pyiid;
int main() {
  const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
  const std::vector<int64_t> one{0, 4}, two{0, 1, 5};  // two: the first chain has no distance
  for (double bad : {nan, inf, -inf, 1e200})
    for (int a = 0; a < 4; ++a)
      for (int k = 0; k < 3; ++k)
        for (int both = 0; both < 2; ++both) {
          double p[5][4] = {{0, 0, 0, 0}, {3, 4, 0, 0}, {1, 2, 2, 0}, {0, 1, 0, 0}, {1, 1, 1, 0}};
          p[a][k] = bad;
          if (both) p[(a + 1) % 4][k] = -bad;
          if (!(chain_extent(&p[0][0], 4, one) == inf)) return std::printf("%g at %d %d\n", bad, a, k), 1;
          float f[5][3];
          for (int i = 0; i < 5; ++i)
            for (int c = 0; c < 3; ++c) f[i][c] = static_cast<float>(p[i][c]);
          if (bad != 1e200 && !(chain_extent(&f[0][0], 3, one) == inf)) return std::printf("float %g\n", bad), 1;
          const double e = chain_extent(&p[0][0], 4, two);  // the atom alone counts for nothing
          if (!both && a == 0 && !(e > 0.0 && e < 10.0)) return std::printf("alone %g\n", e), 1;
        }
  const double q[4][3] = {{0, 0, 0}, {3, 4, 0}, {1, 2, 2}, {0, 1, 0}};
  const double e = chain_extent(&q[0][0], 3, one);
  return e >= 5.0 && e < 5.4 ? 0 : 1;
}
"""


def test_extent_of_positions_that_are_not_finite(tmp_path):
    """The bound of the distances is infinite whichever atom's position is not
    finite (the first one's, or two of opposite sign, too), so that no pair is left
    out on account of it; a chain of one atom has no distances."""
    src, exe = tmp_path / "extent.cpp", tmp_path / "extent"
    src.write_text(EXTENT)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
