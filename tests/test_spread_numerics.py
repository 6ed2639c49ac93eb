"""CPU checks of the spreading kernels' constants and of the code that they
share with the host."""
import os
import re
import shutil
import subprocess

import numpy as np
import pytest

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


ROUTE = r"""
#include "route.h"
#include <cstdio>
using namespace pyiid;
int main() {
  char kind;
  double chains, n, elements, nq, dq, cells;
  while (std::scanf(" %c %lf %lf %lf %lf %lf %lf", &kind, &chains, &n, &elements, &nq, &dq, &cells) == 7) {
    BatchSize s;
    s.chains = static_cast<int64_t>(chains);
    for (int b = 0; b < s.chains; ++b) s.add(static_cast<int64_t>(n));
    const int e = static_cast<int>(elements), q = static_cast<int>(nq);
    const int64_t pairs = e * (e + 1) / 2;
    std::printf("%d\n", kind == 'f'   ? spread_fq_pays(s, e, pairs, q, dq, false)
                        : kind == 'g' ? spread_grad_pays(static_cast<int64_t>(n), e, q, dq)
                                      : force_table_pays(s, e, pairs, q, cells));
  }
}
"""

# kind (F, gradient, forces), chains, atoms, elements, bins, largest Q, cells, and the
# time of the recurrence and of the spreading kernel or table (us, MI355X; for the
# forces without F)
MEASURED = [
    ("f", 1, 55, 1, 250, 25.0, 0, 45, 10), ("f", 1, 7000, 1, 3400, 25.0, 0, 5126, 88),
    ("f", 1, 7000, 1, 100, 1.0, 0, 484, 214), ("f", 1, 7000, 1, 1, 0.1, 0, 450, 600),
    ("f", 1, 4000, 3, 600, 25.0, 0, 403, 66), ("f", 1, 600, 8, 250, 25.0, 0, 62, 30),
    ("f", 1, 600, 32, 250, 25.0, 0, 45, 102), ("f", 1, 60, 16, 250, 25.0, 0, 19, 33),
    ("f", 1, 4000, 16, 250, 25.0, 0, 332, 72), ("f", 1, 300, 128, 250, 25.0, 0, 240, 1127),
    ("f", 1, 7000, 64, 250, 25.0, 0, 627, 394), ("f", 1, 7000, 128, 250, 25.0, 0, 764, 1344),
    ("f", 64, 300, 3, 330, 25.0, 0, 393, 117), ("f", 64, 40, 3, 330, 25.0, 0, 32, 69),
    ("f", 256, 80, 3, 330, 25.0, 0, 93, 223), ("f", 1024, 150, 1, 330, 25.0, 0, 509, 202),
    ("f", 1024, 40, 1, 330, 25.0, 0, 91, 150), ("f", 256, 600, 6, 330, 25.0, 0, 1292, 970),
    ("g", 1, 300, 1, 64, 1.0, 0, 45, 39), ("g", 1, 300, 1, 4, 0.4, 0, 44, 83),
    ("g", 1, 600, 1, 64, 1.0, 0, 45, 56), ("g", 1, 600, 1, 16, 25.0, 0, 42, 33),
    ("g", 1, 1000, 1, 32, 8.0, 0, 47, 66), ("g", 1, 1000, 1, 100, 25.0, 0, 56, 46),
    ("g", 1, 2000, 1, 100, 4.0, 0, 170, 205), ("g", 1, 2000, 1, 100, 12.0, 0, 169, 111),
    ("g", 1, 7000, 1, 16, 2.0, 0, 1311, 1573), ("g", 1, 7000, 1, 64, 8.0, 0, 1373, 1015),
    ("g", 1, 7000, 1, 200, 1.0, 0, 2168, 1740), ("g", 1, 15000, 1, 8, 25.0, 0, 4975, 5878),
    ("g", 1, 300, 16, 250, 25.0, 0, 42, 143), ("g", 1, 2000, 8, 250, 25.0, 0, 297, 163),
    ("g", 1, 2000, 32, 250, 25.0, 0, 397, 643), ("g", 1, 7000, 32, 250, 25.0, 0, 2794, 1816),
    ("t", 1, 2000, 3, 330, 25.0, 1900, 600, 90), ("t", 1, 600, 16, 250, 25.0, 1230, 190, 109),
    ("t", 1, 300, 128, 250, 25.0, 970, 1844, 3472), ("t", 1, 4000, 64, 250, 25.0, 2330, 593, 1305),
    ("t", 256, 300, 6, 330, 25.0, 970, 1013, 1767), ("t", 256, 600, 6, 330, 25.0, 1230, 3102, 2444),
    ("t", 256, 20, 6, 330, 25.0, 360, 1067, 761), ("t", 64, 300, 3, 330, 25.0, 970, 846, 196),
]


def test_rules_of_the_dispatch_take_the_faster_kernel(tmp_path):
    src, exe = tmp_path / "route.cpp", tmp_path / "route"
    src.write_text(ROUTE)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, "-o", str(exe), str(src)], check=True)
    lines = ["%s %d %d %d %d %.9g %d" % (k, b, n, e, nq, q / nq, cells)
             for k, b, n, e, nq, q, cells, _, _ in MEASURED]
    out = subprocess.run([str(exe)], input="\n".join(lines), capture_output=True, text=True, check=True)
    got = [int(x) for x in out.stdout.split()]
    assert len(got) == len(MEASURED)
    for row, new in zip(MEASURED, got):
        assert bool(new) == (row[-1] < row[-2]), row


HIP_STUB = r"""
#pragma once
typedef int hipError_t;
constexpr hipError_t hipSuccess = 0;
constexpr int hipFuncAttributeMaxDynamicSharedMemorySize = 8;
inline int stub_device = 0, stub_calls = 0, stub_fail = 0;
inline hipError_t hipGetDevice(int* d) { return *d = stub_device, hipSuccess; }
inline hipError_t hipFuncSetAttribute(const void*, int, int bytes) {
  ++stub_calls;
  return stub_fail || bytes != 163840 ? 1 : hipSuccess;
}
"""

LDS = r"""
#include "lds_limit.h"
int main() {
  static pyiid::LdsLimit one, two;
  int a, b;
  stub_fail = 1;  // an error is passed on, and asked for again
  if (one.allow({&a, &b}, 163840) == hipSuccess) return 1;
  stub_fail = 0;
  stub_calls = 0;
  for (int round = 0; round < 3; ++round)
    for (stub_device = 0; stub_device < 8; ++stub_device)
      if (one.allow({&a, &b}, 163840) != hipSuccess) return 2;
  if (stub_calls != 16) return 3;  // two kernels on eight devices, once each
  if (two.allow({&a}, 163840) != hipSuccess || stub_calls != 17) return 4;
  stub_device = 200;
  for (int round = 0; round < 2; ++round)
    if (one.allow({&a, &b}, 163840) != hipSuccess) return 5;
  return stub_calls == 21 ? 0 : 6;
}
"""


def test_large_lds_is_asked_for_on_every_device(tmp_path):
    """Each kernel with more than 64 KB of dynamic LDS, once on each device that a
    context runs on; no launcher keeps the answer of one device for all."""
    (tmp_path / "hip").mkdir()
    (tmp_path / "hip" / "hip_runtime.h").write_text(HIP_STUB)
    src, exe = tmp_path / "lds.cpp", tmp_path / "lds"
    src.write_text(LDS)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", str(tmp_path), "-I", CSRC, "-o", str(exe), str(src)],
                   check=True)
    assert subprocess.run([str(exe)]).returncode == 0
    for name in os.listdir(CSRC):
        if name.endswith(".hip"):
            text = open(os.path.join(CSRC, name)).read()
            assert "hipFuncSetAttribute" not in text, name


def vector_registers(source):
    """Vector registers of each kernel of a source, as the compiler reports them."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    flags = re.search(r"^HIPFLAGS := (.*?[^\\])$", open(os.path.join(CSRC, "Makefile")).read(), re.S | re.M)
    flags = flags.group(1).replace("\\\n", " ").replace("$(ARCH)", "gfx950").split()
    out = subprocess.run([hipcc, *flags, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c",
                          os.path.join(CSRC, source), "-o", os.devnull], capture_output=True, text=True)
    assert out.returncode == 0, out.stderr
    found, name = {}, None
    for line in out.stderr.splitlines():
        m = re.search(r"Function Name: (\S+)", line)
        name = m.group(1) if m else name
        m = re.search(r" VGPRs: (\d+)", line)
        if m:
            found[name] = int(m.group(1))
    return found


def test_f_kernels_share_a_cu():
    """A block of the F spreading kernel and one of its transform (16 waves each,
    four a SIMD) fit the 512 registers of a SIMD together, by eights: calls on
    several streams overlap there."""
    regs = vector_registers("spread.hip")
    spread, = [v for k, v in regs.items() if "16spread_fq_kernel" in k]
    transform, = [v for k, v in regs.items() if "transform_fq_kernel" in k]
    assert 4 * 8 * ((spread + 7) // 8 + (transform + 7) // 8) <= 512, (spread, transform)
