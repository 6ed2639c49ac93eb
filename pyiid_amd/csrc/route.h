// Which of the kernels that can take a call is the faster one: the spreading kernels
// and force tables, whose work per pair does not depend on the bins, or the
// recurrence kernels, whose work does.  Plain C++ of sizes only, so that a call's
// route can be checked on the host.
#pragma once

#include <algorithm>
#include <cmath>
#include <cstdint>

namespace pyiid {

// Sizes of a batch.
struct BatchSize {
  int64_t chains = 1, longest = 0;
  double atoms = 0.0, squares = 0.0;  // sum of n and of n^2 over the chains
  void add(int64_t n) {
    longest = std::max(longest, n);
    atoms += static_cast<double>(n);
    squares += static_cast<double>(n) * static_cast<double>(n);
  }
  double pairs() const { return 0.5 * (squares - atoms); }
};

inline int64_t blocks_of_bins(int nq) { return (nq + 63) / 64; }

// F of n_elem elements (n_pair pairs of them), in one launch if `small`.  Every
// grid of a chain and element pair costs its transform, 20 to 40 ns a block of 64
// bins once the chip is full, where the recurrence only cuts its items shorter.
// Measured (us, recurrence and spreading kernel; 25 1/A): 250 bins, 600 atoms of 8,
// 16 and 32 elements 62 30, 40 41, 45 102, 4,000 atoms of 16 and 64 332 72, 291
// 373, 60 atoms of 4 and 16 23 18, 19 33; 330 bins, 256 chains of three elements
// of 80 and 300 atoms 93 223, 423 272; 1,024 chains of 40 and 150 atoms of one
// element 91 150, 509 202.  One structure of up to three elements takes less
// time on the spreading kernel at every size measured (55 to 7,000 atoms, 1 to
// 3,400 bins, 0.3 to 25 1/A), but for a single bin at 0.1 1/A, where all pairs are
// close contacts (7,000 atoms 450 600).
inline bool spread_fq_pays(const BatchSize& s, int n_elem, int64_t n_pair, int nq, double dq,
                           bool small) {
  if (nq < 64 && nq * dq < 0.2) return false;
  if (s.chains == 1 && n_pair <= 6) return true;
  const double chains = static_cast<double>(s.chains), grids = static_cast<double>(n_pair) * chains;
  const double bins = static_cast<double>(blocks_of_bins(nq));
  // points that the distances of a chain reach, about
  const double points = std::min(6.0 * nq, 150.0 * std::cbrt(s.atoms / chains));
  const double spread = small ? 10.0 + 0.0035 * (n_pair + 1.0) * chains * bins
                              : 24.0 + (0.018 + 1.2e-5 * nq + 6e-6 * points) * grids * bins +
                                    2.7e-6 * s.pairs();
  const double recurrence = 20.0 + 0.45 * std::min(static_cast<double>(s.longest) / n_elem, 320.0) +
                            1.05e-7 * nq * (0.5 * s.squares + 16.0 * s.atoms) +
                            (0.01 + 2.5e-5 * nq) * grids;
  return spread <= recurrence;
}

// The gradient of n atoms of `kinds` elements.  Its spreading kernel has 64-bit
// entries and a second look at close pairs where the grid is coarse (distances count
// in grid spacings, 1.4 / Q_max), and its adds meet on few words where there are few
// bins; the recurrence takes the same time for any number of bins up to 256.
// Measured (us, recurrence and spreading kernel): 64 bins to 1 1/A, 600 atoms
// 45 56, 2,000 154 246, 7,000 1373 1737; 64 bins to 8 1/A 48 45, 153 162, 1373
// 1015; 8 bins to 25 1/A 42 36, 142 149, 1308 1337; 200 bins to 2 1/A 66 54, 236
// 231, 2175 1455; 300 atoms 45 39, 45 30, 44 24, 63 33.  The rows and product of
// every element come on top: 250 bins, 200 atoms of 4, 5 and 8 elements 54 42, 46
// 49, 39 67, 1,500 atoms of 12 and 16 204 199, 215 255, 7,000 of 32 2794 1816; up to
// three elements pay at every size measured.
inline bool spread_grad_pays(int64_t n, int kinds, int nq, double dq) {
  const double atoms = static_cast<double>(n), q_max = nq * dq;
  const double most = std::max(3.2 + 0.0035 * atoms * (1.0 + nq / 450.0), atoms / 125.0);
  if (kinds > 3 && kinds > most) return false;
  if (q_max >= 0.95) {
    // from this many bins on whatever the largest Q (from about 1 1/A on)
    const int bins = n <= 400                                ? 1
                     : n < 700                               ? 130
                     : n < 1250 || (n < 2500 && q_max < 2.0) ? 257
                                                             : 190;
    if (nq >= bins) return true;
  }
  const double least = n < 700    ? q_max >= 12.0 ? 190.0 : 512.0
                       : n < 1250 ? 900.0
                       : n < 2500 ? q_max >= 12.0 ? 384.0 : 420.0
                                  : 256.0;
  return nq * q_max >= least;
}

// Forces from tables of n_cell cells.  Each chain and element pair has a table, whose
// making costs its cells times the bins, and which every block that reads it loads;
// the recurrence pays for its tiles of 64 by 64 atoms, whole or not.  Measured
// (us, energy and forces with recurrences alone and with spreading and tables):
// 250 bins, 600 atoms of 16, 32 and 48 elements 230 150, 340 372, 509 724, 4,000 atoms
// of 32 749 507; 330 bins, 256 chains of 6 elements of 20, 300 and 600 atoms 1159
// 1422, 1414 2603, 4394 3414 (of which F 92 661, 401 836, 1292 970).
inline bool force_table_pays(const BatchSize& s, int n_elem, int64_t n_pair, int nq, double n_cell) {
  const double pairs = static_cast<double>(n_pair), chains = static_cast<double>(s.chains);
  if (s.chains == 1)
    return pairs * (0.22 + 6e-7 * nq * n_cell) <=
           40.0 + std::max(pairs * (0.04 + 1.2e-3 * nq), 1.4e-7 * nq * s.pairs());
  const double tiles = n_elem * std::ceil(s.atoms / chains / (64.0 * n_elem));
  return pairs * chains * n_cell * (6.7e-7 * nq + 9.5e-5) <=
         90.0 + 0.5 * tiles * (tiles + 1.0) * chains * (0.02 + 4.5e-4 * nq);
}

}  // namespace pyiid
