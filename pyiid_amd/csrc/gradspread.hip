// Position gradient of F(Q) by spreading (gfx950, wave64).
//
// grad F of atom i is sum_j f_i f_j d_ij K(Q, r_ij), with d_ij = q_i - q_j and
// K(Q, r) = (Q cos(Q r) - sin(Q r) / r) / r^2.  As for F alone, a pair is
// handled once whatever the number of bins:
//
//  1. spread_grad_kernel keeps three grids (x, y, z) of spacing h = 2 pi / (dq
//     n_f), n_f = 4.5 n_q, for its atom and adds every j to 8 points of each:
//     with phi_j(y) the window values and chi_j(y) those of its derivative,
//     sum_g (chi_g / h / r^2 - phi_g / r^3) sin(Q g h) = phihat(Q h) K(Q, r),
//     so one sine transform serves both terms.
//  2. gemm_split_kernel is that transform for all atoms at once: grids (3 N
//     rows) times the n_q x grid sine matrix on the matrix cores, with the
//     weights -1 / na, f_i, f_j and 1 / phihat in its epilogue.
//
// Window: phihat as in the F grid, beta = 19.062 and 8 points; phi and chi are
// least squares over |q| <= pi / 2.25, polynomials of degree 6 and 7.  With
// single-precision values the result is off by 5.8e-8 (phi) and 5.7e-8 (chi,
// of Q_max) r.m.s. over the band.  A grid of n_f = 4 n_q has 1.3e-7 for chi
// and left the gradient 3.8e-7 off at 6,699 atoms.
//
// The product runs on split operands (split_gemm.h).
//
// Reference semantics (pyIID): cpu_flat.py:117-153, cpu_experimental.py:8-15,
// flat_multi_cpu_wrap.py:63-102.
#include <cmath>
#include <type_traits>

#include "fq_grid.h"
#include "lds_limit.h"
#include "split_gemm.h"

namespace pyiid {
namespace {

constexpr int kGw = 8;
constexpr double kGBeta = 19.062;
// phi_j(y) and chi_j(y), j < 4, y in [-1/2, 1/2] about the window's middle;
// phi_{7-j}(y) = phi_j(-y), chi_{7-j}(y) = -chi_j(-y)
constexpr float kPhi[4][7] = {
    {3.40901582e-05f, -0.00027549045f, 0.000964908494f, -0.0018895139f, 0.00225111831f,
     -0.00166305554f, 0.000637135338f},
    {0.00759243827f, -0.0279834767f, 0.0424969158f, -0.0322129548f, 0.00961409082f,
     0.00329632756f, -0.0032371457f},
    {0.11335156f, -0.212225827f, 0.116716452f, 0.0208575311f, -0.0423386611f, 0.006792028f,
     0.00587311726f},
    {0.379021922f, -0.221476835f, -0.160178429f, 0.111719934f, 0.0304739315f, -0.0252178211f,
     -0.0032738704f},
};
constexpr float kChi[4][8] = {
    {-0.000275315306f, 0.00193018817f, -0.0056853555f, 0.00898962606f, -0.00809109359f,
     0.00396534477f, -0.000717389118f, -0.000380087321f},
    {-0.0279849156f, 0.0849923757f, -0.0965007299f, 0.0385146002f, 0.0146398433f, -0.0199819486f,
     0.00589374241f, 0.00149086504f},
    {-0.212221186f, 0.23343518f, 0.0621270564f, -0.169445683f, 0.0399006315f, 0.0361126777f,
     -0.0190095727f, -0.00233059775f},
    {-0.221484802f, -0.320358043f, 0.33592471f, 0.121943086f, -0.136287886f, -0.0200978749f,
     0.032636098f, 0.00121240683f},
};
// Below t = r / h = kGClose K(Q, r), an even function of r, is interpolated in
// r^2 from kGNodes Chebyshev nodes on (0, kGClose h): below 1e-9 for Q h <= pi / 2.25.
constexpr double kGClose = 2.0;
constexpr int kGNodes = 8;
// Fixed point: (chi_j - phi_j / t) (d / h) / t^2 2^s, at most 1.2 2^s / t; s as in
// the F grid (2^24 units at the largest distance), at least 35; from t = 1.2
// 2^(s - 31) on one int32 conversion serves (1.2 A at 25 1/A).
constexpr int kGBits = 24, kGMinScale = 35, kGMaxScale = 48;
// 32-bit entries: 2^kGNarrow, pairs from t = kGNarrowNear = 1.2 2^(kGNarrow - 31) on, and
// structures up to kGNarrowReach grid points across (their quanta add 1e-7 / phihat there;
// denser rows than that outgrow 31 bits in any case).  kGTap bounds |chi_k| + |phi_k| / t.
constexpr int kGNarrow = 33;
constexpr double kGNarrowNear = 4.8, kGNarrowReach = 2048.0;
constexpr float kGTap[4] = {0.0047f, 0.1071f, 0.3521f, 0.3613f};

__host__ __device__ inline double g_node(int k) {
  constexpr double c[kGNodes] = {  // cos((2 k + 1) pi / 32)
      0.99518472667219693, 0.95694033573220882, 0.88192126434835505, 0.77301045336273699,
      0.63439328416364549, 0.47139673682599764, 0.29028467725446233, 0.098017140329560604};
  return kGClose * c[k];
}

// n_f / 2 of the folded grid.
__host__ __device__ inline int half_grid(int nq) { return (9 * nq + 3) / 4; }
// Row length of the grids: nodes, then grid points -4 .. n_f / 2 + 4.
__host__ __device__ inline int row_points(int nq) { return kGNodes + half_grid(nq) + 9; }

// Points of a row in use for distances up to *reach (null: k_fixed).
__device__ __forceinline__ int points_used(const double* reach, double inv_h, int k_fixed, int nq) {
  if (!reach) return k_fixed;
  const int full = row_points(nq);
  const double t = *reach * inv_h + (kGNodes + 10.0);
  return ((t < full ? static_cast<int>(t) : full) + 31) & ~31;
}

// ---- spreading ----

// A pair closer than the fixed point's fast range, or at an infinite
// distance: FP64 and 64-bit conversions.  Pairs from kFarthest on add nothing.
__device__ void spread_grad_rare(unsigned long long* grid, int plane, int* bad, const double* d,
                                 double t, double nf, double scale) {
  if (!(t < 1e300)) {
    atomicOr(bad, 7);
    return;
  }
  auto add = [&](int at, double v) {
    for (int c = 0; c < 3; ++c)
      atomicAdd(&grid[c * plane + at],
                static_cast<unsigned long long>(static_cast<long long>(rint(v * d[c]))));
  };
  if (t < kGClose) {
    const double s = t * t;
#pragma unroll 1
    for (int k = 0; k < kGNodes; ++k) {
      double l = scale;
#pragma unroll 1
      for (int j = 0; j < kGNodes; ++j)
        if (j != k)
          l *= (s - g_node(j) * g_node(j)) / (g_node(k) * g_node(k) - g_node(j) * g_node(j));
      add(k, l);
    }
    return;
  }
  bool neg;
  double u;
  if (!fold(t, nf, u, neg)) return;
  const double fl = floor(u);
  const double y = u - fl - 0.5;
  const int g = kGNodes + static_cast<int>(fl) + 1;
#pragma unroll 1
  for (int j = 0; j < kGw; ++j) {
    const int jj = j < 4 ? j : kGw - 1 - j;
    const double z = j < 4 ? y : -y;
    double phi = kPhi[jj][6], chi = kChi[jj][7];
    for (int k = 5; k >= 0; --k) phi = phi * z + static_cast<double>(kPhi[jj][k]);
    for (int k = 6; k >= 0; --k) chi = chi * z + static_cast<double>(kChi[jj][k]);
    if (j >= 4) chi = -chi;
    // past half the period sin changes sign and cos does not
    add(g + j, (neg ? chi + phi / t : chi - phi / t) * scale / (t * t));
  }
}

// Adds every j of the run to the atom's three grids, WIDE in 64-bit entries, else
// in 32-bit ones with a count of the pairs per cell as a fourth.  Returns
// whether a pair is left out (rare).
template <bool WIDE>
__device__ __forceinline__ bool spread_grad_pairs(const AtomRec* __restrict__ pos, const AtomRec& pi,
                                                  int jb, int je, double inv_h, double nf, float scale,
                                                  double near, unsigned long long* grid, int plane) {
  typedef typename std::conditional<WIDE, unsigned long long, unsigned int>::type entry_t;
  typedef typename std::conditional<WIDE, long long, int>::type signed_t;
  const double half_nf = 0.5 * nf;
  const float fs = scale * static_cast<float>(inv_h);
  bool rare = false;
  for (int j = jb + static_cast<int>(threadIdx.x); j < je; j += blockDim.x) {
    const double dx = pi.x - pos[j].x, dy = pi.y - pos[j].y, dz = pi.z - pos[j].z;
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    double t = scaled_root(r2, inv_h);  // (not a number at r = 0)
    if (!(t >= near && t < kFarthest)) {
      rare = rare || r2 != 0.0;  // the atom itself and duplicates add nothing
      continue;
    }
    float it = __builtin_amdgcn_rcpf(static_cast<float>(t));
    const float w = fs * it * it;
    const float wx = w * static_cast<float>(dx), wy = w * static_cast<float>(dy),
                wz = w * static_cast<float>(dz);
    if (t > half_nf) {
      bool neg;
      (void)fold(t, nf, t, neg);  // (t < kFarthest)
      if (neg) it = -it;
    }
    const float y = static_cast<float>(__builtin_amdgcn_fract(t)) - 0.5f;
    const float y2 = y * y;
    entry_t* gx = reinterpret_cast<entry_t*>(grid) + kGNodes + static_cast<int>(t) + 1;
    entry_t *gy = gx + plane, *gz = gy + plane;
    if (!WIDE) atomicAdd(gz + plane, static_cast<entry_t>(1));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float ec = fmaf(fmaf(fmaf(kChi[k][6], y2, kChi[k][4]), y2, kChi[k][2]), y2, kChi[k][0]);
      const float oc = fmaf(fmaf(fmaf(kChi[k][7], y2, kChi[k][5]), y2, kChi[k][3]), y2, kChi[k][1]);
      const float ep = fmaf(fmaf(fmaf(kPhi[k][6], y2, kPhi[k][4]), y2, kPhi[k][2]), y2, kPhi[k][0]);
      const float op = fmaf(fmaf(kPhi[k][5], y2, kPhi[k][3]), y2, kPhi[k][1]);
      // point k: chi - phi / t at y; point 7 - k: -chi - phi / t at -y
      const float a = fmaf(y, fmaf(-it, op, oc), fmaf(-it, ep, ec));
      const float b = fmaf(y, fmaf(it, op, oc), -fmaf(it, ep, ec));
      auto add = [](entry_t* at, float v) {
        atomicAdd(at, static_cast<entry_t>(static_cast<signed_t>(nearest(v))));
      };
      add(&gx[k], a * wx);
      add(&gy[k], a * wy);
      add(&gz[k], a * wz);
      add(&gx[kGw - 1 - k], b * wx);
      add(&gy[kGw - 1 - k], b * wy);
      add(&gz[kGw - 1 - k], b * wz);
    }
  }
  return rare;
}

// One block per atom and element run: the lanes of its waves take the run's
// atoms in turn and add their 8 points to the block's three grids in LDS.
// The LDS adds bound it: 24 per 64 pairs, at random addresses, which cost
// twice as much as adds without bank conflicts.
//
// narrow: 32-bit entries of 2^kGNarrow.  A count per cell (a 25th add) bounds every
// entry by what its cells' pairs can amount to; where that exceeds 31 bits (or a
// pair is rare) the block starts again with 64-bit entries of `scale`.  With
// 64-bit entries alone LDS was busy for 86% of the kernel, two thirds of that
// bank conflicts; 32-bit ones: F and gradient of 6,699 atoms and 1,250 bins
// 659 -> 538 us, of 20,000 atoms of two elements and 1,500 bins 6.9 -> 5.8 ms
// (error against 64 bits 1.8e-7 -> 2.0e-7 and 2.0e-7 -> 2.5e-7 of the largest
// entry; 5e-7 and 7e-7 with the recurrence).
//
// Afterwards the grids leave as split rows (hi and lo halves), each scaled so
// that its largest entry lies in [2^14, 2^15).
__device__ __forceinline__ void spread_grad_rows(
    const AtomRec* __restrict__ pos, int p0, int n_rows, const int* __restrict__ runs, double inv_h,
    int nf, int plane, int row_len, int k_fixed, const double* __restrict__ reach, int nq,
    float scale, double near, bool narrow, _Float16* __restrict__ rows,
    float* __restrict__ row_scale, unsigned long long* grid) {
  __shared__ int bad;  // a bit per component that is not a number
  __shared__ unsigned int top[3];
  const int p = p0 + blockIdx.x;
  const int n_thread = blockDim.x;
  const int k_used = points_used(reach, inv_h, k_fixed, nq);
  const int k_end = min(k_used, plane);  // no distance reaches past k_used
  const int run = blockIdx.y;
  const int jb = runs[run], je = runs[run + 1];
  unsigned int* grid32 = reinterpret_cast<unsigned int*>(grid);
  if (threadIdx.x == 0) bad = 0;
  if (threadIdx.x < 3) top[threadIdx.x] = 0u;
  const AtomRec pi = pos[p];
  bool wide = !narrow;
  if (narrow) {
    for (int g = threadIdx.x; g < k_end; g += n_thread)
      for (int c = 0; c < 4; ++c) grid32[c * plane + g] = 0u;
    __syncthreads();
    bool over = spread_grad_pairs<false>(pos, pi, jb, je, inv_h, static_cast<double>(nf),
                                         std::ldexp(1.0f, kGNarrow), kGNarrowNear, grid, plane);
    __syncthreads();
    const unsigned int* count = grid32 + 3 * plane;
    for (int g = kGNodes + 1 + static_cast<int>(threadIdx.x); g < k_end; g += n_thread) {
      float m = 0.f;
#pragma unroll
      for (int k = 0; k < kGw; ++k)  // tap k of the cell at g - k
        m = fmaf(static_cast<float>(count[max(g - k, 0)]), kGTap[k < 4 ? k : kGw - 1 - k], m);
      // (the cell at g - 7 is the nearest)
      const int t = max(g - (kGw - 1) - kGNodes - 1, static_cast<int>(kGNarrowNear));
      over = over || !(m < 0.2499f * static_cast<float>(t));  // entry < 2^33 m / t
    }
    wide = __syncthreads_or(over ? 1 : 0) != 0;
  }
  if (wide) {
    for (int c = 0; c < 3; ++c)
      for (int g = threadIdx.x; g < k_end; g += n_thread) grid[c * plane + g] = 0ull;
    __syncthreads();
    const bool rare = spread_grad_pairs<true>(pos, pi, jb, je, inv_h, static_cast<double>(nf), scale,
                                              near, grid, plane);
    // few pairs of a physical structure, if any, are left for a second look
    if (__syncthreads_or(rare ? 1 : 0)) {
      for (int j = jb + static_cast<int>(threadIdx.x); j < je; j += n_thread) {
        const double dx = pi.x - pos[j].x, dy = pi.y - pos[j].y, dz = pi.z - pos[j].z;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        if (!(r2 > 0.0)) {
          // a position that is not a number adds nothing, but shows in the
          // components where it is not
          const int not_finite = (fabs(dx) < HUGE_VAL ? 0 : 1) | (fabs(dy) < HUGE_VAL ? 0 : 2) |
                                 (fabs(dz) < HUGE_VAL ? 0 : 4);
          if (not_finite) atomicOr(&bad, not_finite);
          continue;
        }
        const double t = scaled_root(r2, inv_h);
        if (t >= near && t < kFarthest) continue;
        const double d[3] = {dx * inv_h, dy * inv_h, dz * inv_h};
        spread_grad_rare(grid, plane, &bad, d, sqrt(r2) * inv_h, static_cast<double>(nf),
                         static_cast<double>(scale));
      }
      __syncthreads();
    }
  }
  auto entry = [&](int at) {
    return wide ? static_cast<float>(static_cast<long long>(grid[at]))
                : static_cast<float>(static_cast<int>(grid32[at]));
  };
  // the largest entry of each row, as a non-negative float's bits
  for (int c = 0; c < 3; ++c) {
    float m = 0.f;
    for (int k = threadIdx.x; k < k_end; k += n_thread) m = fmaxf(m, fabsf(entry(c * plane + k)));
    for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
    if ((threadIdx.x & 63) == 0) atomicMax(&top[c], __float_as_uint(m));
  }
  __syncthreads();
  const float unit = wide ? 1.0f / scale : std::ldexp(1.0f, -kGNarrow);
  for (int c = 0; c < 3; ++c) {
    const size_t row = static_cast<size_t>(run) * n_rows + 3 * static_cast<size_t>(blockIdx.x) + c;
    const size_t split_row = static_cast<size_t>(run) * ((n_rows + 127) / 128 * 128) +
                             3 * static_cast<size_t>(blockIdx.x) + c;
    const float m = __uint_as_float(top[c]);
    int e = 0;
    if (m > 0.f) (void)frexpf(m, &e);  // m in [2^(e-1), 2^e)
    const float up = ldexpf(1.0f, 15 - e);
    for (int k = threadIdx.x; k < k_used; k += n_thread) {
      const float x = k < k_end ? entry(c * plane + k) * up : 0.f;
      const _Float16 hi = static_cast<_Float16>(x);
      const size_t at = split_at(split_row, k, row_len);
      rows[at] = hi;
      rows[at + 32] = static_cast<_Float16>(x - static_cast<float>(hi));
    }
    if (threadIdx.x == 0) row_scale[row] = bad >> c & 1 ? __builtin_nanf("") : ldexpf(unit, e - 15);
  }
}

__global__ __launch_bounds__(512, 8) void spread_grad_kernel(
    const AtomRec* __restrict__ pos, int p0, int n_rows, const int* __restrict__ runs, double inv_h,
    int nf, int plane, int row_len, int k_fixed, const double* __restrict__ reach, int nq,
    float scale, double near, bool narrow, _Float16* __restrict__ rows,
    float* __restrict__ row_scale) {
  extern __shared__ unsigned long long grid[];
  spread_grad_rows(pos, p0, n_rows, runs, inv_h, nf, plane, row_len, k_fixed, reach, nq, scale, near,
                   narrow, rows, row_scale, grid);
}

// The same with the work units of F(Q) as further blocks behind the atoms': for a
// structure of a few hundred atoms a launch costs more than either part (505
// atoms, 164 bins: six launches 22.9 us a call among others, four 18.9).
__global__ __launch_bounds__(512, 8) void spread_both_kernel(
    const AtomRec* __restrict__ pos, int n_atoms, const int* __restrict__ runs, double inv_h, int nf,
    int plane, int row_len, int k_fixed, const double* __restrict__ reach, int nq, float scale,
    double near, bool narrow, _Float16* __restrict__ rows, float* __restrict__ row_scale,
    const SpreadUnit* __restrict__ units, const SpreadItem* __restrict__ items, double fq_inv_h,
    int fq_nf, int fq_points, int fq_stride, float fq_scale, double fq_near,
    unsigned long long* __restrict__ grids) {
  extern __shared__ unsigned long long grid[];
  if (static_cast<int>(blockIdx.x) < n_atoms)
    spread_grad_rows(pos, 0, 3 * n_atoms, runs, inv_h, nf, plane, row_len, k_fixed, reach, nq, scale,
                     near, narrow, rows, row_scale, grid);
  else if (blockIdx.y == 0)
    spread_fq_unit(pos, units[blockIdx.x - n_atoms], items, fq_inv_h, fq_nf, fq_points, fq_stride, 0,
                   fq_scale, fq_near, grid, grids);
}

// ---- the sine matrix ----

// w[m][k], split like the rows, scaled by 2^14: node columns
// phihat (q cos(q t) / t^2 - sin(q t) / t^3), grid columns sin(2 pi g m / n_f).
__global__ void sine_matrix_kernel(int nq, int nf, int row_len, _Float16* __restrict__ w,
                                   float* __restrict__ inv_phihat) {
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  const int m = blockIdx.y;
  if (k >= row_len) return;
  const double q = 2.0 * M_PI * m / nf;
  const double a = sqrt(fmax(kGBeta * kGBeta - 0.25 * kGw * kGw * q * q, 1.0));
  const double phihat = (sinh(a) / a) / (sinh(kGBeta) / kGBeta);
  double v = 0.0;
  if (k < kGNodes) {
    const double t = g_node(k);
    v = phihat * (q * cos(q * t) - sin(q * t) / t) / (t * t);
  } else if (k < row_points(nq)) {
    const long long g = k - kGNodes - 4;
    v = sinpi(2.0 * static_cast<double>(g * m % nf) / nf);
  }
  const float x = static_cast<float>(v * 16384.0);
  const _Float16 hi = static_cast<_Float16>(x);
  const size_t at = split_at(m, k, row_len);
  w[at] = hi;
  w[at + 32] = static_cast<_Float16>(static_cast<float>(v * 16384.0 - static_cast<double>(hi)));
  if (k == 0) inv_phihat[m] = static_cast<float>(1.0 / phihat / 16384.0);
}

// ---- rows times sine matrix ----

// out[atom][c][m] = gs[m] f_i(m) / phihat(m) sum_run f_run(m) sum_k rows w.
// Consecutive blocks of an XCD (block id mod 8) share a row tile, which stays in
// its L2.
template <int WM, int WN, int MX, int NY, typename OUT, bool MULTI>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_split_kernel(
    const _Float16* __restrict__ rows, const float* __restrict__ row_scale, int n_rows, int n_run,
    const _Float16* __restrict__ w, const float* __restrict__ inv_phihat, int row_len, int k_fixed,
    const double* __restrict__ reach, double inv_h, int nq, int n_ct, int n_rt, float unit,
    const double* __restrict__ gs, const float* __restrict__ ftab,
    const int* __restrict__ run_elem, const AtomRec* __restrict__ pos,
    const int32_t* __restrict__ perm, int p0, OUT* __restrict__ out, int n_tile,
    ulonglong2* __restrict__ clear, int64_t clear2) {
  __shared__ __align__(16) unsigned char tile[split_lds<WM, WN, MX, NY>()];
  __shared__ float rsc[2][32 * WM * MX];  // the row scales of this and the next run
  const int bid = blockIdx.x;
  if (bid >= n_tile) {  // blocks behind the tiles clear the F grids for the next call
    for (int64_t e = static_cast<int64_t>(bid - n_tile) * blockDim.x + threadIdx.x; e < clear2;
         e += static_cast<int64_t>(gridDim.x - n_tile) * blockDim.x)
      clear[e] = ulonglong2{0ull, 0ull};
    return;
  }
  const int rt = (bid / 8) / n_ct * 8 + bid % 8;
  const int ct = (bid / 8) % n_ct;
  if (rt >= n_rt) return;  // padding block (uniform, before any barrier)
  const int bm = rt * 32 * WM * MX, bn = ct * 32 * WN * NY;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nk = points_used(reach, inv_h, k_fixed, nq) >> 5;
  v16f tot[MX][NY];
#pragma unroll
  for (int x = 0; x < MX; ++x)
#pragma unroll
    for (int y = 0; y < NY; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[x][y][v] = 0.f;
  auto at_run = [&](int run) {
    if (threadIdx.x < 32 * WM * MX)
      rsc[run & 1][threadIdx.x] = row_scale[static_cast<size_t>(run) * n_rows +
                                            min(bm + static_cast<int>(threadIdx.x), n_rows - 1)];
  };
  auto fold = [&](int run, const v16f (&acc)[MX][NY]) {
#pragma unroll
    for (int y = 0; y < NY; ++y) {
      // with several elements weighted by f_run and the row scale
      const int m = min(bn + ((wave % WN) * NY + y) * 32 + (lane & 31), nq - 1);
      const float f = MULTI ? ftab[static_cast<size_t>(run_elem[run]) * nq + m] : 1.f;
#pragma unroll
      for (int x = 0; x < MX; ++x)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          const int r = ((wave / WN) * MX + x) * 32 + (v & 3) + 8 * (v >> 2) + 4 * (lane >> 5);
          tot[x][y][v] = MULTI ? fmaf(acc[x][y][v] * f, rsc[run & 1][r], tot[x][y][v])
                               : tot[x][y][v] + acc[x][y][v];
        }
    }
  };
  split_product<WM, WN, MX, NY>(rows, n_rows, w, row_len, nk, MULTI ? n_run : 1, bm, bn, tile,
                                        fold, at_run);
  split_results<WM, WN, MX, NY>(tot, [&](int i, int j, float t) {
    const int r = bm + i, m = bn + j;
    if (r >= n_rows || m >= nq) return;
    const int p = p0 + r / 3;
    float g;
    if constexpr (MULTI)
      g = t * ftab[static_cast<size_t>(static_cast<int>(pos[p].w)) * nq + m];
    else
      g = t * rsc[0][i];
    const float col = static_cast<float>(gs[m] * static_cast<double>(unit)) * inv_phihat[m];
    out[(3 * static_cast<size_t>(perm ? perm[p] : p) + r % 3) * nq + m] = static_cast<OUT>(g * col);
  });
}

}  // namespace

double grad_reach(int nq, double dq, double r_max) { return r_max * dq * half_grid(nq) / M_PI + kGNodes + 10.0; }
int grad_row_len(int nq) { return (row_points(nq) + 31) & ~31; }
size_t grad_lds_bytes(int nq) {
  return sizeof(unsigned long long) * 3 * static_cast<size_t>(row_points(nq) | 1);
}

hipError_t launch_sine_matrix(hipStream_t st, int nq, void* w, float* inv_phihat) {
  const int len = grad_row_len(nq);
  if (nq > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(sine_matrix_kernel, dim3((len + 255) / 256, nq), dim3(256), 0, st, nq, 2 * half_grid(nq),
                     len, static_cast<_Float16*>(w), inv_phihat);
  return hipGetLastError();
}

namespace {
struct GradLaunch {
  int nf, plane, row_len;
  double inv_h, near;
  float scale;
  size_t lds;
  unsigned threads;
  bool narrow;
};
GradLaunch grad_launch(int64_t n, int nq, double dq, double r_max) {
  GradLaunch g;
  g.nf = 2 * half_grid(nq);
  g.inv_h = dq * half_grid(nq) / M_PI;
  int s = kGMinScale;
  while (s < kGMaxScale && std::ldexp(1.0, s - kGBits) < r_max * g.inv_h && r_max < 1e30) ++s;
  g.scale = std::ldexp(1.0f, s);
  g.near = 1.2 * std::ldexp(1.0, s - 31);
  g.narrow = r_max * g.inv_h <= kGNarrowReach;
  g.plane = row_points(nq) | 1;
  g.row_len = grad_row_len(nq);
  g.lds = grad_lds_bytes(nq);
  // small blocks where six or more fit a CU: their starts and ends overlap better and
  // fewer lanes idle in the last round of atoms (us, alone and among others, 256, 512
  // and 1,024 threads: 1,289 atoms, 330 bins 61 32, 61 34, 66 39; 4,000 atoms of two
  // elements, 600 bins 312 263, 318 268, 343 295; 6,699 atoms, 1,250 bins, whose grids
  // leave two blocks, 683 607, 615 547, 615 550)
  g.threads = n <= 256 || g.lds <= 27 * 1024 ? 256 : 512;
  return g;
}
}  // namespace

hipError_t launch_spread_grad(hipStream_t st, const AtomRec* pos, int p0, int n_atoms, int64_t n,
                              const int* runs, int n_run, int nq, double dq, double r_max,
                              int k_fixed, const double* reach, void* rows, float* row_scale) {
  const GradLaunch g = grad_launch(n, nq, dq, r_max);
  if (g.lds > kGradLds || n_run > 65535) return hipErrorInvalidValue;
  static LdsLimit lds_limit;
  const hipError_t attr = lds_limit.allow({reinterpret_cast<const void*>(spread_grad_kernel)}, kGradLds);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(spread_grad_kernel, dim3(n_atoms, n_run), dim3(g.threads), g.lds, st, pos, p0,
                     3 * n_atoms, runs, g.inv_h, g.nf, g.plane, g.row_len, k_fixed, reach, nq,
                     g.scale, g.near, g.narrow, static_cast<_Float16*>(rows), row_scale);
  return hipGetLastError();
}

hipError_t launch_spread_both(hipStream_t st, const AtomRec* pos, int n_atoms, const int* runs,
                              int n_run, int nq, double dq, double r_max, int k_fixed,
                              const double* reach, void* rows, float* row_scale,
                              const SpreadUnit* units, int n_units, const SpreadItem* items,
                              int scale_bits, unsigned long long* grids) {
  const GradLaunch g = grad_launch(n_atoms, nq, dq, r_max);
  const int fq_nf = 12 * nq, stride = fq_grid_stride(nq);
  const size_t lds = std::max(g.lds, sizeof(unsigned long long) * static_cast<size_t>(stride));
  if (lds > kGradLds || n_run > 65535) return hipErrorInvalidValue;
  static LdsLimit lds_limit;
  const hipError_t attr = lds_limit.allow({reinterpret_cast<const void*>(spread_both_kernel)}, kGradLds);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(spread_both_kernel, dim3(n_atoms + n_units, n_run), dim3(g.threads), lds, st,
                     pos, n_atoms, runs, g.inv_h, g.nf, g.plane, g.row_len, k_fixed, reach, nq,
                     g.scale, g.near, g.narrow, static_cast<_Float16*>(rows), row_scale, units, items,
                     dq * fq_nf / (2.0 * M_PI), fq_nf, fq_grid_points(nq), stride,
                     std::ldexp(1.0f, scale_bits), std::ldexp(1.0, scale_bits - 31), grids);
  return hipGetLastError();
}

hipError_t launch_gemm_split(hipStream_t st, const void* rows, const float* row_scale, int n_atoms,
                             int n_run, const void* w, const float* inv_phihat, int nq, double dq,
                             int k_fixed, const double* reach, const double* gs, const float* ftab,
                             const int* run_elem, bool weighted, const AtomRec* pos,
                             const int32_t* perm, int p0, void* out, bool out_f64,
                             unsigned long long* clear, int64_t clear_words) {
  const int n_rows = 3 * n_atoms;
  const double inv_h = dq * half_grid(nq) / M_PI;
  const float unit = static_cast<float>(inv_h * inv_h);
  const bool large = split_large(n_rows, nq);
  const int n_ct = large ? (nq + 127) / 128 : (nq + 63) / 64, n_rt = (n_rows + 127) / 128;
  const int n_tile = 8 * ((n_rt + 7) / 8) * n_ct;
  const int64_t clear2 = clear ? clear_words / 2 : 0;  // an even number of words
  const dim3 grid(static_cast<unsigned>(n_tile + std::min<int64_t>((clear2 + 511) / 512, 256)));
  const int len = grad_row_len(nq);
#define PYIID_TILES(T, M, WM, WN, MX, NY)                                                       \
  hipLaunchKernelGGL((gemm_split_kernel<WM, WN, MX, NY, T, M>), grid, dim3(64 * WM * WN), 0, st, \
                     static_cast<const _Float16*>(rows), row_scale, n_rows, n_run,              \
                     static_cast<const _Float16*>(w), inv_phihat, len, k_fixed, reach, inv_h, nq, \
                     n_ct, n_rt, unit, gs, ftab, run_elem, pos, perm, p0, static_cast<T*>(out), \
                     n_tile, reinterpret_cast<ulonglong2*>(clear), clear2)
#define PYIID_GEMM(T, M)                 \
  do {                                   \
    if (large)                           \
      PYIID_TILES(T, M, 2, 2, 2, 2);     \
    else                                 \
      PYIID_TILES(T, M, 4, 2, 1, 1);     \
  } while (0)
  if (weighted) {
    if (out_f64)
      PYIID_GEMM(double, true);
    else
      PYIID_GEMM(float, true);
  } else {
    if (out_f64)
      PYIID_GEMM(double, false);
    else
      PYIID_GEMM(float, false);
  }
#undef PYIID_GEMM
#undef PYIID_TILES
  return hipGetLastError();
}

}  // namespace pyiid
