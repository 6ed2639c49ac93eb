// The F(Q) grid of spread.hip: its window, fixed point and the spreading of one
// work unit, shared with gradspread.hip (which runs units beside its own blocks).
#pragma once

#include "pair_math.h"

#include "fold.h"

namespace pyiid {
namespace {

// ---- window of the F grid ----
constexpr int kFqW = 6;             // grid points per pair
constexpr double kFqBeta = 15.160;  // window shape (smallest r.m.s. error at 6 points)
// phi_j(y), j < 3, y in [-1/2, 1/2] about the middle of the window;
// phi_{5-j}(y) = phi_j(-y).  A least squares fit with every coefficient rounded to
// its nearest float had its mean over y 1.7e-8 short of phihat, and v_rcp_f32, which
// makes 1/t, is 6.8e-9 short on average: F was off by one factor, 1 - 2.4e-8, which
// no number of pairs averages out (6,699 atoms, 1,250 bins: 4.7e-8 of the largest F
// at worst).  Here the fit and the choice of floats hold the mean, with v_rcp_f32's,
// within 4e-9 over the band (3.8e-9 r.m.s. of single places).
constexpr float kFqVal[3][6] = {
    {0.000792802835f, -0.00590729201f, 0.0172293913f, -0.0255970359f, 0.0208720788f,
     -0.00801460911f},
    {0.0737483203f, -0.206045285f, 0.198311478f, -0.0387120843f, -0.0626117215f, 0.0401164442f},
    {0.425458878f, -0.352327496f, -0.215540871f, 0.244120404f, 0.0417396985f, -0.0802748948f},
};
// Fixed point of the grid: phi_j 2^s / t, t = r / h.  s is chosen from the
// structure's extent so that a pair at its largest distance still has 2^24
// units (at most 2^25), and s >= 36.  From t = 2^(s - 31) on (0.7 A for a
// particle of 85 A at 25 1/A) the value is below 2^31 and one int32 conversion
// serves; closer pairs take spread_rare.
constexpr int kFqBits = 24;
constexpr int kFqMinScale = 36, kFqMaxScale = 48;
// Below t = kFqClose the window's error over 1/r would show: there sin(Qr)/r,
// an even function of r, is interpolated in r^2 from kFqNodes Chebyshev nodes
// on (0, kFqClose h) (error below 1e-9 for Q h <= pi / 6).  Their weights
// follow the grid, scaled by 2^30.
constexpr double kFqClose = 2.0;
constexpr int kFqNodes = 5;
constexpr double kNodeScale = 1073741824.0;

__host__ __device__ inline double fq_node(int k) {  // t of node k
  constexpr double c[kFqNodes] = {0.98768834059513773, 0.89100652418836787, 0.70710678118654752,
                                  0.45399049973954675, 0.15643446504023087};  // cos((2k+1) pi/20)
  return kFqClose * c[k];
}

// ---- spreading ----

// A pair closer than the fixed point's fast range, or at an infinite
// distance: 64-bit conversions.  Few pairs of a physical structure come here, and
// those from kFarthest on add nothing.  A call of its own: within the kernels its
// constants took 50 of their registers for scalars that did not fit, and a block of
// spread_fq_kernel with 58 vector registers leaves no room for one of
// transform_fq_kernel beside it, where several streams share the chip (F of 6,699
// atoms on three streams in turn 57 us, with up to 56 registers 50; of 20,000 atoms
// of two elements 421 and 406; on one stream alike, also where all pairs are close:
// 7,000 atoms, 64 bins to 2 1/A 200 -> 185 us).
__device__ __noinline__ void spread_rare(unsigned long long* hist, int n_grid, double t, double nf,
                                         double scale) {
  unsigned long long* nodes = hist + n_grid;
  if (!(t < 1e300)) {  // infinite: F is not a number
    atomicAdd(&nodes[kFqNodes], 1ull);
    return;
  }
  if (t < kFqClose) {
    const double s = t * t;
    for (int k = 0; k < kFqNodes; ++k) {
      double l = 1.0;
      for (int j = 0; j < kFqNodes; ++j)
        if (j != k) l *= (s - fq_node(j) * fq_node(j)) / (fq_node(k) * fq_node(k) - fq_node(j) * fq_node(j));
      atomicAdd(&nodes[k], static_cast<unsigned long long>(static_cast<long long>(rint(l * kNodeScale))));
    }
    return;
  }
  bool neg;
  double tf;
  if (!fold(t, nf, tf, neg)) return;
  const double fl = floor(tf);
  const double y = tf - fl - 0.5, w = (neg ? -scale : scale) / t;
  unsigned long long* h = hist + (static_cast<int>(fl) + 1);
  for (int j = 0; j < kFqW; ++j) {
    const float* c = kFqVal[j < 3 ? j : kFqW - 1 - j];
    const double z = j < 3 ? y : -y;
    double p = c[5];
    for (int k = 4; k >= 0; --k) p = p * z + static_cast<double>(c[k]);
    atomicAdd(&h[j], static_cast<unsigned long long>(static_cast<long long>(rint(p * w))));
  }
}

// A pair in the fixed point's fast range; false past kFarthest.
__device__ __forceinline__ bool spread_pair(unsigned long long* hist, double t, double nf,
                                            double half_nf, float scale) {
  float w = scale * __builtin_amdgcn_rcpf(static_cast<float>(t));
  if (t > half_nf) {
    bool neg;
    if (!fold(t, nf, t, neg)) return false;
    if (neg) w = -w;
  }
  const float y = static_cast<float>(__builtin_amdgcn_fract(t)) - 0.5f;
  const float y2 = y * y;
  unsigned long long* h = hist + (static_cast<int>(t) + 1);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float e = fmaf(fmaf(kFqVal[k][4], y2, kFqVal[k][2]), y2, kFqVal[k][0]);
    const float o = y * fmaf(fmaf(kFqVal[k][5], y2, kFqVal[k][3]), y2, kFqVal[k][1]);
    const int a = nearest((e + o) * w), b = nearest((e - o) * w);
    atomicAdd(&h[k], static_cast<unsigned long long>(static_cast<long long>(a)));
    atomicAdd(&h[kFqW - 1 - k], static_cast<unsigned long long>(static_cast<long long>(b)));
  }
  return true;
}

// One block (at least 4 waves) per work unit: a run of items of one chain and element
// pair, whose pairs are spread into the block's grid in LDS, then added to the
// chain's grid in global memory.  An item is an i tile of at most 64 positions
// (one lane each) against a j range; the waves take consecutive slices of
// the range, and a j atom's position is wave-uniform (scalar loads, so the
// FP64 differences take it from SGPRs).
//
// Per 64 pairs about 14 FP64 or conversion instructions (distance to 4e-14:
// a phase of 1,500 rad to 6e-11), 18 FMAs for the window, 6 conversions to
// integer and 6 ds_add_u64.  The LDS adds bound it (64 chains of 5,000 atoms: busy
// 89% of the time, two thirds of that bank conflicts of random addresses) and the
// VALU, busy 95% beside them; 2 blocks (32 waves) per CU hide each other's latency.
// A tile off the diagonal needs two comparisons a pair (1,988 -> 1,930 us for that
// batch, where every pair took five; 1,775 us with settled clocks).
__device__ __forceinline__ void spread_fq_unit(
    const AtomRec* __restrict__ pos, const SpreadUnit& un, const SpreadItem* __restrict__ items,
    double inv_h, int nf, int n_grid, int stride, int shift, float scale, double near,
    unsigned long long* hist, unsigned long long* __restrict__ grids) {
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n_wave = blockDim.x >> 6, wave_bits = __ffs(n_wave) - 1;  // a power of two
  for (int g = threadIdx.x; g < stride; g += blockDim.x) hist[g] = 0ull;
  __syncthreads();
  const double half_nf = 0.5 * nf;
  bool rare = false;
  for (int it = un.begin; it < un.end; ++it) {
    const SpreadItem item = items[it];
    const int64_t len = item.j1 - item.j0;
    const int jb = item.j0 + static_cast<int>(len * wave >> wave_bits);
    const int je = item.j0 + static_cast<int>(len * (wave + 1) >> wave_bits);
    const int i = item.i0 + lane;
    if (i >= item.i1) continue;
    const AtomRec pi = pos[i];
    // (a pair at distance 0, or with a NaN, contributes nothing)
    auto pair = [&](const AtomRec& pj) {
      const double dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
      const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
      const double t = scaled_root(r2, inv_h);
      if (t >= near) {
        if (!spread_pair(hist, t, static_cast<double>(nf), half_nf, scale)) rare = true;
      } else if (r2 > 0.0) {
        rare = true;
      }
    };
    if (item.j1 <= item.i0) {
      for (int j = jb; j < je; ++j) pair(pos[j]);
    } else {
      for (int j = jb; j < je; ++j)
        if (j < i) pair(pos[j]);
    }
  }
  // few pairs of a physical structure, if any, are left for a second look
  if (__syncthreads_or(rare ? 1 : 0)) {
    for (int it = un.begin; it < un.end; ++it) {
      const SpreadItem item = items[it];
      const int i = item.i0 + lane;
      if (i >= item.i1) continue;
      const AtomRec pi = pos[i];
      for (int j = item.j0 + wave; j < item.j1; j += n_wave) {
        const double dx = pi.x - pos[j].x, dy = pi.y - pos[j].y, dz = pi.z - pos[j].z;
        const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
        if (!(j < i && r2 > 0.0)) continue;
        const double t = scaled_root(r2, inv_h);
        if (t >= near && t < kFarthest) continue;
        spread_rare(hist, n_grid, sqrt(r2) * inv_h, static_cast<double>(nf),
                    static_cast<double>(scale));
      }
    }
    __syncthreads();
  }
  unsigned long long* out = grids + static_cast<size_t>(un.grid) * stride;
  for (int g = threadIdx.x; g < stride; g += blockDim.x) {
    const long long v = static_cast<long long>(hist[g]);
    if (v == 0) continue;
    const long long s = (shift == 0 || g == n_grid + kFqNodes) ? v : (v + (1ll << (shift - 1))) >> shift;
    atomicAdd(&out[g], static_cast<unsigned long long>(s));
  }
}

}  // namespace
}  // namespace pyiid
