// F(Q) by spreading the pair distances onto a fine grid (gfx950, wave64).
//
// F needs sum_{pairs} sin(Q_m r) / r on the bins Q_m = m dq: the transform of
// a sum of point weights 1/r at the distances r onto equidistant bins.  A
// recurrence per pair and bin costs pairs x bins; here every pair is handled
// once, whatever the number of bins:
//
//  1. spread_fq_kernel adds the pair's weight to kFqW = 6 points of a grid of
//     spacing h = 2 pi / (dq n_f), n_f = 12 n_q (six times finer than the
//     bins need), with window values phi_j(y) that are polynomials of the
//     pair's place y between the grid points;
//  2. transform_fq_kernel sums grid[g] sin(2 pi g m / n_f) in FP64 and divides
//     by the window's transform phihat(q), q = Q h.
//
// Window: phihat(q) = sinh(a) / a, a = sqrt(beta^2 - (3 q)^2), scaled to 1 at
// q = 0 (the Kaiser-Bessel window's transform), and the phi_j(y) are the least
// squares solution of sum_j phi_j(y) exp(i q (g_j - y)) = phihat(q) over the
// band |q| <= pi / 6, fitted by polynomials of degree 5 in y.  The result is
// exp(i Q r) to 2.6e-8 at worst and 3.8e-9 r.m.s. over the band and y, with the
// float coefficients too; evaluated in single precision 2.3e-8 r.m.s., which pairs
// average out (single-precision sin and cos of the phase have 3e-8).
//
// The grid is folded: sin(2 pi g m / n_f) is odd about g = 0 and g = n_f / 2
// and has period n_f, so a distance of any size is brought into [0, n_f / 2]
// with a sign, and the grid has n_f / 2 + 7 points (3 beyond each end).
//
// Grid sums are 64-bit integers (fixed point): ds_add_u64 adds 64 lanes in
// 4.8 ns per CU (ds_add_f64: 9.1 ns, ds_add_f32: 80 ns, ds_add_u32: 2.7 ns, at
// random addresses), the sums are exact, and they do not depend on the order
// in which waves and blocks add, so results repeat bit for bit.
//
// Reference semantics (pyIID): cpu_flat.py:77-114,
// flat_multi_cpu_wrap.py:22-60.
#include <algorithm>
#include <cmath>

#include "fq_grid.h"
#include "lds_limit.h"

namespace pyiid {
namespace {

__global__ __launch_bounds__(1024, 8) void spread_fq_kernel(
    const AtomRec* __restrict__ pos, const SpreadUnit* __restrict__ units,
    const SpreadItem* __restrict__ items, double inv_h, int nf, int n_grid, int stride, int shift,
    float scale, double near, unsigned long long* __restrict__ grids) {
  extern __shared__ unsigned long long hist[];
  spread_fq_unit(pos, units[blockIdx.x], items, inv_h, nf, n_grid, stride, shift, scale, near, hist,
                 grids);
}

// ---- grid -> F(Q) ----

constexpr int kTrChunk = 2048;  // grid points in LDS at a time (16 KiB)

// What the bins of a block share, made by two of its waves while the others
// spread or load: 1 / phihat, and sine and cosine of 2 pi m / n_f.
struct BinTerms {
  double inv[64], sin1[64], cos1[64];
};

// acc[p] += sum over grid points [lo, hi) of value(p, k) sin(2 pi (first + k - 3) m /
// n_f): the sine starts from an exact phase (reduced as an integer below 2^31:
// n_f <= 12 * 3,400, g + n_f < 1.6 n_f) and follows the FP64 three-term recurrence.
template <int N, typename F>
__device__ __forceinline__ void sine_sum(F value, int lo, int hi, int first, int m, int nf,
                                         double sin1, double cos1, double (&acc)[N]) {
  const unsigned g = static_cast<unsigned>(first + lo - 3 + nf);
  const unsigned s0 = g * static_cast<unsigned>(m) % static_cast<unsigned>(nf);
  const double c2 = 2.0 * cos1;
  double y, c;
  sincospi(2.0 / static_cast<double>(nf) * static_cast<double>(s0), &y, &c);
  double yp = fma(y, cos1, -c * sin1);  // one point before
#pragma unroll 4
  for (int k = lo; k < hi; ++k) {
#pragma unroll
    for (int p = 0; p < N; ++p) acc[p] = fma(value(p, k), y, acc[p]);
    const double yn = fma(c2, y, -yp);
    yp = y;
    y = yn;
  }
}

// 1 / phihat(m) but for its constant sinh(beta) / beta, which comes with the unit
// from fq_unit: sinh(a) = (e^a - e^-a) / 2, where a > 15 leaves e^-2a < 1e-13.
__device__ __forceinline__ double fq_inv_phihat(int m, int nf) {
  const double q = 2.0 * M_PI * m / nf;  // Q h <= pi / 6
  const double a = sqrt(kFqBeta * kFqBeta - 0.25 * kFqW * kFqW * q * q);
  const double e = exp(-a);
  return 2.0 * a * e / (1.0 - e * e);
}

__device__ __forceinline__ void bin_terms(BinTerms& t, int m, int nf, double unit) {
  const int lane = threadIdx.x & 63, from_last = (blockDim.x >> 6) - 1 - (threadIdx.x >> 6);
  if (from_last == 0) t.inv[lane] = unit * fq_inv_phihat(m, nf);
  if (from_last == 1) sincospi(2.0 * m / nf, &t.sin1[lane], &t.cos1[lane]);
}

// h, the fixed point's unit and the window's constant
double fq_unit(double inv_h, int shift, int scale_bits) {
  return std::ldexp(inv_h, shift - scale_bits) * std::sinh(kFqBeta) / kFqBeta;
}

// One more than the last of [0, cnt) at which get(g) is not zero, for the block:
// distances reach the first few hundred of a grid's points (a third of them at
// 55 atoms and 250 bins), and the transform ends there.  top: LDS, zero before;
// a barrier follows.
template <typename G>
__device__ __forceinline__ void last_used(G get, int cnt, int* top) {
  int mine = 0;
  for (int g = threadIdx.x; g < cnt; g += blockDim.x)
    if (get(g)) mine = g + 1;
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mine = max(mine, __shfl_xor(mine, off, 64));
  if ((threadIdx.x & 63) == 0 && mine > 0) atomicMax(top, mine);
}

// The close contacts' part of sum sin(Q r) / r (almost always none)
__device__ __forceinline__ double fq_nodes(const unsigned long long* nodes, int m, int nf,
                                           double inv_h, int shift) {
  const double q = 2.0 * M_PI * m / nf;
  double t = 0.0;
  for (int k = 0; k < kFqNodes; ++k) {
    const long long v = static_cast<long long>(nodes[k]);
    if (v != 0)
      t += static_cast<double>(v) * (ldexp(inv_h, shift) / kNodeScale) * sin(q * fq_node(k)) /
           fq_node(k);
  }
  return nodes[kFqNodes] != 0ull ? __builtin_nan("") : t;
}

// part[b][z][m]: one block takes 64 bins (lanes) of one chain against one of
// the n_split parts of one element pair's grid; its 16 waves take consecutive
// slices of every chunk of points.  The parts are there to fill the chip: one block per 64 bins took 47 us for 1,250 bins and
// 155 us for three element pairs at 1,500.
__global__ __launch_bounds__(1024) void transform_fq_kernel(
    const unsigned long long* __restrict__ grids, int n_pair, int n_split, int nf, int n_grid,
    int stride, int shift, double unit, const float* __restrict__ ftab, int nq, double inv_h,
    int weighted, double* __restrict__ part, const double* __restrict__ scale,
    double* __restrict__ out64, float* __restrict__ out32) {
  __shared__ __align__(16) double buf[kTrChunk];
  __shared__ double sums[16][65];
  __shared__ BinTerms terms;
  __shared__ int top;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = blockIdx.x * 64 + lane;
  const int b = blockIdx.y, z = blockIdx.z;
  const int pair = z / n_split, split = z % n_split;
  const unsigned long long* h = grids + (static_cast<size_t>(b) * n_pair + pair) * stride;
  const int g_lo = static_cast<int>(static_cast<int64_t>(n_grid) * split / n_split);
  const int g_hi = static_cast<int>(static_cast<int64_t>(n_grid) * (split + 1) / n_split);
  double acc[1] = {0.0};
  for (int g0 = g_lo; g0 < g_hi; g0 += kTrChunk) {
    const int cnt = min(kTrChunk, g_hi - g0);
    __syncthreads();
    if (threadIdx.x == 0) top = 0;
    __syncthreads();
    last_used(
        [&](int g) {
          const long long v = static_cast<long long>(h[g0 + g]);
          buf[g] = static_cast<double>(v);
          return v != 0;
        },
        cnt, &top);
    if (g0 == g_lo) bin_terms(terms, m, nf, unit);
    __syncthreads();
    const int used = top;
    if (used > 0)
      sine_sum<1>([&](int, int k) { return buf[k]; }, used * wave / 16, used * (wave + 1) / 16, g0, m, nf,
                  terms.sin1[lane], terms.cos1[lane], acc);
  }
  sums[wave][lane] = acc[0];
  __syncthreads();
  if (wave != 0 || m >= nq) return;
  double total = 0.0;
#pragma unroll
  for (int k = 0; k < 16; ++k) total += sums[k][lane];
  total *= terms.inv[lane];
  if (split == 0) total += fq_nodes(h + n_grid, m, nf, inv_h, shift);
  if (weighted) {
    int ei = 0, ej = pair;
    while (ej > ei) ej -= ++ei;
    total *= static_cast<double>(ftab[static_cast<size_t>(ei) * nq + m]) *
             static_cast<double>(ftab[static_cast<size_t>(ej) * nq + m]);
  }
  if (part) {
    part[(static_cast<size_t>(b) * n_pair * n_split + z) * nq + m] = total;
    return;
  }
  // one part: F itself
  const size_t o = static_cast<size_t>(b) * nq + m;
  const double v = total * scale[o];
  if (out64) out64[o] = v;
  if (out32) out32[o] = static_cast<float>(v);
}

// F from the parts (blocks below n_out, one thread per chain and bin), and the
// grids cleared for the next call (the blocks from n_out).  A launch of its
// own: with the same work in the transform's last blocks, the agent-scope
// fences between 288 blocks took 20 us.
__global__ __launch_bounds__(256) void finish_fq_kernel(
    const double* __restrict__ part, int n_part, int nq, int64_t total, int n_out,
    const double* __restrict__ scale, double* __restrict__ out64, float* __restrict__ out32,
    ulonglong2* __restrict__ grids, int64_t words2) {
  if (static_cast<int>(blockIdx.x) < n_out) {
    const int64_t e = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
    if (e >= total) return;
    const double* p = part + (e / nq) * n_part * nq + e % nq;
    double t = 0.0;
#pragma unroll 8
    for (int z = 0; z < n_part; ++z) t += p[static_cast<size_t>(z) * nq];
    const double v = t * scale[e];
    if (out64) out64[e] = v;
    if (out32) out32[e] = static_cast<float>(v);
    return;
  }
  for (int64_t w = static_cast<int64_t>(blockIdx.x - n_out) * 256 + threadIdx.x; w < words2;
       w += static_cast<int64_t>(gridDim.x - n_out) * 256)
    grids[w] = ulonglong2{0ull, 0ull};
}

// F of small chains in one launch instead of three: every block of 64 bins spreads
// all pairs of its chain again and transforms the grids (N: one for each pair of
// elements) where they lie, in LDS.  A block has a CU of its own and is bound by its
// VALU work: 8 waves, so that the sums' starting phases are few (16 waves 14 us, 4
// waves 12 us, 8 waves 11 us at 55 atoms and 250 bins).
constexpr int kSmallWaves = 8;

template <int N>
__global__ __launch_bounds__(64 * kSmallWaves) void small_fq_kernel(
    const AtomRec* __restrict__ pos, const int* __restrict__ off, int nf, int n_grid, int stride,
    double unit, float scale, double near, const float* __restrict__ ftab, int nq, double inv_h,
    const double* __restrict__ fscale, double* __restrict__ out64, float* __restrict__ out32) {
  extern __shared__ unsigned long long hist[];
  __shared__ double sums[N][kSmallWaves][65];
  __shared__ BinTerms terms;
  __shared__ int top;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int m = blockIdx.x * 64 + lane;
  const int b = blockIdx.y;
  const int i0 = off[b], n = off[b + 1] - i0;
  const int pairs = n * (n - 1) / 2;
  const double half_nf = 0.5 * nf;
  for (int g = threadIdx.x; g < N * stride; g += 64 * kSmallWaves) hist[g] = 0ull;
  if (threadIdx.x == 0) top = 0;
  __syncthreads();
  for (int k = threadIdx.x; k < pairs; k += 64 * kSmallWaves) {
    int i = static_cast<int>((1.0f + __builtin_amdgcn_sqrtf(1.0f + 8.0f * k)) * 0.5f);
    if (i * (i - 1) / 2 > k) --i;
    if ((i + 1) * i / 2 <= k) ++i;
    const AtomRec a = pos[i0 + i], c = pos[i0 + k - i * (i - 1) / 2];
    const double dx = a.x - c.x, dy = a.y - c.y, dz = a.z - c.z;
    const double r2 = fma(dx, dx, fma(dy, dy, dz * dz));
    if (!(r2 > 0.0)) continue;
    unsigned long long* grid = hist;
    if (N > 1) {
      const int x = static_cast<int>(a.w), y = static_cast<int>(c.w), hi = max(x, y);
      grid += (hi * (hi + 1) / 2 + min(x, y)) * stride;
    }
    const double t = scaled_root(r2, inv_h);
    if (!(t >= near && spread_pair(grid, t, static_cast<double>(nf), half_nf, scale)))
      spread_rare(grid, n_grid, sqrt(r2) * inv_h, static_cast<double>(nf), static_cast<double>(scale));
  }
  bin_terms(terms, m, nf, unit);
  __syncthreads();
  double* points = reinterpret_cast<double*>(hist);  // the points in place
  last_used(
      [&](int g) {
        long long any = 0;
#pragma unroll
        for (int p = 0; p < N; ++p) {
          const long long v = static_cast<long long>(hist[p * stride + g]);
          points[p * stride + g] = static_cast<double>(v);
          any |= v;
        }
        return any != 0;
      },
      n_grid, &top);
  __syncthreads();
  const int used = top;
  double acc[N] = {};
  if (used > 0)
    sine_sum<N>([&](int p, int k) { return points[p * stride + k]; }, used * wave / kSmallWaves,
                used * (wave + 1) / kSmallWaves, 0, m, nf, terms.sin1[lane], terms.cos1[lane], acc);
#pragma unroll
  for (int p = 0; p < N; ++p) sums[p][wave][lane] = acc[p];
  __syncthreads();
  if (wave != 0 || m >= nq) return;
  double total = 0.0;
  int ei = 0, ej = 0;
#pragma unroll
  for (int p = 0; p < N; ++p) {
    double v = 0.0;
#pragma unroll
    for (int k = 0; k < kSmallWaves; ++k) v += sums[p][k][lane];
    v = v * terms.inv[lane] + fq_nodes(hist + p * stride + n_grid, m, nf, inv_h, 0);
    if (ftab)
      v *= static_cast<double>(ftab[static_cast<size_t>(ei) * nq + m]) *
           static_cast<double>(ftab[static_cast<size_t>(ej) * nq + m]);
    total += v;
    if (++ej > ei) {
      ++ei;
      ej = 0;
    }
  }
  const size_t o = static_cast<size_t>(b) * nq + m;
  const double v = total * fscale[o];
  if (out64) out64[o] = v;
  if (out32) out32[o] = static_cast<float>(v);
}

// Bound of the distances between the block's positions x[3] per call of get(a):
// the diameter of the sphere about the middle of their box.  Waves reduce by
// shuffles, then each reduces the waves' values the same way.  Latency and the
// shuffles of the waves on one CU bound it, so few waves: with the packing 3.9 us
// at 55 atoms (1 wave), 4.4 at 300 (4), 6.9 at 1,500 (8), where 16 waves that
// each read all waves' values took 9 to 10.
template <typename G>
__device__ double block_reach(G get, int n) {
  __shared__ double box[16][6];
  __shared__ double rad[16];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, n_wave = blockDim.x >> 6;
  double v[6];  // max of x, y, z and of -x, -y, -z
  for (int k = 0; k < 6; ++k) v[k] = -1e308;
  bool bad = false;
  for (int a = threadIdx.x; a < n; a += blockDim.x) {
    double x[3];
    get(a, x);
    for (int k = 0; k < 3; ++k) {
      bad = bad || !(fabs(x[k]) < 1e150);
      v[k] = fmax(v[k], x[k]);
      v[k + 3] = fmax(v[k + 3], -x[k]);
    }
  }
  for (int off = 32; off > 0; off >>= 1)
    for (int k = 0; k < 6; ++k) v[k] = fmax(v[k], __shfl_xor(v[k], off, 64));
  if (lane == 0)
    for (int k = 0; k < 6; ++k) box[wave][k] = v[k];
  const int any_bad = __syncthreads_or(bad ? 1 : 0);
  if (n_wave > 1) {
    const int w = min(lane & 15, n_wave - 1);
    for (int k = 0; k < 6; ++k) v[k] = box[w][k];
    for (int off = 8; off > 0; off >>= 1)
      for (int k = 0; k < 6; ++k) v[k] = fmax(v[k], __shfl_xor(v[k], off, 64));
  }
  double r2 = 0.0;
  for (int a = threadIdx.x; a < n; a += blockDim.x) {
    double x[3];
    get(a, x);
    double d = 0.0;
    for (int k = 0; k < 3; ++k) d += (x[k] - 0.5 * (v[k] - v[k + 3])) * (x[k] - 0.5 * (v[k] - v[k + 3]));
    r2 = fmax(r2, d);
  }
  for (int off = 32; off > 0; off >>= 1) r2 = fmax(r2, __shfl_xor(r2, off, 64));
  if (lane == 0) rad[wave] = r2;
  __syncthreads();
  if (n_wave > 1) {
    r2 = rad[min(lane & 15, n_wave - 1)];
    for (int off = 8; off > 0; off >>= 1) r2 = fmax(r2, __shfl_xor(r2, off, 64));
  }
  return any_bad ? __builtin_inf() : 2.0 * sqrt(r2) * 1.000001;
}

__global__ __launch_bounds__(1024) void reach_kernel(const AtomRec* __restrict__ pos, int n,
                                                     double* __restrict__ reach) {
  const double r = block_reach(
      [&](int a, double* x) {
        const AtomRec p = pos[a];
        x[0] = p.x;
        x[1] = p.y;
        x[2] = p.z;
      },
      n);
  if (threadIdx.x == 0) *reach = r;
}

__device__ __forceinline__ void pack_one(const float* __restrict__ p, const int32_t* __restrict__ e,
                                         int64_t i, AtomRec* __restrict__ out,
                                         float* __restrict__ keep, const int32_t* __restrict__ place,
                                         AtomRec* __restrict__ ordered) {
  const float x = p[3 * i + 0], y = p[3 * i + 1], z = p[3 * i + 2];
  AtomRec a;
  a.x = x;
  a.y = y;
  a.z = z;
  a.w = static_cast<double>(e[i]);
  out[i] = a;
  if (place) ordered[place[i]] = a;
  if (keep) {
    keep[3 * i + 0] = x;
    keep[3 * i + 1] = y;
    keep[3 * i + 2] = z;
  }
}

__global__ void pack_kernel(const float* __restrict__ p, const int32_t* __restrict__ e, int64_t n,
                            AtomRec* __restrict__ out, float* __restrict__ keep,
                            const int32_t* __restrict__ place, AtomRec* __restrict__ ordered) {
  const int64_t i = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (i < n) pack_one(p, e, i, out, keep, place, ordered);
}

__global__ __launch_bounds__(1024) void pack_reach_kernel(const float* __restrict__ p,
                                                          const int32_t* __restrict__ e, int n,
                                                          AtomRec* __restrict__ out,
                                                          float* __restrict__ keep,
                                                          double* __restrict__ reach,
                                                          const int32_t* __restrict__ place,
                                                          AtomRec* __restrict__ ordered) {
  for (int i = threadIdx.x; i < n; i += blockDim.x)
    pack_one(p, e, i, out, keep, place, ordered);
  const double r = block_reach(
      [&](int a, double* x) {
        for (int k = 0; k < 3; ++k) x[k] = p[3 * a + k];
      },
      n);
  if (threadIdx.x == 0) *reach = r;
}

__global__ void gather_kernel(const AtomRec* __restrict__ pos, const int32_t* __restrict__ perm,
                              int n, AtomRec* __restrict__ out) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p < n) out[p] = pos[perm[p]];
}

}  // namespace

int fq_grid_points(int nq) { return 6 * nq + 7; }
int fq_grid_stride(int nq) { return (fq_grid_points(nq) + kFqNodes + 2) & ~1; }
int fq_scale_bits(int nq, double dq, double r_max) {
  const double t = r_max * dq * 12.0 * nq / (2.0 * M_PI);
  if (!(t < 1e30)) return kFqMinScale;
  int e = kFqMinScale;
  while (e < kFqMaxScale && std::ldexp(1.0, e - kFqBits) < t) ++e;
  return e;
}

hipError_t launch_spread_fq(hipStream_t st, const AtomRec* pos, const SpreadUnit* units,
                            int n_units, const SpreadItem* items, int nq, double dq, int shift,
                            int scale_bits, unsigned long long* grids) {
  if (n_units == 0) return hipSuccess;
  const int nf = 12 * nq, stride = fq_grid_stride(nq);
  const size_t lds = sizeof(unsigned long long) * static_cast<size_t>(stride);
  if (lds > kSpreadLds) return hipErrorInvalidValue;
  static LdsLimit lds_limit;
  const hipError_t attr = lds_limit.allow({reinterpret_cast<const void*>(spread_fq_kernel)}, kSpreadLds);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(spread_fq_kernel, dim3(n_units), dim3(1024), lds, st, pos, units, items,
                     dq * nf / (2.0 * M_PI), nf, fq_grid_points(nq), stride, shift,
                     std::ldexp(1.0f, scale_bits), std::ldexp(1.0, scale_bits - 31), grids);
  return hipGetLastError();
}

// About 512 blocks, and at least 32 grid points for each of a block's waves.
int fq_transform_parts(int nq, int n_chain, int n_pair) {
  const int64_t blocks = static_cast<int64_t>((nq + 63) / 64) * n_chain * n_pair;
  return static_cast<int>(
      std::max<int64_t>(1, std::min<int64_t>((512 + blocks - 1) / blocks, fq_grid_points(nq) / 512)));
}

hipError_t launch_transform_fq(hipStream_t st, unsigned long long* grids, int n_chain, int n_pair,
                               bool weighted, const float* ftab, int nq, double dq, int shift,
                               int scale_bits, const double* scale, double* part, double* out_f64,
                               float* out_f32, bool one_part) {
  const int nf = 12 * nq, stride = fq_grid_stride(nq);
  const int n_split = one_part ? 1 : fq_transform_parts(nq, n_chain, n_pair);
  const double inv_h = dq * nf / (2.0 * M_PI);
  if (n_chain > 65535 || n_pair * n_split > 65535) return hipErrorInvalidValue;
  hipLaunchKernelGGL(transform_fq_kernel, dim3((nq + 63) / 64, n_chain, n_pair * n_split),
                     dim3(1024), 0, st, grids, n_pair, n_split, nf, fq_grid_points(nq), stride,
                     shift, fq_unit(inv_h, shift, scale_bits), ftab, nq, inv_h, weighted ? 1 : 0,
                     one_part ? nullptr : part, scale, out_f64, out_f32);
  if (one_part) return hipGetLastError();
  const int64_t total = static_cast<int64_t>(n_chain) * nq;
  const int64_t words2 = static_cast<int64_t>(n_chain) * n_pair * stride / 2;  // stride is even
  const int64_t n_out = (total + 255) / 256;
  const int64_t n_clear = std::min<int64_t>((words2 + 511) / 512, 1024);
  hipLaunchKernelGGL(finish_fq_kernel, dim3(static_cast<unsigned>(n_out + n_clear)), dim3(256), 0,
                     st, part, n_pair * n_split, nq, total, static_cast<int>(n_out), scale, out_f64,
                     out_f32, reinterpret_cast<ulonglong2*>(grids), words2);
  return hipGetLastError();
}

size_t small_fq_lds(int nq, int n_pair) {
  return sizeof(unsigned long long) * static_cast<size_t>(fq_grid_stride(nq)) * n_pair;
}

hipError_t launch_small_fq(hipStream_t st, const AtomRec* pos, const int* off, int n_chain,
                           int n_pair, bool weighted, const float* ftab, int nq, double dq,
                           int scale_bits, const double* scale, double* out_f64, float* out_f32) {
  const int nf = 12 * nq, stride = fq_grid_stride(nq);
  const double inv_h = dq * nf / (2.0 * M_PI);
  const size_t lds = small_fq_lds(nq, n_pair);
  if (lds > kSmallFqLds || n_chain > 65535 || (n_pair != 1 && n_pair != 3 && n_pair != 6))
    return hipErrorInvalidValue;
  static LdsLimit lds_limit;
  const hipError_t attr = lds_limit.allow({reinterpret_cast<const void*>(small_fq_kernel<1>),
                                           reinterpret_cast<const void*>(small_fq_kernel<3>),
                                           reinterpret_cast<const void*>(small_fq_kernel<6>)},
                                          kSmallFqLds);
  if (attr != hipSuccess) return attr;
  const dim3 grid((nq + 63) / 64, n_chain), block(64 * kSmallWaves);
  const double unit = fq_unit(inv_h, 0, scale_bits), near = std::ldexp(1.0, scale_bits - 31);
  const float one = std::ldexp(1.0f, scale_bits);
  const float* f = weighted ? ftab : nullptr;
#define PYIID_SMALL(N)                                                                            \
  hipLaunchKernelGGL(small_fq_kernel<N>, grid, block, lds, st, pos, off, nf, fq_grid_points(nq),  \
                     stride, unit, one, near, f, nq, inv_h, scale, out_f64, out_f32)
  if (n_pair == 1)
    PYIID_SMALL(1);
  else if (n_pair == 3)
    PYIID_SMALL(3);
  else
    PYIID_SMALL(6);
#undef PYIID_SMALL
  return hipGetLastError();
}

hipError_t launch_pack(hipStream_t st, const float* p, const int32_t* e, int64_t n, AtomRec* out,
                       float* keep, double* reach, const int32_t* place, AtomRec* ordered) {
  if (n == 0) return hipSuccess;
  if (reach && n <= kReachAtoms)
    hipLaunchKernelGGL(pack_reach_kernel, dim3(1), dim3(n <= 256 ? 64 : n <= 1024 ? 256 : 512), 0, st,
                       p, e, static_cast<int>(n), out, keep, reach, place, ordered);
  else
    hipLaunchKernelGGL(pack_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st,
                       p, e, n, out, keep, place, ordered);
  return hipGetLastError();
}

hipError_t launch_reach(hipStream_t st, const AtomRec* pos, int64_t n, double* reach) {
  hipLaunchKernelGGL(reach_kernel, dim3(1), dim3(1024), 0, st, pos, static_cast<int>(n), reach);
  return hipGetLastError();
}

hipError_t launch_gather(hipStream_t st, const AtomRec* pos, const int32_t* perm, int64_t n,
                         AtomRec* out) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(gather_kernel, dim3(static_cast<unsigned>((n + 255) / 256)), dim3(256), 0, st,
                     pos, perm, static_cast<int>(n), out);
  return hipGetLastError();
}

}  // namespace pyiid
