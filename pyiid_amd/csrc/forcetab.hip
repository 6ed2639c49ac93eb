// Contracted forces from a table of the pair force (gfx950, wave64).
//
// Forces need sum_q u_q grad F(q) only, so a pair of elements (I, J) at
// distance r acts on its atoms with P(r) (q_i - q_j),
//   P(r) = sum_q u_q f_I f_J (Q cos(Q r) - sin(Q r) / r) / r^2,
// one function of r for all pairs of a chain and element pair.
//
//  1. force_table_kernel tabulates P on cells of width h = pi / (5 n_q dq) as
//     polynomials of degree 5 through the cell's Chebyshev nodes, where the Q
//     sums run in FP64.  The highest frequency turns by pi / 5 in a cell, so
//     the interpolation error is 2 (pi / 20)^6 / 6! = 4.2e-8 of its amplitude.
//  2. table_force_kernel forms every ordered pair's distance in FP64, reads
//     its cell's six coefficients from LDS and adds P (q_i - q_j) to atom i.
//
// A recurrence per pair and bin took 5.8 VALU instructions for each; the table
// takes 34 instructions per ordered pair, whatever the number of bins.
//
// Reference semantics (pyIID): calc_1d.py:78-95 through cpu_flat.py:117-153.
#include <cmath>
#include <type_traits>

#include "lds_limit.h"
#include "pair_math.h"

namespace pyiid {
namespace {

constexpr int kNodes = 6;

struct NodeFit {
  double y[kNodes];           // Chebyshev nodes on [-1/2, 1/2]
  double c[kNodes][kNodes];   // monomial coefficient k of the interpolant: sum_n c[k][n] P(y_n)
};

NodeFit node_fit() {
  NodeFit f;
  for (int n = 0; n < kNodes; ++n) f.y[n] = 0.5 * std::cos(M_PI * (2 * n + 1) / (2 * kNodes));
  for (int n = 0; n < kNodes; ++n) {
    // Lagrange basis polynomial of node n, expanded
    double p[kNodes] = {1.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    int deg = 0;
    for (int m = 0; m < kNodes; ++m) {
      if (m == n) continue;
      const double s = 1.0 / (f.y[n] - f.y[m]);
      ++deg;
      for (int k = deg; k >= 0; --k) p[k] = s * ((k > 0 ? p[k - 1] : 0.0) - f.y[m] * (k < deg ? p[k] : 0.0));
    }
    for (int k = 0; k < kNodes; ++k) f.c[k][n] = p[k];
  }
  return f;
}

constexpr int kTabSplit = 2;     // halves of a chunk of bins, side by side in a block
constexpr int kTabChunk = 1024;  // bins staged in LDS at a time (PARTS > 1)

// Block: CELLS cells x 6 nodes x 2 halves of every chunk of bins of one table
// (chain, element pair); a wave holds the cells of 64 / CELLS nodes, or PARTS parts
// of its half side by side.  sin and cos of Q r follow the FP64 three-term
// recurrence along Q from the part's first bin.  Tables of 64 chains are bound by
// their FP64 operations (PARTS = 1: the two starting phases of a chain of 165 bins
// are a few percent); a single table of 400 cells by the chain's length (PARTS = 4).
// TABLES tables of a block share the sines and cosines, half of the operations of
// one alone; their coefficients, the same for a whole wave, come by scalar loads,
// for LDS reads of every bin by every wave bound the kernel (256 tables of 2,100
// cells: one a block from LDS 208 us, by scalar loads 240, four from LDS 241, by
// scalar loads 127).
template <int CELLS, int PARTS, int TABLES>
__global__ __launch_bounds__(64 * kNodes * kTabSplit * CELLS * PARTS / 64) void force_table_kernel(
    const double2* __restrict__ coef, int nq, double dq, int n_table, int n_cell, double h, NodeFit fit,
    float4* __restrict__ t4, float2* __restrict__ t2) {
  constexpr int kNodesPer = 64 / (CELLS * PARTS);  // of a wave
  constexpr int kWaves = kNodes / kNodesPer;       // of a half
  __shared__ double val[kTabSplit][2][kNodes][CELLS * PARTS];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int in_cell = lane % CELLS, part = lane / CELLS % PARTS;
  const int node = wave % kWaves * kNodesPer + lane / (CELLS * PARTS), half = wave / kWaves;
  const int cell = blockIdx.x * CELLS + in_cell;
  const int sub = half * PARTS + part;
  const int table0 = blockIdx.y * TABLES;
  const double x = dq * ((cell + 0.5 + fit.y[node]) * h) / M_PI;  // phase per bin / pi
  double s1, c1;
  sincospi(x, &s1, &c1);
  const double k2 = 2.0 * c1;
  double a[TABLES] = {}, b[TABLES] = {};
  auto start = [&](int m, double& s, double& c, double& sp, double& cp) {
    s = 0.0;
    c = 1.0;
    if (m > 0) sincospi(x * m, &s, &c);
    sp = s * c1 - c * s1;  // one bin before
    cp = c * c1 + s * s1;
  };
  double s, c, sp, cp;
  if constexpr (TABLES > 1) {
    static_assert(PARTS == 1, "the bins are the wave's");
    const double2* w[TABLES];
#pragma unroll
    for (int k = 0; k < TABLES; ++k) w[k] = coef + static_cast<size_t>(min(table0 + k, n_table - 1)) * nq;
    const int lo = nq * half / kTabSplit, hi = nq * (half + 1) / kTabSplit;
    start(lo, s, c, sp, cp);
#pragma unroll 4
    for (int m = lo; m < hi; ++m) {
#pragma unroll
      for (int k = 0; k < TABLES; ++k) {
        a[k] = fma(w[k][m].x, c, a[k]);
        b[k] = fma(w[k][m].y, s, b[k]);
      }
      const double sn = fma(k2, s, -sp), cn = fma(k2, c, -cp);
      sp = s;
      cp = c;
      s = sn;
      c = cn;
    }
  } else {
    __shared__ double2 cf[kTabChunk];
    for (int m0 = 0; m0 < nq; m0 += kTabChunk) {
      const int cnt = min(kTabChunk, nq - m0);
      if (m0 > 0) __syncthreads();
      for (int m = threadIdx.x; m < cnt; m += blockDim.x)
        cf[m] = coef[static_cast<size_t>(table0) * nq + m0 + m];
      const int lo = cnt * sub / (kTabSplit * PARTS), hi = cnt * (sub + 1) / (kTabSplit * PARTS);
      start(m0 + lo, s, c, sp, cp);
      __syncthreads();
#pragma unroll 8
      for (int m = lo; m < hi; ++m) {
        a[0] = fma(cf[m].x, c, a[0]);
        b[0] = fma(cf[m].y, s, b[0]);
        const double sn = fma(k2, s, -sp), cn = fma(k2, c, -cp);
        sp = s;
        cp = c;
        s = sn;
        c = cn;
      }
    }
  }
#pragma unroll
  for (int k = 0; k < TABLES; ++k) {
    if (k > 0) __syncthreads();  // the table before is done
    val[half][0][node][part * CELLS + in_cell] = a[k];
    val[half][1][node][part * CELLS + in_cell] = b[k];
    __syncthreads();
    const int table = table0 + k;
    if (cell >= n_cell || half != 0 || part != 0 || table >= n_table) continue;
    double p = 0.0;
#pragma unroll
    for (int n = 0; n < kNodes; ++n) {
      const double inv = 1.0 / ((cell + 0.5 + fit.y[n]) * h);
      double an = 0.0, bn = 0.0;
#pragma unroll
      for (int q = 0; q < PARTS; ++q) {
        an += val[0][0][n][q * CELLS + in_cell] + val[1][0][n][q * CELLS + in_cell];
        bn += val[0][1][n][q * CELLS + in_cell] + val[1][1][n][q * CELLS + in_cell];
      }
      p = fma(fit.c[node][n], (an - bn * inv) * (inv * inv), p);
    }
    const size_t at = static_cast<size_t>(table) * n_cell + cell;
    // node k holds coefficient k: 0..3 in t4, 4 and 5 in t2
    if (node < 4)
      reinterpret_cast<float*>(t4 + at)[node] = static_cast<float>(p);
    else
      reinterpret_cast<float*>(t2 + at)[node - 4] = static_cast<float>(p);
  }
}

// P(r) beyond the table (an atom that has left the extent the table was made
// for): the sums themselves.
__device__ double pair_force_far(double r, const float* u, const float* fi,
                                             const float* fj, int nq, double dq, double* far_seen) {
  if (far_seen) *far_seen = 1.0;
  double s1, c1;
  sincos(dq * r, &s1, &c1);
  const double k2 = 2.0 * c1;
  double s = 0.0, sp = -s1, c = 1.0, cp = c1, a = 0.0, b = 0.0;
  for (int m = 0; m < nq; ++m) {
    const double w = fi ? static_cast<double>(u[m]) * fi[m] * fj[m] : static_cast<double>(u[m]);
    a = fma(w * (dq * m), c, a);
    b = fma(w, s, b);
    const double sn = fma(k2, s, -sp), cn = fma(k2, c, -cp);
    sp = s;
    cp = c;
    s = sn;
    c = cn;
  }
  return (a - b / r) / (r * r);
}

constexpr int kAhead = 3;
constexpr double kLeast = 1e-30;  // r^2 of an atom and itself: within float's range

// Block (16 waves): the unit's 64-position i tiles against its j range, its
// table in LDS.  Wave w takes tile w mod tiles and slice w / tiles of the
// range; a j atom's position is wave-uniform (scalar loads).  Each lane owns
// its atom: FP32 sums over 64 j atoms, FP64 across them, then across slices
// through LDS and across planes in reduce_force_kernel, in a fixed order.
//
// VALU issue bounds it: 34 instructions for 64 ordered pairs, 11 of them FP64 and 8
// conversions or roots, and one ds_read_b128 + ds_read_b64 gather.  The range check
// is on r^2, no check singles out the atom itself, and three pairs side by side
// in one basic block cover each other's latency: 64 chains of 5,000 atoms 1.64 ->
// 1.44 ms (two pairs 1.49, four, which spill, 1.70).  Forming
// every pair from both sides keeps the accumulators in registers: the
// exchange of unordered pairs between lanes would cost about as much as the
// distance saved.
__global__ __launch_bounds__(1024, 8) void table_force_kernel(
    const AtomRec* __restrict__ pos, const ForceUnit* __restrict__ units, int n_cell, double inv_h,
    const float4* __restrict__ t4, const float2* __restrict__ t2, const float* __restrict__ u,
    const float* __restrict__ ftab, int nq, double dq, int64_t n, double* __restrict__ part,
    const int32_t* __restrict__ perm, double conv, double* __restrict__ out,
    double* __restrict__ far_seen) {
  extern __shared__ __align__(16) unsigned char lds[];
  float4* l4 = reinterpret_cast<float4*>(lds);
  float2* l2 = reinterpret_cast<float2*>(lds + sizeof(float4) * static_cast<size_t>(n_cell));
  const ForceUnit un = units[blockIdx.x];
  {
    const float4* g4 = t4 + static_cast<size_t>(un.table) * n_cell;
    const float2* g2 = t2 + static_cast<size_t>(un.table) * n_cell;
    for (int e = threadIdx.x; e < n_cell; e += blockDim.x) {
      l4[e] = g4[e];
      l2[e] = g2[e];
    }
  }
  __syncthreads();
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  // (tiles and the block's waves are powers of two)
  const int tile_bits = __ffs(un.tiles) - 1, slice_bits = __ffs(blockDim.x >> 6) - 1 - tile_bits;
  const int n_slice = 1 << slice_bits;
  const int tile = wave & (un.tiles - 1), slice = wave >> tile_bits;
  const int i = un.i0 + tile * 64 + lane;
  const bool have = i < un.i1;
  const int64_t len = un.j1 - un.j0;
  // (wave-uniform, so that the j atoms come by scalar loads)
  const int jb = __builtin_amdgcn_readfirstlane(un.j0 + static_cast<int>(len * slice >> slice_bits));
  const int je = __builtin_amdgcn_readfirstlane(un.j0 + static_cast<int>(len * (slice + 1) >> slice_bits));
  const AtomRec pi = pos[have ? i : un.i0];
  // r^2 up to which a pair takes the table (half a cell short of its end, so that
  // rounding cannot lead past it)
  const double limit = (n_cell - 0.5) / inv_h * ((n_cell - 0.5) / inv_h);
  double gx = 0.0, gy = 0.0, gz = 0.0;
  bool far = false;
  float fx, fy, fz;
  auto pairs = [&](int j, auto count) {  // j .. side by side: loads and chains overlap
    constexpr int kN = decltype(count)::value;
    double dx[kN], dy[kN], dz[kN], r2[kN], t[kN];
    float y[kN], p[kN];
    float4 a[kN];
    float2 b[kN];
#pragma unroll
    for (int e = 0; e < kN; ++e) {
      dx[e] = pi.x - pos[j + e].x;
      dy[e] = pi.y - pos[j + e].y;
      dz[e] = pi.z - pos[j + e].z;
    }
#pragma unroll
    for (int e = 0; e < kN; ++e) {
      // (the atom itself and duplicates: a finite P times a zero difference)
      r2[e] = fma(dx[e], dx[e], fma(dy[e], dy[e], fma(dz[e], dz[e], kLeast)));
      t[e] = scaled_root(r2[e], inv_h);
    }
#pragma unroll
    for (int e = 0; e < kN; ++e) {
      y[e] = static_cast<float>(__builtin_amdgcn_fract(t[e])) - 0.5f;
      const int cell = r2[e] < limit ? static_cast<int>(t[e]) : 0;
      a[e] = l4[cell];
      b[e] = l2[cell];
    }
#pragma unroll
    for (int e = 0; e < kN; ++e) {
      p[e] = fmaf(fmaf(fmaf(fmaf(fmaf(b[e].y, y[e], b[e].x), y[e], a[e].w), y[e], a[e].z), y[e],
                       a[e].y), y[e], a[e].x);
      far = far || r2[e] >= limit;
      p[e] = r2[e] < limit ? p[e] : 0.f;
      fx = fmaf(p[e], static_cast<float>(dx[e]), fx);
      fy = fmaf(p[e], static_cast<float>(dy[e]), fy);
      fz = fmaf(p[e], static_cast<float>(dz[e]), fz);
    }
  };
  for (int j0 = jb; j0 < je; j0 += 64) {
    const int j1 = min(je, j0 + 64);
    fx = fy = fz = 0.f;
    int j = j0;
    for (; j + kAhead <= j1; j += kAhead) pairs(j, std::integral_constant<int, kAhead>());
    for (; j < j1; ++j) pairs(j, std::integral_constant<int, 1>());
    gx += static_cast<double>(fx);
    gy += static_cast<double>(fy);
    gz += static_cast<double>(fz);
  }
  if (far) {  // atoms that have left the extent the table was made for
    const float* uc = u + static_cast<size_t>(un.chain) * nq;
    const float* fi = un.ei < 0 ? nullptr : ftab + static_cast<size_t>(un.ei) * nq;
    const float* fj = un.ei < 0 ? nullptr : ftab + static_cast<size_t>(un.ej) * nq;
    for (int j = jb; j < je; ++j) {
      const double dx = pi.x - pos[j].x, dy = pi.y - pos[j].y, dz = pi.z - pos[j].z;
      const double r2 = fma(dx, dx, fma(dy, dy, fma(dz, dz, kLeast)));
      if (!(r2 >= limit)) continue;
      const double p = pair_force_far(sqrt(r2), uc, fi, fj, nq, dq, far_seen);
      gx = fma(p, dx, gx);
      gy = fma(p, dy, gy);
      gz = fma(p, dz, gz);
    }
  }
  if (n_slice > 1) {
    __syncthreads();  // the table is no longer read
    double* red = reinterpret_cast<double*>(lds);
    double* mine = red + (static_cast<size_t>(wave) * 64 + lane) * 3;
    mine[0] = gx;
    mine[1] = gy;
    mine[2] = gz;
    __syncthreads();
    if (slice != 0) return;
    for (int k = 1; k < n_slice; ++k) {
      const double* o = red + (static_cast<size_t>(k * un.tiles + tile) * 64 + lane) * 3;
      gx += o[0];
      gy += o[1];
      gz += o[2];
    }
  }
  if (have) {
    double* o = out ? out + static_cast<size_t>(perm ? perm[i] : i) * 3
                    : part + (static_cast<size_t>(un.plane) * n + i) * 3;
    const double f = out ? conv : 1.0;
    o[0] = f * gx;
    o[1] = f * gy;
    o[2] = f * gz;
  }
}

// out[perm[p]][c] = conv * sum over the position's planes
__global__ void reduce_force_kernel(const double* __restrict__ part, int64_t n,
                                    const int32_t* __restrict__ planes,
                                    const int32_t* __restrict__ perm, double conv,
                                    double* __restrict__ out) {
  const int64_t e = blockIdx.x * static_cast<int64_t>(blockDim.x) + threadIdx.x;
  if (e >= 3 * n) return;
  const int64_t p = e / 3;
  double s = 0.0;
  const int np = planes[p];
  for (int k = 0; k < np; ++k) s += part[static_cast<size_t>(k) * n * 3 + e];
  out[static_cast<size_t>(perm ? perm[p] : p) * 3 + (e - 3 * p)] = conv * s;
}

}  // namespace

double force_cell(int nq, double dq) { return M_PI / (5.0 * std::max(1, nq) * dq); }

size_t force_lds_bytes(int64_t n_cell) {
  const size_t table = (sizeof(float4) + sizeof(float2)) * static_cast<size_t>(n_cell);
  const size_t red = sizeof(double) * 16 * 64 * 3;
  return table > red ? table : red;
}

hipError_t launch_force_table(hipStream_t st, const double2* coef, int nq, double dq, int n_table,
                              int n_cell, float4* t4, float2* t2) {
  static const NodeFit fit = node_fit();
  // four parts while their blocks fit the chip at once (two per CU): 10 us
  // instead of 16 for one table of 1,600 cells; beyond, the starting phases of
  // the parts cost more than the shorter chains save (16 tables of 1,080 cells:
  // 20 us against 15).  Up to about four blocks of 64 cells per CU half blocks
  // leave the CUs more even (14.0 us against 15.4).  Many tables go by fours (64 of
  // 2,400 cells: 50 us against 70)
  const int64_t blocks = static_cast<int64_t>((n_cell + 63) / 64) * n_table;
#define PYIID_TABLE(CELLS, PARTS, TABLES)                                                        \
  hipLaunchKernelGGL((force_table_kernel<CELLS, PARTS, TABLES>),                               \
                     dim3((n_cell + CELLS - 1) / CELLS, (n_table + TABLES - 1) / TABLES),      \
                     dim3(kNodes * kTabSplit * CELLS * PARTS), 0, st, coef, nq, dq, n_table,   \
                     n_cell, force_cell(nq, dq), fit, t4, t2)
  if (static_cast<int64_t>((n_cell + 15) / 16) * n_table <= 512)
    PYIID_TABLE(16, 4, 1);
  else if (blocks <= 1024)
    PYIID_TABLE(32, 1, 1);
  else if (blocks <= 2048)
    PYIID_TABLE(64, 1, 1);
  else
    PYIID_TABLE(64, 1, 4);
#undef PYIID_TABLE
  return hipGetLastError();
}

hipError_t launch_table_force(hipStream_t st, const AtomRec* pos, const ForceUnit* units,
                              int n_units, int n_cell, const float4* t4, const float2* t2,
                              const float* u, const float* ftab, int nq, double dq, int64_t n,
                              double* part, const int32_t* perm, double conv, double* out,
                              double* far_seen) {
  if (n_units == 0) return hipSuccess;
  const size_t lds = force_lds_bytes(n_cell);
  if (lds > kForceLds) return hipErrorInvalidValue;
  static LdsLimit lds_limit;
  const hipError_t attr = lds_limit.allow({reinterpret_cast<const void*>(table_force_kernel)}, kForceLds);
  if (attr != hipSuccess) return attr;
  hipLaunchKernelGGL(table_force_kernel, dim3(n_units), dim3(1024), lds, st, pos, units, n_cell,
                     1.0 / force_cell(nq, dq), t4, t2, u, ftab, nq, dq, n, part, perm, conv, out,
                     far_seen);
  return hipGetLastError();
}

hipError_t launch_reduce_force(hipStream_t st, const double* part, int64_t n,
                               const int32_t* planes, const int32_t* perm, double conv,
                               double* out) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(reduce_force_kernel, dim3(static_cast<unsigned>((3 * n + 255) / 256)),
                     dim3(256), 0, st, part, n, planes, perm, conv, out);
  return hipGetLastError();
}

}  // namespace pyiid
