// F(Q) -> G(r) transform on the FP32 matrix cores, and the FP64 potential
// (Rw / chi^2) reductions with their adjoint vectors.
//
// The reference transform (kernels/master_kernel.py:39-203) is an odd-extended
// zero-padded inverse FFT followed by linear interpolation onto the r grid;
// it is exactly G = T . F with a dense R x Q matrix T (built on the host in
// FP64, stored here as FP32).  grad G = grad F . T^T runs on split operands
// (split_gemm.h), smaller products on v_mfma_f32_16x16x4_f32.
#include <algorithm>
#include <cmath>

#include "split_gemm.h"

namespace pyiid {
namespace {

using v4f = float __attribute__((ext_vector_type(4)));

// C[m][n] = sum_k A[m][k] * B[n][k] for few rows (F -> G of a batch of chains).
// Block: one 16 x 16 tile, its 4 waves a quarter of k each, added through LDS.
// The product is far too small for the chip (64 chains: 0.17 GFLOP), so what
// counts is the length of a block's chain: with 64 x 64 tiles staged through
// LDS it took 23 to 50 us, in 63 blocks of 21 barriers each; here a wave loads
// its operands straight from L2, 16 of k at a time, and runs 6 steps at 330
// bins.  Lane l holds k0 + 4 (l / 16) .. + 3 of row l % 16 of both operands and
// MFMA step s takes element s: any order of k gives the same sum.
template <bool A64>
__global__ __launch_bounds__(256) void gemm_rows_kernel(const void* __restrict__ a_raw, int64_t m,
                                                        int k, const float* __restrict__ b, int n,
                                                        double* __restrict__ c64,
                                                        float* __restrict__ c32) {
  __shared__ float red[3][4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int64_t bm = static_cast<int64_t>(blockIdx.y) * 16;
  const int bn = blockIdx.x * 16;
  const int64_t ar = min(bm + (lane & 15), m - 1);
  const int br = min(bn + (lane & 15), n - 1);
  const int steps = (k + 15) / 16;
  const int s0 = steps * wave / 4, s1 = steps * (wave + 1) / 4;
  v4f acc = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll 2
  for (int s = s0; s < s1; ++s) {
    const int kk = s * 16 + 4 * (lane >> 4);
    float av[4], bv[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool in = kk + e < k;
      const int at = in ? kk + e : 0;
      if constexpr (A64)
        av[e] = static_cast<float>(static_cast<const double*>(a_raw)[ar * k + at]);
      else
        av[e] = static_cast<const float*>(a_raw)[ar * k + at];
      bv[e] = b[static_cast<int64_t>(br) * k + at];
      av[e] = in ? av[e] : 0.f;
      bv[e] = in ? bv[e] : 0.f;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(av[e], bv[e], acc, 0, 0, 0);
  }
  if (wave != 0)
#pragma unroll
    for (int v = 0; v < 4; ++v) red[wave - 1][v][lane] = acc[v];
  __syncthreads();
  if (wave != 0) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const float t = ((acc[v] + red[0][v][lane]) + red[1][v][lane]) + red[2][v][lane];
    const int64_t row = bm + 4 * (lane >> 4) + v;
    const int col = bn + (lane & 15);
    if (row < m && col < n) {
      if (c64) c64[row * n + col] = static_cast<double>(t);
      if (c32) c32[row * n + col] = t;
    }
  }
}

// The same product for more rows: block tile 64 x 64, 4 waves of 32 x 32,
// each wave 2 x 2 MFMA 16x16x4 tiles; K staged through LDS 16 at a time.
// MFMA f32 16x16x4 operand layout (lane l): A[l%16][l/16], B[l/16][l%16];
// result register v holds C[4*(l/16)+v][l%16].
template <bool A64>
__global__ __launch_bounds__(256) void gemm_nt_kernel(const void* __restrict__ a_raw, int64_t m,
                                                      int k, const float* __restrict__ b, int n,
                                                      double* __restrict__ c64,
                                                      float* __restrict__ c32) {
  constexpr int KS = 16;
  __shared__ float as[64][KS + 1];
  __shared__ float bs[64][KS + 1];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t bm = static_cast<int64_t>(blockIdx.y) * 64;
  const int bn = blockIdx.x * 64;
  v4f acc[2][2];
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) acc[x][y] = v4f{0.f, 0.f, 0.f, 0.f};

  for (int k0 = 0; k0 < k; k0 += KS) {
    __syncthreads();
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int idx = threadIdx.x + e * 256;
      const int row = idx / KS, kk = idx % KS;
      const int64_t ar = bm + row;
      float av = 0.0f;
      if (ar < m && k0 + kk < k) {
        if constexpr (A64)
          av = static_cast<float>(static_cast<const double*>(a_raw)[ar * k + k0 + kk]);
        else
          av = static_cast<const float*>(a_raw)[ar * k + k0 + kk];
      }
      as[row][kk] = av;
      const int br = bn + row;
      bs[row][kk] = (br < n && k0 + kk < k) ? b[(int64_t)br * k + k0 + kk] : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < KS; kk += 4) {
      float af[2], bf[2];
#pragma unroll
      for (int x = 0; x < 2; ++x) af[x] = as[wm * 32 + x * 16 + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
      for (int y = 0; y < 2; ++y) bf[y] = bs[wn * 32 + y * 16 + (lane & 15)][kk + (lane >> 4)];
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[x], bf[y], acc[x][y], 0, 0, 0);
    }
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t row = bm + wm * 32 + x * 16 + 4 * (lane >> 4) + v;
        const int col = bn + wn * 32 + y * 16 + (lane & 15);
        if (row < m && col < n) {
          if (c64) c64[row * n + col] = static_cast<double>(acc[x][y][v]);
          if (c32) c32[row * n + col] = acc[x][y][v];
        }
      }
}

// The same product for tall A: block tile 128 x 128,
// 4 waves of 64 x 64 (4 x 4 MFMA 16x16x4 tiles), K in chunks of 16 through
// double-buffered LDS; the next chunk's global loads are in flight during the
// current chunk's MFMAs, one barrier per chunk.  Blocks are dispatched round
// robin to the 8 XCDs (block id mod 8); the block -> tile map gives each XCD
// its own column tiles, so the rows of B (the transform) that it reads stay
// in that XCD's L2 while it sweeps the row tiles.
constexpr int kG2 = 128, kG2K = 16, kG2Ld = kG2K + 1;

template <bool A64>
__global__ __launch_bounds__(256) void gemm_nt128_kernel(const void* __restrict__ a_raw,
                                                         int64_t m, int k,
                                                         const float* __restrict__ b, int n,
                                                         int n_ct, int64_t n_rt,
                                                         double* __restrict__ c64,
                                                         float* __restrict__ c32) {
  __shared__ float as[2][kG2 * kG2Ld];
  __shared__ float bs[2][kG2 * kG2Ld];
  const int64_t bid = blockIdx.x;
  const int ct_per = (n_ct + 7) / 8;
  const int ct = static_cast<int>(bid % 8) + 8 * static_cast<int>((bid / 8) % ct_per);
  const int64_t rt = (bid / 8) / ct_per;
  if (ct >= n_ct || rt >= n_rt) return;  // padding block (uniform, before any barrier)
  const int64_t bm = rt * kG2;
  const int bn = ct * kG2;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  float ra[8], rb[8];
  auto load = [&](int k0) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int idx = threadIdx.x + e * 256;
      const int row = idx / kG2K, kk = idx % kG2K;
      const int64_t ar = bm + row;
      float av = 0.0f;
      if (ar < m && k0 + kk < k) {
        if constexpr (A64)
          av = static_cast<float>(static_cast<const double*>(a_raw)[ar * k + k0 + kk]);
        else
          av = static_cast<const float*>(a_raw)[ar * k + k0 + kk];
      }
      ra[e] = av;
      const int br = bn + row;
      rb[e] = (br < n && k0 + kk < k) ? b[static_cast<int64_t>(br) * k + k0 + kk] : 0.0f;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int idx = threadIdx.x + e * 256;
      const int row = idx / kG2K, kk = idx % kG2K;
      as[buf][row * kG2Ld + kk] = ra[e];
      bs[buf][row * kG2Ld + kk] = rb[e];
    }
  };

  v4f acc[4][4];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y) acc[x][y] = v4f{0.f, 0.f, 0.f, 0.f};

  const int nk = (k + kG2K - 1) / kG2K;
  load(0);
  store(0);
  __syncthreads();
  for (int c = 0; c < nk; ++c) {
    const int cur = c & 1;
    if (c + 1 < nk) load((c + 1) * kG2K);
    const float* a_s = as[cur];
    const float* b_s = bs[cur];
#pragma unroll
    for (int kk = 0; kk < kG2K; kk += 4) {
      float af[4], bf[4];
#pragma unroll
      for (int x = 0; x < 4; ++x)
        af[x] = a_s[(wm * 64 + x * 16 + (lane & 15)) * kG2Ld + kk + (lane >> 4)];
#pragma unroll
      for (int y = 0; y < 4; ++y)
        bf[y] = b_s[(wn * 64 + y * 16 + (lane & 15)) * kG2Ld + kk + (lane >> 4)];
#pragma unroll
      for (int x = 0; x < 4; ++x)
#pragma unroll
        for (int y = 0; y < 4; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(af[x], bf[y], acc[x][y], 0, 0, 0);
    }
    if (c + 1 < nk) store(cur ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 4; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t row = bm + wm * 64 + x * 16 + 4 * (lane >> 4) + v;
        const int col = bn + wn * 64 + y * 16 + (lane & 15);
        if (row < m && col < n) {
          if (c64) c64[row * n + col] = static_cast<double>(acc[x][y][v]);
          if (c32) c32[row * n + col] = acc[x][y][v];
        }
      }
}

// ---- the gradient's transform on split operands ----

// Rows of a (m x k) as a split operand, each scaled so that its largest entry
// lies in [2^14, 2^15); scale gives the way back, or NaN for a row with an entry
// that is not finite or a largest one outside [1e-20, 1e20].  A wave per row.
template <bool A64>
__global__ __launch_bounds__(256) void split_rows_kernel(const void* __restrict__ a_raw, int64_t m,
                                                         int k, int row_len,
                                                         _Float16* __restrict__ rows,
                                                         float* __restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int64_t r = blockIdx.x * 4ll + (threadIdx.x >> 6);
  if (r >= m) return;
  auto at = [&](int i) {
    if constexpr (A64)
      return static_cast<float>(static_cast<const double*>(a_raw)[r * k + i]);
    else
      return static_cast<const float*>(a_raw)[r * k + i];
  };
  float top = 0.f;
  bool bad = false;
  for (int i = lane; i < k; i += 64) {
    const float v = fabsf(at(i));
    bad = bad || !(v <= 1e20f);
    top = fmaxf(top, v);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) top = fmaxf(top, __shfl_xor(top, off, 64));
  bad = __any(bad || (top > 0.f && top < 1e-20f));
  int e = 0;
  if (top > 0.f && !bad) (void)frexpf(top, &e);  // top in [2^(e-1), 2^e)
  const float up = ldexpf(1.0f, 15 - e);
  for (int i = lane; i < row_len; i += 64) {
    const float x = i < k && !bad ? at(i) * up : 0.f;
    const _Float16 hi = static_cast<_Float16>(x);
    const size_t o = split_at(r, i, row_len);
    rows[o] = hi;
    rows[o + 32] = static_cast<_Float16>(x - static_cast<float>(hi));
  }
  if (lane == 0) scale[r] = bad ? __builtin_nanf("") : ldexpf(1.0f, e - 15);
}

// c[r][t] = sum_q a[r][q] T[t][q] for the rows [r0, r0 + m) that split_rows_kernel
// made, against T split alike.  Rows it could not scale are summed as they are.
// 3,867 rows of 330 bins to 4,000 points (31 GFLOP in FP16, 124 MB of results):
// 65 us with the rows' split, against 136 us on the FP32 matrix cores, which
// reached 75 TFLOP/s of their 157.
template <int WM, int WN, int MX, int NY, bool A64>
__global__ __launch_bounds__(64 * WM * WN, 2) void gemm_grad_kernel(
    const _Float16* __restrict__ rows, const float* __restrict__ row_scale, int m,
    const _Float16* __restrict__ ts, const float* __restrict__ t_scale, int n, int row_len,
    const void* __restrict__ a_raw, const float* __restrict__ t, int k, int n_ct, int n_rt,
    double* __restrict__ c64) {
  __shared__ __align__(16) unsigned char tile[split_lds<WM, WN, MX, NY>()];
  __shared__ float rs[32 * WM * MX], cs[32 * WN * NY];
  // consecutive blocks of an XCD (block id mod 8) share a row tile
  const int rt = static_cast<int>(blockIdx.x / 8) / n_ct * 8 + static_cast<int>(blockIdx.x % 8);
  const int ct = static_cast<int>(blockIdx.x / 8) % n_ct;
  if (rt >= n_rt) return;  // padding block (uniform, before any barrier)
  const int bm = rt * 32 * WM * MX, bn = ct * 32 * WN * NY;
  v16f tot[MX][NY];
#pragma unroll
  for (int x = 0; x < MX; ++x)
#pragma unroll
    for (int y = 0; y < NY; ++y)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[x][y][v] = 0.f;
  auto at_run = [&](int) {
    const int i = threadIdx.x;
    if (i < 32 * WM * MX) rs[i] = row_scale[min(bm + i, m - 1)];
    if (i < 32 * WN * NY) cs[i] = t_scale[min(bn + i, n - 1)];
  };
  auto fold = [&](int, const v16f (&acc)[MX][NY]) {
#pragma unroll
    for (int x = 0; x < MX; ++x)
#pragma unroll
      for (int y = 0; y < NY; ++y)
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[x][y][v] += acc[x][y][v];
  };
  split_product<WM, WN, MX, NY>(rows, m, ts, row_len, row_len >> 5, 1, bm, bn, tile, fold, at_run);
  split_results<WM, WN, MX, NY>(tot, [&](int i, int j, float v) {
    const int r = bm + i, col = bn + j;
    if (r >= m || col >= n) return;
    float g = v * rs[i] * cs[j];
    if (rs[i] != rs[i] || cs[j] != cs[j]) {
      g = 0.f;
      for (int q = 0; q < k; ++q) {
        const size_t at = static_cast<size_t>(r) * k + q;
        const float av = A64 ? static_cast<float>(static_cast<const double*>(a_raw)[at])
                             : static_cast<const float*>(a_raw)[at];
        g = fmaf(av, t[static_cast<size_t>(col) * k + q], g);
      }
    }
    c64[static_cast<size_t>(r) * n + col] = static_cast<double>(g);
  });
}

// The block's sums of three values, in every thread (one pass through LDS).
__device__ void block_sum3(double& x, double& y, double& z, double (*sh)[16]) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    x += __shfl_xor(x, off, 64);
    y += __shfl_xor(y, off, 64);
    z += __shfl_xor(z, off, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __syncthreads();
  if (lane == 0) {
    sh[0][wave] = x;
    sh[1][wave] = y;
    sh[2][wave] = z;
  }
  __syncthreads();
  x = y = z = 0.0;
  const int nw = blockDim.x >> 6;
  for (int w = 0; w < nw; ++w) {
    x += sh[0][w];
    y += sh[1][w];
    z += sh[2][w];
  }
}

// The block's chain.  Rw: master_kernel.py:206-236; chi^2: :239-266; the adjoint
// w is d(potential)/d(gcalc) as get_grad_rw / get_grad_chi_sq apply it
// (:293-375): grad = gradG . w with
//   w = c * (s * res + (g.res)/(g.g) * (o - 2 a g)),
//   c = -value/|res|^2 (Rw) or -2 (chi^2), res = o - s g, a = optimal scale.
constexpr int kPotKeep = 6;
// mix (nullable): w as a combination of o and g, w = mix.x o + mix.y g.
__device__ __forceinline__ void potential_block(int potential, const double* __restrict__ o,
                                                const double* __restrict__ g, int n,
                                                double* __restrict__ out5, double* __restrict__ w,
                                                double2* __restrict__ mix, double (*sh)[16]) {
  // the thread's points stay in registers between the passes (kPotKeep of them;
  // longer arrays are read again)
  double ok[kPotKeep], gk[kPotKeep];
#pragma unroll
  for (int e = 0; e < kPotKeep; ++e) {
    const int t = threadIdx.x + e * 1024;
    ok[e] = t < n ? o[t] : 0.0;
    gk[e] = t < n ? g[t] : 0.0;
  }
  double go = 0.0, gg = 0.0, oo = 0.0;
  auto first = [&](double ot, double gt) {
    go += gt * ot;
    gg += gt * gt;
    oo += ot * ot;
  };
#pragma unroll
  for (int e = 0; e < kPotKeep; ++e) first(ok[e], gk[e]);
  for (int t = threadIdx.x + kPotKeep * 1024; t < n; t += 1024) first(o[t], g[t]);
  block_sum3(go, gg, oo, sh);
  const double a = go / gg;
  const double s = (a <= 0.0) ? 1.0 : a;
  double rr = 0.0, gr = 0.0, none = 0.0;
  auto second = [&](double ot, double gt) {
    const double res = ot - s * gt;
    rr += res * res;
    gr += gt * res;
  };
#pragma unroll
  for (int e = 0; e < kPotKeep; ++e)
    if (threadIdx.x + e * 1024 < n) second(ok[e], gk[e]);
  for (int t = threadIdx.x + kPotKeep * 1024; t < n; t += 1024) second(o[t], g[t]);
  block_sum3(rr, gr, none, sh);
  double value, coef;
  if (potential == 0) {
    value = (a <= 0.0) ? 1.0 : sqrt(rr / oo);
    coef = -value / rr;
  } else {
    value = rr;
    coef = -2.0;
  }
  if (w) {
    const double gfac = gr / gg;
    auto third = [&](int t, double ot, double gt) {
      const double res = ot - s * gt;
      w[t] = coef * (s * res + gfac * (ot - 2.0 * a * gt));
    };
#pragma unroll
    for (int e = 0; e < kPotKeep; ++e)
      if (threadIdx.x + e * 1024 < n) third(threadIdx.x + e * 1024, ok[e], gk[e]);
    for (int t = threadIdx.x + kPotKeep * 1024; t < n; t += 1024) third(t, o[t], g[t]);
  }
  if (threadIdx.x == 0) {
    out5[0] = value;
    out5[1] = s;
    out5[2] = a;
    out5[3] = rr;
    out5[4] = gr;
    if (mix) {
      const double gfac = gr / gg;
      *mix = double2{coef * (s + gfac), -coef * (s * s + 2.0 * a * gfac)};
    }
  }
}

__global__ __launch_bounds__(1024) void potential_kernel(int potential,
                                                         const double* __restrict__ o,
                                                         const double* __restrict__ g, int n,
                                                         double* __restrict__ out5,
                                                         double* __restrict__ w) {
  __shared__ double sh[3][16];
  potential_block(potential, o, g, n, out5, w, nullptr, sh);
}

__global__ void gemv_rows_kernel(const double* __restrict__ x, int64_t rows, int n,
                                 const double* __restrict__ w, double* __restrict__ y) {
  const int lane = threadIdx.x & 63;
  const int64_t row = blockIdx.x * (int64_t)(blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= rows) return;
  double acc = 0.0;
  for (int t = lane; t < n; t += 64) acc += x[row * n + t] * w[t];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off, 64);
  if (lane == 0) y[row] = acc;
}

// What the force table reads for bin q of chain b: u and, per element pair,
// (u f_I f_J Q, u f_I f_J).
__device__ __forceinline__ void put_u(double v, int b, int q, int nq, double dq,
                                      const float* __restrict__ ftab, int weighted, int n_pair,
                                      float* __restrict__ u, double2* __restrict__ coef) {
  const float uf = static_cast<float>(v);
  u[static_cast<size_t>(b) * nq + q] = uf;
  if (!coef) return;
  int ei = 0, ej = 0;
  for (int p = 0; p < n_pair; ++p) {
    double w = uf;
    if (weighted)
      w *= static_cast<double>(ftab[static_cast<size_t>(ei) * nq + q]) *
           static_cast<double>(ftab[static_cast<size_t>(ej) * nq + q]);
    coef[(static_cast<size_t>(b) * n_pair + p) * nq + q] = double2{w * (dq * q), w};
    if (++ej > ei) {
      ++ei;
      ej = 0;
    }
  }
}

// part[z][x][b][q] = sum over slice z of t of x[b][t] T[t][q] in FP64 (T float), on
// the FP64 matrix cores, for x the target o and the computed g: a block takes
// 16 chains x 16 bins, its 16 waves consecutive parts of its slice, 4 of t per
// MFMA, added in wave order through LDS.  All chains of a tile share the read of T.
// It is latency and the reach of a few CUs' loads that count (one block per 64
// bins and chain, reading T for each, took 25 us for one chain and 52 us for 64;
// the tiles in one slice 31 us): four slices give 84 blocks at 330 bins, and a
// wave has a group's loads in flight.
// Layout of v_mfma_f64_16x16x4 (lane l): A[l % 16][l / 16], B[l / 16][l % 16];
// result v: row 4 v + l / 16, column l % 16.
using v4d = double __attribute__((ext_vector_type(4)));
constexpr int kAdjWaves = 16;

__device__ __forceinline__ void adjoint_block(const float* __restrict__ t, int n_r, int nq,
                                              const double* __restrict__ o,
                                              const double* __restrict__ g, int n_chain, int bx,
                                              int by, int bz, double* __restrict__ part,
                                              double (*red)[8][64]) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int q = min(bx * 16 + (lane & 15), nq - 1);
  const int b = min(by * 16 + (lane & 15), n_chain - 1);
  // groups of 16 of t: lane l takes 4 (l / 16) .. + 3 of them, one in each of four
  // MFMAs (any order of t gives the same sum), so that the lanes of a chain read a
  // line of o and g
  const int groups = (n_r + 15) / 16;
  constexpr int kSub = kAdjointSlices * kAdjWaves;
  const int sub = bz * kAdjWaves + wave;
  const int s0 = static_cast<int>(static_cast<int64_t>(groups) * sub / kSub);
  const int s1 = static_cast<int>(static_cast<int64_t>(groups) * (sub + 1) / kSub);
  const double *ob = o + static_cast<size_t>(b) * n_r, *gb = g + static_cast<size_t>(b) * n_r;
  v4d acc_o = v4d{0.0, 0.0, 0.0, 0.0}, acc_g = acc_o;
  for (int s = s0; s < s1; ++s) {
    double x[4], z[4];
    float y[4];
    const int at = s * 16 + 4 * (lane >> 4);
    if (at + 3 < n_r) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        x[e] = ob[at + e];
        z[e] = gb[at + e];
        y[e] = t[static_cast<size_t>(at + e) * nq + q];
      }
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int i = min(at + e, n_r - 1);
        x[e] = at + e < n_r ? ob[i] : 0.0;
        z[e] = at + e < n_r ? gb[i] : 0.0;
        y[e] = at + e < n_r ? t[static_cast<size_t>(i) * nq + q] : 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const double tv = static_cast<double>(y[e]);
      acc_o = __builtin_amdgcn_mfma_f64_16x16x4f64(x[e], tv, acc_o, 0, 0, 0);
      acc_g = __builtin_amdgcn_mfma_f64_16x16x4f64(z[e], tv, acc_g, 0, 0, 0);
    }
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    red[wave][v][lane] = acc_o[v];
    red[wave][4 + v][lane] = acc_g[v];
  }
  __syncthreads();
  if (wave >= 8) return;
  double v = 0.0;  // wave v adds result v % 4 of factor v / 4
#pragma unroll
  for (int k = 0; k < kAdjWaves; ++k) v += red[k][wave][lane];
  const int row = by * 16 + 4 * (wave & 3) + (lane >> 4), col = bx * 16 + (lane & 15);
  if (row < n_chain && col < nq)
    part[(static_cast<size_t>(bz * 2 + (wave >> 2)) * n_chain + row) * nq + col] = v;
}

// The potential of every chain (the first n_chain blocks) and, beside it, the
// adjoint product: the adjoint vector w is a combination of o and g (mix), so
// T^T o and T^T g need not wait for the sums that w takes.  One after the other they
// took 14 us for one chain and 18 for 16 (4,000 points, 330 bins), together 9
// and 11.  The blocks behind clear the F grids for the next call.
__global__ __launch_bounds__(1024) void score_kernel(
    int potential, const double* __restrict__ o, const double* __restrict__ g, int n_r, int n_chain,
    double* __restrict__ out5, double2* __restrict__ mix, const float* __restrict__ t, int nq,
    int n_bx, int n_adj, double* __restrict__ part, ulonglong2* __restrict__ clear, int64_t clear2) {
  __shared__ union {
    double sh[3][16];
    double red[kAdjWaves][8][64];
  } lds;
  const int bid = blockIdx.x;
  if (bid < n_chain) {
    const size_t at = static_cast<size_t>(bid) * n_r;
    potential_block(potential, o + at, g + at, n_r, out5 + 5 * static_cast<size_t>(bid), nullptr,
                    mix + bid, lds.sh);
  } else if (bid < n_chain + n_adj) {
    const int a = bid - n_chain;
    adjoint_block(t, n_r, nq, o, g, n_chain, a % n_bx, a / n_bx / kAdjointSlices,
                  a / n_bx % kAdjointSlices, part, lds.red);
  } else {
    const int64_t first = bid - n_chain - n_adj;
    for (int64_t w = first * 1024 + threadIdx.x; w < clear2;
         w += (static_cast<int64_t>(gridDim.x) - n_chain - n_adj) * 1024)
      clear[w] = ulonglong2{0ull, 0ull};
  }
}

__global__ void adjoint_sum_kernel(const double* __restrict__ part, const double2* __restrict__ mix,
                                   int n_chain, int nq, const double* __restrict__ gscale, double dq,
                                   const float* __restrict__ ftab, int weighted, int n_pair,
                                   float* __restrict__ u, double2* __restrict__ coef) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x, b = blockIdx.y;
  if (q >= nq) return;
  const size_t e = static_cast<size_t>(b) * nq + q, total = static_cast<size_t>(n_chain) * nq;
  double vo = 0.0, vg = 0.0;
#pragma unroll
  for (int s = 0; s < kAdjointSlices; ++s) {
    vo += part[2 * s * total + e];
    vg += part[(2 * s + 1) * total + e];
  }
  put_u(fma(mix[b].x, vo, mix[b].y * vg) * gscale[e], b, q, nq, dq, ftab, weighted, n_pair, u, coef);
}

__global__ void adjoint_fq_kernel(int nq, int q_first, const double* __restrict__ w,
                                  const double* __restrict__ gscale, double dq,
                                  const float* __restrict__ ftab, int weighted, int n_pair,
                                  float* __restrict__ u, double2* __restrict__ coef) {
  const int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nq) return;
  put_u(q >= q_first ? w[q - q_first] * gscale[q] : 0.0, 0, q, nq, dq, ftab, weighted, n_pair, u,
        coef);
}

__global__ void f64_to_f32_kernel(const double* __restrict__ x, int64_t n, float* __restrict__ y) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x)
    y[e] = static_cast<float>(x[e]);
}

__global__ void f32_to_f64_kernel(const float* __restrict__ x, int64_t n, double* __restrict__ y) {
  for (int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; e < n;
       e += (int64_t)gridDim.x * blockDim.x)
    y[e] = static_cast<double>(x[e]);
}

int blocks_for(int64_t total, int block) {
  int64_t g = (total + block - 1) / block;
  if (g > 65536) g = 65536;
  if (g < 1) g = 1;
  return static_cast<int>(g);
}

}  // namespace

hipError_t launch_gemm_nt(hipStream_t st, const void* a, bool a_f64, int64_t m, int k,
                          const float* b, int n, double* c_f64, float* c_f32) {
  if (m >= 1024) {
    const int n_ct = (n + kG2 - 1) / kG2;
    const int64_t n_rt = (m + kG2 - 1) / kG2;
    const int64_t blocks = 8LL * ((n_ct + 7) / 8) * n_rt;
    if (blocks > 2147483647LL) return hipErrorInvalidValue;
    const dim3 grid(static_cast<unsigned>(blocks));
    if (a_f64)
      hipLaunchKernelGGL(gemm_nt128_kernel<true>, grid, dim3(256), 0, st, a, m, k, b, n, n_ct,
                         n_rt, c_f64, c_f32);
    else
      hipLaunchKernelGGL(gemm_nt128_kernel<false>, grid, dim3(256), 0, st, a, m, k, b, n, n_ct,
                         n_rt, c_f64, c_f32);
    return hipGetLastError();
  }
  if (m < 1) return hipSuccess;
  // few rows: many short blocks (66 rows of 330 bins to 4,000 points: 20 us, 29 in
  // 64 x 64 tiles); from 81 on the tiles read less (96 rows of 128 bins: 12 us, 14
  // in 16 x 16 tiles; 960 rows: 26, 110)
  if (m <= 80) {
    const dim3 grid((n + 15) / 16, static_cast<unsigned>((m + 15) / 16));
    if (a_f64)
      hipLaunchKernelGGL(gemm_rows_kernel<true>, grid, dim3(256), 0, st, a, m, k, b, n, c_f64, c_f32);
    else
      hipLaunchKernelGGL(gemm_rows_kernel<false>, grid, dim3(256), 0, st, a, m, k, b, n, c_f64, c_f32);
    return hipGetLastError();
  }
  const dim3 grid((n + 63) / 64, static_cast<unsigned>((m + 63) / 64));
  if (a_f64)
    hipLaunchKernelGGL(gemm_nt_kernel<true>, grid, dim3(256), 0, st, a, m, k, b, n, c_f64, c_f32);
  else
    hipLaunchKernelGGL(gemm_nt_kernel<false>, grid, dim3(256), 0, st, a, m, k, b, n, c_f64, c_f32);
  return hipGetLastError();
}

hipError_t launch_split_rows(hipStream_t st, const void* a, bool a_f64, int64_t m, int k, void* rows,
                             float* scale) {
  if (m < 1) return hipSuccess;
  const dim3 grid(static_cast<unsigned>((m + 3) / 4));
  const int len = split_row_len(k);
  if (a_f64)
    hipLaunchKernelGGL(split_rows_kernel<true>, grid, dim3(256), 0, st, a, m, k, len,
                       static_cast<_Float16*>(rows), scale);
  else
    hipLaunchKernelGGL(split_rows_kernel<false>, grid, dim3(256), 0, st, a, m, k, len,
                       static_cast<_Float16*>(rows), scale);
  return hipGetLastError();
}

hipError_t launch_gemm_grad(hipStream_t st, const void* rows, const float* row_scale, const void* a,
                            bool a_f64, int m, int k, const void* ts, const float* t_scale,
                            const float* t, int n, double* out) {
  const bool large = split_large(m, n);
  const int n_ct = large ? (n + 127) / 128 : (n + 63) / 64, n_rt = (m + 127) / 128;
  const int64_t blocks = 8ll * ((n_rt + 7) / 8) * n_ct;
  if (blocks > 2147483647LL) return hipErrorInvalidValue;
  const dim3 grid(static_cast<unsigned>(blocks));
#define PYIID_TILES(A64, WM, WN, MX, NY)                                                          \
  hipLaunchKernelGGL((gemm_grad_kernel<WM, WN, MX, NY, A64>), grid, dim3(64 * WM * WN), 0, st,    \
                     static_cast<const _Float16*>(rows), row_scale, m,                            \
                     static_cast<const _Float16*>(ts), t_scale, n, split_row_len(k), a, t, k,     \
                     n_ct, n_rt, out)
  if (large && a_f64)
    PYIID_TILES(true, 2, 2, 2, 2);
  else if (large)
    PYIID_TILES(false, 2, 2, 2, 2);
  else if (a_f64)
    PYIID_TILES(true, 4, 2, 1, 1);
  else
    PYIID_TILES(false, 4, 2, 1, 1);
#undef PYIID_TILES
  return hipGetLastError();
}

hipError_t launch_potential(hipStream_t st, int potential, const double* gobs,
                            const double* gcalc, int n, double* out5, double* w) {
  hipLaunchKernelGGL(potential_kernel, dim3(1), dim3(1024), 0, st, potential, gobs, gcalc, n, out5, w);
  return hipGetLastError();
}

hipError_t launch_gemv_rows(hipStream_t st, const double* x, int64_t rows, int n, const double* w,
                            double* y) {
  const int64_t blocks = (rows + 3) / 4;
  hipLaunchKernelGGL(gemv_rows_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, st, x,
                     rows, n, w, y);
  return hipGetLastError();
}

hipError_t launch_score(hipStream_t st, int potential, const double* gobs, const double* gcalc,
                        int n_r, int n_chain, double* out5, double2* mix, const float* t, int nq,
                        double* part, unsigned long long* clear, int64_t clear_words) {
  const int n_bx = (nq + 15) / 16;
  const int64_t n_adj = part ? static_cast<int64_t>(n_bx) * ((n_chain + 15) / 16) * kAdjointSlices : 0;
  const int64_t clear2 = clear ? clear_words / 2 : 0;  // an even number of words
  const int64_t n_clear = std::min<int64_t>((clear2 + 4095) / 4096, 256);
  const int64_t blocks = n_chain + n_adj + n_clear;
  if (blocks > 2147483647LL) return hipErrorInvalidValue;
  hipLaunchKernelGGL(score_kernel, dim3(static_cast<unsigned>(blocks)), dim3(1024), 0, st, potential,
                     gobs, gcalc, n_r, n_chain, out5, mix, t, nq, n_bx, static_cast<int>(n_adj), part,
                     reinterpret_cast<ulonglong2*>(clear), clear2);
  return hipGetLastError();
}

hipError_t launch_adjoint_sum(hipStream_t st, const double* part, const double2* mix, int n_chain,
                              int nq, const double* gscale, double dq, const float* ftab,
                              bool weighted, int n_pair, float* u, double2* coef) {
  hipLaunchKernelGGL(adjoint_sum_kernel, dim3((nq + 63) / 64, n_chain), dim3(64), 0, st, part, mix,
                     n_chain, nq, gscale, dq, ftab, weighted ? 1 : 0, n_pair, u, coef);
  return hipGetLastError();
}

hipError_t launch_adjoint_fq(hipStream_t st, int nq, int q_first, const double* w,
                             const double* gscale, double dq, const float* ftab, bool weighted,
                             int n_pair, float* u, double2* coef) {
  hipLaunchKernelGGL(adjoint_fq_kernel, dim3((nq + 255) / 256), dim3(256), 0, st, nq, q_first, w,
                     gscale, dq, ftab, weighted ? 1 : 0, n_pair, u, coef);
  return hipGetLastError();
}

hipError_t launch_f64_to_f32(hipStream_t st, const double* x, int64_t n, float* y) {
  hipLaunchKernelGGL(f64_to_f32_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, x, n, y);
  return hipGetLastError();
}

hipError_t launch_f32_to_f64(hipStream_t st, const float* x, int64_t n, double* y) {
  hipLaunchKernelGGL(f32_to_f64_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, x, n, y);
  return hipGetLastError();
}

}  // namespace pyiid
