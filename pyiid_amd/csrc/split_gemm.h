// FP32 products on the FP16 matrix cores (gfx950, wave64), shared by
// gradspread.hip and transform.hip.
//
// An operand is split into two halves, x = hi + lo, each 11 bits, its rows scaled
// by powers of two: hi hi + hi lo + lo hi in FP32 leaves 2^-22 of an entry, at
// three FP16 products for one in FP32, whose matrix rate is 16 times lower.
// Sums leave the MFMA accumulators every 128 points: a single FP32 chain over
// a row rounds at the size of its running sum, and left the gradient 3.9e-7 off
// at 6,699 atoms (1.8e-7 with it).
#pragma once

#include "internal.h"

namespace pyiid {
namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));

// Element k of row r of an operand of row_len points (a multiple of 32), its lo
// half 32 elements on: tiles of 128 rows, in them steps of 32 points, in them a
// line of 32 hi and 32 lo values per row, so that what a block reads in a step is
// contiguous.
__host__ __device__ __forceinline__ size_t split_at(size_t r, int k, int row_len) {
  return ((r >> 7) * (row_len >> 5) + (k >> 5)) * (128 * 64) + (r & 127) * 64 + (k & 31);
}

constexpr int kFold = 4;  // steps of 32 points between folds

// A block of 4 waves makes 128 x 128 results (2 x 2 MFMA tiles a wave), where
// these fill the chip, two blocks per CU; else one of 8 waves makes 128 x 64 (one
// tile a wave).  F and gradient, among others: 6,699 atoms, 1,250 bins (1,570
// tiles of 128 x 128) 541 and 561 us, 3,000 atoms, 800 bins (497) 145 and 143,
// 1,289 atoms, 330 bins (93) 37 and 33, one alone 84 and 63.
inline bool split_large(int64_t rows, int64_t cols) {
  return (rows + 127) / 128 * ((cols + 127) / 128) >= 512;
}

// LDS bytes of a block of WM x WN waves, each of MX x NY tiles.
template <int WM, int WN, int MX, int NY>
constexpr int split_lds() {
  return 2 * 32 * (WM * MX + WN * NY) * 128;
}

// Rows [bm, bm + 32 WM MX) of a (m rows for each of n_run runs) times rows
// [bn, bn + 32 WN NY) of b, nk steps of 32 points of each run: WM x WN waves of
// MX x NY tiles (MFMA 32x32x16 in FP16, three products each), steps through
// double-buffered LDS.  A row's line of a step is 128 bytes, whose eight 16-byte
// chunks are permuted in LDS (chunk ^ row / 2 mod 8), so that the 16 rows which are
// read together meet different banks.  fold(run, acc) is called every kFold steps
// and at the end of a run; at_run(run) before a run's first step, with a
// barrier behind it.  Rows past the operands' ends (up to a multiple of 128)
// are read and their results left out.
//
// What bounds it (128 x 128, 60,000 rows, 1,500 columns, two runs): the matrix
// cores are busy for 45% of the time, and for 66% without the loads and LDS
// writes; products, LDS and loads together also lower the clock from 2.15 to
// 1.9 GHz.  2.58 -> 2.36 ms by conflict-free reads, contiguous loads and the
// operands of one half of a step coming in during the other's products.
// Operand layout (lane l): A[l % 32][8 (l / 32) + i], B likewise; result
// register v: row v % 4 + 8 (v / 4) + 4 (l / 32), column l % 32.
template <int WM, int WN, int MX, int NY, class Fold, class AtRun>
__device__ __forceinline__ void split_product(const _Float16* __restrict__ a, int m,
                                              const _Float16* __restrict__ b, int row_len, int nk,
                                              int n_run, int bm, int bn, unsigned char* lds,
                                              Fold fold, AtRun at_run) {
  constexpr int kStride = WM * WN * 8;  // rows that the block's threads move together
  constexpr int kRa = 32 * WM * MX / kStride, kRb = 32 * WN * NY / kStride;
  constexpr int kA = 32 * WM * MX * 128, kBuf = kA + 32 * WN * NY * 128;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  constexpr int kStep = 128 * 128;  // bytes of a step of a tile of rows
  const int wm = wave / WN, wn = wave % WN;
  // a thread moves chunk threadIdx.x % 8 of rows threadIdx.x / 8 + kStride s; the
  // block's rows of each operand lie in one tile of 128
  static_assert(32 * WM * MX <= 128 && 32 * WN * NY <= 128, "a tile of rows");
  const int chunk = threadIdx.x & 7, trow = threadIdx.x >> 3;
  const unsigned mine = trow * 128 + chunk * 16;
  const char* next_a = reinterpret_cast<const char*>(a + split_at(bm, 0, row_len));
  const char* next_b = reinterpret_cast<const char*>(b + split_at(bn, 0, row_len));
  const size_t skip = (static_cast<size_t>((m + 127) / 128) * (row_len >> 5) - nk) * kStep;
  int left = nk * n_run, ahead = 0;  // steps to load; the next one within its run
  v4u ra[kRa], rb[kRb];
  auto load = [&]() {
#pragma unroll
    for (int s = 0; s < kRa; ++s)
      ra[s] = *reinterpret_cast<const v4u*>(next_a + (mine + s * kStride * 128));
#pragma unroll
    for (int s = 0; s < kRb; ++s)
      rb[s] = *reinterpret_cast<const v4u*>(next_b + (mine + s * kStride * 128));
    --left;
    next_a += kStep;
    next_b += kStep;
    if (++ahead == nk) {
      ahead = 0;
      next_a += skip;
      next_b -= nk * kStep;
    }
  };
  unsigned char* put = lds + trow * 128 + (chunk ^ ((trow >> 1) & 7)) * 16;
  auto store = [&](int buf) {
#pragma unroll
    for (int s = 0; s < kRa; ++s) *reinterpret_cast<v4u*>(put + buf * kBuf + s * kStride * 128) = ra[s];
#pragma unroll
    for (int s = 0; s < kRb; ++s) *reinterpret_cast<v4u*>(put + buf * kBuf + kA + s * kStride * 128) = rb[s];
  };
  v16f acc[MX][NY];
  // chunk c of a lane's row: c = 2 h + lane / 32, its lo half 4 chunks on
  const int frow = lane & 31, sw = ((lane >> 5) ^ ((frow >> 1) & 7)) * 16;
  const unsigned char* get_a = lds + (wm * 32 * MX + frow) * 128;
  const unsigned char* get_b = lds + kA + (wn * 32 * NY + frow) * 128;
  struct Half {  // the operands of 16 of a step's 32 points
    v8h ah[MX], al[MX], bh[NY], bl[NY];
  } half[2];
  auto get = [&](int buf, int h) {
    const int hi = buf * kBuf + (sw ^ (h * 32)), lo = buf * kBuf + (sw ^ (h * 32 + 64));
#pragma unroll
    for (int x = 0; x < MX; ++x) {
      half[h].ah[x] = *reinterpret_cast<const v8h*>(get_a + x * 32 * 128 + hi);
      half[h].al[x] = *reinterpret_cast<const v8h*>(get_a + x * 32 * 128 + lo);
    }
#pragma unroll
    for (int y = 0; y < NY; ++y) {
      half[h].bh[y] = *reinterpret_cast<const v8h*>(get_b + y * 32 * 128 + hi);
      half[h].bl[y] = *reinterpret_cast<const v8h*>(get_b + y * 32 * 128 + lo);
    }
  };
  auto products = [&](int h, bool first) {
    // one product of every tile after another: neighbours are independent
#pragma unroll
    for (int z = 0; z < 3; ++z)
#pragma unroll
      for (int x = 0; x < MX; ++x)
#pragma unroll
        for (int y = 0; y < NY; ++y) {
          const v16f zero = {};
          acc[x][y] = __builtin_amdgcn_mfma_f32_32x32x16_f16(
              z == 0 ? half[h].al[x] : half[h].ah[x], z == 1 ? half[h].bl[y] : half[h].bh[y],
              first && z == 0 ? zero : acc[x][y], 0, 0, 0);
        }
  };
  load();
  store(0);
  if (left > 0) load();
  at_run(0);
  __syncthreads();
  get(0, 0);
  int buf = 0, todo = nk * n_run;
  // While one half's products run, the other half's operands come from LDS; the
  // barrier in the middle finds the next step stored and this one read.
  auto step = [&](bool first) {
    const bool more = --todo > 0;
    get(buf, 1);
    if (more) store(buf ^ 1);
    if (left > 0) load();
    __builtin_amdgcn_sched_barrier(0);
    products(0, first);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();
    if (more) get(buf ^ 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    products(1, false);
    __builtin_amdgcn_sched_barrier(0);
    buf ^= 1;
  };
  for (int run = 0; run < n_run; ++run) {
    for (int k0 = 0; k0 < nk; k0 += kFold) {
      const int k1 = min(k0 + kFold, nk);
      step(true);
      for (int k = k0 + 1; k < k1; ++k) step(false);
      fold(run, acc);
      if (k1 == nk && run + 1 < n_run) at_run(run + 1);
    }
  }
}

// Calls f(row of the tile, column of the tile, value) for the lane's results.
template <int WM, int WN, int MX, int NY, class F>
__device__ __forceinline__ void split_results(const v16f (&t)[MX][NY], F f) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int y = 0; y < NY; ++y)
#pragma unroll
    for (int x = 0; x < MX; ++x)
#pragma unroll
      for (int v = 0; v < 16; ++v)
        f((wave / WN) * 32 * MX + x * 32 + (v & 3) + 8 * (v >> 2) + 4 * (lane >> 5),
          (wave % WN) * 32 * NY + y * 32 + (lane & 31), t[x][y][v]);
}

}  // namespace
}  // namespace pyiid
