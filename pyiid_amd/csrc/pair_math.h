// Device math shared by the kernels that handle each pair once (spread.hip,
// gradspread.hip, forcetab.hip).
#pragma once

#include "internal.h"

namespace pyiid {
namespace {

// t = r / h from r^2: r^2 z with z the FP32 inverse root, refined by one step in FP64
// with the scale in it (relative error 4e-14).  Where r^2 leaves float's range the
// result is not a number or below every positive t.
__device__ __forceinline__ double scaled_root(double r2, double inv_h) {
  const double z = static_cast<double>(__builtin_amdgcn_rsqf(static_cast<float>(r2)));
  const double a = r2 * z;
  return a * fma(fma(-a, z, 1.0), 0.5 * inv_h, inv_h);
}

// Nearest integer of a float below 2^31 (one instruction; ties upwards).
__device__ __forceinline__ int nearest(float v) {
  int r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

}  // namespace
}  // namespace pyiid
