// Device math shared by the kernels that handle each pair once (spread.hip,
// gradspread.hip, forcetab.hip).
#pragma once

#include "internal.h"

namespace pyiid {
namespace {

// t = r / h from r^2, the root refined from FP32 by one Newton step in FP64
// (relative error 1e-14; not a number where r^2 leaves float's range).
__device__ __forceinline__ double scaled_root(double r2, double inv_h) {
  const float r2f = static_cast<float>(r2);
  const float y0 = __builtin_amdgcn_rsqf(r2f);
  const float rf = r2f * y0;
  const double rd = static_cast<double>(rf);
  return fma(fma(-rd, rd, r2), static_cast<double>(0.5f * y0), rd) * inv_h;
}

// Nearest integer of a float below 2^31 (one instruction; ties upwards).
__device__ __forceinline__ int nearest(float v) {
  int r;
  asm("v_cvt_rpi_i32_f32 %0, %1" : "=v"(r) : "v"(v));
  return r;
}

}  // namespace
}  // namespace pyiid
