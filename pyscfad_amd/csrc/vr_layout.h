// Scratch layout of the V-bar reductions (k_vr) and the sums its readers take.
#pragma once
#include "ccsdt_common.h"

namespace pamd {

// Part s of kVRS of the b-sums (k_vr_a) and a-sums (k_vr_b): arrays that are
// sums over the split index are written per part; part 0 uses the slots of R
// listed above, parts 1.. an extension after them (vr_part, vr_part_vec).  The
// vectors have kVRS x ncb parts (index cb * kVRS + s); blocks 0, 1, 8, 9 have
// ncb parts (vr_cpart), column block cb >= 1 in a second extension.
__device__ __forceinline__ double *vr_part(double *R, int v, int s, int q) {
  const size_t vv = (size_t)v * v;
  if (s == 0) return R + (size_t)q * vv;
  return R + 10 * vv + 2 * (size_t)v + ((size_t)(s - 1) * 6 + (q - 2)) * vv;
}
__device__ __forceinline__ double *vr_part_vec(double *R, int v, int s, int which) {
  const size_t vv = (size_t)v * v;
  if (s == 0) return R + 10 * vv + (size_t)which * v;
  return R + 10 * vv + 2 * (size_t)v + (size_t)(kVRS - 1) * 6 * vv + ((size_t)(s - 1) * 2 + which) * v;
}
__device__ __forceinline__ double *vr_cpart(double *R, int v, int cb, int q) {
  const size_t vv = (size_t)v * v;
  if (cb == 0) return R + (size_t)q * vv;
  const int slot = q < 2 ? q : q - 6;  // 0, 1, 8, 9 -> 0, 1, 2, 3
  return R + 10 * vv + 2 * (size_t)v + (size_t)(kVRS - 1) * 6 * vv +
         (size_t)(kVRS * vr_col_blocks(v) - 1) * 2 * v + ((size_t)(cb - 1) * 4 + slot) * vv;
}

// sums over the parts, in part order
__device__ __forceinline__ double vr_sum(const double *R, int v, int q, size_t idx) {
  double x = 0.0;
#pragma unroll
  for (int s = 0; s < kVRS; ++s) x += vr_part(const_cast<double *>(R), v, s, q)[idx];
  return x;
}
__device__ __forceinline__ double vr_sum_vec(const double *R, int v, int which, int idx) {
  double x = 0.0;
  const int np = kVRS * vr_col_blocks(v);
  for (int s = 0; s < np; ++s) x += vr_part_vec(const_cast<double *>(R), v, s, which)[idx];
  return x;
}
__device__ __forceinline__ double vr_csum(const double *R, int v, int q, size_t idx) {
  double x = 0.0;
  const int ncb = vr_col_blocks(v);
  for (int cb = 0; cb < ncb; ++cb) x += vr_cpart(const_cast<double *>(R), v, cb, q)[idx];
  return x;
}

}  // namespace pamd
