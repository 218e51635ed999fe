// 16x16x4 MFMA of one element type and the wave-level scalars of the small
// factorisations (gfx950).
#pragma once

#include "common.h"

namespace mbd {

// Both forms take one A and one B element per lane per K = 4 step:
//   A operand: lane l -> A[row l%16][k l/16], B operand: lane l -> B[k l/16][col l%16]
//   D: lane l -> D[row(l/16, v)][col l%16], v = 0..3
template <typename T>
struct Mfma;
template <>
struct Mfma<double> {
  using acc_t = v4d;
  __device__ static int row(int g, int v) { return g + 4 * v; }
  __device__ static acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
};
template <>
struct Mfma<float> {
  using acc_t = v4f;
  __device__ static int row(int g, int v) { return 4 * g + v; }
  __device__ static acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
};

// 1 / sqrt(x) and 1 / x for x > 0 from the hardware estimates refined by
// Newton steps (the correctly rounded square root and division are long
// dependent chains on the factorisations' critical path).  The last step adds
// a correction formed from the residual, an error of 1.5 units of 2^-53 (FP32:
// 2^-24) against 2 of 1 / sqrt(x) from the two rounded operations; the form
// y (3/2 - x y^2 / 2) of the same length has 2.5.
__device__ inline double rsq_fast(double x) {
  double y = __builtin_amdgcn_rsq(x);
  y = y * fma(-0.5 * x, y * y, 1.5);
  return fma(0.5 * y, fma(-(x * y), y, 1.0), y);
}
__device__ inline double rcp_fast(double x) {
  double r = __builtin_amdgcn_rcp(x);
  r = fma(r, fma(-x, r, 1.0), r);
  r = fma(r, fma(-x, r, 1.0), r);
  return r;
}
__device__ inline float rsq_fast(float x) {
  const float y = __builtin_amdgcn_rsqf(x);
  return fmaf(0.5f * y, fmaf(-(x * y), y, 1.0f), y);
}
__device__ inline float rcp_fast(float x) {
  float r = __builtin_amdgcn_rcpf(x);
  return fmaf(r, fmaf(-x, r, 1.0f), r);
}

// The value of lane src, wave-uniform.
__device__ inline double lane_value(double v, int src) {
  const unsigned long long u = (unsigned long long)__double_as_longlong(v);
  const unsigned lo = __builtin_amdgcn_readlane((unsigned)u, src);
  const unsigned hi = __builtin_amdgcn_readlane((unsigned)(u >> 32), src);
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ inline float lane_value(float v, int src) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), src));
}

}  // namespace mbd
