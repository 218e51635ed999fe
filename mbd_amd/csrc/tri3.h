// Products of a column-major matrix block, and of its transpose, with three
// right-hand sides in LDS, by one workgroup of kTriNT threads.
#pragma once

#include "common.h"

namespace mbd {

constexpr int kTriNT = 256, kTriU = 16;  // threads; columns in flight per thread
constexpr int kTriPW = kTriNT + 16;      // partial buffer row

// emit(r, s0, s1, s2) with s_b = sum_c M[r + c ld] x[b S + c] for r < rows:
// threads on rows, so loads are coalesced and nothing is reduced across
// lanes; few rows share their columns among 2 or 4 groups of threads.
template <typename T, typename F>
__device__ __forceinline__ void mv3(const T *__restrict__ M, long ld, int rows, int cols,
                                    const double *x, int S, double *P, F emit) {
  const int t = threadIdx.x;
  const int G = rows <= 64 ? 4 : (rows <= 128 ? 2 : 1), W = kTriNT / G;
  const int cw = (cols + G * kTriU - 1) / (G * kTriU) * kTriU, cb = min(cols, (t / W) * cw), ce = min(cols, cb + cw);
  for (int r0 = 0; r0 < rows; r0 += W) {
    const int r = r0 + t % W, rr = min(r, rows - 1);
    double s[3] = {0.0, 0.0, 0.0};
    for (int c = cb; c < ce; c += kTriU) {
      T v[kTriU];
#pragma unroll
      for (int i = 0; i < kTriU; ++i) v[i] = M[rr + (long)min(c + i, ce - 1) * ld];
      if (c + kTriU <= ce) {
#pragma unroll
        for (int i = 0; i < kTriU; ++i)
#pragma unroll
          for (int b = 0; b < 3; ++b) s[b] = fma((double)v[i], x[b * S + c + i], s[b]);
      } else {
        for (int i = 0; i < kTriU; ++i)
          if (c + i < ce)
#pragma unroll
            for (int b = 0; b < 3; ++b) s[b] = fma((double)v[i], x[b * S + c + i], s[b]);
      }
    }
    if (G > 1) {  // one pass over r0: rows <= W
#pragma unroll
      for (int b = 0; b < 3; ++b) P[b * kTriPW + t] = s[b];
      __syncthreads();
      if (t < W)
        for (int g = 1; g < G; ++g)
#pragma unroll
          for (int b = 0; b < 3; ++b) s[b] += P[b * kTriPW + g * W + t];
      if (t < W && r < rows) emit(r, s[0], s[1], s[2]);
      __syncthreads();
    } else if (r < rows) {
      emit(r, s[0], s[1], s[2]);
    }
  }
}

// emit(c, s0, s1, s2) with s_b = sum_r M[r + c ld] x[b S + r] for c < cols: a
// wave takes 16 columns, lanes on rows; at the end the 16 x 3 sums are halved
// four times across the lanes (51 exchanges instead of 6 for each).
template <typename T, typename F>
__device__ __forceinline__ void dot3(const T *__restrict__ M, long ld, int rows, int cols,
                                     const double *x, int S, F emit) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int c0 = kTriU * wave; c0 < cols; c0 += kTriU * (kTriNT / 64)) {
    double a[kTriU][3];
#pragma unroll
    for (int i = 0; i < kTriU; ++i)
#pragma unroll
      for (int b = 0; b < 3; ++b) a[i][b] = 0.0;
    for (int r0 = 0; r0 < rows; r0 += 64) {
      const int r = min(r0 + lane, rows - 1);
      const bool in = r0 + lane < rows;
      T v[kTriU];
#pragma unroll
      for (int i = 0; i < kTriU; ++i) v[i] = M[r + (long)min(c0 + i, cols - 1) * ld];
      double y[3];
#pragma unroll
      for (int b = 0; b < 3; ++b) y[b] = in ? x[b * S + r] : 0.0;
#pragma unroll
      for (int i = 0; i < kTriU; ++i)
#pragma unroll
        for (int b = 0; b < 3; ++b) a[i][b] = fma((double)v[i], y[b], a[i][b]);
    }
#pragma unroll
    for (int h = kTriU / 2, o = 32; h >= 1; h /= 2, o /= 2) {
      const bool up = lane & o;
#pragma unroll
      for (int i = 0; i < h; ++i)
#pragma unroll
        for (int b = 0; b < 3; ++b) {
          const double keep = up ? a[i + h][b] : a[i][b], send = up ? a[i][b] : a[i + h][b];
          a[i][b] = keep + __shfl_xor(send, o, 64);
        }
    }
#pragma unroll
    for (int b = 0; b < 3; ++b) {
      a[0][b] += __shfl_xor(a[0][b], 2, 64);
      a[0][b] += __shfl_xor(a[0][b], 1, 64);
    }
    const int c = c0 + (lane >> 2);  // lane bits 5 4 3 2: the halves kept
    if ((lane & 3) == 0 && c < cols) emit(c, a[0][0], a[0][1], a[0][2]);
  }
}

}  // namespace mbd
