// Solves and per-molecule sums of the larger batched molecules (mol.h).
#include <cmath>

#include "mol.h"
#include "tri3.h"

namespace mbd {

namespace {

constexpr int NT = kTriNT, PW = kTriPW;

// X <- (L L^T)^-1 X, three right-hand sides X[b S + r] in LDS.
template <typename T>
__device__ void solve3(const T *L, long ld, int n, const T *inv, double *X, int S, double *P) {
  constexpr int NB = kCholNB;
  double *Y = P;  // [b PW + r]
  for (int k0 = 0; k0 < n; k0 += NB) {
    const int kb = min(NB, n - k0), k1 = k0 + kb;
    // kb <= 128 rows: emitted between two barriers, after every read of X
    mv3(inv + (long)k0 * NB, NB, kb, kb, X + k0, S, P, [&](int r, double a, double b, double c) {
      X[k0 + r] = a;
      X[S + k0 + r] = b;
      X[2 * S + k0 + r] = c;
    });
    if (k1 < n)
      mv3(L + k1 + (long)k0 * ld, ld, n - k1, kb, X + k0, S, P, [&](int r, double a, double b, double c) {
        X[k1 + r] -= a;
        X[S + k1 + r] -= b;
        X[2 * S + k1 + r] -= c;
      });
    __syncthreads();
  }
  for (int k0 = ((n - 1) / NB) * NB; k0 >= 0; k0 -= NB) {
    const int kb = min(NB, n - k0), k1 = k0 + kb;
    if (k1 < n) {
      dot3(L + k1 + (long)k0 * ld, ld, n - k1, kb, X + k1, S, [&](int r, double a, double b, double c) {
        X[k0 + r] -= a;
        X[S + k0 + r] -= b;
        X[2 * S + k0 + r] -= c;
      });
      __syncthreads();
    }
    dot3(inv + (long)k0 * NB, NB, kb, kb, X + k0, S, [&](int r, double a, double b, double c) {
      Y[r] = a;
      Y[PW + r] = b;
      Y[2 * PW + r] = c;
    });
    __syncthreads();
    for (int e = threadIdx.x; e < 3 * kb; e += NT) X[(e / kb) * S + k0 + e % kb] = Y[(e / kb) * PW + e % kb];
    __syncthreads();
  }
}

__device__ inline double block_sum(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int q = 0; q < NT / 64; ++q) s += red[q];
  return s;
}
// NaN-keeping maximum of non-negative values.
__device__ inline double block_max(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) {
    const double w = __shfl_xor(v, o, 64);
    v = (w > v || w != w) ? w : v;
  }
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = red[0];
  for (int q = 1; q < NT / 64; ++q) s = (red[q] > s || red[q] != red[q]) ? red[q] : s;
  return s;
}

}  // namespace

// One workgroup per matrix, which is read from memory twice per solve and
// once per residual (HBM bound); the right-hand sides stay in LDS.
template <typename T>
__global__ __launch_bounds__(NT, 2) void k_mol_solve(int S, int natoms, const MolInfo *__restrict__ mols,
                                                     const double *__restrict__ A,
                                                     const T *__restrict__ L, const T *__restrict__ inv,
                                                     const int *__restrict__ info, double tol, int maxit,
                                                     double *alpha, int *stat, double *resid, int *redo) {
  extern __shared__ __align__(16) double sm[];
  double *X = sm, *R = X + 3 * S, *P = R + 3 * S, *red = P + 3 * PW;
  const MolMat z = mol_mat(nullptr, blockIdx.x);
  const MolInfo mi = mols[z.mol];
  const int t = threadIdx.x, n = mi.n;
  const long ld = mi.ld, at = mi.a + (long)z.slot * n * ld;
  if (info[blockIdx.x] != 0) {
    if (t == 0) redo[mi.id] = 1;
    return;
  }
  const T *Lm = L + at, *im = inv + mi.inv + z.slot * mol_inv_size(n);
  for (int e = t; e < n; e += NT)
    for (int b = 0; b < 3; ++b) X[b * S + e] = (e % 3 == b) ? 1.0 : 0.0;
  __syncthreads();
  solve3(Lm, ld, n, im, X, S, P);
  double rmax = 0.0;
  int iters = 0;
  for (;;) {
    double m = 0.0;
    mv3(A + at, ld, n, n, X, S, P, [&](int r, double a, double b, double c) {
      const int q = r % 3;
      const double r0 = (q == 0 ? 1.0 : 0.0) - a, r1 = (q == 1 ? 1.0 : 0.0) - b,
                   r2 = (q == 2 ? 1.0 : 0.0) - c;
      R[r] = r0;
      R[S + r] = r1;
      R[2 * S + r] = r2;
      const double w = fabs(r0) + fabs(r1) + fabs(r2);
      m = w != w ? w : fmax(m, fmax(fabs(r0), fmax(fabs(r1), fabs(r2))));
    });
    rmax = block_max(m, red);
    if (rmax <= tol || iters >= maxit) break;
    solve3(Lm, ld, n, im, R, S, P);
    for (int e = t; e < n; e += NT)
      for (int b = 0; b < 3; ++b) X[b * S + e] += R[b * S + e];
    __syncthreads();
    ++iters;
  }
  for (int i = t; i < n / 3; i += NT) {
    double s = 0.0;
    s += X[3 * i] / 3.0;
    s += X[S + 3 * i + 1] / 3.0;
    s += X[2 * S + 3 * i + 2] / 3.0;
    alpha[(long)z.slot * natoms + mi.atom0 + i] = s;
  }
  if (t == 0) {
    if (!(rmax <= tol)) redo[mi.id] = 1;
    atomicMax(&stat[4 * mi.id + 2], iters);
    atomicMax((unsigned long long *)&resid[mi.id], (unsigned long long)__double_as_longlong(rmax));
  }
}

template <typename T>
void solve_mols(hipStream_t s, int nmol, int nmax, int natoms, const MolInfo *mols, const double *A,
                const T *L, const T *inv, const int *info, double tol, int maxit, double *alpha,
                int *stat, double *resid, int *redo) {
  const int S = mol_ld(nmax);
  const size_t lds = sizeof(double) * (6 * (size_t)S + 3 * PW + 8);
  MBD_HIP(hipFuncSetAttribute((const void *)k_mol_solve<T>, hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)lds));
  hipLaunchKernelGGL((k_mol_solve<T>), dim3(nmol * kNumFreq), dim3(NT), lds, s, S, natoms, mols, A, L, inv,
                     info, tol, maxit, alpha, stat, resid, redo);
  MBD_LAUNCH_CHECK();
}
template void solve_mols<double>(hipStream_t, int, int, int, const MolInfo *, const double *,
                                 const double *, const double *, const int *, double, int, double *, int *,
                                 double *, int *);
template void solve_mols<float>(hipStream_t, int, int, int, const MolInfo *, const double *, const float *,
                                const float *, const int *, double, int, double *, int *, double *, int *);

// One workgroup per molecule (UTILS.f90:302-313, 737-739), the sums in the
// persistent kernel's order.
__global__ __launch_bounds__(NT) void k_mol_params(int natoms, const MolInfo *__restrict__ mols,
                                                   const double *__restrict__ weight,
                                                   const double *__restrict__ a0,
                                                   const double *__restrict__ r0,
                                                   const double *__restrict__ alpha, double *c6,
                                                   double *omega, double *reff, double *c6_mol,
                                                   double *w2) {
  __shared__ double red[NT / 64];
  const MolInfo mi = mols[blockIdx.x];
  const int t = threadIdx.x, N = mi.n / 3;
  double top = 0.0, neg = 0.0;  // largest omega^2 and largest 1 / omega^2
  for (int i = t; i < N; i += NT) {
    const int o = mi.atom0 + i;
    const double ae = alpha[o];
    double s = 0.0;
    for (int k = 1; k < kNumFreq; ++k) {
      const double ak = alpha[(long)k * natoms + o];
      s = s + weight[k] * (ak * ak);
    }
    const double c = s * kThreeOverPi, w = (4.0 / 3.0) * c / (ae * ae);
    c6[o] = c;
    omega[o] = w;
    reff[o] = r0[o] * pow(ae / a0[o], kOtd);
    const double q = w * w, iq = 1.0 / q;
    top = (q > top || q != q) ? q : top;
    neg = (iq > neg || iq != iq) ? iq : neg;
  }
  double c6m = 0.0;
  for (int k = 1; k < kNumFreq; ++k) {
    double part = 0.0;
    for (int i = t; i < N; i += NT) part += alpha[(long)k * natoms + mi.atom0 + i];
    const double iso = block_sum(part, red);
    c6m = c6m + weight[k] * (iso * iso);
  }
  top = block_max(top, red);
  neg = block_max(neg, red);
  if (t == 0) {
    c6_mol[mi.id] = kThreeOverPi * c6m;
    w2[2 * blockIdx.x] = 1.0 / neg;
    w2[2 * blockIdx.x + 1] = top;
  }
}

void params_mols(hipStream_t s, int nmol, int natoms, const MolInfo *mols, const double *weight,
                 const double *a0, const double *r0, const double *alpha, double *c6, double *omega,
                 double *reff, double *c6_mol, double *w2) {
  hipLaunchKernelGGL(k_mol_params, dim3(nmol), dim3(NT), 0, s, natoms, mols, weight, a0, r0, alpha, c6,
                     omega, reff, c6_mol, w2);
  MBD_LAUNCH_CHECK();
}

__global__ void k_mol_reset(int n, const int *list, int *counter, int *stat, double *resid) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i == 0) counter[0] = 0;
  if (i >= n) return;
  const int m = list[i];
  counter[1 + m] = 0;
  resid[m] = 0.0;
  for (int k = 0; k < 4; ++k) stat[4 * m + k] = 0;
}

void reset_mols(hipStream_t s, int n, const int *list, int *counter, int *stat, double *resid) {
  hipLaunchKernelGGL(k_mol_reset, dim3(ceil_div(n, 256)), dim3(256), 0, s, n, list, counter, stat, resid);
  MBD_LAUNCH_CHECK();
}

}  // namespace mbd
