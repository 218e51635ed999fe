// Dipole-tensor builders: per-atom frequency parameters, the SCS relay
// matrices A(i w) = diag(1/alpha) + T_sr and the coupled-QHO matrix C.
//
// Both builders tile the lower triangle of the atom (or supercell-site) pair
// space in 16 x 16 tiles, one thread per pair.  A thread scans the lattice
// image box with the reference's FP64 inclusion test r <= rc (computed without
// FMA contraction, so the image set equals the reference's; a squared-distance
// prefilter with a rounding margin skips the square root of every image that
// is certainly outside), sums the damped tensors of the included images, and
// drops its 3x3 block into an LDS tile; the 48 x 48 tile is written with
// coalesced column-major stores, and its transpose too when the caller needs
// the full matrix (the factorisations and the eigen reduction read only the
// lower triangle).
// The SCS builder scans the image box once per group of kFreqGroup grid
// points: the image set, distances, products d_a d_b and the Fermi damping do
// not depend on the frequency; only sigma (erf and the Gaussian) does.
//
// Reference formulas: UTILS.f90:637-696 (SR tensor), 1098-1153 (LR tensor),
// 543-633 (SCS blocks), 883-1094 (supercell / CFDM blocks), 1157-1184
// (alpha(i w), sigma), 737-739 (R_eff, omega).
#include "common.h"
#include "kernels.h"
#include "mol.h"
#include "profile.h"
#include "tensor.h"

namespace mbd {

namespace {

constexpr int kFullTiles = 512;  // tiles that fill the 256 CUs with two workgroups each
constexpr int kFreqGroup = 7;   // grid points per image scan of the SCS builder
constexpr int TILE = 16;        // atoms (sites) per tile edge
constexpr int TB = 3 * TILE;    // matrix rows per tile edge
constexpr int TBP = TB + 1;     // padded LDS column

__device__ inline void tri_index(int idx, int &ti, int &tj) {
  int t = (int)((sqrt(8.0 * idx + 1.0) - 1.0) * 0.5);
  while ((t + 1) * (t + 2) / 2 <= idx) ++t;
  while (t * (t + 1) / 2 > idx) --t;
  ti = t;
  tj = idx - t * (t + 1) / 2;
}

// The reference's inclusion test r <= rc with r = sqrt(dx^2 + dy^2 + dz^2)
// rounded as exact_dist: s2 is the rounded sum of squares, rc2x the rounded
// rc^2 times (1 + 4 eps).  s2 > rc2x implies r > rc (sqrt is monotonic and
// correctly rounded), so the square root is taken only near or inside the
// sphere, where r itself is needed.
__device__ inline bool in_sphere(double dx, double dy, double dz, double rc, double rc2x,
                                 double &r) {
  double s2;
  {
#pragma clang fp contract(off)
    s2 = dx * dx + dy * dy;
    s2 = s2 + dz * dz;
  }
  if (s2 > rc2x) return false;
  r = sqrt(s2);
  return r <= rc;
}

// Image loops of the builders: a wave-uniform pass over a chunk of 32 images
// (scalar loads) marks in a per-lane mask the images that may lie in the
// sphere (rounded r^2 <= rc2x), other than image `skip`; each lane then runs
// the tensor only over its own marked images (in_sphere decides exactly).  A
// wave so runs the tensor once per marked image of its fullest pair in each
// chunk rather than once per image marked by any of its 64 pairs (at a 100 A
// cutoff in a 38 A cell about 76 of 343 images per pair, scattered
// differently over the lanes).  Each pair sums its images in table order, or
// with several slices of a workgroup (k_scs_build) each slice's in that order
// and then the slices.
constexpr int kImgChunk = 32;
// NEAR: near is set if an image's r^2 is so close to rc^2 that another
// rounding of the same displacement could decide otherwise.
template <bool NEAR = false>
__device__ inline unsigned sphere_mask(double d0x, double d0y, double d0z,
                                       const double *__restrict__ img, int c0, int cn, int skip,
                                       double rc2x, bool *near = nullptr) {
  unsigned m = 0;
  for (int b = 0; b < cn; ++b) {
    double dx, dy, dz, s2;
    add3(d0x, d0y, d0z, img[3 * (c0 + b)], img[3 * (c0 + b) + 1], img[3 * (c0 + b) + 2], dx, dy, dz);
    {
#pragma clang fp contract(off)
      s2 = dx * dx + dy * dy;
      s2 = s2 + dz * dz;
    }
    if (s2 <= rc2x && c0 + b != skip) m |= 1u << b;
    if (NEAR) *near = *near || fabs(s2 - rc2x) <= 3e-14 * rc2x;
  }
  return m;
}

// Next marked image of a mask (cleared from it): its displacement and, if it
// lies in the sphere, r; false if it does not.
__device__ inline bool take_marked(double d0x, double d0y, double d0z,
                                   const double *__restrict__ img, int c0, unsigned &m, double rc,
                                   double rc2x, double &dx, double &dy, double &dz, double &r) {
  const int s = c0 + __builtin_ctz(m);
  m &= m - 1;
  add3(d0x, d0y, d0z, img[3 * s], img[3 * s + 1], img[3 * s + 2], dx, dy, dz);
  return in_sphere(dx, dy, dz, rc, rc2x, r);
}

// Six unique entries of a symmetric 3x3: xx, yy, zz, xy, xz, yz.
template <typename T>
struct Sym6 {
  T v[6];
};

// Write a symmetric 3x3 (6 entries) into the LDS tile at block (bi, bj).
template <typename T>
__device__ inline void put_block(T (*S)[TBP], int bi, int bj, const T *v6) {
  const int idx[3][3] = {{0, 3, 4}, {3, 1, 5}, {4, 5, 2}};
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int r = 0; r < 3; ++r) S[3 * bj + c][3 * bi + r] = v6[idx[r][c]];
}

// Store the LDS tile at (ti, tj) and, off the diagonal, its transpose.
template <typename T>
__device__ inline void store_tile(T (*S)[TBP], T *M, long ld, int n, int ti,
                                  int tj, bool full) {
  const int r0 = TB * ti, c0 = TB * tj;
  for (int e = threadIdx.x; e < TB * TB; e += blockDim.x) {
    const int r = e % TB, c = e / TB;
    if (r0 + r < n && c0 + c < n) M[(r0 + r) + (long)(c0 + c) * ld] = S[c][r];
  }
  if (full && ti != tj) {
    for (int e = threadIdx.x; e < TB * TB; e += blockDim.x) {
      const int a = e % TB, b = e / TB;  // row c0+a, column r0+b
      if (c0 + a < n && r0 + b < n) M[(c0 + a) + (long)(r0 + b) * ld] = S[a][b];
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
// Per-atom parameters at each grid point (UTILS.f90:251-255, 1172-1179).
__global__ void k_atom_params(int N, int nf, const double *__restrict__ omega,
                              const double *__restrict__ hirsh,
                              const double *__restrict__ a0,
                              const double *__restrict__ c60,
                              const double *__restrict__ r0,
                              double *__restrict__ alpha_w,
                              double *__restrict__ sgm,
                              double *__restrict__ rvdw) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int f = blockIdx.y;
  if (i >= N) return;
  const double w = omega[f];
  const double wp = (4.0 / 3.0) * c60[i] / (a0[i] * a0[i]);
  const double aw = (hirsh[i] * a0[i]) / (1.0 + (w * w) / (wp * wp));
  alpha_w[(long)f * N + i] = aw;
  sgm[(long)f * N + i] = pow((aw / 3.0) * sqrt(2.0 / kPi), kOtd);
  if (f == 0) rvdw[i] = pow(hirsh[i], kOtd) * r0[i];
}

void atom_params(hipStream_t s, int N, int nf, const double *omega,
                 const double *hirsh, const double *a0, const double *c60,
                 const double *r0, double *alpha_w, double *sgm,
                 double *rvdw) {
  dim3 grid(ceil_div(N, 256), nf);
  hipLaunchKernelGGL(k_atom_params, grid, dim3(256), 0, s, N, nf, omega, hirsh,
                     a0, c60, r0, alpha_w, sgm, rvdw);
  MBD_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// SCS relay matrices of nf consecutive grid points (UTILS.f90:543-633): a
// workgroup per 16 x 16 atom-pair tile, one image scan per group of
// kFreqGroup grid points.  Off-diagonal block (i, j): sum over images n of
// T_sr(r_i - r_j + L_n; sqrt(s_i^2 + s_j^2), R_i + R_j); diagonal block:
// (1/alpha_i) I + sum over n != 0 of T_sr(L_n; s_i, 2 R_i).
template <typename T, int F, int IS>
__global__ __launch_bounds__(256 * IS) void k_scs_build(
    int N, const double *__restrict__ xyz, int nimg, int center,
    const double *__restrict__ img, double rc, double beta,
    const double *__restrict__ alpha_w, const double *__restrict__ sgm,
    const double *__restrict__ rvdw, T *__restrict__ A, int lda,
    long stride, int nf, bool full) {
  __shared__ T S[TB][TBP];
  __shared__ double part[IS > 1 ? IS - 1 : 1][6][IS > 1 ? 256 : 1];
  int ti, tj;
  tri_index(blockIdx.x, ti, tj);
  const int n = 3 * N;
  const int pair = threadIdx.x % 256, slice = IS > 1 ? threadIdx.x / 256 : 0;
  const int lx = pair % TILE, ly = pair / TILE;
  const int i = TILE * ti + lx, j = TILE * tj + ly;
  const bool active = (i < N && j < N && (ti != tj || i >= j));
  const bool diag = (i == j);
  const double rc2x = (rc * rc) * (1.0 + 4.0 * 2.220446049250313e-16);
  double d0x = 0.0, d0y = 0.0, d0z = 0.0, R12 = 0.0;
  if (active) {
    if (diag) {
      R12 = 2.0 * rvdw[i];
    } else {
      d0x = xyz[3 * i] - xyz[3 * j];
      d0y = xyz[3 * i + 1] - xyz[3 * j + 1];
      d0z = xyz[3 * i + 2] - xyz[3 * j + 2];
      R12 = rvdw[i] + rvdw[j];
    }
  }
  for (int f0 = blockIdx.y * F; f0 < nf; f0 += gridDim.y * F) {
    const int nfg = min(F, nf - f0);
    double acc[F][6];
#pragma unroll
    for (int g = 0; g < F; ++g)
#pragma unroll
      for (int e = 0; e < 6; ++e) acc[g][e] = 0.0;
    if (active) {
      // sigma of the pair at each grid point of the group
      double sg12[F];
#pragma unroll
      for (int g = 0; g < F; ++g) {
        const int f = f0 + min(g, nfg - 1);
        const double si = sgm[(long)f * N + i], sj = sgm[(long)f * N + j];
        sg12[g] = diag ? si : sqrt(si * si + sj * sj);
      }
      if (sizeof(T) == 8) {
        double isg[F];
#pragma unroll
        for (int g = 0; g < F; ++g) isg[g] = 1.0 / sg12[g];
        for (int c0 = kImgChunk * slice; c0 < nimg; c0 += kImgChunk * IS) {
          unsigned m = sphere_mask(d0x, d0y, d0z, img, c0, min(kImgChunk, nimg - c0),
                                   diag ? center : -1, rc2x);
          while (m) {
            double dx, dy, dz, r;
            if (!take_marked(d0x, d0y, d0z, img, c0, m, rc, rc2x, dx, dy, dz, r)) continue;
            const double ir = 1.0 / r, damp = sr_damp64(r, R12, beta);
#pragma unroll
            for (int g = 0; g < F; ++g)
              if (g < nfg) sr_tensor_add64h(dx, dy, dz, r, ir, isg[g], damp, acc[g]);
          }
        }
      } else {
        // FP32 terms summed in FP64: a conversion and an add per term
        // against the eight operations of a compensated FP32 sum, with the
        // same registers and a smaller error (FP64 adds run at the FP32 rate)
        const float fb = (float)beta, fR = (float)R12;
        const float ibR = 1.0f / (fb * fR);
        // per grid point 1 / sigma and 2/sqrt(pi) / sigma^3, per image the
        // powers of 1 / r: one division per image instead of three per image
        // and grid point (the hardware reciprocal estimate, biased, had
        // raised the molecular C6 error tenfold)
        float isg[F], zc[F];
#pragma unroll
        for (int g = 0; g < F; ++g) {
          isg[g] = 1.0f / (float)sg12[g];
          zc[g] = 2.25675833f * isg[g] * isg[g] * isg[g];
        }
        for (int c0 = kImgChunk * slice; c0 < nimg; c0 += kImgChunk * IS) {
          unsigned m = sphere_mask(d0x, d0y, d0z, img, c0, min(kImgChunk, nimg - c0),
                                   diag ? center : -1, rc2x);
          while (m) {
            double dx, dy, dz, r;
            if (!take_marked(d0x, d0y, d0z, img, c0, m, rc, rc2x, dx, dy, dz, r)) continue;
            // frequency-independent parts: products, powers of r, damping
            const float x0 = (float)dx, x1 = (float)dy, x2 = (float)dz, rf = (float)r;
            const float r2 = rf * rf;
            const float ir = 1.0f / rf, ir2 = ir * ir, ir5 = ir2 * ir2 * ir;
            const float ef = __expf(-6.0f * (rf * ibR - 1.0f));
            const float damp = isinf(ef) ? 1.0f : ef / (1.0f + ef);
            const float dd[6] = {x0 * x0, x1 * x1, x2 * x2, x0 * x1, x0 * x2, x1 * x2};
#pragma unroll
            for (int g = 0; g < F; ++g) {
              if (g < nfg) {
                const float x = rf * isg[g];
                const float ex = __expf(-(x * x));
                const float zl = (erff(x) - 1.12837917f * x * ex) * ir5;
                const float zr = ex * zc[g] * ir2;
#pragma unroll
                for (int e = 0; e < 6; ++e) {
                  const float t = 3.0f * dd[e] - (e < 3 ? r2 : 0.0f);
                  acc[g][e] += (double)((-t * zl + dd[e] * zr) * damp);
                }
              }
            }
          }
        }
      }
    }
#pragma unroll
    for (int g = 0; g < F; ++g) {
      if (g < nfg) {
        __syncthreads();
        if (IS > 1) {  // the slices' sums, in their order
          if (slice > 0)
#pragma unroll
            for (int e = 0; e < 6; ++e) part[slice - 1][e][pair] = acc[g][e];
          __syncthreads();
          if (slice == 0)
            for (int q = 0; q < IS - 1; ++q)
#pragma unroll
              for (int e = 0; e < 6; ++e) acc[g][e] += part[q][e][pair];
        }
        if (active && slice == 0) {
          const double inv = diag ? 1.0 / alpha_w[(long)(f0 + g) * N + i] : 0.0;
          T out[6];
#pragma unroll
          for (int e = 0; e < 6; ++e) out[e] = (T)(acc[g][e] + (e < 3 ? inv : 0.0));
          put_block(S, lx, ly, out);
          if (ti == tj && !diag) put_block(S, ly, lx, out);
        }
        __syncthreads();
        store_tile(S, A + (long)(f0 + g) * stride, lda, n, ti, tj, full);
      }
    }
  }
}

template <typename T>
void scs_build(hipStream_t s, int N, const double *xyz, int nimg, int center,
               const double *img, double rc_bohr, double beta,
               const double *alpha_w, const double *sgm, const double *rvdw,
               T *A, int lda, long stride, int nf, bool full) {
  const int tn = ceil_div(N, TILE), nt = tn * (tn + 1) / 2;
  // algorithmic output: the lower 3x3 blocks of each matrix
  ProfScope ps(K_SCS_BUILD, s, 9.0 * sizeof(T) * 0.5 * N * (N + 1.0) * nf, 0.0);
  auto go = [&](auto *kern, int f, int is) {
    hipLaunchKernelGGL(kern, dim3(nt, ceil_div(nf, f)), dim3(256 * is), 0, s, N, xyz, nimg, center, img,
                       rc_bohr, beta, alpha_w, sgm, rvdw, A, lda, stride, nf, full);
  };
  // Few tiles leave the chip idle: the grid points go to workgroups of their
  // own (a tile's distances are formed again for each group of them), and a
  // long image list to two or four slices of a workgroup (FP64: a sheet of 60
  // atoms 2.23 -> 0.18 ms, a cell of 60 3.9 -> 0.31, of 150 1.9 -> 0.56, of
  // 400 1.28 -> 1.06; with the chip full the shared distances win).
  const bool split = nimg >= 4 * kImgChunk;
  if (nt >= kFullTiles)
    hipLaunchKernelGGL((k_scs_build<T, kFreqGroup, 1>), dim3(nt), dim3(256), 0, s, N, xyz, nimg, center,
                       img, rc_bohr, beta, alpha_w, sgm, rvdw, A, lda, stride, nf, full);
  else if (!split)
    go(k_scs_build<T, 1, 1>, 1, 1);
  else if (nt >= kFullTiles / 14)
    go(k_scs_build<T, 3, 2>, 3, 2);
  else
    go(k_scs_build<T, 1, 4>, 1, 4);
  MBD_LAUNCH_CHECK();
}
template void scs_build<double>(hipStream_t, int, const double *, int, int,
                                const double *, double, double, const double *,
                                const double *, const double *, double *, int,
                                long, int, bool);
template void scs_build<float>(hipStream_t, int, const double *, int, int,
                               const double *, double, double, const double *,
                               const double *, const double *, float *, int,
                               long, int, bool);

// ---------------------------------------------------------------------------
// MBD per-atom quantities (UTILS.f90:737-739).
__global__ void k_mbd_params(int N, const double *__restrict__ alpha_eff,
                             const double *__restrict__ c6_eff,
                             const double *__restrict__ a0,
                             const double *__restrict__ r0,
                             double *__restrict__ omega,
                             double *__restrict__ reff) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double a = alpha_eff[i];
  reff[i] = r0[i] * pow(a / a0[i], kOtd);
  omega[i] = (4.0 / 3.0) * c6_eff[i] / (a * a);
}

void mbd_params(hipStream_t s, int N, const double *alpha_eff,
                const double *c6_eff, const double *a0, const double *r0,
                double *omega, double *reff) {
  hipLaunchKernelGGL(k_mbd_params, dim3(ceil_div(N, 256)), dim3(256), 0, s, N,
                     alpha_eff, c6_eff, a0, r0, omega, reff);
  MBD_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// Coupled-QHO matrix over supercell sites s = p * ncell + a (rows 3s..3s+2).
// cell[3*a + k] are the integer cell coordinates of cell a; lat the unit-cell
// lattice; img the supercell image translations.
__global__ __launch_bounds__(256) void k_cfdm_build(
    int N, int ncell, const double *__restrict__ xyz,
    const int *__restrict__ cell, const double *__restrict__ lat, int nimg,
    int center, const double *__restrict__ img, double rc, double beta,
    const double *__restrict__ alpha_eff, const double *__restrict__ omega,
    const double *__restrict__ reff, double *__restrict__ C, long ldc, bool full) {
  __shared__ double S[TB][TBP];
  const double rc2x = (rc * rc) * (1.0 + 4.0 * 2.220446049250313e-16);
  int ti, tj;
  tri_index(blockIdx.x, ti, tj);
  const int nsite = N * ncell;
  const int n = 3 * nsite;
  const int lx = threadIdx.x % TILE, ly = threadIdx.x / TILE;
  const int si = TILE * ti + lx, sj = TILE * tj + ly;
  const bool active = (si < nsite && sj < nsite && (ti != tj || si >= sj));
  if (active) {
    const int p = si / ncell, a = si % ncell;
    const int q = sj / ncell, b = sj % ncell;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    if (si == sj) {
      // cfdm_diag_block, UTILS.f90:998-1043
      const double pref = omega[p] * omega[p] * alpha_eff[p];
      const double R2 = 2.0 * reff[p];
      for (int s = 0; s < nimg; ++s) {
        if (s == center) continue;
        const double dx = img[3 * s], dy = img[3 * s + 1], dz = img[3 * s + 2];
        double r;
        if (in_sphere(dx, dy, dz, rc, rc2x, r)) lr_tensor_add64(dx, dy, dz, r, R2, beta, pref, acc);
      }
      const double w2 = omega[p] * omega[p];
      acc[0] += w2;
      acc[1] += w2;
      acc[2] += w2;
    } else {
      // cfdm_offdiag_block, UTILS.f90:1047-1094
      const double pref = omega[p] * omega[q] * sqrt(alpha_eff[p] * alpha_eff[q]);
      const double R12 = reff[p] + reff[q];
      const double di = (double)(cell[3 * a] - cell[3 * b]);
      const double dj = (double)(cell[3 * a + 1] - cell[3 * b + 1]);
      const double dk = (double)(cell[3 * a + 2] - cell[3 * b + 2]);
      double dcx, dcy, dcz, d0x, d0y, d0z;
      {
#pragma clang fp contract(off)
        dcx = (di * lat[0] + dj * lat[3]) + dk * lat[6];
        dcy = (di * lat[1] + dj * lat[4]) + dk * lat[7];
        dcz = (di * lat[2] + dj * lat[5]) + dk * lat[8];
        d0x = (xyz[3 * p] - xyz[3 * q]) + dcx;
        d0y = (xyz[3 * p + 1] - xyz[3 * q + 1]) + dcy;
        d0z = (xyz[3 * p + 2] - xyz[3 * q + 2]) + dcz;
      }
      for (int c0 = 0; c0 < nimg; c0 += kImgChunk) {
        unsigned m = sphere_mask(d0x, d0y, d0z, img, c0, min(kImgChunk, nimg - c0), -1, rc2x);
        while (m) {
          double dx, dy, dz, r;
          if (take_marked(d0x, d0y, d0z, img, c0, m, rc, rc2x, dx, dy, dz, r))
            lr_tensor_add64(dx, dy, dz, r, R12, beta, pref, acc);
        }
      }
    }
    put_block(S, lx, ly, acc);
    if (ti == tj && si != sj) put_block(S, ly, lx, acc);
  }
  __syncthreads();
  store_tile(S, C, ldc, n, ti, tj, full);
}

// The same matrix of a supercell by cell differences: B_a[p, q] is the block
// of atom p in cell a and atom q in cell 0 (lower 3 x 3 blocks p >= q of N
// atoms, matrix a of B).  near[0] is set where an image lies on the cutoff
// sphere to rounding, so that another pair of cells with the same difference
// could have included it or not.
__global__ __launch_bounds__(256) void k_cfdm_cells(
    int N, const double *__restrict__ xyz, const int *__restrict__ cell,
    const double *__restrict__ lat, int nimg, int center, const double *__restrict__ img, double rc,
    double beta, const double *__restrict__ alpha_eff, const double *__restrict__ omega,
    const double *__restrict__ reff, double *__restrict__ B, int *__restrict__ near) {
  __shared__ double S[TB][TBP];
  const double rc2x = (rc * rc) * (1.0 + 4.0 * 2.220446049250313e-16);
  int ti, tj;
  tri_index(blockIdx.x, ti, tj);
  const int a = blockIdx.y, n = 3 * N;
  const int lx = threadIdx.x % TILE, ly = threadIdx.x / TILE;
  const int p = TILE * ti + lx, q = TILE * tj + ly;
  if (p < N && q < N && p >= q) {
    double acc[6] = {0, 0, 0, 0, 0, 0};
    const bool self = p == q && a == 0;
    const double pref = omega[p] * omega[q] * sqrt(alpha_eff[p] * alpha_eff[q]);
    const double R12 = reff[p] + reff[q];
    const double di = (double)cell[3 * a], dj = (double)cell[3 * a + 1], dk = (double)cell[3 * a + 2];
    double d0x, d0y, d0z;
    {
#pragma clang fp contract(off)
      const double dcx = (di * lat[0] + dj * lat[3]) + dk * lat[6];
      const double dcy = (di * lat[1] + dj * lat[4]) + dk * lat[7];
      const double dcz = (di * lat[2] + dj * lat[5]) + dk * lat[8];
      d0x = (xyz[3 * p] - xyz[3 * q]) + dcx;
      d0y = (xyz[3 * p + 1] - xyz[3 * q + 1]) + dcy;
      d0z = (xyz[3 * p + 2] - xyz[3 * q + 2]) + dcz;
    }
    bool nr = false;
    for (int c0 = 0; c0 < nimg; c0 += kImgChunk) {
      unsigned m = sphere_mask<true>(d0x, d0y, d0z, img, c0, min(kImgChunk, nimg - c0),
                                     self ? center : -1, rc2x, &nr);
      while (m) {
        double dx, dy, dz, r;
        if (take_marked(d0x, d0y, d0z, img, c0, m, rc, rc2x, dx, dy, dz, r))
          lr_tensor_add64(dx, dy, dz, r, R12, beta, pref, acc);
      }
    }
    if (nr) atomicOr(near, 1);
    if (self) {
      const double w2 = omega[p] * omega[p];
      acc[0] += w2;
      acc[1] += w2;
      acc[2] += w2;
    }
    put_block(S, lx, ly, acc);
  }
  __syncthreads();
  store_tile(S, B + (long)a * n * n, n, n, ti, tj, false);
}

void cfdm_cells(hipStream_t s, int N, int ncell, const double *xyz, const int *cell,
                const double *lat, int nimg, int center, const double *img, double rc_bohr,
                double beta, const double *alpha_eff, const double *omega, const double *reff,
                double *B, int *near) {
  const int tn = ceil_div(N, TILE);
  ProfScope ps(K_CFDM_BUILD, s, 72.0 * 0.5 * N * (N + 1.0) * ncell, 0.0);
  hipLaunchKernelGGL(k_cfdm_cells, dim3(tn * (tn + 1) / 2, ncell), dim3(256), 0, s, N, xyz, cell, lat,
                     nimg, center, img, rc_bohr, beta, alpha_eff, omega, reff, B, near);
  MBD_LAUNCH_CHECK();
}

// Phases of the cells' Fourier transform, (nreal + npair) x ncell cosines and
// then the pairs' sines: every k.a / S is a multiple of 1 / L, L the least
// common multiple of the cells along the axes, whose cosines and sines cs
// holds, then the wave vectors, real ones first (one upload).
__global__ __launch_bounds__(256) void k_cell_phase(int s1, int s2, int s3, int L, int nreal, int npair,
                                                    const double *__restrict__ cs,
                                                    double *__restrict__ phase) {
  const int nc = s1 * s2 * s3, a = blockIdx.x * 256 + threadIdx.x, k = blockIdx.y;
  if (a >= nc) return;
  const double *kv = cs + 2 * L + 3 * k;
  const int m1 = (int)kv[0] * (a % s1) % s1 * (L / s1), m2 = (int)kv[1] * (a / s1 % s2) % s2 * (L / s2),
            m3 = (int)kv[2] * (a / s1 / s2) % s3 * (L / s3);
  const int m = (m1 + m2 + m3) % L;
  phase[(long)k * nc + a] = cs[m];
  if (k >= nreal) phase[(long)(k + npair) * nc + a] = cs[L + m];
}

// H_k = sum_a exp(2 pi i k.a / S) B_a for r >= c: the nreal real matrices of
// order n (Hr), and per pair k, -k the real [Re -Im; Im Re] of order 2 n (Hp),
// lower triangles.  Workgroups of blockIdx.z take every gridDim.z-th wave
// vector: with all of them in one workgroup each B_a is read once from HBM and
// again from the caches (a cell of 1024 atoms has 75 MB a block), but a
// primitive cell's blocks of a few KB leave that form a handful of threads
// with cells^2 / 2 steps in a row (energies, with the phases formed on the
// host: 1 atom in 343 cells 9.6 -> 0.6 ms, 3 atoms in 1000 cells 74 -> 1.6 ms;
// 1024 atoms in 8 cells 1.8 ms for the blocks and this either way).
__global__ __launch_bounds__(256) void k_cell_dft(int n, int ncell, int nreal, int npair,
                                                  const double *__restrict__ phase,
                                                  const double *__restrict__ B,
                                                  double *__restrict__ Hr, double *__restrict__ Hp) {
  const int r = blockIdx.x * 256 + threadIdx.x, c = blockIdx.y;
  if (r < c || r >= n) return;
  const long nn = (long)n * n;
  const double *b = B + r + (long)c * n;
  for (int q = blockIdx.z; q < nreal + npair; q += gridDim.z) {
    const double *cs = phase + (long)q * ncell;
    if (q < nreal) {
      double v = 0.0;
      for (int a = 0; a < ncell; ++a) v += cs[a] * b[a * nn];
      Hr[q * nn + r + (long)c * n] = v;
      continue;
    }
    const double *sn = cs + (long)npair * ncell;
    double re = 0.0, im = 0.0;
    for (int a = 0; a < ncell; ++a) {
      const double v = b[a * nn];
      re += cs[a] * v;
      im += sn[a] * v;
    }
    double *H = Hp + 4 * (q - nreal) * nn;
    const long ld = 2L * n;
    H[r + c * ld] = re;
    H[n + r + (n + c) * ld] = re;
    H[n + r + c * ld] = r == c ? 0.0 : im;
    if (r != c) H[n + c + r * ld] = -im;
  }
}

void cell_dft(hipStream_t s, int n, const int *cells, int L, int nreal, int npair, const double *cs,
              double *phase, const double *B, double *Hr, double *Hp) {
  const int nc = cells[0] * cells[1] * cells[2], nk = nreal + npair;
  ProfScope ps(K_CFDM_BUILD, s, 4.0 * n * (n + 1.0) * (nc + nreal + 4.0 * npair), 0.0);
  hipLaunchKernelGGL(k_cell_phase, dim3(ceil_div(nc, 256), nk), dim3(256), 0, s, cells[0], cells[1],
                     cells[2], L, nreal, npair, cs, phase);
  // 8 workgroups per CU, half of them above the diagonal
  const int nz = std::min(nk, ceil_div(8 * 256, ceil_div(n, 256) * n));
  hipLaunchKernelGGL(k_cell_dft, dim3(ceil_div(n, 256), n, nz), dim3(256), 0, s, n, nc, nreal, npair,
                     phase, B, Hr, Hp);
  MBD_LAUNCH_CHECK();
}

void cfdm_build(hipStream_t s, int N, int ncell, const double *xyz,
                const int *cell, const double *lat, int nimg, int center,
                const double *img, double rc_bohr, double beta,
                const double *alpha_eff, const double *omega,
                const double *reff, double *C, long ldc, bool full) {
  const int tn = ceil_div((long)N * ncell, TILE);
  dim3 grid((unsigned)((long)tn * (tn + 1) / 2));
  const double ns = (double)N * ncell;
  ProfScope ps(K_CFDM_BUILD, s, 72.0 * 0.5 * ns * (ns + 1.0), 0.0);
  hipLaunchKernelGGL(k_cfdm_build, grid, dim3(256), 0, s, N, ncell, xyz, cell,
                     lat, nimg, center, img, rc_bohr, beta, alpha_eff, omega,
                     reff, C, ldc, full);
  MBD_LAUNCH_CHECK();
}

// ---------------------------------------------------------------------------
// The same two matrices for many non-periodic molecules (one image): molecule
// blockIdx.x, tile blockIdx.y.  The relay matrices of all grid points are
// formed per pair (distance, 1 / r and damping once); A both triangles, L the
// lower one in the factorisation's type.
template <typename T>
__global__ __launch_bounds__(256) void k_mol_scs(int natoms, const MolInfo *__restrict__ mols,
                                                 const double *__restrict__ xyz, double rc, double beta,
                                                 const double *__restrict__ alpha_w,
                                                 const double *__restrict__ sgm,
                                                 const double *__restrict__ rvdw,
                                                 double *__restrict__ A, T *__restrict__ L) {
  __shared__ double S[TB][TBP];
  const MolInfo mi = mols[blockIdx.x];
  const int n = mi.n, N = n / 3, o = mi.atom0;
  int ti, tj;
  tri_index(blockIdx.y, ti, tj);
  if (TILE * ti >= N) return;
  const int lx = threadIdx.x % TILE, ly = threadIdx.x / TILE;
  const int i = TILE * ti + lx, j = TILE * tj + ly;
  const bool active = i < N && j < N && i >= j, diag = i == j;
  const int gi = o + min(i, N - 1), gj = o + min(j, N - 1);
  double dx = 0.0, dy = 0.0, dz = 0.0, r = 1.0, ir = 0.0, damp = 0.0;
  bool in = false;
  if (active && !diag) {
    dx = xyz[3 * gi] - xyz[3 * gj];
    dy = xyz[3 * gi + 1] - xyz[3 * gj + 1];
    dz = xyz[3 * gi + 2] - xyz[3 * gj + 2];
    r = exact_dist(dx, dy, dz);
    in = r <= rc;
    ir = 1.0 / r;
    damp = sr_damp64(r, rvdw[gi] + rvdw[gj], beta);
  }
  for (int f = 0; f < kNumFreq; ++f) {
    double acc[6] = {0, 0, 0, 0, 0, 0};
    if (in) {
      const double si = sgm[(long)f * natoms + gi], sj = sgm[(long)f * natoms + gj];
      sr_tensor_add64h(dx, dy, dz, r, ir, 1.0 / sqrt(si * si + sj * sj), damp, acc);
    }
    if (diag) acc[0] = acc[1] = acc[2] = 1.0 / alpha_w[(long)f * natoms + gi];
    __syncthreads();
    if (active) {
      put_block(S, lx, ly, acc);
      if (ti == tj && !diag) put_block(S, ly, lx, acc);
    }
    __syncthreads();
    const long at = mi.a + (long)f * n * mi.ld;
    store_tile(S, A + at, mi.ld, n, ti, tj, true);
    for (int e = threadIdx.x; e < TB * TB; e += 256) {
      const int row = TB * ti + e % TB, col = TB * tj + e / TB;
      if (row < n && col <= row) L[at + row + (long)col * mi.ld] = (T)S[e / TB][e % TB];
    }
  }
}

template <typename T>
void scs_build_mols(hipStream_t s, int nmol, int nmax, int natoms, const MolInfo *mols,
                    const double *xyz, double rc, double beta, const double *alpha_w,
                    const double *sgm, const double *rvdw, double *A, T *L) {
  const int tn = ceil_div(nmax / 3, TILE);
  hipLaunchKernelGGL((k_mol_scs<T>), dim3(nmol, tn * (tn + 1) / 2), dim3(256), 0, s, natoms, mols, xyz, rc,
                     beta, alpha_w, sgm, rvdw, A, L);
  MBD_LAUNCH_CHECK();
}
template void scs_build_mols<double>(hipStream_t, int, int, int, const MolInfo *, const double *, double,
                                     double, const double *, const double *, const double *, double *,
                                     double *);
template void scs_build_mols<float>(hipStream_t, int, int, int, const MolInfo *, const double *, double,
                                    double, const double *, const double *, const double *, double *,
                                    float *);

__global__ __launch_bounds__(256) void k_mol_cfdm(const MolInfo *__restrict__ mols,
                                                  const double *__restrict__ xyz, double rc, double beta,
                                                  const double *__restrict__ alpha,
                                                  const double *__restrict__ omega,
                                                  const double *__restrict__ reff,
                                                  double *__restrict__ C) {
  __shared__ double S[TB][TBP];
  const MolInfo mi = mols[blockIdx.x];
  const int n = mi.n, N = n / 3, o = mi.atom0;
  int ti, tj;
  tri_index(blockIdx.y, ti, tj);
  if (TILE * ti >= N) return;
  const int lx = threadIdx.x % TILE, ly = threadIdx.x / TILE;
  const int i = TILE * ti + lx, j = TILE * tj + ly;
  if (i < N && j < N && i >= j) {
    const int gi = o + i, gj = o + j;
    double acc[6] = {0, 0, 0, 0, 0, 0};
    if (i == j) {
      acc[0] = acc[1] = acc[2] = omega[gi] * omega[gi];
    } else {
      const double dx = xyz[3 * gi] - xyz[3 * gj], dy = xyz[3 * gi + 1] - xyz[3 * gj + 1],
                   dz = xyz[3 * gi + 2] - xyz[3 * gj + 2], r = exact_dist(dx, dy, dz);
      if (r <= rc)
        lr_tensor_add64(dx, dy, dz, r, reff[gi] + reff[gj], beta,
                        omega[gi] * omega[gj] * sqrt(alpha[gi] * alpha[gj]), acc);
    }
    put_block(S, lx, ly, acc);
  }
  __syncthreads();
  // lower triangle only: the upper blocks of a diagonal tile were not formed
  for (int e = threadIdx.x; e < TB * TB; e += 256) {
    const int row = TB * ti + e % TB, col = TB * tj + e / TB;
    if (row < n && col <= row) C[mi.c + row + (long)col * mi.ld] = S[e / TB][e % TB];
  }
}

void cfdm_build_mols(hipStream_t s, int nmol, int nmax, const MolInfo *mols, const double *xyz,
                     double rc, double beta, const double *alpha, const double *omega,
                     const double *reff, double *C) {
  const int tn = ceil_div(nmax / 3, TILE);
  hipLaunchKernelGGL(k_mol_cfdm, dim3(nmol, tn * (tn + 1) / 2), dim3(256), 0, s, mols, xyz, rc, beta,
                     alpha, omega, reff, C);
  MBD_LAUNCH_CHECK();
}

}  // namespace mbd
