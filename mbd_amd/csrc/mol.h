// Batched molecules of order above kMolMinOrder: every step of the solve is
// one launch over all of their matrices (mol.hip, and the matrix-of-its-own-
// order forms of the kernels in build.hip, gemm.hip, chol.hip and logdet.hip).
// Smaller molecules keep the persistent kernel (batch.h).
#pragma once

#include <functional>

#include "common.h"
#include "kernels.h"
#include "logdet.h"

namespace mbd {

// The persistent kernel gives each matrix one workgroup with a barrier per
// column; the launches here spread a matrix over workgroups in 128-column
// blocks (512 molecules of 8 to 256 atoms, mixed: 183 -> 24 ms).  Up to order
// 96, the largest that the entry point without allocations takes (its results
// are those of the batch bit for bit), a matrix fits one diagonal block and
// the persistent kernel needs no launch per step.
constexpr int kMolMinOrder = 96;
// A molecule owns kNumFreq matrices: its relay matrices, later the shifted
// ones of its energy.
static_assert(kLdMaxNodes + 1 <= kNumFreq, "the energy's matrices reuse the relay matrices' room");

struct MolInfo {
  int n, ld;       // order, leading dimension (a multiple of 16; the rows past n are never written)
  int atom0;       // first atom in the batch's arrays
  int id;          // molecule in the batch
  long a, c, inv;  // element offsets of its matrices, coupled matrix, inverted diagonal blocks
};
struct MolMat {
  int mol, slot;
};

__host__ __device__ inline int mol_ld(int n) { return (n + 15) / 16 * 16; }
__host__ __device__ inline long mol_inv_size(int n) {
  return (long)((n + kCholNB - 1) / kCholNB) * kCholNB * kCholNB;
}
// Matrix x of a list, or of kNumFreq matrices per molecule in order.
__device__ inline MolMat mol_mat(const MolMat *mats, int x) {
  return mats ? mats[x] : MolMat{x / kNumFreq, x % kNumFreq};
}

// gemm.hip
template <typename T>
void gemm_mols(hipStream_t s, bool upd, int k0, int nmax, int nmat, const MolInfo *mols,
               const MolMat *mats, T *L, const T *inv);
// chol.hip
template <typename T>
void potrf_mols(hipStream_t s, int nmax, const MolInfo *mols, const MolMat *mats,
                const std::function<int(int)> &atleast, T *L, T *inv, int *info);
// build.hip: the FP64 relay matrices (both triangles) and, in L, their lower triangles; the coupled
// matrices (lower triangles).  natoms: stride of the per-grid-point arrays.
template <typename T>
void scs_build_mols(hipStream_t s, int nmol, int nmax, int natoms, const MolInfo *mols,
                    const double *xyz, double rc, double beta, const double *alpha_w,
                    const double *sgm, const double *rvdw, double *A, T *L);
void cfdm_build_mols(hipStream_t s, int nmol, int nmax, const MolInfo *mols, const double *xyz,
                     double rc, double beta, const double *alpha, const double *omega,
                     const double *reff, double *C);
// logdet.hip: as ld_bounds, ld_shift and ld_sums; hi has ceil(nmax / 64) entries per molecule.
void ld_bounds_mols(hipStream_t s, int nmol, int nmax, const MolInfo *mols, const double *C, double *hi);
void ld_shift_mols(hipStream_t s, int nmat, int nmax, const MolInfo *mols, const MolMat *mats,
                   const double *shift, const double *C, double *A);
void ld_sums_mols(hipStream_t s, int nmat, const MolInfo *mols, const MolMat *mats, const double *shift,
                  const double *A, const double *omega, double *g);
// mol.hip.  X = A^-1 B from the factors and the inverted diagonal blocks, refined against A while
// max |B - A X| exceeds tol, at most maxit times; alpha[f natoms + atom]; iterations and residuals
// into stat and resid as the persistent kernel keeps them.  redo[id] is set where a factor failed
// or the refinement did not converge.
template <typename T>
void solve_mols(hipStream_t s, int nmol, int nmax, int natoms, const MolInfo *mols, const double *A,
                const T *L, const T *inv, const int *info, double tol, int maxit, double *alpha,
                int *stat, double *resid, int *redo);
// C6, omega, R_eff and molecular C6; w2[2 m], w2[2 m + 1]: smallest and largest omega^2 (inf if
// one is not finite).
void params_mols(hipStream_t s, int nmol, int natoms, const MolInfo *mols, const double *weight,
                 const double *a0, const double *r0, const double *alpha, double *c6, double *omega,
                 double *reff, double *c6_mol, double *w2);
// Counters, statistics and residuals of the molecules in list back to zero.
void reset_mols(hipStream_t s, int n, const int *list, int *counter, int *stat, double *resid);

}  // namespace mbd
