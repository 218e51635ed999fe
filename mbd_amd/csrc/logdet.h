// E_MBD from Cholesky log-determinants (logdet.hip).
#pragma once

#include <vector>

#include "common.h"
#include "refine.h"

namespace mbd {

// Quadrature nodes of the energy: E = sum_b w[b] (ln det(C + t[b]) - ln det(D + t[b])) / cells with
// D = diag(omega^2); one more entry, t = -lo without a weight, whose factorisation proves that
// every eigenvalue of C lies above lo.
constexpr int kLdMaxNodes = 20;
// Order of the coupled matrix up to which its energy is by log-determinants.  They cost 12 n^3 / 3
// operations on the GEMM, the band reduction 4 n^3 / 3 behind panels and a bulge chase whose share falls
// with n: order 16800 299 / 366 ms, 20001 488 / 542, 24576 865 / 823, 30000 (two passes within
// 64 GB) 1574 / 1341.
constexpr long kLdMaxOrder = 22000;
struct LdNodes {
  int n = 0;  // nodes; entry n is the proof's shift
  double t[kLdMaxNodes + 1];
  double w[kLdMaxNodes + 1];
};
// Nodes for eigenvalues in [lo, hi]; false if more than kLdMaxNodes would be needed.
bool ld_nodes(double lo, double hi, LdNodes &nd);

// Gershgorin discs of `batch` symmetric n x n matrices (lower triangle read): hi[b nblk + i] is the
// largest right end over rows 64 i ... 64 i + 63 of matrix b, nblk = ceil(n / 64).
void ld_bounds(hipStream_t s, int n, const double *H, long ld, long sH, int batch, double *hi);
// kLzSteps Lanczos steps on each matrix from three start vectors at once (V, P, Q: batch x 3 n; sv,
// part as symv3_lower takes them, ceil(n / 256) partials per matrix); ab[((3 b + k) kLzSteps + j) 2]:
// the tridiagonal matrices' diagonals and off-diagonals.
constexpr int kLzSteps = 16;
void ld_lanczos(hipStream_t s, int n, const double *H, long ld, long sH, int batch, double *V, double *P,
                double *Q, const Symv3Work &sv, double *part, double *ab);
// Smallest and largest Ritz value of the `count` tridiagonal matrices; false if one is not finite.
bool ld_ritz(const double *ab, int count, double &lo, double &hi);
// Lower triangle of H_r + t[b0 + b] I as matrix r nb + b of A (leading dimension lda), r < batch, b < nb.
void ld_shift(hipStream_t s, int n, const double *H, long ld, long sH, int batch, const LdNodes &nd,
              int b0, int nb, double *A, long lda, long sA);
// g[m nblk + i], nblk = ceil(n / 64): the part of rows 64 i ... 64 i + 63 in ln det(H_r + t) - ln det(D +
// t) from the factor L_m of m < batch nb; row r of a matrix belongs to atom (r % (3 N cells)) / (3 cells).
// Nothing for the entry without a weight.
void ld_sums(hipStream_t s, int n, const double *H, long ld, long sH, const double *L, long lda, long sA,
             int batch, const LdNodes &nd, int b0, int nb, const double *omega, int N, int cells, double *g);

}  // namespace mbd
