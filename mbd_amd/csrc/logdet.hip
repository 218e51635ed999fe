// E_MBD without eigenvalues (the sum 1/2 sum sqrt(lambda) - 1/2 sum omega of
// UTILS.f90:835-877, for a matrix whose eigenvalues are all positive).
//
// With D = diag(omega^2), sqrt(x) - sqrt(d) = 1/pi int_0^inf ln((x + y^2) /
// (d + y^2)) dy, so
//   E = 1/(2 pi) int_0^inf [ln det(C + y^2) - ln det(D + y^2)] dy,
// and a Cholesky factor gives each log-determinant.  With all eigenvalues (and
// omega^2) in [lo, hi], y = sqrt(lo) sc(u | k') with k^2 = lo / hi turns the
// integrand into an even periodic function of u, analytic for |Im u| < K, and
// the midpoint rule with N points on [0, K'] converges as
// exp(-2 pi K N / K') = exp(-2 pi^2 N / ln(16 hi / lo)) (the substitution of
// Hale, Higham and Trefethen for contour integrals of matrix functions; SIAM
// J. Numer. Anal. 46, 2008).  N nodes (8 to 13 for the first guess of lo on
// what has been measured, up to kLdMaxNodes taken) and one more factorisation
// replace the reduction to tridiagonal form and the bisection: (N + 1) n^3 / 3
// flops on the GEMM against 4 n^3 / 3 in panels, a bulge chase and Sturm counts
// bound by latency.
// hi is Gershgorin's bound, or for large orders the largest Ritz value of 16
// Lanczos steps from three fixed start vectors and a fifth of the Ritz values'
// spread.  That one is a heuristic: nothing proves it.  For start vectors
// uniform on the sphere the largest eigenvalue would lie beyond it with a
// probability of some 1e-10 at order 12288 (Kuczynski and Wozniakowski, SIAM J.
// Matrix Anal. Appl. 13, 1992: 1.65 sqrt(n) exp(-sqrt(e) (2 kLzSteps - 1)) for
// each vector, e = 1/6).  The rule loses accuracy gradually: with the largest
// eigenvalue 5, 20, 50 and 100 % beyond the interval the energy's relative
// error is 1e-14, 3e-13 to 7e-13, 1e-11 to 9e-11 and 2e-9 to 6e-9 (spectra of
// cells of 600 and 1000 atoms).
// lo is a guess that one more Cholesky factorisation, of C - lo I, proves (it
// exists exactly if every eigenvalue exceeds lo); the caller takes the
// eigenvalue path when it does not exist.
#include <algorithm>
#include <cmath>
#include <vector>

#include "common.h"
#include "logdet.h"
#include "mol.h"

namespace mbd {

namespace {

double agm(double a, double b) {
  for (int i = 0; i < 40 && std::fabs(a - b) > 1e-16 * a; ++i) {
    const double t = 0.5 * (a + b);
    b = std::sqrt(a * b);
    a = t;
  }
  return 0.5 * (a + b);
}

// sn, cn, dn of u with complementary modulus kc, by the arithmetic-geometric
// mean (Abramowitz and Stegun 16.4)
void jacobi(double u, double kc, double &sn, double &cn, double &dn) {
  constexpr int M = 16;
  double a[M + 1], c[M + 1], b = kc;
  a[0] = 1.0;
  c[0] = std::sqrt((1.0 - kc) * (1.0 + kc));
  int n = 0;
  while (n < M && c[n] > 1e-17 * a[n]) {
    a[n + 1] = 0.5 * (a[n] + b);
    c[n + 1] = 0.5 * (a[n] - b);
    b = std::sqrt(a[n] * b);
    ++n;
  }
  double phi = std::ldexp(a[n] * u, n);
  for (; n > 0; --n) phi = 0.5 * (phi + std::asin(c[n] / a[n] * std::sin(phi)));
  sn = std::sin(phi);
  cn = std::cos(phi);
  dn = std::sqrt(cn * cn + kc * kc * sn * sn);
}

// The midpoint rule's relative error.  Its error alone, of energies of order 36
// to 1800 (rings, chains, cells): 1e-13 up to 8e-13 of the energy, 1e-14 up to
// 2e-14, 1e-15 up to 1e-15 (for one node more).
constexpr double kLdEps = 1e-14;
constexpr int GB = 64;            // rows of a bounds workgroup
constexpr int GW = 8;             // its waves
constexpr int SC = 8;             // columns of a shift workgroup

}  // namespace

bool ld_nodes(double lo, double hi, LdNodes &nd) {
  if (!(lo > 0.0) || !(hi > lo) || !std::isfinite(hi)) return false;
  const double pi = 3.14159265358979323846;
  const double kc = std::sqrt(lo / hi);  // k: the complementary modulus of k'
  const double Kp = pi / (2.0 * agm(1.0, kc));
  const double K = pi / (2.0 * agm(1.0, std::sqrt((1.0 - kc) * (1.0 + kc))));
  nd.n = std::max(2, (int)std::ceil(std::log(2.0 / kLdEps) * Kp / (2.0 * pi * K)));
  if (nd.n > kLdMaxNodes) return false;
  const double h = Kp / nd.n;
  for (int b = 0; b < nd.n; ++b) {
    double sn, cn, dn;
    jacobi((b + 0.5) * h, kc, sn, cn, dn);
    nd.t[b] = lo * (sn / cn) * (sn / cn);
    nd.w[b] = h * std::sqrt(lo) * dn / (cn * cn) / (2.0 * pi);
  }
  nd.t[nd.n] = -lo;
  nd.w[nd.n] = 0.0;
  return true;
}

// Lanczos from three start vectors, so that the interval of the quadrature is
// the spectrum's and not Gershgorin's (a cell of 4096 atoms: 13 -> 11
// nodes, each a factorisation of 11 ms, for 3.3 ms).  One workgroup per vector: the
// products before each step take longer than its pass over three vectors.
__device__ inline double lz_sum(double v, double *red) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double s = 0.0;
  for (int i = 0; i < 16; ++i) s += red[i];
  return s;
}

__global__ __launch_bounds__(1024) void k_lz_init(int n, double *V, double *P) {
  __shared__ double red[16];
  const long at = ((long)blockIdx.y * 3 + blockIdx.x) * n;
  double ss = 0.0;
  for (int i = threadIdx.x; i < n; i += 1024) {
    // an integer hash of the position as a number in (-1, 1)
    unsigned z = (unsigned)(at + i) * 2654435769u + 0x9E3779B9u;
    z = (z ^ (z >> 16)) * 0x85EBCA6Bu;
    z = (z ^ (z >> 13)) * 0xC2B2AE35u;
    z ^= z >> 16;
    const double x = ((double)z + 0.5) * (2.0 / 4294967296.0) - 1.0;
    V[at + i] = x;
    P[at + i] = 0.0;
    ss += x * x;
  }
  const double is = 1.0 / sqrt(lz_sum(ss, red));
  for (int i = threadIdx.x; i < n; i += 1024) V[at + i] *= is;
}

__global__ __launch_bounds__(1024) void k_lz_step(int n, int j, int npart, const double *part, double *V,
                                                  double *P, const double *Q, double *ab) {
  __shared__ double red[16];
  const int k = blockIdx.x, b = blockIdx.y, t = threadIdx.x;
  const long at = ((long)b * 3 + k) * n;
  double *o = ab + ((long)b * 3 + k) * kLzSteps * 2;
  double a = 0.0;
  for (int i = t; i < npart; i += 1024) a += part[((long)b * npart + i) * 4 + k];
  a = lz_sum(a, red);
  const double bp = j ? o[2 * j - 1] : 0.0;
  double ss = 0.0;
  for (int i = t; i < n; i += 1024) {
    const double w = Q[at + i] - a * V[at + i] - bp * P[at + i];
    P[at + i] = w;
    ss += w * w;
  }
  const double be = sqrt(lz_sum(ss, red)), ib = be > 0.0 ? 1.0 / be : 0.0;
  for (int i = t; i < n; i += 1024) {
    const double w = P[at + i];
    P[at + i] = V[at + i];
    V[at + i] = w * ib;
  }
  if (t == 0) {
    o[2 * j] = a;
    o[2 * j + 1] = be;
  }
}

void ld_lanczos(hipStream_t s, int n, const double *H, long ld, long sH, int batch, double *V, double *P,
                double *Q, const Symv3Work &sv, double *part, double *ab) {
  hipLaunchKernelGGL(k_lz_init, dim3(3, batch), dim3(1024), 0, s, n, V, P);
  MBD_LAUNCH_CHECK();
  const int np = ceil_div(n, 256);
  for (int j = 0; j < kLzSteps; ++j) {
    symv3_lower<double>(s, n, H, (int)ld, sH, batch, V, n, 3L * n, Q, n, 3L * n, sv, 0, part, np, nullptr,
                        nullptr, 0);
    hipLaunchKernelGGL(k_lz_step, dim3(3, batch), dim3(1024), 0, s, n, j, np, part, V, P, Q, ab);
    MBD_LAUNCH_CHECK();
  }
}

bool ld_ritz(const double *ab, int count, double &lo, double &hi) {
  lo = 1e300;
  hi = -1e300;
  for (int c = 0; c < count; ++c, ab += 2 * kLzSteps) {
    double g0 = 1e300, g1 = -1e300, scale = 0.0;
    int m = kLzSteps;
    for (int j = 0; j < kLzSteps; ++j) {
      if (!std::isfinite(ab[2 * j]) || !std::isfinite(ab[2 * j + 1])) return false;
      scale = std::max(scale, std::fabs(ab[2 * j]));
      if (ab[2 * j + 1] <= 1e-8 * scale) {  // an invariant subspace: the rest is rounding
        m = j + 1;
        break;
      }
    }
    for (int j = 0; j < m; ++j) {
      const double r = (j ? ab[2 * j - 1] : 0.0) + (j + 1 < m ? ab[2 * j + 1] : 0.0);
      g0 = std::min(g0, ab[2 * j] - r);
      g1 = std::max(g1, ab[2 * j] + r);
    }
    auto below = [&](double x) {  // Ritz values below x
      int cnt = 0;
      double q = 1.0;
      for (int j = 0; j < m; ++j) {
        const double e = j ? ab[2 * j - 1] : 0.0;
        q = ab[2 * j] - x - e * e / (q != 0.0 ? q : 1e-300);
        cnt += q < 0.0;
      }
      return cnt;
    };
    for (int side = 0; side < 2; ++side) {
      double a = g0, b = g1;
      for (int i = 0; i < 50; ++i) {
        const double x = 0.5 * (a + b);
        (below(x) >= (side ? m : 1) ? b : a) = x;
      }
      (side ? hi : lo) = side ? std::max(hi, b) : std::min(lo, a);
    }
  }
  return true;
}

// Row sums of |H| for 64 rows: the part left of the diagonal block with lanes
// on rows, the diagonal block, and the columns below it (the rows' part right
// of the diagonal) with lanes down a column; every partial has one owner and
// a fixed order.  Each element off the diagonal blocks is read twice; HBM
// bound (0.4 ms at n = 12288).
__device__ void bounds_block(int n, const double *__restrict__ M, long ld, int r0, double *hi) {
  __shared__ double part[GW][GB], diag[GB], below[GB];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int nr = min(GB, n - r0);
  const int row = r0 + min(lane, nr - 1);
  double s = 0.0;
  for (int c = w; c < r0; c += 8 * GW) {
    double v[8];
#pragma unroll
    for (int q = 0; q < 8; ++q) v[q] = M[row + (long)min(c + q * GW, r0 - 1) * ld];
#pragma unroll
    for (int q = 0; q < 8; ++q) s += (c + q * GW < r0) ? fabs(v[q]) : 0.0;
  }
  // the diagonal block: row `lane`, its columns dealt to the waves
  for (int c = w; c < nr; c += GW) {
    const int a = max(lane, c), b = min(lane, c);
    const double v = M[r0 + min(a, nr - 1) + (long)(r0 + b) * ld];
    s += (lane < nr && c != lane) ? fabs(v) : 0.0;
    if (c == lane) diag[lane] = v;
  }
  part[w][lane] = s;
  // columns r0 + w, r0 + w + GW, ... below the diagonal block
  double q[GB / GW];
#pragma unroll
  for (int i = 0; i < GB / GW; ++i) q[i] = 0.0;
  for (int r = r0 + GB + lane; r < n; r += 64) {
#pragma unroll
    for (int i = 0; i < GB / GW; ++i) q[i] += fabs(M[r + (long)min(r0 + w + i * GW, n - 1) * ld]);
  }
#pragma unroll
  for (int i = 0; i < GB / GW; ++i) {
    for (int o = 32; o > 0; o >>= 1) q[i] += __shfl_xor(q[i], o, 64);
    if (lane == 0) below[w + i * GW] = q[i];
  }
  __syncthreads();
  if (w == 0) {
    double t = below[lane];
    for (int i = 0; i < GW; ++i) t += part[i][lane];
    t += lane < nr ? diag[lane] : 0.0;
    // a NaN row must not be lost in the maximum
    bool bad = lane < nr && !(t < 1e300);
    double m = lane < nr ? t : -1e300;
    for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
    if (__any(bad)) m = INFINITY;
    if (lane == 0) *hi = m;
  }
}

__global__ __launch_bounds__(64 * GW) void k_ld_bounds(int n, const double *__restrict__ H, long ld,
                                                       long sH, double *__restrict__ hi) {
  bounds_block(n, H + (long)blockIdx.y * sH, ld, blockIdx.x * GB,
               hi + (long)blockIdx.y * gridDim.x + blockIdx.x);
}

// Molecule blockIdx.x, rows of blockIdx.y.
__global__ __launch_bounds__(64 * GW) void k_ld_bounds_mols(const MolInfo *__restrict__ mols,
                                                            const double *__restrict__ C,
                                                            double *__restrict__ hi) {
  const MolInfo mi = mols[blockIdx.x];
  if ((int)blockIdx.y * GB < mi.n)
    bounds_block(mi.n, C + mi.c, mi.ld, blockIdx.y * GB, hi + (long)blockIdx.x * gridDim.y + blockIdx.y);
}

void ld_bounds_mols(hipStream_t s, int nmol, int nmax, const MolInfo *mols, const double *C, double *hi) {
  hipLaunchKernelGGL(k_ld_bounds_mols, dim3(nmol, ceil_div(nmax, GB)), dim3(64 * GW), 0, s, mols, C, hi);
  MBD_LAUNCH_CHECK();
}

void ld_bounds(hipStream_t s, int n, const double *H, long ld, long sH, int batch, double *hi) {
  hipLaunchKernelGGL(k_ld_bounds, dim3(ceil_div(n, GB), batch), dim3(64 * GW), 0, s, n, H, ld, sH, hi);
  MBD_LAUNCH_CHECK();
}

// Each element of the lower triangle read once and written once per node.
__global__ __launch_bounds__(256) void k_ld_shift(int n, const double *__restrict__ H, long ld,
                                                  long sH, LdNodes nd, int b0, int nb,
                                                  double *__restrict__ A, long lda, long sA) {
  const int r = blockIdx.x * 256 + threadIdx.x, c0 = blockIdx.y * SC;
  if (blockIdx.x * 256 + 255 < c0 || r >= n) return;
  const double *M = H + (long)blockIdx.z * sH;
  double v[SC];
#pragma unroll
  for (int i = 0; i < SC; ++i) v[i] = M[r + (long)min(c0 + i, n - 1) * ld];
  double *out = A + (long)blockIdx.z * nb * sA + r;
  for (int b = 0; b < nb; ++b, out += sA) {
    const double t = nd.t[b0 + b];
#pragma unroll
    for (int i = 0; i < SC; ++i) {
      const int c = c0 + i;
      if (c <= r) out[(long)c * lda] = r == c ? v[i] + t : v[i];
    }
  }
}

void ld_shift(hipStream_t s, int n, const double *H, long ld, long sH, int batch, const LdNodes &nd,
              int b0, int nb, double *A, long lda, long sA) {
  hipLaunchKernelGGL(k_ld_shift, dim3(ceil_div(n, 256), ceil_div(n, SC), batch), dim3(256), 0, s, n, H,
                     ld, sH, nd, b0, nb, A, lda, sA);
  MBD_LAUNCH_CHECK();
}

// Matrix blockIdx.x of a list, 256 rows by SCM columns per workgroup.
constexpr int SCM = 32;
__global__ __launch_bounds__(256) void k_ld_shift_mols(const MolInfo *__restrict__ mols,
                                                       const MolMat *__restrict__ mats,
                                                       const double *__restrict__ shift,
                                                       const double *__restrict__ C,
                                                       double *__restrict__ A) {
  const MolMat z = mats[blockIdx.x];
  const MolInfo mi = mols[z.mol];
  const int r = blockIdx.y * 256 + threadIdx.x, n = mi.n;
  const double t = shift[blockIdx.x];
  const int c1 = min(n, (int)(blockIdx.z + 1) * SCM);
  const double *M = C + mi.c;
  double *out = A + mi.a + (long)z.slot * n * mi.ld;
  if (r >= n) return;
  for (int c0 = blockIdx.z * SCM; c0 < c1 && c0 <= r; c0 += SC) {
    double v[SC];
#pragma unroll
    for (int i = 0; i < SC; ++i) v[i] = M[r + (long)min(c0 + i, n - 1) * mi.ld];
#pragma unroll
    for (int i = 0; i < SC; ++i)
      if (c0 + i <= r) out[r + (long)(c0 + i) * mi.ld] = r == c0 + i ? v[i] + t : v[i];
  }
}

void ld_shift_mols(hipStream_t s, int nmat, int nmax, const MolInfo *mols, const MolMat *mats,
                   const double *shift, const double *C, double *A) {
  hipLaunchKernelGGL(k_ld_shift_mols, dim3(nmat, ceil_div(nmax, 256), ceil_div(nmax, SCM)), dim3(256), 0, s,
                     mols, mats, shift, C, A);
  MBD_LAUNCH_CHECK();
}

// Matrix blockIdx.x of a list: as k_ld_sums.
__global__ __launch_bounds__(256) void k_ld_sums_mols(const MolInfo *__restrict__ mols,
                                                      const MolMat *__restrict__ mats,
                                                      const double *__restrict__ shift,
                                                      const double *__restrict__ A,
                                                      const double *__restrict__ omega,
                                                      double *__restrict__ g) {
  __shared__ double red[4];
  const MolMat z = mats[blockIdx.x];
  const MolInfo mi = mols[z.mol];
  const int t = threadIdx.x;
  const double *M = A + mi.a + (long)z.slot * mi.n * mi.ld;
  double s = 0.0;
  for (int j = t; j < mi.n; j += 256) {
    const double l = M[j + (long)j * mi.ld], w = omega[mi.atom0 + j / 3];
    s += log(l * l / (w * w + shift[blockIdx.x]));
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((t & 63) == 0) red[t >> 6] = s;
  __syncthreads();
  if (t == 0) g[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

void ld_sums_mols(hipStream_t s, int nmat, const MolInfo *mols, const MolMat *mats, const double *shift,
                  const double *A, const double *omega, double *g) {
  hipLaunchKernelGGL(k_ld_sums_mols, dim3(nmat), dim3(256), 0, s, mols, mats, shift, A, omega, g);
  MBD_LAUNCH_CHECK();
}

// Sum over the rows of ln(L_jj^2 / (omega_j^2 + t)) in a fixed order, 64 rows
// per workgroup.  In exact arithmetic L_jj^2 = C_jj + t - d_j with d_j the sum
// of the squares left of the diagonal, and the term is log1p((C_jj - omega_j^2
// - d_j) / (omega_j^2 + t)): it has no rounding of the diagonal's size, which
// at a large shift is far above the term (d_j / t is 1e-5 and 1e-7 at the last
// two nodes) and has the largest weights (the last node's 1 to 3, the third
// last's 0.08).  So the last kLdRowNodes nodes' rows are read, the others'
// diagonal only.  Relative errors against 80-bit energies, of the eigenvalue
// path / all nodes by the diagonal / the last two by rows / all by rows: ring
// of 12 (order 36) 1.7e-13 / 3.6e-13 / 1.3e-14 / 1.0e-14, order 42 1.1e-13 /
// 1.5e-13 / 1.5e-14 / 6.5e-15, 1584 2.5e-14 / 1.8e-14 / 5.6e-15 / 4.6e-15,
// periodic of order 3993 2.6e-14 / 8.8e-14 / 7e-16 / 1.4e-15; 104 matrices of
// order 3072 16 us / 169 us / 0.8 ms of a pass of 34 ms.
constexpr int kLdRowNodes = 2;
constexpr int SW = 16;  // waves of a sums workgroup
__global__ __launch_bounds__(64 * SW) void k_ld_sums(int n, const double *__restrict__ H, long ld, long sH,
                                                     const double *__restrict__ L, long lda, long sA,
                                                     LdNodes nd, int b0, int nb,
                                                     const double *__restrict__ omega, int N, int cells,
                                                     double *__restrict__ g) {
  __shared__ double part[SW][GB];
  const int m = blockIdx.y, b = b0 + m % nb, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (b == nd.n) return;  // the proof has no weight
  const int r0 = blockIdx.x * GB, row = min(r0 + lane, n - 1), end = min(r0 + GB - 1, n - 1);
  const double *M = L + (long)m * sA + row;
  const bool rows = b >= nd.n - kLdRowNodes;
  double s = 0.0;
  if (rows) {
    for (int c = w; c < end; c += 8 * SW) {
      double v[8];
#pragma unroll
      for (int q = 0; q < 8; ++q) v[q] = M[(long)min(c + q * SW, end) * lda];
#pragma unroll
      for (int q = 0; q < 8; ++q) s = c + q * SW < row ? fma(v[q], v[q], s) : s;
    }
    part[w][lane] = s;
    __syncthreads();
  }
  if (w) return;
  const double om = omega[(row % (3 * N * cells)) / (3 * cells)], w2 = om * om, d = w2 + nd.t[b];
  if (rows) {
    for (int i = 1; i < SW; ++i) s += part[i][lane];
    s = log1p(((H[(long)(m / nb) * sH + row + row * ld] - w2) - s) / d);
  } else {
    const double l = M[row * lda];
    s = log(l * l / d);
  }
  s = r0 + lane < n ? s : 0.0;
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if (lane == 0) g[(long)m * gridDim.x + blockIdx.x] = s;
}

void ld_sums(hipStream_t s, int n, const double *H, long ld, long sH, const double *L, long lda, long sA,
             int batch, const LdNodes &nd, int b0, int nb, const double *omega, int N, int cells, double *g) {
  hipLaunchKernelGGL(k_ld_sums, dim3(ceil_div(n, GB), batch * nb), dim3(64 * SW), 0, s, n, H, ld, sH, L, lda,
                     sA, nd, b0, nb, omega, N, cells, g);
  MBD_LAUNCH_CHECK();
}

}  // namespace mbd
