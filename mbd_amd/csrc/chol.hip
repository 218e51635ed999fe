// Batched blocked Cholesky of the SCS relay matrices and the solve with the
// stacked-identity right-hand side (the operations PDPOTRF('L') and
// PDPOTRS('L', NRHS=3) perform at UTILS.f90:469,473), the contraction to
// alpha_SCS and the molecular tensor (UTILS.f90:479-495), and the C6 sums
// (UTILS.f90:273-276, 302-315).
//
// Right-looking with two block sizes: per block column of NB one workgroup per
// matrix factors the NB x NB diagonal block in LDS and inverts it; the panel
// below becomes A21 * inv(L11)^T, and its update A22 -= A21 A21^T reaches only
// the rest of an outer block of NBO columns; the columns after that are
// updated once per outer block, both on the MFMA GEMM.  An update of K
// columns moves 2 sizeof(T) bytes per 2 K flops of the trailing triangle: at
// K = NB that is as long as the MFMAs take (21 matrices of order 8709 in
// FP64, trailing updates per factorisation with NBO = 128, 256, 512, 1024:
// 109, 90, 83, 82 ms; order 12288 in FP32: 133, 115, 107, 106 ms).  The
// inverted diagonal blocks are kept for the triangular solves, which then
// need only matrix-vector work per block.
#include "common.h"
#include "kernels.h"
#include "mfma.h"
#include "mol.h"
#include "profile.h"
#include "tri3.h"

#include <algorithm>
#include <functional>

namespace mbd {

namespace {

constexpr int DB = 32;                             // sub-block of a diagonal block
constexpr int DNB = kCholNB / DB;                  // sub-blocks per edge
constexpr int DTRI = DNB * (DNB + 1) / 2;
static_assert(DNB == 4, "the inverse's doubling steps are written for 4 x 4 sub-blocks");

template <typename T>
using Sub = T[DB][DB + 1];  // row-major sub-block in LDS

// LDS of k_potrf_diag: the lower sub-blocks, R^{-1} of the diagonal ones
// (R = L^T), and two scratch blocks.
template <typename T>
struct DiagLds {
  Sub<T> l[DTRI];
  Sub<T> ri[DNB];
  Sub<T> w[2];
};

__device__ constexpr int sub_index(int i, int j) { return i * (i + 1) / 2 + j; }

// The 16 x 16 tile (wave >> 1, wave & 1) of op(A) op(B) added to acc, on
// MFMA; op transposes where TA / TB is set.
template <typename T, bool TA, bool TB>
__device__ inline void sub_mm(typename Mfma<T>::acc_t &acc, const Sub<T> &A, const Sub<T> &Bm) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
  const int r = 16 * (wv >> 1) + lr, c = 16 * (wv & 1) + lr;
#pragma unroll
  for (int k = 0; k < DB; k += 4) {
    const T a = TA ? A[k + lk][r] : A[r][k + lk];
    const T b = TB ? Bm[c][k + lk] : Bm[k + lk][c];
    acc = Mfma<T>::mma(a, b, acc);
  }
}

// C = alpha acc (+ C): each wave its tile.
template <typename T, bool ADD>
__device__ inline void sub_put(Sub<T> &C, const typename Mfma<T>::acc_t &acc, T alpha) {
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, lr = lane & 15, lk = lane >> 4;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    T *p = &C[16 * (wv >> 1) + Mfma<T>::row(lk, v)][16 * (wv & 1) + lr];
    *p = ADD ? *p + alpha * acc[v] : alpha * acc[v];
  }
}

// Lower Cholesky of the 32 x 32 sub-block G (lower triangle read) by one
// wave, without barriers: lanes 0..31 hold G's columns and lanes 32..63 the
// identity's, step k applies the same row operations to both with pivot
// column k read from lane k through the scalar unit, and the identity ends as
// the inverse factor (32 steps at one barrier and one LDS round trip each
// cost 20 us, this 9 us in FP64).  Writes L over G and L^{-T} to Ri, zeros
// outside the triangles; returns the first non-positive pivot, or DB (such
// steps divide by 1 and carry on).
template <typename T>
__device__ __forceinline__ int wave_chol(Sub<T> &G, Sub<T> &Ri) {
  const int lane = threadIdx.x & 63, j = lane & (DB - 1);
  const bool ih = lane >= DB;  // identity half
  T x[DB];
#pragma unroll
  for (int i = 0; i < DB; ++i) x[i] = G[i > j ? i : j][i > j ? j : i];
#pragma unroll
  for (int i = 0; i < DB; ++i) x[i] = ih ? (i == j ? T(1) : T(0)) : x[i];
  int bad = DB;
#pragma unroll
  for (int k = 0; k < DB; ++k) {
    const T d = lane_value(x[k], k);
    if (!(d > T(0)) && bad == DB) bad = k;
    const T dd = d > T(0) ? d : T(1);
    // column k of L and of L^{-T} are final
    const bool in = ih ? (j <= k) : (k <= j);
    T *p = ih ? &Ri[j][k] : &G[j][k];
    const T rs = rsq_fast(dd);
    T v = x[k] * rs;
    // the diagonal correctly rounded (one Newton step of the square root): an
    // error of one sign in every pivot would add up in the log-determinants
    v = (!ih && j == k) ? fma(T(0.5) * rs, fma(-v, v, dd), v) : v;
    *p = in ? v : T(0);
    if (k == DB - 1) break;
    const T a = (ih || j > k) ? x[k] * rcp_fast(dd) : T(0);
#pragma unroll
    for (int i = k + 1; i < DB; ++i) x[i] = fma(-lane_value(x[i], k), a, x[i]);
  }
  return bad;
}

}  // namespace

// Factor the kb x kb diagonal block M at (k0, k0) of a matrix, write L11 back,
// and write inv(L11) (kb x kb, zero above the diagonal) to I with leading
// dimension NB.  info records the first non-positive pivot as k0 + j + 1
// (LAPACK convention).
//
// One workgroup per matrix, so a chain of dependent steps bounds it: four
// 32 x 32 factorisations by one wave each with the panel and trailing
// sub-blocks on MFMA between them, then the inverse by doubling (2 + 6
// products).  A column at a time with a barrier per step took 610 us for a
// 128 x 128 block, FP32 and FP64 alike.
template <typename T>
__device__ __forceinline__ void potrf_diag_block(T *M, int lda, int k0, int kb, T *I, int *info) {
  extern __shared__ unsigned char smem_raw[];
  DiagLds<T> &s = *reinterpret_cast<DiagLds<T> *>(smem_raw);
  using acc_t = typename Mfma<T>::acc_t;
  const acc_t zero = {0, 0, 0, 0};
  const int t = threadIdx.x;

  // lower triangle into the sub-blocks, 16 columns in flight per thread
  // (clamped addresses); the identity past kb
  const int r = t & (kCholNB - 1), rc = min(r, kb - 1), ch = t >> 7;
  for (int c0 = 0; c0 < kCholNB; c0 += 32) {
    T v[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) v[i] = M[rc + (long)min(c0 + ch + 2 * i, kb - 1) * lda];
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int c = c0 + ch + 2 * i;
      if (r / DB >= c / DB)
        s.l[sub_index(r / DB, c / DB)][r % DB][c % DB] =
            (r < kb && c < kb) ? v[i] : (r == c ? T(1) : T(0));
    }
  }
  __syncthreads();
  const int nb = (kb + DB - 1) / DB;
  for (int k = 0; k < nb; ++k) {
    if (t < 64) {
      const int bad = wave_chol<T>(s.l[sub_index(k, k)], s.ri[k]);
      if (t == 0 && bad < DB && *info == 0) *info = k0 + k * DB + bad + 1;
    }
    __syncthreads();
    if (k + 1 == nb) break;
    // sub-blocks below: L_ik = A_ik L_kk^{-T}
    acc_t p[DNB - 1] = {zero, zero, zero};
#pragma unroll
    for (int i = 0; i < DNB - 1; ++i)
      if (k + 1 + i < nb) sub_mm<T, false, false>(p[i], s.l[sub_index(k + 1 + i, k)], s.ri[k]);
    __syncthreads();
#pragma unroll
    for (int i = 0; i < DNB - 1; ++i)
      if (k + 1 + i < nb) sub_put<T, false>(s.l[sub_index(k + 1 + i, k)], p[i], T(1));
    __syncthreads();
    for (int i = k + 1; i < nb; ++i)
      for (int j = k + 1; j <= i; ++j) {
        acc_t q = zero;
        sub_mm<T, false, true>(q, s.l[sub_index(i, k)], s.l[sub_index(j, k)]);
        sub_put<T, true>(s.l[sub_index(i, j)], q, T(-1));
      }
    __syncthreads();
  }
  for (int c0 = 0; c0 < kCholNB; c0 += 2) {
    const int c = c0 + ch;
    if (r >= c && r < kb) M[r + (long)c * lda] = s.l[sub_index(r / DB, c / DB)][r % DB][c % DB];
  }
  // inverse X of the factor, X_ii = ri_i^T, the others over L's sub-blocks
  // (the unused ones past nb are formed from whatever LDS holds and dropped)
  __syncthreads();
  Sub<T> *L = s.l;
  auto X = [&](int i, int j) -> Sub<T> & { return L[sub_index(i, j)]; };
  if (nb > 1) {
    // X_10 = -X_11 (L_10 X_00), X_32 = -X_33 (L_32 X_22)
    acc_t a0 = zero, a1 = zero;
    sub_mm<T, false, true>(a0, X(1, 0), s.ri[0]);
    if (nb > 3) sub_mm<T, false, true>(a1, X(3, 2), s.ri[2]);
    sub_put<T, false>(s.w[0], a0, T(1));
    sub_put<T, false>(s.w[1], a1, T(1));
    __syncthreads();
    a0 = zero;
    a1 = zero;
    sub_mm<T, true, false>(a0, s.ri[1], s.w[0]);
    if (nb > 3) sub_mm<T, true, false>(a1, s.ri[3], s.w[1]);
    sub_put<T, false>(X(1, 0), a0, T(-1));
    if (nb > 3) sub_put<T, false>(X(3, 2), a1, T(-1));
    __syncthreads();
  }
  if (nb > 2) {
    // W = [L_20 L_21; L_30 L_31] [X_00 0; X_10 X_11], then -[X_22 0; X_32 X_33] W
    acc_t q[4] = {zero, zero, zero, zero};
    sub_mm<T, false, true>(q[0], X(2, 0), s.ri[0]);
    sub_mm<T, false, false>(q[0], X(2, 1), X(1, 0));
    sub_mm<T, false, true>(q[1], X(2, 1), s.ri[1]);
    if (nb > 3) {
      sub_mm<T, false, true>(q[2], X(3, 0), s.ri[0]);
      sub_mm<T, false, false>(q[2], X(3, 1), X(1, 0));
      sub_mm<T, false, true>(q[3], X(3, 1), s.ri[1]);
    }
    __syncthreads();
    sub_put<T, false>(X(2, 0), q[0], T(1));
    sub_put<T, false>(X(2, 1), q[1], T(1));
    if (nb > 3) {
      sub_put<T, false>(X(3, 0), q[2], T(1));
      sub_put<T, false>(X(3, 1), q[3], T(1));
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = zero;
    sub_mm<T, true, false>(q[0], s.ri[2], X(2, 0));
    sub_mm<T, true, false>(q[1], s.ri[2], X(2, 1));
    if (nb > 3) {
      sub_mm<T, false, false>(q[2], X(3, 2), X(2, 0));
      sub_mm<T, true, false>(q[2], s.ri[3], X(3, 0));
      sub_mm<T, false, false>(q[3], X(3, 2), X(2, 1));
      sub_mm<T, true, false>(q[3], s.ri[3], X(3, 1));
    }
    __syncthreads();
    sub_put<T, false>(X(2, 0), q[0], T(-1));
    sub_put<T, false>(X(2, 1), q[1], T(-1));
    if (nb > 3) {
      sub_put<T, false>(X(3, 0), q[2], T(-1));
      sub_put<T, false>(X(3, 1), q[3], T(-1));
    }
    __syncthreads();
  }
  for (int c0 = 0; c0 < kCholNB; c0 += 2) {
    const int c = c0 + ch;
    if (r < kb && c < kb)
      I[r + (long)c * kCholNB] =
          r < c ? T(0)
                : (r / DB == c / DB ? s.ri[r / DB][c % DB][r % DB]
                                    : s.l[sub_index(r / DB, c / DB)][r % DB][c % DB]);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void k_potrf_diag(T *A, int lda, long sA, int k0, int kb, T *inv,
                                                    long sinv, int *info) {
  const int b = blockIdx.x;
  potrf_diag_block(A + (long)b * sA + k0 + (long)k0 * lda, lda, k0, kb, inv + (long)b * sinv, info + b);
}

// The same for matrix blockIdx.x of matrices of different orders.
template <typename T>
__global__ __launch_bounds__(256) void k_potrf_diag_mols(int k0, const MolInfo *__restrict__ mols,
                                                         const MolMat *__restrict__ mats, T *L, T *inv,
                                                         int *info) {
  const MolMat z = mol_mat(mats, blockIdx.x);
  const MolInfo mi = mols[z.mol];
  if (k0 >= mi.n) return;
  potrf_diag_block(L + mi.a + (long)z.slot * mi.n * mi.ld + k0 + (long)k0 * mi.ld, mi.ld, k0,
                   min(kCholNB, mi.n - k0),
                   inv + mi.inv + z.slot * mol_inv_size(mi.n) + (long)k0 * kCholNB, info + blockIdx.x);
}

// energy: matrices of log-determinants.  proof > 0: of every `proof`
// consecutive ones the others are useless if the last is not positive definite,
// and their updates are left out once it has shown that (not the short panel
// products: the look took 2 % of them).
template <typename T>
void potrf_batched(hipStream_t s, int n, T *A, int lda, long sA, int batch,
                   T *inv, long sinv_blk, int *info, bool energy, int proof) {
  const int NB = kCholNB, per = std::max(1, proof);
  const int *stop = proof ? info : nullptr;
  const size_t smem = sizeof(DiagLds<T>);
  static bool attr_set = false;
  if (!attr_set) {
    MBD_HIP(hipFuncSetAttribute((const void *)k_potrf_diag<T>,
                                hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)smem));
    attr_set = true;
  }
  constexpr int NBO = kCholNBO;
  for (int o0 = 0; o0 < n; o0 += NBO) {
    const int o1 = std::min(n, o0 + NBO);  // this outer block's end
    for (int k0 = o0; k0 < o1; k0 += NB) {
      const int kb = std::min(NB, n - k0);
      T *invk = inv + (long)(k0 / NB) * NB * NB;
      {
        ProfScope ps(energy ? K_LD_DIAG : K_CHOL_DIAG, s, 0.0, batch * (2.0 / 3.0) * kb * (double)kb * kb);
        hipLaunchKernelGGL((k_potrf_diag<T>), dim3(batch), dim3(256), smem, s, A,
                           lda, sA, k0, kb, invk, sinv_blk, info);
        MBD_LAUNCH_CHECK();
      }
      const int k1 = k0 + kb;
      const int m2 = n - k1;
      if (m2 <= 0) break;
      T *A21 = A + k1 + (long)k0 * lda;
      // A21 <- A21 inv(L11)^T (in place: one column tile per row tile);
      // algorithmic work of the triangular solve: m2 kb^2 flops
      {
        ProfScope ps(energy ? K_LD_TRSM : K_CHOL_TRSM, s, 0.0, batch * (double)m2 * kb * kb);
        gemm_nt(s, false, m2, kb, kb, T(1), A21, lda, sA, invk, NB, sinv_blk,
                T(0), A21, lda, sA, batch);
      }
      // the rest of the outer block's columns, on and below the diagonal
      const int w2 = o1 - k1;
      if (w2 > 0) {
        ProfScope ps(energy ? K_LD_SYRK : K_CHOL_SYRK, s, 0.0, batch * (double)kb * w2 * (2.0 * m2 - w2 + 1.0));
        gemm_nt(s, true, m2, w2, kb, T(-1), A21, lda, sA, A21, lda, sA, T(1),
                A + k1 + (long)k1 * lda, lda, sA, batch, stop, per);
      }
    }
    // trailing A22 -= A21 A21^T on the lower triangle, A21 the outer block's
    // columns below it: m2 (m2 + 1) (o1 - o0) flops
    const int m2 = n - o1;
    if (m2 <= 0) break;
    const T *A21 = A + o1 + (long)o0 * lda;
    ProfScope ps(energy ? K_LD_SYRK : K_CHOL_SYRK, s, 0.0, batch * (double)m2 * (m2 + 1.0) * (o1 - o0));
    gemm_nt(s, true, m2, m2, o1 - o0, T(-1), A21, lda, sA, A21, lda, sA, T(1),
            A + o1 + (long)o1 * lda, lda, sA, batch, stop, per);
  }
}

// Left-looking: block column k0 of every matrix that reaches it is updated by
// all columns before it at once, so each element is written twice and the
// update's K grows with k0 (orders up to about 1000: the outer blocks of the
// right-looking form would be the whole matrix).  atleast(k) matrices, the
// first of the list, have an order above k.
template <typename T>
void potrf_mols(hipStream_t s, int nmax, const MolInfo *mols, const MolMat *mats,
                const std::function<int(int)> &atleast, T *L, T *inv, int *info) {
  const size_t smem = sizeof(DiagLds<T>);
  MBD_HIP(hipFuncSetAttribute((const void *)k_potrf_diag_mols<T>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem));
  for (int k0 = 0; k0 < nmax; k0 += kCholNB) {
    const int cnt = atleast(k0);
    if (k0) gemm_mols<T>(s, true, k0, nmax, cnt, mols, mats, L, inv);
    hipLaunchKernelGGL((k_potrf_diag_mols<T>), dim3(cnt), dim3(256), smem, s, k0, mols, mats, L, inv, info);
    MBD_LAUNCH_CHECK();
    gemm_mols<T>(s, false, k0, nmax, atleast(k0 + kCholNB), mols, mats, L, inv);
  }
}
template void potrf_mols<double>(hipStream_t, int, const MolInfo *, const MolMat *,
                                 const std::function<int(int)> &, double *, double *, int *);
template void potrf_mols<float>(hipStream_t, int, const MolInfo *, const MolMat *,
                                const std::function<int(int)> &, float *, float *, int *);

template void potrf_batched<double>(hipStream_t, int, double *, int, long,
                                    int, double *, long, int *, bool, int);
template void potrf_batched<float>(hipStream_t, int, float *, int, long, int,
                                   float *, long, int *, bool, int);

// ---------------------------------------------------------------------------
// Triangular solves with NRHS = 3, X column-major n x 3 (ldx) per matrix,
// accumulated in double (X is double; L may be float).

// HBM bound: 16 coalesced loads in flight per thread on both sides (a column
// per thread and one load at a time moved 1.8 TB/s, now 2.7; the SCS stage of a
// 4096-atom mixed solve 158.5 -> 147 ms, of a sheet of 2048 32.3 -> 27.6).
__device__ inline void load_rhs(const double *X, int ldx, int kb, double (*xs)[kCholNB]) {
  for (int e = threadIdx.x; e < 3 * kCholNB; e += kTriNT) {
    const int b = e / kCholNB, r = e % kCholNB;
    xs[b][r] = r < kb ? X[r + (long)b * ldx] : 0.0;
  }
  __syncthreads();
}

template <typename T>
__global__ __launch_bounds__(kTriNT) void k_trsv_diag(const T *inv, long sinv, int k0, int kb, double *X,
                                                      int ldx, long sX, int transposed) {
  __shared__ double xs[3][kCholNB], P[3 * kTriPW];
  const T *I = inv + (long)blockIdx.x * sinv;
  double *Xb = X + (long)blockIdx.x * sX + k0;
  load_rhs(Xb, ldx, kb, xs);
  auto put = [&](int r, double a, double b, double c) {
    Xb[r] = a;
    Xb[r + ldx] = b;
    Xb[r + 2L * ldx] = c;
  };
  if (transposed)
    dot3(I, kCholNB, kb, kb, xs[0], kCholNB, put);
  else
    mv3(I, kCholNB, kb, kb, xs[0], kCholNB, P, put);
}

// forward update: X[r] -= L[r, k0:k1] X[k0:k1] for r >= k1, kTriNT rows per
// workgroup
template <typename T>
__global__ __launch_bounds__(kTriNT) void k_trsv_upd_fwd(int n, const T *A, int lda, long sA, int k0,
                                                         int kb, double *X, int ldx, long sX) {
  __shared__ double xs[3][kCholNB], P[3 * kTriPW];
  double *Xb = X + (long)blockIdx.y * sX;
  load_rhs(Xb + k0, ldx, kb, xs);
  const int r0 = k0 + kb + blockIdx.x * kTriNT;
  mv3(A + (long)blockIdx.y * sA + r0 + (long)k0 * lda, lda, min(kTriNT, n - r0), kb, xs[0], kCholNB, P,
      [&](int r, double a, double b, double c) {
        Xb[r0 + r] -= a;
        Xb[r0 + r + ldx] -= b;
        Xb[r0 + r + 2L * ldx] -= c;
      });
}

// backward update: X[j] -= L[k0:k1, j]^T X[k0:k1] for j < k0, kTrsvCols
// columns per workgroup
constexpr int kTrsvCols = kTriNT / 64 * kTriU;
template <typename T>
__global__ __launch_bounds__(kTriNT) void k_trsv_upd_bwd(const T *A, int lda, long sA, int k0, int kb,
                                                         double *X, int ldx, long sX) {
  __shared__ double xs[3][kCholNB];
  double *Xb = X + (long)blockIdx.y * sX;
  load_rhs(Xb + k0, ldx, kb, xs);
  const int j0 = blockIdx.x * kTrsvCols;
  dot3(A + (long)blockIdx.y * sA + k0 + (long)j0 * lda, lda, kb, min(kTrsvCols, k0 - j0), xs[0], kCholNB,
       [&](int c, double a, double b, double d) {
         Xb[j0 + c] -= a;
         Xb[j0 + c + ldx] -= b;
         Xb[j0 + c + 2L * ldx] -= d;
       });
}

template <typename T>
void potrs3_batched(hipStream_t s, int n, const T *L, int lda, long sA,
                    int batch, const T *inv, long sinv_blk, double *X, int ldx,
                    long sX) {
  const int NB = kCholNB;
  const int nblk = ceil_div(n, NB);
  for (int kbk = 0; kbk < nblk; ++kbk) {  // L y = b
    const int k0 = kbk * NB, kb = (n - k0 < NB) ? n - k0 : NB;
    hipLaunchKernelGGL((k_trsv_diag<T>), dim3(batch), dim3(256), 0, s,
                       inv + (long)kbk * NB * NB, sinv_blk, k0, kb, X, ldx, sX, 0);
    MBD_LAUNCH_CHECK();
    const int rest = n - k0 - kb;
    if (rest > 0) {
      ProfScope ps(K_TRSV, s, batch * (double)rest * kb * sizeof(T), 2.0 * 3 * batch * rest * kb);
      hipLaunchKernelGGL((k_trsv_upd_fwd<T>), dim3(ceil_div(rest, 256), batch),
                         dim3(256), 0, s, n, L, lda, sA, k0, kb, X, ldx, sX);
      MBD_LAUNCH_CHECK();
    }
  }
  for (int kbk = nblk - 1; kbk >= 0; --kbk) {  // L^T x = y
    const int k0 = kbk * NB, kb = (n - k0 < NB) ? n - k0 : NB;
    hipLaunchKernelGGL((k_trsv_diag<T>), dim3(batch), dim3(256), 0, s,
                       inv + (long)kbk * NB * NB, sinv_blk, k0, kb, X, ldx, sX, 1);
    MBD_LAUNCH_CHECK();
    if (k0 > 0) {
      ProfScope ps(K_TRSV, s, batch * (double)k0 * kb * sizeof(T), 2.0 * 3 * batch * k0 * kb);
      hipLaunchKernelGGL((k_trsv_upd_bwd<T>), dim3(ceil_div(k0, kTrsvCols), batch),
                         dim3(256), 0, s, L, lda, sA, k0, kb, X, ldx, sX);
      MBD_LAUNCH_CHECK();
    }
  }
}
template void potrs3_batched<double>(hipStream_t, int, const double *, int,
                                     long, int, const double *, long,
                                     double *, int, long);
template void potrs3_batched<float>(hipStream_t, int, const float *, int, long,
                                    int, const float *, long, double *, int,
                                    long);

// ---------------------------------------------------------------------------
// Right-hand side: the stacked 3x3 identities (UTILS.f90:435-439).
__global__ void k_set_rhs(int n, double *X, int ldx, long sX) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  const int b = blockIdx.y;
  if (r >= n) return;
  double *Xb = X + (long)b * sX;
  const int c = r % 3;
  Xb[r] = (c == 0) ? 1.0 : 0.0;
  Xb[r + ldx] = (c == 1) ? 1.0 : 0.0;
  Xb[r + 2L * ldx] = (c == 2) ? 1.0 : 0.0;
}

void set_rhs(hipStream_t s, int n, double *X, int ldx, long sX, int batch) {
  hipLaunchKernelGGL(k_set_rhs, dim3(ceil_div(n, 256), batch), dim3(256), 0, s,
                     n, X, ldx, sX);
  MBD_LAUNCH_CHECK();
}

// alpha_SCS,i = tr(X_i)/3 and P = sum_i X_i per matrix (one workgroup each,
// fixed-order tree reduction).
__global__ __launch_bounds__(256) void k_contract(int N, const double *X,
                                                  int ldx, long sX,
                                                  double *alpha, double *P) {
  __shared__ double red[9][256];
  const int b = blockIdx.x, t = threadIdx.x;
  const double *Xb = X + (long)b * sX;
  double acc[9] = {0, 0, 0, 0, 0, 0, 0, 0, 0};
  for (int i = t; i < N; i += blockDim.x) {
    const double x00 = Xb[3 * i], x11 = Xb[3 * i + 1 + ldx], x22 = Xb[3 * i + 2 + 2L * ldx];
    double s = 0.0;
    s += x00 / 3.0;
    s += x11 / 3.0;
    s += x22 / 3.0;
    alpha[(long)b * N + i] = s;
    for (int c = 0; c < 3; ++c)
      for (int r = 0; r < 3; ++r) acc[r + 3 * c] += Xb[3 * i + r + (long)c * ldx];
  }
  for (int e = 0; e < 9; ++e) red[e][t] = acc[e];
  __syncthreads();
  for (int w = blockDim.x / 2; w > 0; w >>= 1) {
    if (t < w)
      for (int e = 0; e < 9; ++e) red[e][t] += red[e][t + w];
    __syncthreads();
  }
  if (t < 9) P[9 * b + t] = red[t][0];
}

void contract(hipStream_t s, int N, const double *X, int ldx, long sX,
              int batch, double *alpha, double *P) {
  hipLaunchKernelGGL(k_contract, dim3(batch), dim3(256), 0, s, N, X, ldx, sX,
                     alpha, P);
  MBD_LAUNCH_CHECK();
}

// Eigenvalues (ascending) of the symmetric 3x3 built from the upper
// triangle of P, as DSYEV('V','U',3) reads it (UTILS.f90:273): cyclic Jacobi.
__device__ void sym3_eig(const double *P, double *w) {
  double a[3][3];
  for (int r = 0; r < 3; ++r)
    for (int c = r; c < 3; ++c) a[r][c] = a[c][r] = P[r + 3 * c];
  for (int sweep = 0; sweep < 50; ++sweep) {
    const double off = fabs(a[0][1]) + fabs(a[0][2]) + fabs(a[1][2]);
    if (off == 0.0) break;
    for (int p = 0; p < 2; ++p)
      for (int q = p + 1; q < 3; ++q) {
        if (a[p][q] == 0.0) continue;
        const double theta = (a[q][q] - a[p][p]) / (2.0 * a[p][q]);
        const double tt = copysign(1.0, theta) / (fabs(theta) + sqrt(theta * theta + 1.0));
        const double c = 1.0 / sqrt(tt * tt + 1.0), sn = tt * c;
        for (int k = 0; k < 3; ++k) {
          const double akp = a[k][p], akq = a[k][q];
          a[k][p] = c * akp - sn * akq;
          a[k][q] = sn * akp + c * akq;
        }
        for (int k = 0; k < 3; ++k) {
          const double apk = a[p][k], aqk = a[q][k];
          a[p][k] = c * apk - sn * aqk;
          a[q][k] = sn * apk + c * aqk;
        }
      }
  }
  double e[3] = {a[0][0], a[1][1], a[2][2]};
  for (int i = 0; i < 3; ++i)
    for (int j = i + 1; j < 3; ++j)
      if (e[j] < e[i]) {
        const double tmp = e[i];
        e[i] = e[j];
        e[j] = tmp;
      }
  w[0] = e[0];
  w[1] = e[1];
  w[2] = e[2];
}

// Molecular C6 and the per-point eigenvalues (UTILS.f90:273-278, 288): one
// lane per grid point (a Jacobi iteration is a chain of dependent divisions:
// 600 us for the 21 points one after another), the sum in the reference's
// order by one lane.
__global__ void k_molpol(const double *P, const double *weight, double *eig,
                         double *c6_mol) {
  __shared__ double term[kNumFreq];
  const int k = threadIdx.x;
  if (k < kNumFreq) {
    double w[3];
    sym3_eig(P + 9 * k, w);
    eig[3 * k] = w[0];
    eig[3 * k + 1] = w[1];
    eig[3 * k + 2] = w[2];
    const double iso = (w[0] + w[1] + w[2]) / 3.0;
    term[k] = weight[k] * (iso * iso);
  }
  __syncthreads();
  if (k == 0) {
    double acc = 0.0;
    for (int q = 1; q < kNumFreq; ++q) acc = acc + term[q];
    *c6_mol = kThreeOverPi * acc;
  }
}

// Per-atom C6 (UTILS.f90:302-313): alpha layout [k * N + i], k = 0..20.
__global__ void k_c6_atoms(int N, const double *alpha, const double *weight,
                           double *c6) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  double s = 0.0;
  for (int k = 1; k < kNumFreq; ++k) {
    const double a = alpha[(long)k * N + i];
    s = s + weight[k] * (a * a);
  }
  c6[i] = s * kThreeOverPi;
}

void c6_sums(hipStream_t s, int N, const double *alpha, const double *P,
             const double *weight, double *eig, double *c6_mol, double *c6) {
  hipLaunchKernelGGL(k_molpol, dim3(1), dim3(64), 0, s, P, weight, eig, c6_mol);
  MBD_LAUNCH_CHECK();
  hipLaunchKernelGGL(k_c6_atoms, dim3(ceil_div(N, 256)), dim3(256), 0, s, N,
                     alpha, weight, c6);
  MBD_LAUNCH_CHECK();
}

}  // namespace mbd
