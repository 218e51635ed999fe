// MFMA GEMM "NT" update for CDNA4: C = alpha * A * B^T + beta * C.
//
// This is the trailing-update engine of the blocked factorisations: the
// Cholesky panel solve (as a product with the inverted diagonal block) and
// symmetric rank-k update, and the two-sided Householder SYR2K of the
// tridiagonalisation.  One 256-thread workgroup owns a 128 x 128 tile of C;
// its four wave64s each own a 64 x 64 sub-tile held as 4 x 4 MFMA 16x16
// accumulators (v_mfma_f64_16x16x4_f64, v_mfma_f32_16x16x4_f32).  K is staged
// through double-buffered LDS in steps of 16 with the next global tile
// prefetched into registers while the MFMAs run.
//
// Rows are dealt to the 16 x 16 blocks so that a lane's blocks hold V
// consecutive rows (V = 16 bytes of elements: 4 in FP32, 2 in FP64): block i
// of a wave covers rows V (16 (i / V) + l) + i % V.  One 16-byte LDS read
// then feeds V blocks, and with the blocks computed transposed (the B tile as
// the MFMA's first operand) a lane holds V consecutive rows of each of its
// columns of C, so global accesses are 16 bytes a lane on both sides.  The
// matrix cores bound it: 56 TFLOP/s in FP64 and 121 in FP32 over the updates
// of a 21-matrix Cholesky of order 8709 / 12288 (35 and 73 with 8-byte
// accesses, branches between the loads and K = 128 updates), against 77 and
// 155 of the MFMAs alone.
#include "common.h"
#include "kernels.h"
#include "mfma.h"
#include "mol.h"

namespace mbd {

namespace {

constexpr int BM = 128, BN = 128, BK = 16, NT = 256;

template <typename T>
struct Vec16;  // 16 bytes of elements, element-aligned
template <>
struct Vec16<double> {
  typedef double t __attribute__((ext_vector_type(2), aligned(8)));
  static constexpr int n = 2;
};
template <>
struct Vec16<float> {
  typedef float t __attribute__((ext_vector_type(4), aligned(4)));
  static constexpr int n = 4;
};

// Two waves per SIMD (launch bound): the FP64 form otherwise takes 202 VGPRs
// plus 128 AGPRs, one workgroup per CU, and each workgroup's prologue,
// barriers and epilogue stall the matrix cores.
// LOWER: the tiles on and below the diagonal of an m x n trapezoid (n <= m).
// GEN: operands read an element at a time, for fewer than V rows or columns
// and for ta: op(A)[r][k] = A[k + r lda] instead of A[r + k lda];
// tb: op(B)[c][k] = B[k + c ldb] instead of B[c + k ldb].
// No load of the K loop sits under a branch: past the edges of A, B and K the
// addresses are clamped and the values put right (uniform branch, edge tiles
// only) before they go to LDS; branches between the loads had made the
// compiler wait for each one.
// ml, nl: rows of A and of B that may be read (m, n or more).  A wave whose
// 64 x 64 sub-tile lies past m or n computes nothing.
// STOP: *stop set leaves the tile as it is (looked at behind the first loads,
// whose latency covers the look's).
template <typename T, bool LOWER, bool GEN, bool STOP = false>
__device__ __forceinline__ void gemm_tile(int m, int n, int ml, int nl, int k, T alpha,
                                          const T *__restrict__ A, int lda, const T *__restrict__ B,
                                          int ldb, T beta, T *__restrict__ C, int ldc, int tm, int tn,
                                          int ta, int tb, const int *stop = nullptr) {
  using vec = typename Vec16<T>::t;
  constexpr int V = Vec16<T>::n, G = 4 / V;  // row groups of a wave
  constexpr int NV = BM * BK / V / NT;       // operand vectors per thread
  constexpr int KS = NT / (BM / V);          // their distance in k
  const int row0 = tm * BM, col0 = tn * BN;

  __shared__ __align__(16) T As[2][BK][BM];
  __shared__ __align__(16) T Bs[2][BK][BN];

  const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int lr = lane & 15, lk = lane >> 4;

  typename Mfma<T>::acc_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = typename Mfma<T>::acc_t{0, 0, 0, 0};

  // this thread's vectors: rows sr ... sr + V - 1 of the tiles, columns
  // sk + KS i; at the edges the last V rows, shifted back into place below
  const int sr = (t % (BM / V)) * V, sk = t / (BM / V);
  const int ar = min(row0 + sr, ml - V), br = min(col0 + sr, nl - V);
  const bool edge = row0 + BM > m || col0 + BN > n;
  vec ra[NV], rb[NV];
  auto gload = [&](int k0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int kc = min(k0 + sk + KS * i, k - 1);
      if (GEN) {
#pragma unroll
        for (int q = 0; q < V; ++q) {
          const int r = min(row0 + sr + q, ml - 1), c = min(col0 + sr + q, nl - 1);
          ra[i][q] = A[ta ? kc + (long)r * lda : r + (long)kc * lda];
          rb[i][q] = B[tb ? kc + (long)c * ldb : c + (long)kc * ldb];
        }
      } else {
        ra[i] = *(const vec *)(A + ar + (long)kc * lda);
        rb[i] = *(const vec *)(B + br + (long)kc * ldb);
      }
    }
  };
  auto sstore = [&](int buf, int k0) {
    if (!GEN && edge) {
      const int da = row0 + sr - ar, db = col0 + sr - br;
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int q = 0; q < V; ++q)
#pragma unroll
          for (int z = V - 1; z > q; --z) {
            ra[i][q] = da == z - q ? ra[i][z] : ra[i][q];
            rb[i][q] = db == z - q ? rb[i][z] : rb[i][q];
          }
    }
    if (k0 + BK > k) {
#pragma unroll
      for (int i = 0; i < NV; ++i) {
        const bool in = k0 + sk + KS * i < k;
#pragma unroll
        for (int q = 0; q < V; ++q) {
          ra[i][q] = in ? ra[i][q] : T(0);
          rb[i][q] = in ? rb[i][q] : T(0);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      *(vec *)__builtin_assume_aligned(&As[buf][sk + KS * i][sr], 16) = ra[i];
      *(vec *)__builtin_assume_aligned(&Bs[buf][sk + KS * i][sr], 16) = rb[i];
    }
  };
  // the MFMAs of one staged K tile, the next step's fragments read ahead
  auto compute = [&](int cur) {
    vec af[2][G], bf[2][G];
    auto frag = [&](int b, int kk) {
#pragma unroll
      for (int g = 0; g < G; ++g) {
        af[b][g] = *(const vec *)__builtin_assume_aligned(&As[cur][kk + lk][wm * 64 + V * (16 * g + lr)], 16);
        bf[b][g] = *(const vec *)__builtin_assume_aligned(&Bs[cur][kk + lk][wn * 64 + V * (16 * g + lr)], 16);
      }
    };
    frag(0, 0);
#pragma unroll
    for (int q = 0; q < BK / 4; ++q) {
      if (q + 1 < BK / 4) frag((q + 1) & 1, 4 * (q + 1));
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[i][j] = Mfma<T>::mma(bf[q & 1][j / V][j % V], af[q & 1][i / V][i % V], acc[i][j]);
    }
  };

  const bool idle = row0 + wm * 64 >= m || col0 + wn * 64 >= n;
  const int nk = (k + BK - 1) / BK;
  const int halt = STOP ? *stop : 0;
  gload(0);
  if (STOP) {
    __builtin_amdgcn_sched_barrier(0);
    if (halt) return;
  }
  sstore(0, 0);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    if (kt + 1 < nk) gload((kt + 1) * BK);
    __builtin_amdgcn_s_setprio(1);  // its MFMAs before the other waves' loads
    if (!idle) compute(kt & 1);
    __builtin_amdgcn_s_setprio(0);
    if (kt + 1 < nk) sstore((kt & 1) ^ 1, (kt + 1) * BK);
    __syncthreads();
  }

  // C in G^2 blocks of 16 V rows by 16 V columns per wave: block (g, h) holds
  // rows crow(g) ... + V - 1 and columns ccol(h, j, v) of the lane
  auto crow = [&](int g) { return row0 + wm * 64 + V * (16 * g + lr); };
  auto ccol = [&](int h, int j, int v) {
    return col0 + wn * 64 + V * (16 * h + Mfma<T>::row(lk, v)) + j;
  };
  if (!edge && (!LOWER || tm > tn)) {
    // a block's C is loaded while the block before it is stored
    vec cv[2][V][4];
    auto cload = [&](int b) {
#pragma unroll
      for (int j = 0; j < V; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          cv[b & 1][j][v] = *(const vec *)(C + crow(b / G) + (long)ccol(b % G, j, v) * ldc);
    };
    if (beta != T(0)) cload(0);
#pragma unroll
    for (int b = 0; b < G * G; ++b) {
      __builtin_amdgcn_sched_barrier(0);  // no earlier loads: their registers would spill
      if (beta != T(0) && b + 1 < G * G) cload(b + 1);
#pragma unroll
      for (int j = 0; j < V; ++j)
#pragma unroll
        for (int v = 0; v < 4; ++v) {
          vec x;
#pragma unroll
          for (int q = 0; q < V; ++q) {
            const T p = alpha * acc[V * (b / G) + q][V * (b % G) + j][v];
            x[q] = beta != T(0) ? p + beta * cv[b & 1][j][v][q] : p;
          }
          *(vec *)(C + crow(b / G) + (long)ccol(b % G, j, v) * ldc) = x;
        }
    }
    return;
  }
  // edge and diagonal tiles, an element at a time: a column group's loads
  // before its first store (a load after a store to C, which may alias it,
  // would wait for the previous element's round trip)
#pragma unroll
  for (int b = 0; b < G * G; ++b)
#pragma unroll
    for (int j = 0; j < V; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      T x[4][V];
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int q = 0; q < V; ++q)
          x[v][q] = C[min(crow(b / G) + q, m - 1) + (long)min(ccol(b % G, j, v), n - 1) * ldc];
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int q = 0; q < V; ++q) {
          const T p = alpha * acc[V * (b / G) + q][V * (b % G) + j][v];
          x[v][q] = beta != T(0) ? p + beta * x[v][q] : p;
          asm volatile("" : "+v"(x[v][q]));  // computed here, not sunk into the stores' branches
        }
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int q = 0; q < V; ++q) {
          const int r = crow(b / G) + q, c = ccol(b % G, j, v);
          if (r < m && c < n && (!LOWER || r >= c)) C[r + (long)c * ldc] = x[v][q];
        }
    }
}

// One uniform batch: matrix blockIdx.z of each operand, tile blockIdx.x.
// STOP: nothing for the matrices whose entry of stop says so (an instance of
// its own: the look alone costs the short products of every other caller 1 to 2 %).
template <typename T, bool LOWER, bool GEN, bool STOP>
__global__ __launch_bounds__(NT, 2) void k_gemm_nt(
    int m, int n, int k, T alpha, const T *__restrict__ A, int lda, long sA,
    const T *__restrict__ B, int ldb, long sB, T beta, T *__restrict__ C,
    int ldc, long sC, int tiles_n, int ta, int tb, const int *stop, int per) {
  int tm, tn;
  const int idx = blockIdx.x;
  if (LOWER && idx < tiles_n * (tiles_n + 1) / 2) {
    tm = (int)((sqrt(8.0 * idx + 1.0) - 1.0) * 0.5);
    while ((tm + 1) * (tm + 2) / 2 <= idx) ++tm;
    while (tm * (tm + 1) / 2 > idx) --tm;
    tn = idx - tm * (tm + 1) / 2;
  } else {
    const int rest = LOWER ? idx - tiles_n * (tiles_n + 1) / 2 : idx;
    tm = rest / tiles_n + (LOWER ? tiles_n : 0);
    tn = rest % tiles_n;
  }
  const long bz = blockIdx.z;
  gemm_tile<T, LOWER, GEN, STOP>(m, n, m, n, k, alpha, A + bz * sA, lda, B + bz * sB, ldb, beta,
                                 C + bz * sC, ldc, tm, tn, ta, tb,
                                 STOP ? stop + (bz / per + 1) * per - 1 : nullptr);
}

// The two products of a left-looking Cholesky's block column k0 over matrices
// of different orders, matrix blockIdx.x, row tile blockIdx.y:
// UPD:  L[k0:, k0:k0+NB] -= L[k0:, 0:k0] L[k0:k0+NB, 0:k0]^T on and below the diagonal;
// else: L[k0+NB:, k0:k0+NB] <- itself times inv(L11)^T.
// Rows between the order and the leading dimension may be read (they reach
// only elements that are not stored).
template <typename T, bool UPD>
__global__ __launch_bounds__(NT, 2) void k_gemm_mols(int k0, const MolInfo *__restrict__ mols,
                                                     const MolMat *__restrict__ mats, T *L,
                                                     const T *inv) {
  const MolMat z = mol_mat(mats, blockIdx.x);
  const MolInfo mi = mols[z.mol];
  const int r0 = UPD ? k0 : k0 + kCholNB, m = mi.n - r0, tm = blockIdx.y;
  if (tm * BM >= m) return;
  T *M = L + mi.a + (long)z.slot * mi.n * mi.ld;
  if (UPD)
    gemm_tile<T, true, false>(m, min(m, kCholNB), mi.ld - r0, mi.ld - r0, k0, T(-1), M + r0, mi.ld,
                              M + r0, mi.ld, T(1), M + r0 + (long)k0 * mi.ld, mi.ld, tm, 0, 0, 0);
  else
    gemm_tile<T, false, false>(m, kCholNB, mi.ld - r0, kCholNB, kCholNB, T(1), M + r0 + (long)k0 * mi.ld,
                               mi.ld, inv + mi.inv + z.slot * mol_inv_size(mi.n) + (long)k0 * kCholNB,
                               kCholNB, T(0), M + r0 + (long)k0 * mi.ld, mi.ld, tm, 0, 0, 0);
}

// Tall-skinny FP64 update C = alpha (A1 B1^T + A2 B2^T) + beta C for at most
// TS_N columns and TS_K terms of each product (A2, B2 may be null).  A
// 128 x 128 tile would leave three quarters of its MFMA work on zero columns
// and give a tall matrix only m / 128 workgroups; here a workgroup owns 64
// rows of C, each wave 16 rows by the 32 columns as two 16 x 16 MFMA blocks,
// computed transposed (the B columns as the MFMA's first operand) so that the
// 16 lanes of a group hold 16 consecutive rows of one column of C.  K goes
// through LDS in chunks of TS_KC (25 KB of LDS, so that a workgroup fits on
// a CU beside two workgroups of the square-tile kernel running on another
// stream), the next chunk's loads issued before the current chunk's MFMAs.
constexpr int TS_M = 64, TS_N = 32, TS_K = 128, TS_KC = 32;

__global__ __launch_bounds__(256) void k_gemm_ts(int m, int n, int k, double alpha,
                                                 const double *__restrict__ A1,
                                                 const double *__restrict__ B1,
                                                 const double *__restrict__ A2,
                                                 const double *__restrict__ B2, int lda, int ldb,
                                                 double beta, double *__restrict__ C, int ldc) {
  __shared__ double As[TS_KC][TS_M + 1];  // As[kk][row]
  __shared__ double Bs[TS_KC][TS_N + 1];  // Bs[kk][col]
  const int t = threadIdx.x, lane = t & 63, w = t >> 6, lr = lane & 15, lk = lane >> 4;
  const int row0 = blockIdx.x * TS_M;
  const int r = lane, rr = min(row0 + r, m - 1);
  v4d acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
  const int nch = (k + TS_KC - 1) / TS_KC, nterm = A2 ? 2 : 1, nstep = nterm * nch;
  // A chunk: element e = t + 256 i is row e % 64, column w + 4 i; B chunk:
  // row e % 32, column e / 32; clamped addresses, zeros past m, n and k.
  // Up to TS_G chunks (every chunk of the panel updates, K <= 128) are loaded
  // at once, and C with them, so that one memory latency covers the kernel.
  constexpr int TS_G = 4;
  double ra[TS_G][TS_M * TS_KC / 256], rb[TS_G][TS_N * TS_KC / 256];
  auto gload = [&](int st, int j) {
    const int term = st / nch, k0 = (st % nch) * TS_KC;
    const double *A = term ? A2 : A1, *Bm = term ? B2 : B1;
#pragma unroll
    for (int i = 0; i < TS_M * TS_KC / 256; ++i) {
      const int kk = k0 + w + 4 * i;
      const double v = A[rr + (long)min(kk, k - 1) * lda];
      ra[j][i] = (kk < k && row0 + r < m) ? v : 0.0;
    }
#pragma unroll
    for (int i = 0; i < TS_N * TS_KC / 256; ++i) {
      const int e = t + 256 * i, c = e & (TS_N - 1), kk = k0 + (e >> 5);
      const double v = Bm[min(c, n - 1) + (long)min(kk, k - 1) * ldb];
      rb[j][i] = (c < n && kk < k) ? v : 0.0;
    }
  };
  // transposed blocks: lane (lk, lr) holds C[row 16 w + lr][col lk + 4 v] (+16)
  const int row = row0 + 16 * w + lr, crow = min(row, m - 1);
  double cv[8];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    cv[v] = beta != 0.0 ? C[crow + (long)min(lk + 4 * v, n - 1) * ldc] : 0.0;
    cv[4 + v] = beta != 0.0 ? C[crow + (long)min(16 + lk + 4 * v, n - 1) * ldc] : 0.0;
  }
  for (int g0 = 0; g0 < nstep; g0 += TS_G) {
#pragma unroll
    for (int j = 0; j < TS_G; ++j) gload(min(g0 + j, nstep - 1), j);
#pragma unroll
    for (int j = 0; j < TS_G; ++j) {
      if (g0 + j >= nstep) break;
      __syncthreads();  // the previous chunk's LDS reads are done
#pragma unroll
      for (int i = 0; i < TS_M * TS_KC / 256; ++i) As[w + 4 * i][r] = ra[j][i];
#pragma unroll
      for (int i = 0; i < TS_N * TS_KC / 256; ++i) {
        const int e = t + 256 * i;
        Bs[e >> 5][e & (TS_N - 1)] = rb[j][i];
      }
      __syncthreads();
#pragma unroll
      for (int q = 0; q < TS_KC / 4; ++q) {
        const double a = As[4 * q + lk][16 * w + lr];
        const double b0 = Bs[4 * q + lk][lr], b1 = Bs[4 * q + lk][16 + lr];
        acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(b0, a, acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(b1, a, acc1, 0, 0, 0);
      }
    }
  }
  if (row < m) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int c0 = lk + 4 * v, c1 = 16 + lk + 4 * v;
      if (c0 < n) C[row + (long)c0 * ldc] = alpha * acc0[v] + beta * cv[v];
      if (c1 < n) C[row + (long)c1 * ldc] = alpha * acc1[v] + beta * cv[4 + v];
    }
  }
}

template <typename T>
void launch(hipStream_t s, bool lower, int m, int n, int k, T alpha,
            const T *A, int lda, long sA, const T *B, int ldb, long sB,
            T beta, T *C, int ldc, long sC, int batch, int ta = 0, int tb = 0,
            const int *stop = nullptr, int per = 1) {
  if (m <= 0 || n <= 0 || batch <= 0) return;
  const int tmn = ceil_div(m, BM), tnn = ceil_div(n, BN);
  const bool gen = ta || tb || m < Vec16<T>::n || n < Vec16<T>::n;
  const dim3 grid(lower ? tnn * (tnn + 1) / 2 + (tmn - tnn) * tnn : tmn * tnn, 1, batch);
  auto *f = lower ? (gen ? k_gemm_nt<T, true, true, false> : k_gemm_nt<T, true, false, false>)
                  : (gen ? k_gemm_nt<T, false, true, false> : k_gemm_nt<T, false, false, false>);
  if (stop && lower && !gen) f = k_gemm_nt<T, true, false, true>;
  hipLaunchKernelGGL(f, grid, dim3(NT), 0, s, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C, ldc,
                     sC, tnn, ta, tb, stop, per);
  MBD_LAUNCH_CHECK();
}

}  // namespace

void gemm_f32(hipStream_t s, int ta, int tb, int m, int n, int k, float alpha, const float *A,
              int lda, const float *B, int ldb, float beta, float *C, int ldc) {
  launch<float>(s, false, m, n, k, alpha, A, lda, 0, B, ldb, 0, beta, C, ldc, 0, 1, ta, tb);
}

void gemm_ts2(hipStream_t s, int m, int n, int k, double alpha, const double *A1, const double *B1,
              const double *A2, const double *B2, int lda, int ldb, double beta, double *C, int ldc) {
  if (m <= 0 || n <= 0) return;
  hipLaunchKernelGGL(k_gemm_ts, dim3(ceil_div(m, TS_M)), dim3(256), 0, s, m, n, k, alpha, A1, B1, A2,
                     B2, lda, ldb, beta, C, ldc);
  MBD_LAUNCH_CHECK();
}

template <typename T>
void gemm_mols(hipStream_t s, bool upd, int k0, int nmax, int nmat, const MolInfo *mols,
               const MolMat *mats, T *L, const T *inv) {
  const int m = nmax - (upd ? k0 : k0 + kCholNB);
  if (m <= 0 || nmat <= 0) return;
  hipLaunchKernelGGL((upd ? k_gemm_mols<T, true> : k_gemm_mols<T, false>), dim3(nmat, ceil_div(m, BM)),
                     dim3(NT), 0, s, k0, mols, mats, L, inv);
  MBD_LAUNCH_CHECK();
}
template void gemm_mols<double>(hipStream_t, bool, int, int, int, const MolInfo *, const MolMat *,
                                double *, const double *);
template void gemm_mols<float>(hipStream_t, bool, int, int, int, const MolInfo *, const MolMat *, float *,
                               const float *);

void gemm_nt(hipStream_t s, bool lower, int m, int n, int k, double alpha,
             const double *A, int lda, long sA, const double *B, int ldb,
             long sB, double beta, double *C, int ldc, long sC, int batch, const int *stop, int per) {
  if (!lower && batch == 1 && n <= TS_N && k >= 1 && k <= TS_K) {
    gemm_ts2(s, m, n, k, alpha, A, B, nullptr, nullptr, lda, ldb, beta, C, ldc);
    return;
  }
  launch<double>(s, lower, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C,
                 ldc, sC, batch, 0, 0, stop, per);
}

void gemm_nt(hipStream_t s, bool lower, int m, int n, int k, float alpha,
             const float *A, int lda, long sA, const float *B, int ldb,
             long sB, float beta, float *C, int ldc, long sC, int batch, const int *stop, int per) {
  launch<float>(s, lower, m, n, k, alpha, A, lda, sA, B, ldb, sB, beta, C,
                ldc, sC, batch, 0, 0, stop, per);
}

}  // namespace mbd
