// C ABI of libmbd_hip.so: handle, system set-up, and the orchestration of
// the SCS / C6 / MBD stages on one HIP stream (see include/mbd_hip.h for the
// reference interface each entry point replaces).
//
// Device memory plan (3N = n, all column-major):
//   relay matrices     nf_batch x n x n   (FP64, or FP32 + FP32 factor copy)
//   inverted diagonal  nf_batch x ceil(n/NB) x NB x NB
//   solutions          21 x n x 3 (FP64)
//   C matrix           (n Ncell) x (n Ncell) FP64 + Householder workspace
// Up to all 21 frequencies are processed per batch, bounded by a memory
// budget (MBD_SCS_MEM_GB, default 64 GB) so one launch sequence factors every
// frequency at once.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <numeric>
#include <string>
#include <vector>

#include "../../include/mbd_hip.h"
#include "common.h"
#include "kernels.h"
#include "net.h"
#include "batch.h"
#include "logdet.h"
#include "mol.h"
#include "pcg.h"
#include "profile.h"
#include "refine.h"

using namespace mbd;

namespace {

template <typename T>
struct DevBuf {
  T *p = nullptr;
  size_t n = 0;
  void ensure(size_t count) {
    if (count <= n && p) return;
    if (p) MBD_HIP(hipFree(p));
    p = nullptr;
    n = 0;
    if (count == 0) return;
    MBD_HIP(hipMalloc(&p, count * sizeof(T)));
    n = count;
  }
  void release() {
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
  }
};

struct Elem {
  const char *sym;
  float alpha, c6, r0;
};

// Free-atom polarisability, C6 and vdW radius (UTILS.f90:1338-1691), kept as
// float literals because the reference assigns REAL(4) literals.
const Elem kElements[] = {
    {"H", 4.5f, 6.5f, 3.1f},          {"He", 1.38f, 1.46f, 2.65f},
    {"Li", 164.2f, 1387.0f, 4.16f},   {"Be", 38.0f, 214.0f, 4.17f},
    {"B", 21.0f, 99.5f, 3.89f},       {"C", 12.0f, 46.6f, 3.59f},
    {"N", 7.4f, 24.2f, 3.34f},        {"O", 5.4f, 15.6f, 3.19f},
    {"F", 3.8f, 9.52f, 3.04f},        {"Ne", 2.67f, 6.38f, 2.91f},
    {"Na", 162.7f, 1556.0f, 3.73f},   {"Mg", 71.0f, 627.0f, 4.27f},
    {"Al", 60.0f, 528.0f, 4.33f},     {"Si", 37.0f, 305.0f, 4.2f},
    {"P", 25.0f, 185.0f, 4.01f},      {"S", 19.6f, 134.0f, 3.86f},
    {"Cl", 15.0f, 94.6f, 3.71f},      {"Ar", 11.1f, 64.3f, 3.55f},
    {"K", 292.9f, 3897.0f, 3.71f},    {"Ca", 160.0f, 2221.0f, 4.65f},
    {"Sc", 120.0f, 1383.0f, 4.59f},   {"Ti", 98.0f, 1044.0f, 4.51f},
    {"V", 84.0f, 832.0f, 4.44f},      {"Cr", 78.0f, 602.0f, 3.99f},
    {"Mn", 63.0f, 552.0f, 3.97f},     {"Fe", 56.0f, 482.0f, 4.23f},
    {"Co", 50.0f, 408.0f, 4.18f},     {"Ni", 48.0f, 373.0f, 3.82f},
    {"Cu", 42.0f, 253.0f, 3.76f},     {"Zn", 40.0f, 284.0f, 4.02f},
    {"Ga", 60.0f, 498.0f, 4.19f},     {"Ge", 41.0f, 354.0f, 4.2f},
    {"As", 29.0f, 246.0f, 4.11f},     {"Se", 25.0f, 210.0f, 4.04f},
    {"Br", 20.0f, 162.0f, 3.93f},     {"Kr", 16.8f, 129.6f, 3.82f},
    {"Rb", 319.2f, 4691.0f, 3.72f},   {"Sr", 199.0f, 3170.0f, 4.54f},
    {"Y", 126.737f, 1968.58f, 4.8151f}, {"Zr", 119.97f, 1677.91f, 4.53f},
    {"Nb", 101.603f, 1263.61f, 4.2365f}, {"Mo", 88.4225785f, 1028.73f, 4.099f},
    {"Tc", 80.083f, 1390.87f, 4.076f}, {"Ru", 65.895f, 609.754f, 3.9953f},
    {"Rh", 56.1f, 469.0f, 3.95f},     {"Pd", 23.68f, 157.5f, 3.66f},
    {"Ag", 50.6f, 339.0f, 3.82f},     {"Cd", 39.7f, 452.0f, 3.99f},
    {"In", 70.22f, 707.046f, 4.23198f}, {"Sn", 55.95f, 587.417f, 4.303f},
    {"Sb", 43.67197f, 459.322f, 4.276f}, {"Te", 37.65f, 396.0f, 4.22f},
    {"I", 35.0f, 385.0f, 4.17f},      {"Xe", 27.3f, 285.9f, 4.08f},
    {"Cs", 427.12f, 6582.08f, 3.78f}, {"Ba", 275.0f, 5727.0f, 4.77f},
    {"Hf", 99.52f, 1274.8f, 4.21f},   {"Ta", 82.53f, 1019.92f, 4.15f},
    {"W", 71.041f, 847.93f, 4.08f},   {"Re", 63.04f, 710.2f, 4.02f},
    {"Os", 55.055f, 596.67f, 3.84f},  {"Ir", 42.51f, 359.1f, 4.0f},
    {"Pt", 39.68f, 347.1f, 3.92f},    {"Au", 36.5f, 298.0f, 3.86f},
    {"Hg", 33.9f, 392.0f, 3.98f},     {"Tl", 69.92f, 717.44f, 3.91f},
    {"Pb", 61.8f, 697.0f, 4.31f},     {"Bi", 49.02f, 571.0f, 4.32f},
    {"Po", 45.013f, 530.92f, 4.097f}, {"At", 38.93f, 457.53f, 4.07f},
    {"Rn", 33.54f, 390.63f, 4.23f},
};

// Casimir-Polder grid (UTILS.f90:1188-1211), REAL(4) literals.
const float kOmega[21] = {0.0f,      0.0392901f, 0.118358f, 0.198912f, 0.282029f,
                          0.368919f, 0.461006f,  0.560027f, 0.668179f, 0.788336f,
                          0.92439f,  1.08179f,   1.26849f,  1.49661f,  1.78563f,
                          2.16917f,  2.71062f,   3.54573f,  5.02734f,  8.44896f,
                          25.4517f};
const float kWeight[21] = {0.0f,      0.0786611f, 0.07964f,  0.0816475f, 0.0847872f,
                           0.0892294f, 0.0952317f, 0.103172f, 0.113605f,  0.12735f,
                           0.145652f, 0.170453f,  0.204917f, 0.254456f,  0.328962f,
                           0.448092f, 0.655606f,  1.06596f,  2.06357f,   5.6851f,
                           50.9558f};

struct Timer {
  hipEvent_t a, b;
  Timer() {
    MBD_HIP(hipEventCreate(&a));
    MBD_HIP(hipEventCreate(&b));
  }
  ~Timer() {
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
  }
  void start(hipStream_t s) { MBD_HIP(hipEventRecord(a, s)); }
  void stop(hipStream_t s) { MBD_HIP(hipEventRecord(b, s)); }
  double ms() {
    MBD_HIP(hipEventSynchronize(b));
    float v = 0.f;
    MBD_HIP(hipEventElapsedTime(&v, a, b));
    return v;
  }
};

// Lattice translations ((0-i) a1 + (0-j) a2) + (0-k) a3 over the box, i
// outermost, in the reference's loop order (UTILS.f90:561-568).
std::vector<double> image_box(const double *lat, const int *half) {
  std::vector<double> t;
  for (int i = -half[0]; i <= half[0]; ++i)
    for (int j = -half[1]; j <= half[1]; ++j)
      for (int k = -half[2]; k <= half[2]; ++k)
        for (int c = 0; c < 3; ++c)
          t.push_back(((double)(0 - i) * lat[c] + (double)(0 - j) * lat[3 + c]) +
                      (double)(0 - k) * lat[6 + c]);
  return t;
}

double norm3(const double *v) { return std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]); }

// Whether the image box of the coupled matrix (half images to either side of
// each supercell vector) holds every image inside the cutoff sphere for every
// pair of atoms and cells.  A displacement at f (in supercell vectors) plus
// image L has |f_k + L_k| h_k <= r with h_k the distance between the lattice
// planes, so along k only images |L_k| <= rc / h_k + max |f_k| can reach.  An
// axis without images (vacuum) has one cell and nothing to cover.
bool images_cover(int n_atoms, const double *xyz, const double *lat, const int *S, const int *half,
                  const int *vac, double rc) {
  double cr[3][3], vol = 0.0;  // cr[k] = a_i x a_j: the planes' normals
  for (int k = 0; k < 3; ++k) {
    const double *a = lat + 3 * ((k + 1) % 3), *b = lat + 3 * ((k + 2) % 3);
    for (int c = 0; c < 3; ++c)
      cr[k][c] = a[(c + 1) % 3] * b[(c + 2) % 3] - a[(c + 2) % 3] * b[(c + 1) % 3];
  }
  for (int c = 0; c < 3; ++c) vol += lat[c] * cr[0][c];
  for (int k = 0; k < 3; ++k) {
    if (vac[k]) continue;
    double lo = 1e300, hi = -1e300;
    for (int i = 0; i < n_atoms; ++i) {
      double f = 0.0;
      for (int c = 0; c < 3; ++c) f += xyz[3 * i + c] * cr[k][c];
      lo = std::min(lo, f / vol);
      hi = std::max(hi, f / vol);
    }
    const double plane = S[k] * std::fabs(vol) / norm3(cr[k]);
    const double reach = rc / plane + (hi - lo + (S[k] - 1)) / S[k];
    if (!(reach < half[k] + 1 - 1e-9)) return false;
  }
  return true;
}

}  // namespace

// Scratch of mbd_batch_run_noalloc: the persistent kernel's per-workgroup
// matrix slots, the task and per-molecule counters, the residual maxima and
// the phase timers, in one fixed device array (each GPU the library runs on
// holds its own copy until the process ends).  Host code uses only the
// device address that hipGetSymbolAddress returns for the current device.
namespace {
constexpr int kNaMaxAtoms = 32;     // atoms per molecule
constexpr int kNaMaxMol = 16384;    // molecules per call
constexpr int kNaSlots = 256;       // workgroups (one matrix slot each)
constexpr size_t kNaSlotBytes = 180224;  // batch_slot_bytes(3 * kNaMaxAtoms)
constexpr size_t kNaCountOff = (size_t)kNaSlots * kNaSlotBytes;
constexpr size_t kNaResidOff = kNaCountOff + 4 * (size_t)(kNaMaxMol + 64);
constexpr size_t kNaPhaseOff = kNaResidOff + 8 * (size_t)kNaMaxMol;
constexpr size_t kNaBytes = kNaPhaseOff + 8 * 16;
constexpr int kNaMaxDevices = 64;
void *na_ptr[kNaMaxDevices] = {nullptr};
}  // namespace
static __device__ __align__(256) char scratch[kNaBytes];

struct mbd_handle {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  bool has_sys = false;
  // system
  int N = 0;
  int periodic = 0;
  double lat[9] = {0};
  double latSL[9] = {0};
  double beta = 1.0, rc_scs = 120.0, rc_cfdm = 100.0, rc_sc = 25.0;
  int scs_img[3] = {0, 0, 0}, supercell[3] = {1, 1, 1}, cfdm_img[3] = {0, 0, 0};
  int nimg_scs = 1, nimg_cfdm = 1, ncell = 1;
  std::vector<double> a0_h, r0_h;
  // device: system
  DevBuf<double> xyz, hirsh, a0, c60, r0, omega, weight, img_scs, img_cfdm, lat_d;
  DevBuf<int> cell;
  // device: SCS
  DevBuf<double> alpha_w, sgm, rvdw;
  DevBuf<double> A64, inv64, X, alpha, P, eig3, c6mol, c6, R, D;
  DevBuf<float> A32, L32, inv32;
  DevBuf<int> info;
  DevBuf<double> rnorm;
  // FP64 re-solve of single grid points (fallback of the FP32 / iterative
  // forms) and the LU fallback of a failed FP64 Cholesky
  DevBuf<double> A1, inv1, luUt;
  DevBuf<int> info1, luPiv;
  // device: iterative (learned) form; preconditioner clusters of the system
  DevBuf<double> pMinv, pR, pZ, pP, pQ, pscal, ppart, alpha_pred;
  Clusters cl;  // formed by the system's first iterative solve
  bool cl_ready = false;
  std::vector<double> xyz_h, hirsh_h;
  DevBuf<int> clOff, clAtoms;
  DevBuf<long> clMoff;
  // partials of the lower-triangle products (refinement residuals, block-PCG)
  DevBuf<double> svU, svV;
  bool have_net = false;
  DevBuf<float> net_blob, net_X, net_Xn, net_act;
  DevBuf<float4> net_nbl;
  DevBuf<int> net_cnt;
  DevBuf<double> img_net;  // SCS images that can reach within the descriptor cutoff
  int nimg_net = 1, center_net = 0;
  // device: MBD
  DevBuf<double> C, om_at, reff, lam, e2, bounds, E, VW, tau, dd, ee, alph, pa, pb, py, qred, ps;
  DevBuf<double> ext_alpha, ext_c6;
  DevBuf<int> nneg;
  // batched molecules (small ones: one persistent launch, replayed from a hipGraph)
  struct Batch {
    int nmol = 0, natoms = 0, nmax = 0, ncu = 0;
    double beta = 1.0, rc_scs = 0.0, rc_cfdm = 0.0;  // bohr
    DevBuf<int> off, order, counter, stat, phase;
    DevBuf<double> xyz, hirsh, a0, c60, r0, alpha, c6, energy, c6_mol, resid;
    DevBuf<char> work;
    int cfg = -1;  // tuned candidate, -1 = default
    hipGraphExec_t exec[2] = {nullptr, nullptr};
    int exec_cfg[2] = {-1, -1};
    // molecules above kMolMinOrder, the first `nlarge` of the order: solved by
    // launches over all of them (mol.h)
    int nlarge = 0, exec_first[2] = {0, 0};
    hipStream_t side = nullptr;  // the persistent kernel beside them
    hipEvent_t fork = nullptr, join = nullptr;
    std::vector<int> ord, size;  // order; matrix order of each molecule in it
    std::vector<int> first;      // first atom of each molecule
    DevBuf<double> par, wA, wC, wHi, wG, wShift, wInv;
    DevBuf<char> wL, wInfo, wMat, again;
    DevBuf<int> wFac, wRedo, wList;
  } bt;
  // tridiagonalisation replayed from a captured graph (36k small launches at
  // n = 12288); rebuilt when the size or any buffer address changes
  hipGraphExec_t trd_exec = nullptr;
  std::vector<const void *> trd_key;
  // two-stage eigen reduction work space; eig_flag is the bulge-chasing abort
  // flag of the last run_energy, read back with the energy
  DevBuf<double> sbrV, sbrT, sbrR, sbrX, sbrY, sbrMp, sbrM, sbrAB;
  DevBuf<int> sbrCnt, sbrMcnt, sbrProg, sbrFlag;
  DevBuf<unsigned long long> sbrMail;
  DevBuf<int> sbrCq;
  DevBuf<double> sbrCqR;
  // look-ahead: second factor buffer, the stream the pair updates run on, and
  // the events that fork to it and join from it
  DevBuf<double> sbrVW2;
  hipStream_t stream2 = nullptr;
  hipEvent_t sbr_fork = nullptr, sbr_join = nullptr;
  int eig_used = 1;
  int eig_flag = 0;
  // log-determinant energy: shifted matrices and their inverted diagonal
  // blocks share A64 / inv64; bounds and sums on the device and the host
  DevBuf<double> ldHi, ldG, lzV, lzPart;
  DevBuf<int> ldInfo;
  // supercells by cell differences: blocks, their Fourier transform, phases
  DevBuf<double> cellB, cellH, cellPh;
  DevBuf<int> cellNear;
  bool cells_cover = false;  // the image box covers the cutoff sphere for every pair
  // result of the last run_energy
  double e_val = 0.0;
  int n_neg = 0;
  // instrumentation
  bool prof_on = false;
  Profiler prof;

  int n() const { return 3 * N; }
};

namespace {
// Makes the handle's profiler the active one for the duration of a call.
struct ProfGuard {
  explicit ProfGuard(mbd_handle *h) { active_profiler() = h->prof_on ? &h->prof : nullptr; }
  ~ProfGuard() { active_profiler() = nullptr; }
};
}  // namespace

namespace {

void batch_drop_graphs(mbd_handle *h) {
  for (int m = 0; m < 2; ++m) {
    if (h->bt.exec[m]) (void)hipGraphExecDestroy(h->bt.exec[m]);
    h->bt.exec[m] = nullptr;
    h->bt.exec_cfg[m] = -1;
  }
}

void batch_release(mbd_handle *h) {
  batch_drop_graphs(h);
  auto &b = h->bt;
  DevBuf<double> *d[] = {&b.xyz, &b.hirsh, &b.a0, &b.c60, &b.r0, &b.alpha,
                         &b.c6, &b.energy, &b.c6_mol, &b.resid};
  for (auto *x : d) x->release();
  b.off.release();
  b.order.release();
  b.counter.release();
  b.stat.release();
  b.phase.release();
  b.work.release();
  DevBuf<double> *w[] = {&b.par, &b.wA, &b.wC, &b.wHi, &b.wG, &b.wShift, &b.wInv};
  for (auto *x : w) x->release();
  DevBuf<char> *wc[] = {&b.wL, &b.wInfo, &b.wMat, &b.again};
  for (auto *x : wc) x->release();
  if (b.side) {
    (void)hipStreamSynchronize(b.side);
    (void)hipEventDestroy(b.fork);
    (void)hipEventDestroy(b.join);
    (void)hipStreamDestroy(b.side);
    b.side = nullptr;
  }
  b.wFac.release();
  b.wRedo.release();
  b.wList.release();
  b.nmol = 0;
}

int fail(mbd_handle *h, const HipError &e) {
  char buf[256];
  snprintf(buf, sizeof buf, "HIP error %d (%s) at capi.hip:%d in %s", (int)e.err,
           hipGetErrorString(e.err), e.line, e.what);
  if (h) h->err = buf;
  fprintf(stderr, "libmbd_hip: %s\n", buf);
  return MBD_ERR_HIP;
}

size_t mem_budget() {
  const char *s = getenv("MBD_SCS_MEM_GB");
  double gb = s ? atof(s) : 64.0;
  if (gb <= 0) gb = 64.0;
  return (size_t)(gb * 1e9);
}

// Iteration cap of the block-PCG (MBD_PCG_MAXITER overrides; a tiny cap
// forces the residual gate to fail, which exercises the Cholesky fallback).
int pcg_maxit() {
  const char *s = getenv("MBD_PCG_MAXITER");
  const int v = s ? atoi(s) : 0;
  return v > 0 ? v : kPcgMaxIter;
}

// Leading dimension of the matrices that are factored: columns start on cache
// lines, and not a multiple of 2 KB apart (every column in the same memory
// channels).  Cells of 1331 and 2903 atoms (odd orders) 18.8 -> 18.2 and
// 176.5 -> 171.4 ms, of 4096 atoms (order 12288, mixed) 307.4 -> 305.0 ms;
// 16 more rows at every multiple of 32 or 64 measured 306.1 and 306.6.
int lead_dim(int n) {
  const int l = (n + 15) / 16 * 16;
  return l % 256 ? l : l + 32;
}

int freq_batch(const mbd_handle *h, size_t bytes_per_matrix) {
  size_t b = mem_budget() / std::max<size_t>(bytes_per_matrix, 1);
  return (int)std::max<size_t>(1, std::min<size_t>(kNumFreq, b));
}

struct DirectStats {
  int iters = 0;
  std::vector<double> res;  // final max |B - A X| per matrix
  std::vector<int> info;    // FP32 Cholesky info per matrix
};

// FP32 Cholesky of matrices [b0, b0 + bs) of h->A32 (copied to h->L32) and
// the solve with FP64 iterative refinement against the FP32 tensor; X holds
// those matrices' solutions (stride sX).  Refinement stops once every matrix
// meets kRefineTol or after kRefineMaxIter sweeps; the caller re-solves the
// matrices that failed (a non-positive FP32 pivot or a residual above the
// tolerance) in FP64.
DirectStats solve_mixed_direct(mbd_handle *h, int n, int lda, long sA, long sinv, long sX,
                               int b0, int bs, double *X, int *info) {
  hipStream_t s = h->stream;
  const float *A = h->A32.p + (long)b0 * sA;
  float *L = h->L32.p + (long)b0 * sA;
  float *inv = h->inv32.p + (long)b0 * sinv;
  double *R = h->R.p + (long)b0 * sX;
  MBD_HIP(hipMemcpyAsync(L, A, sizeof(float) * (size_t)bs * sA, hipMemcpyDeviceToDevice, s));
  potrf_batched<float>(s, n, L, lda, sA, bs, inv, sinv, info);
  set_rhs(s, n, X, n, sX, bs);
  potrs3_batched<float>(s, n, L, lda, sA, bs, inv, sinv, X, n, sX);
  DirectStats st;
  st.res.assign(bs, 0.0);
  st.info.assign(bs, 0);
  MBD_HIP(hipMemcpyAsync(st.info.data(), info, sizeof(int) * bs, hipMemcpyDeviceToHost, s));
  std::vector<double> rn(2 * bs);
  for (st.iters = 0; st.iters < kRefineMaxIter; ++st.iters) {
    residual3<float>(s, n, A, lda, sA, bs, X, n, sX, R, n, sX, h->rnorm.p,
                     Symv3Work{h->svU.p, h->svV.p});
    MBD_HIP(hipMemcpyAsync(rn.data(), h->rnorm.p, sizeof(double) * 2 * bs,
                           hipMemcpyDeviceToHost, s));
    MBD_HIP(hipStreamSynchronize(s));
    // ||b||_inf = 1 for the stacked identity, so max |r| is relative; a NaN
    // residual (broken factor) fails the test below
    bool done = true;
    for (int b = 0; b < bs; ++b) {
      st.res[b] = rn[2 * b];
      if (!(rn[2 * b] <= kRefineTol) && st.info[b] == 0) done = false;
    }
    if (done) break;
    potrs3_batched<float>(s, n, L, lda, sA, bs, inv, sinv, R, n, sX);
    axpy3(s, n, bs, R, n, sX, X, n, sX);
  }
  return st;
}

// Grid point k solved by LU with partial pivoting on its FP64 relay matrix
// (rebuilt into the single-matrix buffer A1): the fallback when the FP64
// Cholesky meets a non-positive pivot.  Xk receives A^-1 B.
void solve_point_lu(mbd_handle *h, int k, double *Xk) {
  const int N = h->N, n = h->n();
  hipStream_t s = h->stream;
  const long sA = (long)n * n;
  h->A1.ensure((size_t)sA);
  h->luPiv.ensure((size_t)n);
  h->luUt.ensure((size_t)std::max(1, n - kLuNB) * kLuNB);
  h->info1.ensure(1);
  MBD_HIP(hipMemsetAsync(h->info1.p, 0, sizeof(int), s));
  scs_build<double>(s, N, h->xyz.p, h->nimg_scs, h->nimg_scs / 2, h->img_scs.p, h->rc_scs / kBohr,
                    h->beta, h->alpha_w.p + (long)k * N, h->sgm.p + (long)k * N, h->rvdw.p,
                    h->A1.p, n, sA, 1, true);
  getrf_batched(s, n, h->A1.p, n, sA, 1, h->luPiv.p, h->luUt.p, 0, h->info1.p);
  set_rhs(s, n, Xk, n, 3L * n, 1);
  getrs3_batched(s, n, h->A1.p, n, sA, 1, h->luPiv.p, Xk, n, 3L * n);
}

// Grid point k solved in FP64 (relay matrix, Cholesky, and LU when the
// Cholesky fails): the fallback of the FP32 and iterative forms.  Returns the
// FP64 Cholesky info (0 when it succeeded).
int solve_point_fp64(mbd_handle *h, int k, double *Xk) {
  const int N = h->N, n = h->n();
  hipStream_t s = h->stream;
  const long sA = (long)n * n;
  const long sinv = (long)ceil_div(n, kCholNB) * kCholNB * kCholNB;
  h->A1.ensure((size_t)sA);
  h->inv1.ensure((size_t)sinv);
  h->info1.ensure(1);
  MBD_HIP(hipMemsetAsync(h->info1.p, 0, sizeof(int), s));
  scs_build<double>(s, N, h->xyz.p, h->nimg_scs, h->nimg_scs / 2, h->img_scs.p, h->rc_scs / kBohr,
                    h->beta, h->alpha_w.p + (long)k * N, h->sgm.p + (long)k * N, h->rvdw.p,
                    h->A1.p, n, sA, 1, false);
  potrf_batched<double>(s, n, h->A1.p, n, sA, 1, h->inv1.p, sinv, h->info1.p);
  int info = 0;
  MBD_HIP(hipMemcpyAsync(&info, h->info1.p, sizeof(int), hipMemcpyDeviceToHost, s));
  MBD_HIP(hipStreamSynchronize(s));
  if (info == 0) {
    set_rhs(s, n, Xk, n, 3L * n, 1);
    potrs3_batched<double>(s, n, h->A1.p, n, sA, 1, h->inv1.p, sinv, Xk, n, 3L * n);
  } else {
    solve_point_lu(h, k, Xk);
  }
  return info;
}

// Atom clusters of the iterative solve's block preconditioner, formed on the
// host while the device builds the relay matrices (formed with the system they
// cost a 4096-atom learned solve 8 of 184 ms before its first launch, and the
// other forms, which do not use them, as much).
void system_clusters(mbd_handle *h) {
  if (h->cl_ready) return;
  h->cl = build_clusters(h->N, h->xyz_h.data(), h->lat, h->periodic != 0, h->hirsh_h.data(),
                         h->a0_h.data(), h->r0_h.data(), h->beta);
  h->clOff.ensure(h->cl.off.size());
  h->clAtoms.ensure(h->cl.atoms.size());
  h->clMoff.ensure(h->cl.moff.size());
  MBD_HIP(hipMemcpyAsync(h->clOff.p, h->cl.off.data(), sizeof(int) * h->cl.off.size(),
                         hipMemcpyHostToDevice, h->stream));
  MBD_HIP(hipMemcpyAsync(h->clAtoms.p, h->cl.atoms.data(), sizeof(int) * h->cl.atoms.size(),
                         hipMemcpyHostToDevice, h->stream));
  MBD_HIP(hipMemcpyAsync(h->clMoff.p, h->cl.moff.data(), sizeof(long) * h->cl.moff.size(),
                         hipMemcpyHostToDevice, h->stream));
  h->cl_ready = true;
}

// SCS at all 21 points into h->alpha (21 x N), h->P (21 x 9), then C6.
void run_scs(mbd_handle *h, int mode, mbd_diag *d) {
  const int N = h->N, n = h->n();
  hipStream_t s = h->stream;
  h->alpha_w.ensure((size_t)kNumFreq * N);
  h->sgm.ensure((size_t)kNumFreq * N);
  h->rvdw.ensure(N);
  atom_params(s, N, kNumFreq, h->omega.p, h->hirsh.p, h->a0.p, h->c60.p, h->r0.p,
              h->alpha_w.p, h->sgm.p, h->rvdw.p);
  const int lda = lead_dim(n);
  const long sA = (long)n * lda;
  const int nblk = ceil_div(n, kCholNB);
  const long sinv = (long)nblk * kCholNB * kCholNB;
  const long sX = 3L * n;
  h->X.ensure((size_t)kNumFreq * sX);
  h->alpha.ensure((size_t)kNumFreq * N);
  h->P.ensure(9 * kNumFreq);
  h->info.ensure(kNumFreq);
  MBD_HIP(hipMemsetAsync(h->info.p, 0, sizeof(int) * kNumFreq, s));
  const double rc = h->rc_scs / kBohr;
  const int center = h->nimg_scs / 2;
  int max_it = 0;
  double max_res = 0.0;
  // per grid point: FP64 Cholesky info where an FP64 factorisation ran (all
  // points in the FP64 form, the fallback points otherwise)
  std::vector<int> info64(kNumFreq, 0);
  std::vector<char> fell(kNumFreq, 0);  // points re-solved by a fallback
  if (mode == MBD_MODE_FP64) {
    const int nb = freq_batch(h, (size_t)sA * 8 + (size_t)sinv * 8);
    h->A64.ensure((size_t)nb * sA);
    h->inv64.ensure((size_t)nb * sinv);
    for (int f0 = 0; f0 < kNumFreq; f0 += nb) {
      const int bs = std::min(nb, kNumFreq - f0);
      scs_build<double>(s, N, h->xyz.p, h->nimg_scs, center, h->img_scs.p, rc, h->beta,
                        h->alpha_w.p + (long)f0 * N, h->sgm.p + (long)f0 * N, h->rvdw.p,
                        h->A64.p, lda, sA, bs, false);
      potrf_batched<double>(s, n, h->A64.p, lda, sA, bs, h->inv64.p, sinv, h->info.p + f0);
      set_rhs(s, n, h->X.p + f0 * sX, n, sX, bs);
      potrs3_batched<double>(s, n, h->A64.p, lda, sA, bs, h->inv64.p, sinv,
                             h->X.p + f0 * sX, n, sX);
      MBD_HIP(hipMemcpyAsync(info64.data() + f0, h->info.p + f0, sizeof(int) * bs,
                             hipMemcpyDeviceToHost, s));
      MBD_HIP(hipStreamSynchronize(s));
      // a non-positive pivot: that point's system is solved by LU instead
      for (int b = 0; b < bs; ++b)
        if (info64[f0 + b] != 0) {
          fell[f0 + b] = 1;
          solve_point_lu(h, f0 + b, h->X.p + (f0 + b) * sX);
        }
      contract(s, N, h->X.p + f0 * sX, n, sX, bs, h->alpha.p + (long)f0 * N, h->P.p + 9 * f0);
    }
  } else {
    const int nb = freq_batch(h, (size_t)sA * 8 + (size_t)sinv * 4);
    h->A32.ensure((size_t)nb * sA);
    h->L32.ensure((size_t)nb * sA);
    h->inv32.ensure((size_t)nb * sinv);
    h->R.ensure((size_t)nb * sX);
    h->rnorm.ensure((size_t)2 * kNumFreq);
    const Symv3Sizes svz = symv3_sizes(n);
    h->svU.ensure((size_t)nb * svz.upart);
    h->svV.ensure((size_t)nb * svz.vpart);
    if (mode == MBD_MODE_LEARNED) {
      h->pR.ensure((size_t)nb * sX);
      h->pZ.ensure((size_t)nb * sX);
      h->pP.ensure((size_t)nb * sX);
      h->pQ.ensure((size_t)nb * sX);
      h->pscal.ensure((size_t)nb * kPcgScal);
    }
    if (mode == MBD_MODE_LEARNED && h->have_net) {
      // network warm start: descriptors and forward pass for every atom and
      // grid point, alpha_pred = alpha(i w) exp(y)
      const long S = (long)kNumFreq * N;
      ProfScope ps(K_NET, s, 0.0, 2.0 * S * (double)net_param_count());
      h->net_X.ensure((size_t)kNetIn * S);
      h->net_Xn.ensure((size_t)kNetIn * S);
      h->net_act.ensure((size_t)S * (3 * kNetHidden + 1));
      h->alpha_pred.ensure((size_t)S);
      h->net_nbl.ensure((size_t)N * kNetCap);
      h->net_cnt.ensure((size_t)N);
      net_descriptors(s, N, kNumFreq, h->xyz.p, h->nimg_net, h->center_net, h->img_net.p,
                      h->beta, h->alpha_w.p, h->hirsh.p, h->rvdw.p, h->omega.p, h->net_nbl.p,
                      h->net_cnt.p, h->net_X.p);
      mlp_gather(s, (int)S, nullptr, h->net_X.p, S, h->net_blob.p, h->net_Xn.p);
      float *act[4] = {h->net_act.p, h->net_act.p + S * kNetHidden,
                       h->net_act.p + 2 * S * kNetHidden, h->net_act.p + 3 * S * kNetHidden};
      mlp_forward(s, (int)S, h->net_blob.p + 2 * kNetIn, h->net_Xn.p, act);
      net_alpha(s, (int)S, act[3], h->alpha_w.p, h->alpha_pred.p);
    }
    for (int f0 = 0; f0 < kNumFreq; f0 += nb) {
      const int bs = std::min(nb, kNumFreq - f0);
      scs_build<float>(s, N, h->xyz.p, h->nimg_scs, center, h->img_scs.p, rc, h->beta,
                       h->alpha_w.p + (long)f0 * N, h->sgm.p + (long)f0 * N, h->rvdw.p,
                       h->A32.p, lda, sA, bs, false);
      double *Xb = h->X.p + f0 * sX;
      // matrices of this batch whose FP32 / iterative solve failed
      std::vector<int> redo;
      if (mode == MBD_MODE_MIXED) {
        DirectStats st = solve_mixed_direct(h, n, lda, sA, sinv, sX, 0, bs, Xb, h->info.p + f0);
        max_it = std::max(max_it, st.iters);
        for (int b = 0; b < bs; ++b) {
          if (st.info[b] == 0 && st.res[b] <= kRefineTol)
            max_res = std::max(max_res, st.res[b]);
          else
            redo.push_back(b);
        }
      } else {
        system_clusters(h);
        const int npart = std::max(h->cl.n, ceil_div(n, 256));
        h->pMinv.ensure((size_t)nb * h->cl.mtot);
        h->ppart.ensure((size_t)nb * npart * 4);
        PcgWork wk;
        wk.cl_off = h->clOff.p;
        wk.cl_atoms = h->clAtoms.p;
        wk.cl_moff = h->clMoff.p;
        wk.ncl = h->cl.n;
        wk.cl_mtot = h->cl.mtot;
        wk.Minv = h->pMinv.p;
        wk.R = h->pR.p;
        wk.Z = h->pZ.p;
        wk.P = h->pP.p;
        wk.Q = h->pQ.p;
        wk.scal = h->pscal.p;
        wk.part = h->ppart.p;
        wk.npart = npart;
        wk.rnorm = h->rnorm.p;
        wk.sv = Symv3Work{h->svU.p, h->svV.p};
        const double *a0 = h->have_net ? h->alpha_pred.p + (long)f0 * N : nullptr;
        PcgResult pr = pcg_solve<float>(s, N, h->A32.p, lda, sA, bs, a0, Xb, wk, kPcgTol,
                                        pcg_maxit());
        for (int b = 0; b < bs; ++b) {
          max_it = std::max(max_it, pr.iters[b]);
          if (pr.residual[b] <= kPcgGate) {
            max_res = std::max(max_res, pr.residual[b]);
            continue;
          }
          // the iterative residual failed: direct FP32 Cholesky + FP64 refinement
          fell[f0 + b] = 1;
          DirectStats st =
              solve_mixed_direct(h, n, lda, sA, sinv, sX, b, 1, Xb + b * sX, h->info.p + f0 + b);
          if (st.info[0] == 0 && st.res[0] <= kRefineTol)
            max_res = std::max(max_res, st.res[0]);
          else
            redo.push_back(b);
        }
      }
      // FP32 factor not positive definite or refinement not converged: the
      // point is solved in FP64 (Cholesky, LU if that fails too)
      for (int b : redo) {
        fell[f0 + b] = 1;
        info64[f0 + b] = solve_point_fp64(h, f0 + b, Xb + b * sX);
      }
      contract(s, N, Xb, n, sX, bs, h->alpha.p + (long)f0 * N, h->P.p + 9 * f0);
    }
  }
  if (d) d->fallback_used = (int)std::count(fell.begin(), fell.end(), 1);
  h->eig3.ensure(3 * kNumFreq);
  h->c6mol.ensure(1);
  h->c6.ensure(N);
  c6_sums(s, N, h->alpha.p, h->P.p, h->weight.p, h->eig3.p, h->c6mol.p, h->c6.p);
  MBD_HIP(hipStreamSynchronize(s));
  if (d) {
    d->info_scs = 0;
    for (int k = 0; k < kNumFreq; ++k)
      if (info64[k] != 0) {
        d->info_scs = info64[k];
        break;
      }
    d->refine_iters = max_it;
    d->residual = max_res;
  }
}

// The energy by log-determinants rather than eigenvalues: unless
// MBD_EIG_METHOD asks for one of the eigenvalue methods.
bool use_logdet() { return !getenv("MBD_EIG_METHOD"); }

constexpr int kLzMinOrder = 7000;
// From this n^3 (summed over the matrices) on, a guess of the lower end after
// one that failed is proved before its nodes are factored (the matrix most
// likely has an eigenvalue that is not positive), and, without Ritz values, a
// set's updates end once its proof has failed (the look costs the updates of a
// positive definite matrix 0.2 %).  Energies of matrices with negative eigenvalues (a
// factorisation of order 3000 fails at row 231), without either / proof first /
// both / by eigenvalues alone: order 2100 31.3 / 30.3 / 28.5 / 25.1 ms, 3000
// 47.8 / 44.5 / 41.3 / 36.3, 6000 130 / 107 / 88 / 77, 6900 168 / 134 / 104 /
// 92.  Below, one matrix takes about as long as a set (order 900: 31.5 / 31.3 /
// 30.7 / 29.2).
constexpr double kLdProofWork = 2048.0 * 2048.0 * 2048.0;
void fetch(mbd_handle *h, double *dst, const double *src, size_t count);

// `batch` symmetric matrices of order n (lower triangles, leading dimension
// n, back to back) whose eigenvalues together are the coupled matrix's.
struct LdGroup {
  int n, batch;
  const double *H;
};

// Extreme Ritz values over the matrices of `groups`, from kLzMinOrder on: a
// node of the quadrature costs n^3 / 3 operations, a Lanczos step one pass
// over n^2 / 2 elements and three launches.  Energy stage without and with
// them: order 3993 12.2 / 12.8 ms (12 -> 10 nodes), 6144 22.7 / 22.9, 8709
// 72.2 / 66.0, 12288 162.9 / 146.5 (13 -> 11).
bool ritz_values(mbd_handle *h, const std::vector<LdGroup> &groups, double &lo, double &hi) {
  hipStream_t s = h->stream;
  size_t nv = 0, nu = 0, nw = 0, np = 0, nab = 0;
  for (const LdGroup &g : groups) {
    if (g.n < kLzMinOrder) return false;
    const Symv3Sizes z = symv3_sizes(g.n);
    nv = std::max(nv, 9 * (size_t)g.n * g.batch);
    nu = std::max(nu, z.upart * g.batch);
    nw = std::max(nw, z.vpart * g.batch);
    np = std::max(np, 4 * (size_t)ceil_div(g.n, 256) * g.batch);
    nab += 6 * (size_t)kLzSteps * g.batch;
  }
  h->lzV.ensure(nv);
  h->svU.ensure(nu);
  h->svV.ensure(nw);
  h->lzPart.ensure(np + nab);
  double *ab = h->lzPart.p + np;
  for (const LdGroup &g : groups) {
    const size_t m = 3 * (size_t)g.n * g.batch;
    ld_lanczos(s, g.n, g.H, g.n, (long)g.n * g.n, g.batch, h->lzV.p, h->lzV.p + m, h->lzV.p + 2 * m,
               Symv3Work{h->svU.p, h->svV.p}, h->lzPart.p, ab);
    ab += 6 * (size_t)kLzSteps * g.batch;
  }
  std::vector<double> v(nab);
  fetch(h, v.data(), h->lzPart.p + np, nab);
  MBD_HIP(hipStreamSynchronize(s));
  return ld_ritz(v.data(), (int)(nab / (2 * kLzSteps)), lo, hi);
}

// n^3 over the matrices.
double ld_work(const std::vector<LdGroup> &groups) {
  double w = 0.0;
  for (const LdGroup &g : groups) w += g.batch * (double)g.n * g.n * g.n;
  return w;
}

// Factors entries b0 ... b1 - 1 of `nd` for every matrix of `groups` and adds
// the nodes' terms to e.  1: done; 0: a matrix is not positive definite; -1:
// no room for one shifted matrix.  watch: updates end once the proof, if it is
// among the entries, has failed.
int ld_factor(mbd_handle *h, const std::vector<LdGroup> &groups, int cells, const LdNodes &nd, int b0,
              int b1, bool watch, double &e) {
  hipStream_t s = h->stream;
  const size_t budget = mem_budget();
  const int all = b1 - b0;
  size_t nmat = 0, npart = 0;
  for (const LdGroup &g : groups) {
    nmat += (size_t)g.batch * all;
    npart += (size_t)g.batch * all * ceil_div(g.n, 64);
  }
  h->ldG.ensure(npart);
  h->ldInfo.ensure(nmat);
  batch_zero(s, h->ldInfo.p, (int)nmat);
  std::vector<int> node;  // of each factored matrix, in order
  size_t p0 = 0;          // their sums' parts
  for (const LdGroup &g : groups) {
    const int lda = lead_dim(g.n);
    const long sH = (long)g.n * g.n, sA = (long)g.n * lda,
               sinv = (long)ceil_div(g.n, kCholNB) * kCholNB * kCholNB;
    const size_t one = 8 * (size_t)(sA + sinv);
    // shifted matrices per pass: the SCS stage's memory budget, and what is free
    size_t fit = std::min<size_t>(budget / one, (size_t)g.batch * all);
    if (fit < 1) return -1;
    if (h->A64.n < fit * sA || h->inv64.n < fit * sinv) {
      size_t freeb = 0, total = 0;
      MBD_HIP(hipMemGetInfo(&freeb, &total));
      fit = std::min(fit, (freeb / 10 * 9 + 8 * (h->A64.n + h->inv64.n)) / one);
      if (fit < 1) return -1;
      try {
        h->A64.ensure(fit * sA);
        h->inv64.ensure(fit * sinv);
      } catch (const HipError &x) {
        if (x.err != hipErrorOutOfMemory) throw;
        (void)hipGetLastError();
        return -1;
      }
    }
    const int rb = std::max<int>(1, (int)(fit / all)), nbmax = std::min<int>((int)fit, all);
    for (int r0 = 0; r0 < g.batch; r0 += rb)
      for (int q0 = b0; q0 < b1; q0 += nbmax) {
        const int rn = std::min(rb, g.batch - r0), nb = std::min(nbmax, b1 - q0);
        const size_t m0 = node.size();
        ld_shift(s, g.n, g.H + r0 * sH, g.n, sH, rn, nd, q0, nb, h->A64.p, lda, sA);
        potrf_batched<double>(s, g.n, h->A64.p, lda, sA, rn * nb, h->inv64.p, sinv,
                              h->ldInfo.p + m0, true, watch && q0 + nb == nd.n + 1 ? nb : 0);
        ld_sums(s, g.n, g.H + r0 * sH, g.n, sH, h->A64.p, lda, sA, rn, nd, q0, nb, h->om_at.p, h->N, cells,
                h->ldG.p + p0);
        for (int m = 0; m < rn * nb; ++m) node.push_back(q0 + m % nb);
        p0 += (size_t)rn * nb * ceil_div(g.n, 64);
      }
  }
  std::vector<double> part(p0);
  std::vector<int> info(node.size());
  MBD_HIP(hipMemcpyAsync(part.data(), h->ldG.p, 8 * p0, hipMemcpyDeviceToHost, s));
  MBD_HIP(hipMemcpyAsync(info.data(), h->ldInfo.p, 4 * info.size(), hipMemcpyDeviceToHost, s));
  MBD_HIP(hipStreamSynchronize(s));
  if (std::any_of(info.begin(), info.end(), [](int i) { return i != 0; })) return 0;
  size_t m = 0, at = 0;
  for (const LdGroup &g : groups)
    for (int q = 0; q < g.batch * all; ++q, ++m) {
      double sum = 0.0;
      for (int i = 0; i < ceil_div(g.n, 64); ++i) sum += part[at++];
      if (node[m] < nd.n) e += nd.w[node[m]] * sum;
    }
  return 1;
}

// E_MBD of the matrices of `groups` by log-determinants into h->e_val; row r
// belongs to atom (r % (3 N cells)) / (3 cells).  false, with nothing
// decided, when they have an eigenvalue below 0.03 of the smallest omega^2
// (negative ones among them), an omega that is not positive, a value that is
// not finite, or no room for one shifted matrix.
bool energy_by_logdet(mbd_handle *h, const std::vector<LdGroup> &groups, int cells) {
  hipStream_t s = h->stream;
  const int N = h->N;
  long nhi = 0;
  for (const LdGroup &g : groups) nhi += (long)g.batch * ceil_div(g.n, 64);
  h->ldHi.ensure(nhi);
  std::vector<double> hi(nhi), om(N);
  long at = 0;
  for (const LdGroup &g : groups) {
    ld_bounds(s, g.n, g.H, g.n, (long)g.n * g.n, g.batch, h->ldHi.p + at);
    at += (long)g.batch * ceil_div(g.n, 64);
  }
  MBD_HIP(hipMemcpyAsync(hi.data(), h->ldHi.p, 8 * nhi, hipMemcpyDeviceToHost, s));
  MBD_HIP(hipMemcpyAsync(om.data(), h->om_at.p, 8 * N, hipMemcpyDeviceToHost, s));
  MBD_HIP(hipStreamSynchronize(s));
  double top = 0.0, w2min = 1e300, w2max = 0.0;
  for (double v : hi) {
    if (!std::isfinite(v)) return false;
    top = std::max(top, v);
  }
  for (double w : om) {
    // the log-determinants know omega^2 only: a negative omega (of a negative
    // C6) would enter the sum of -3/2 omega with the wrong sign
    if (!(w > 0.0) || !std::isfinite(w)) return false;
    w2min = std::min(w2min, w * w);
    w2max = std::max(w2max, w * w);
  }
  top = std::max(top, w2max);
  // the smallest eigenvalue is 0.38 (graphene) to 0.97 (water) of the
  // smallest omega^2 on the reference's examples and the benchmark's systems
  std::vector<std::pair<double, double>> guess = {{0.3 * w2min, top}, {0.03 * w2min, top}};
  double rlo, rhi, above = INFINITY;  // the smallest eigenvalue is not above this
  if (ritz_values(h, groups, rlo, rhi)) {
    if (rlo <= 0.0) return false;  // an eigenvalue is not positive
    above = rlo;
    const double up = std::max(w2max, std::min(top, rhi + 0.2 * (rhi - rlo)));
    guess.insert(guess.begin(), {0.65 * std::min(rlo, w2min), up});
  }
  // (with Ritz values above zero a proof hardly fails: no watching)
  const bool big = ld_work(groups) >= kLdProofWork, watch = big && above == INFINITY;
  bool failed = false;
  for (const auto &[lo, up] : guess) {
    if (lo >= above) continue;  // its proof cannot hold
    LdNodes nd;
    if (!ld_nodes(lo, up, nd)) return false;
    double e = 0.0;
    int pd = 1;
    if (failed && big) {
      pd = ld_factor(h, groups, cells, nd, nd.n, nd.n + 1, watch, e);
      if (pd > 0) pd = ld_factor(h, groups, cells, nd, 0, nd.n, false, e);
    } else {
      pd = ld_factor(h, groups, cells, nd, 0, nd.n + 1, watch, e);
    }
    if (pd < 0 || !std::isfinite(e)) return false;
    if (pd) {
      h->e_val = e / h->ncell;
      h->n_neg = 0;
      return true;
    }
    above = lo;
    failed = true;
  }
  return false;
}

// The energy of a supercell from the Fourier transform of its blocks over the
// cells: C's eigenvalues are those of one Hermitian matrix of order 3 N per
// wave vector, (3 N cells)^3 operations fall to about cells (3 N)^3.  Taken
// where the image box covers the cutoff sphere for every pair of atoms and
// cells (h->cells_cover: then a block depends on the cells' difference
// alone).  kBlocks: an image lies on the sphere to rounding, the blocks cannot
// be used; kSpectrum: energy_by_logdet decided nothing on them, and would not
// on the whole matrix, which has the same eigenvalues (tried there too, a 2 x
// 2 x 2 supercell of 64 atoms with negative eigenvalues took 22.0 ms instead
// of 18.6, against 17.9 by eigenvalues alone; 3 x 3 x 3 cells of 27 atoms
// 34.0, 27.3 and 26.5).
enum class ByCells { kDone, kBlocks, kSpectrum };
ByCells energy_by_cells(mbd_handle *h, const double *alpha_eff_d) {
  hipStream_t s = h->stream;
  const int N = h->N, n = h->n(), nc = h->ncell, *S = h->supercell;
  const size_t nn = (size_t)n * n;
  // wave vectors k = -k, then one of each pair
  std::vector<int> kv, pair;
  auto index = [&](int i, int j, int k) { return (k * S[1] + j) * S[0] + i; };
  for (int k = 0; k < S[2]; ++k)
    for (int j = 0; j < S[1]; ++j)
      for (int i = 0; i < S[0]; ++i) {
        const int q = index(i, j, k);
        const int m = index((S[0] - i) % S[0], (S[1] - j) % S[1], (S[2] - k) % S[2]);
        if (m == q)
          kv.insert(kv.end(), {i, j, k});
        else if (q < m)
          pair.insert(pair.end(), {i, j, k});
      }
  const int nr = (int)kv.size() / 3, np = (int)pair.size() / 3;
  kv.insert(kv.end(), pair.begin(), pair.end());
  const int L = std::lcm(S[0], std::lcm(S[1], S[2]));
  std::vector<double> cs(2 * (size_t)L);  // and the wave vectors
  for (int m = 0; m < L; ++m) {
    cs[m] = std::cos(2.0 * kPi * m / L);
    cs[L + m] = std::sin(2.0 * kPi * m / L);
  }
  cs.insert(cs.end(), kv.begin(), kv.end());
  h->cellPh.ensure(cs.size() + (size_t)(nr + 2 * np) * nc);
  h->cellB.ensure(nc * nn);
  h->cellH.ensure((nr + 4 * (size_t)np) * nn);
  h->cellNear.ensure(1);
  MBD_HIP(hipMemcpyAsync(h->cellPh.p, cs.data(), 8 * cs.size(), hipMemcpyHostToDevice, s));
  batch_zero(s, h->cellNear.p, 1);
  cfdm_cells(s, N, nc, h->xyz.p, h->cell.p, h->lat_d.p, h->nimg_cfdm, h->nimg_cfdm / 2, h->img_cfdm.p,
             h->rc_cfdm / kBohr, h->beta, alpha_eff_d, h->om_at.p, h->reff.p, h->cellB.p,
             h->cellNear.p);
  cell_dft(s, n, S, L, nr, np, h->cellPh.p, h->cellPh.p + cs.size(), h->cellB.p, h->cellH.p,
           h->cellH.p + nr * nn);
  int near = 0;
  MBD_HIP(hipMemcpyAsync(&near, h->cellNear.p, sizeof near, hipMemcpyDeviceToHost, s));
  MBD_HIP(hipStreamSynchronize(s));
  if (near) return ByCells::kBlocks;
  std::vector<LdGroup> groups;
  if (nr) groups.push_back({n, nr, h->cellH.p});
  if (np) groups.push_back({2 * n, np, h->cellH.p + nr * nn});
  return energy_by_logdet(h, groups, 1) ? ByCells::kDone : ByCells::kSpectrum;
}

// E_MBD from device alpha_eff / c6_eff.
void run_energy(mbd_handle *h, const double *alpha_eff_d, const double *c6_d,
                mbd_diag *d) {
  const int N = h->N;
  hipStream_t s = h->stream;
  h->om_at.ensure(N);
  h->reff.ensure(N);
  mbd_params(s, N, alpha_eff_d, c6_d, h->a0.p, h->r0.p, h->om_at.p, h->reff.p);
  const long nm = 3L * N * h->ncell;
  if (d) {
    d->info_eig = 0;
    for (int k = 0; k < 3; ++k) d->supercell[k] = h->supercell[k];
  }
  h->eig_flag = 0;
  bool logdet = use_logdet();
  if (h->ncell > 1 && h->cells_cover && logdet) {
    const ByCells r = energy_by_cells(h, alpha_eff_d);
    if (r == ByCells::kDone) return;
    logdet = r == ByCells::kBlocks;
  }
  h->C.ensure((size_t)nm * nm);
  cfdm_build(s, N, h->ncell, h->xyz.p, h->cell.p, h->lat_d.p, h->nimg_cfdm,
             h->nimg_cfdm / 2, h->img_cfdm.p, h->rc_cfdm / kBohr, h->beta,
             alpha_eff_d, h->om_at.p, h->reff.p, h->C.p, nm, false);
  if (logdet && nm <= kLdMaxOrder &&
      energy_by_logdet(h, {LdGroup{(int)nm, 1, h->C.p}}, h->ncell))
    return;
  TrdWork wk;
  h->VW.ensure((size_t)nm * 3 * kTrdNB);
  h->tau.ensure(nm);
  h->dd.ensure(nm);
  h->ee.ensure(nm);
  h->alph.ensure(kTrdNB);
  wk.pald = (int)(nm / 64 + 2);
  h->pa.ensure((size_t)wk.pald * kTrdQuant);
  h->pb.ensure((size_t)wk.pald);
  const size_t nbt = (size_t)ceil_div(nm, kTrdTile);
  h->py.ensure(nbt * nbt * kTrdTile);
  wk.py = h->py.p;
  h->qred.ensure(kTrdQred);
  wk.qred = h->qred.p;
  h->ps.ensure(nbt + 1);
  wk.ps = h->ps.p;
  wk.VW = h->VW.p;
  wk.ldv = nm;
  wk.tau = h->tau.p;
  wk.d = h->dd.p;
  wk.e = h->ee.p;
  wk.alpha = h->alph.p;
  wk.pa = h->pa.p;
  wk.pb = h->pb.p;
  const int method = eig_method((int)nm);
  h->eig_used = method;
  SbrWork sw{};
  if (method == 2) {
    const SbrSizes z = sbr_sizes((int)nm);
    h->sbrV.ensure(z.V);
    h->sbrT.ensure(z.TR);
    h->sbrR.ensure(z.TR);
    h->sbrX.ensure(z.X);
    h->sbrY.ensure(z.Yp);
    h->sbrMp.ensure(z.Mp);
    h->sbrM.ensure((size_t)3 * kSbrB * kSbrB);
    h->sbrAB.ensure(z.AB);
    h->sbrCnt.ensure(z.cnt);
    h->sbrMcnt.ensure(z.mcnt);
    h->sbrProg.ensure(z.prog);
    h->sbrFlag.ensure(4);
    h->sbrMail.ensure(z.mail);
    h->sbrCq.ensure(z.cq);
    h->sbrCqR.ensure(z.cqR);
    sw = SbrWork{h->sbrV.p, h->sbrT.p, h->sbrR.p, h->sbrCnt.p, h->sbrX.p, h->sbrY.p,
                 h->sbrMp.p, h->sbrM.p, h->sbrMcnt.p, h->sbrAB.p, h->sbrProg.p, h->sbrFlag.p,
                 h->sbrMail.p, h->sbrCq.p, h->sbrCqR.p, h->VW.p, nm, h->dd.p, h->ee.p};
    if (sbr_lookahead()) {
      h->sbrVW2.ensure((size_t)nm * 6 * kSbrB);
      if (!h->stream2) {
        // The look-ahead SYR2K fills every CU it may use with two workgroups
        // of 64 KB of LDS each, and the panel kernels of the main stream (up
        // to 157 KB) then wait for whole CUs to drain: its stream leaves
        // kSbrFreeCus CUs to the main stream (a stream's CU mask holds for
        // eager launches only, not for a replayed graph).
        int ncu = 0;
        MBD_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device));
        const char *fe = getenv("MBD_SBR_FREE_CUS");
        const int nfree = fe ? atoi(fe) : kSbrFreeCus;
        if (nfree > 0 && nfree < ncu) {
          std::vector<uint32_t> mask((ncu + 31) / 32, 0u);
          for (int c = 0; c < ncu - nfree; ++c) mask[c / 32] |= 1u << (c % 32);
          MBD_HIP(hipExtStreamCreateWithCUMask(&h->stream2, (uint32_t)mask.size(), mask.data()));
        } else {
          MBD_HIP(hipStreamCreateWithFlags(&h->stream2, hipStreamNonBlocking));
        }
      }
      if (!h->sbr_fork) MBD_HIP(hipEventCreateWithFlags(&h->sbr_fork, hipEventDisableTiming));
      if (!h->sbr_join) MBD_HIP(hipEventCreateWithFlags(&h->sbr_join, hipEventDisableTiming));
      sw.VW2 = h->sbrVW2.p;
      sw.s2 = h->stream2;
      sw.fork = h->sbr_fork;
      sw.join = h->sbr_join;
    }
  }
  auto reduce = [&]() {
    if (method == 2)
      sbr_tridiagonalize(s, (int)nm, h->C.p, nm, sw);
    else
      tridiagonalize(s, (int)nm, h->C.p, nm, wk);
  };
  // The one-stage reduction (thousands of small launches) replays a captured
  // graph; the two-stage one launches eagerly, which measured faster (with
  // the look-ahead stream's CU mask in force).  MBD_TRD_GRAPH=0|1 forces
  // either way.
  const char *g = getenv("MBD_TRD_GRAPH");
  const bool graph = g ? g[0] != '0' : method != 2;
  if (h->prof_on || !graph) {
    reduce();
  } else {
    const std::vector<const void *> key = {(const void *)(intptr_t)nm, (const void *)(intptr_t)method,
                                           h->C.p, h->VW.p, h->tau.p, h->dd.p, h->ee.p, h->alph.p,
                                           h->pa.p, h->pb.p, h->py.p, h->qred.p, h->ps.p,
                                           sw.Vn, sw.Tn, sw.Rn, sw.cnt, sw.X, sw.Yp, sw.Mp, sw.M,
                                           sw.mcnt, sw.AB, sw.prog, sw.flag, sw.mail, sw.cq,
                                           sw.cqR, sw.VW2, (const void *)sw.s2};
    if (!h->trd_exec || h->trd_key != key) {
      if (h->trd_exec) (void)hipGraphExecDestroy(h->trd_exec);
      h->trd_exec = nullptr;
      h->trd_key.clear();
      tridiag_prepare();
      hipGraph_t gr = nullptr;
      MBD_HIP(hipStreamBeginCapture(s, hipStreamCaptureModeRelaxed));
      try {
        reduce();
      } catch (const HipError &) {
        (void)hipStreamEndCapture(s, &gr);
        if (gr) (void)hipGraphDestroy(gr);
        throw;
      }
      MBD_HIP(hipStreamEndCapture(s, &gr));
      const hipError_t ie = hipGraphInstantiate(&h->trd_exec, gr, nullptr, nullptr, 0);
      (void)hipGraphDestroy(gr);
      MBD_HIP(ie);
      h->trd_key = key;
    }
    MBD_HIP(hipGraphLaunch(h->trd_exec, s));
  }
  if (method == 2)
    MBD_HIP(hipMemcpyAsync(&h->eig_flag, sw.flag, sizeof(int), hipMemcpyDeviceToHost, s));
  h->lam.ensure(nm);
  h->e2.ensure(nm);
  h->bounds.ensure(kBisectBounds);
  tridiag_eigvals(s, (int)nm, h->dd.p, h->ee.p, h->e2.p, h->bounds.p, h->lam.p);
  h->E.ensure(4);
  h->nneg.ensure(1);
  energy(s, (int)nm, h->lam.p, N, h->om_at.p, h->ncell, h->E.p, h->nneg.p);
  MBD_HIP(hipMemcpyAsync(&h->e_val, h->E.p, sizeof(double), hipMemcpyDeviceToHost, s));
  MBD_HIP(hipMemcpyAsync(&h->n_neg, h->nneg.p, sizeof(int), hipMemcpyDeviceToHost, s));
  MBD_HIP(hipStreamSynchronize(s));
}

void fetch(mbd_handle *h, double *dst, const double *src, size_t count) {
  if (dst && count) MBD_HIP(hipMemcpyAsync(dst, src, sizeof(double) * count, hipMemcpyDeviceToHost, h->stream));
}

void fetch_scs_outputs(mbd_handle *h, double *alpha_eff, double *coupled_pol,
                       double *molpol_eig, double *c6_eff, double *c6_mol) {
  const int N = h->N;
  fetch(h, alpha_eff, h->alpha.p, N);
  if (coupled_pol) {
    std::vector<double> a((size_t)kNumFreq * N);
    fetch(h, a.data(), h->alpha.p, a.size());
    MBD_HIP(hipStreamSynchronize(h->stream));
    for (int i = 0; i < N; ++i)
      for (int k = 1; k < kNumFreq; ++k) coupled_pol[(k - 1) + 20L * i] = a[(size_t)k * N + i];
  }
  fetch(h, molpol_eig, h->eig3.p, 3 * kNumFreq);
  fetch(h, c6_eff, h->c6.p, N);
  fetch(h, c6_mol, h->c6mol.p, 1);
  MBD_HIP(hipStreamSynchronize(h->stream));
}

struct DevScratch {
  std::vector<void *> ptrs;
  template <typename T>
  T *get(size_t count) {
    void *p = nullptr;
    MBD_HIP(hipMalloc(&p, sizeof(T) * std::max<size_t>(count, 1)));
    ptrs.push_back(p);
    return static_cast<T *>(p);
  }
  ~DevScratch() {
    for (void *p : ptrs) (void)hipFree(p);
  }
};
long blob_floats() { return 2L * kNetIn + net_param_count(); }

bool valid_mode(int mode) {
  return mode == MBD_MODE_FP64 || mode == MBD_MODE_MIXED || mode == MBD_MODE_LEARNED;
}

}  // namespace

namespace {

template <typename T>
int debug_cholesky(int device, int n, int batch, const T *A, T *L, int *info) {
  if (n <= 0) return -2;
  if (batch <= 0) return -3;
  if (!A) return -4;
  if (!L) return -5;
  if (!info) return -6;
  T *dA = nullptr, *dinv = nullptr;
  int *dinfo = nullptr;
  int rc = 0;
  try {
    MBD_HIP(hipSetDevice(device));
    const long sA = (long)n * n;
    const long sinv = (long)ceil_div(n, kCholNB) * kCholNB * kCholNB;
    MBD_HIP(hipMalloc(&dA, sizeof(T) * sA * batch));
    MBD_HIP(hipMalloc(&dinv, sizeof(T) * sinv * batch));
    MBD_HIP(hipMalloc(&dinfo, sizeof(int) * batch));
    MBD_HIP(hipMemcpy(dA, A, sizeof(T) * sA * batch, hipMemcpyHostToDevice));
    MBD_HIP(hipMemset(dinfo, 0, sizeof(int) * batch));
    potrf_batched<T>(nullptr, n, dA, n, sA, batch, dinv, sinv, dinfo);
    MBD_HIP(hipDeviceSynchronize());
    MBD_HIP(hipMemcpy(L, dA, sizeof(T) * sA * batch, hipMemcpyDeviceToHost));
    MBD_HIP(hipMemcpy(info, dinfo, sizeof(int) * batch, hipMemcpyDeviceToHost));
  } catch (const HipError &e) {
    rc = fail(nullptr, e);
  }
  if (dA) (void)hipFree(dA);
  if (dinv) (void)hipFree(dinv);
  if (dinfo) (void)hipFree(dinfo);
  return rc;
}

}  // namespace

extern "C" {

int mbd_create(int device, mbd_handle **out) {
  if (!out) return -2;
  mbd_handle *h = new mbd_handle;
  h->device = device;
  try {
    MBD_HIP(hipSetDevice(device));
    MBD_HIP(hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking));
    h->omega.ensure(kNumFreq);
    h->weight.ensure(kNumFreq);
    double w[kNumFreq], g[kNumFreq];
    mbd_casimir_grid(w, g);
    MBD_HIP(hipMemcpy(h->omega.p, w, sizeof w, hipMemcpyHostToDevice));
    MBD_HIP(hipMemcpy(h->weight.p, g, sizeof g, hipMemcpyHostToDevice));
    // device address of the no-allocation scratch on this device (once)
    if (device >= 0 && device < kNaMaxDevices && !na_ptr[device]) {
      void *p = nullptr;
      MBD_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
      na_ptr[device] = p;
    }
  } catch (const HipError &e) {
    int rc = fail(h, e);
    delete h;
    *out = nullptr;
    return rc;
  }
  *out = h;
  return 0;
}

int mbd_destroy(mbd_handle *h) {
  if (!h) return 0;
  (void)hipSetDevice(h->device);
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  DevBuf<double> *dbufs[] = {&h->xyz, &h->hirsh, &h->a0, &h->c60, &h->r0, &h->omega,
                             &h->weight, &h->img_scs, &h->img_cfdm, &h->lat_d, &h->alpha_w,
                             &h->sgm, &h->rvdw, &h->A64, &h->inv64, &h->X, &h->alpha,
                             &h->P, &h->eig3, &h->c6mol, &h->c6, &h->R, &h->D, &h->rnorm,
                             &h->C, &h->om_at, &h->reff, &h->lam, &h->e2, &h->bounds,
                             &h->E, &h->VW, &h->tau, &h->dd, &h->ee, &h->alph, &h->pa,
                             &h->pb, &h->py, &h->qred, &h->ps, &h->pMinv, &h->pR, &h->pZ, &h->pP, &h->pQ, &h->pscal, &h->ppart, &h->alpha_pred, &h->img_net, &h->ext_alpha, &h->ext_c6};
  for (auto *b : dbufs) b->release();
  h->A32.release();
  h->L32.release();
  h->net_blob.release();
  h->net_X.release();
  h->net_Xn.release();
  h->net_act.release();
  h->net_nbl.release();
  h->net_cnt.release();
  h->inv32.release();
  h->info.release();
  h->A1.release();
  h->inv1.release();
  h->svU.release();
  h->svV.release();
  h->clOff.release();
  h->clAtoms.release();
  h->clMoff.release();
  h->luUt.release();
  h->info1.release();
  h->luPiv.release();
  h->cell.release();
  h->nneg.release();
  DevBuf<double> *sbufs[] = {&h->sbrV, &h->sbrT, &h->sbrR, &h->sbrX, &h->sbrY, &h->sbrMp,
                             &h->sbrM, &h->sbrAB, &h->sbrCqR, &h->sbrVW2};
  for (auto *b : sbufs) b->release();
  DevBuf<int> *sibufs[] = {&h->sbrCnt, &h->sbrMcnt, &h->sbrProg, &h->sbrFlag, &h->sbrCq};
  for (auto *b : sibufs) b->release();
  h->sbrMail.release();
  h->ldHi.release();
  h->ldG.release();
  h->lzV.release();
  h->lzPart.release();
  h->ldInfo.release();
  h->cellB.release();
  h->cellH.release();
  h->cellPh.release();
  h->cellNear.release();
  batch_release(h);
  if (h->trd_exec) (void)hipGraphExecDestroy(h->trd_exec);
  if (h->stream2) (void)hipStreamSynchronize(h->stream2);
  if (h->sbr_fork) (void)hipEventDestroy(h->sbr_fork);
  if (h->sbr_join) (void)hipEventDestroy(h->sbr_join);
  if (h->stream2) (void)hipStreamDestroy(h->stream2);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
  return 0;
}

const char *mbd_last_error(const mbd_handle *h) { return h ? h->err.c_str() : ""; }

int mbd_free_atom_params(const char *symbol, double *c6, double *alpha, double *r0) {
  if (!symbol) return -1;
  char s[3] = {0, 0, 0};
  int k = 0;
  for (const char *p = symbol; *p && k < 2; ++p)
    if (*p != ' ') s[k++] = *p;
  for (const auto &e : kElements)
    if (strcmp(e.sym, s) == 0) {
      if (c6) *c6 = (double)e.c6;
      if (alpha) *alpha = (double)e.alpha;
      if (r0) *r0 = (double)e.r0;
      return 0;
    }
  return -1;
}

double mbd_beta(int flag_xc) {
  switch (flag_xc) {
    case 1: return (double)0.83f;
    case 2:
    case 3: return (double)0.85f;
    default: return 1.0;
  }
}

void mbd_casimir_grid(double *omega21, double *weight21) {
  for (int k = 0; k < kNumFreq; ++k) {
    if (omega21) omega21[k] = (double)kOmega[k];
    if (weight21) weight21[k] = (double)kWeight[k];
  }
}

int mbd_set_system(mbd_handle *h, int n_atoms, const double *xyz, const double *hirshfeld,
                   const double *alpha0, const double *c6_0, const double *r0,
                   const double *lattice, int periodic, const int *vacuum, double beta,
                   double rc_scs, double rc_cfdm, double rc_supercell) {
  if (!h) return -1;
  if (n_atoms <= 0) return -2;
  if (!xyz) return -3;
  if (!hirshfeld) return -4;
  if (!alpha0) return -5;
  if (!c6_0) return -6;
  if (!r0) return -7;
  if (periodic && !lattice) return -8;
  try {
    MBD_HIP(hipSetDevice(h->device));
    h->N = n_atoms;
    h->periodic = periodic ? 1 : 0;
    for (int c = 0; c < 9; ++c) h->lat[c] = periodic ? lattice[c] : 0.0;
    h->beta = beta;
    h->rc_scs = rc_scs;
    h->rc_cfdm = rc_cfdm;
    h->rc_sc = rc_supercell;
    int vac[3] = {0, 0, 0};
    if (vacuum)
      for (int k = 0; k < 3; ++k) vac[k] = vacuum[k] ? 1 : 0;
    // image ranges and supercell (UTILS.f90:1215-1320)
    for (int k = 0; k < 3; ++k) {
      h->scs_img[k] = 0;
      h->supercell[k] = 1;
      h->cfdm_img[k] = 0;
      if (h->periodic && !vac[k]) {
        const double la = norm3(h->lat + 3 * k);
        h->scs_img[k] = (int)std::ceil((rc_scs / kBohr) / la);
        h->supercell[k] = (int)std::ceil((rc_supercell / kBohr) / la);
      }
    }
    for (int k = 0; k < 3; ++k)
      for (int c = 0; c < 3; ++c) h->latSL[3 * k + c] = h->lat[3 * k + c] * h->supercell[k];
    for (int k = 0; k < 3; ++k)
      if (h->periodic && !vac[k])
        h->cfdm_img[k] = (int)std::ceil((rc_cfdm / kBohr) / norm3(h->latSL + 3 * k));
    h->cells_cover = h->periodic && images_cover(n_atoms, xyz, h->lat, h->supercell, h->cfdm_img, vac,
                                                 rc_cfdm / kBohr);
    std::vector<double> ti = image_box(h->lat, h->scs_img);
    std::vector<double> tc = image_box(h->latSL, h->cfdm_img);
    h->nimg_scs = (int)(ti.size() / 3);
    h->nimg_cfdm = (int)(tc.size() / 3);
    const int S1 = h->supercell[0], S2 = h->supercell[1], S3 = h->supercell[2];
    h->ncell = S1 * S2 * S3;
    std::vector<int> cells(3 * h->ncell);
    for (int c1 = 0; c1 < S1; ++c1)
      for (int c2 = 0; c2 < S2; ++c2)
        for (int c3 = 0; c3 < S3; ++c3) {
          const int a = c3 * S2 * S1 + c2 * S1 + c1;  // UTILS.f90:915
          cells[3 * a] = c1;
          cells[3 * a + 1] = c2;
          cells[3 * a + 2] = c3;
        }
    auto up = [&](DevBuf<double> &b, const double *src, size_t cnt) {
      b.ensure(cnt);
      MBD_HIP(hipMemcpyAsync(b.p, src, sizeof(double) * cnt, hipMemcpyHostToDevice, h->stream));
    };
    up(h->xyz, xyz, 3L * n_atoms);
    up(h->hirsh, hirshfeld, n_atoms);
    up(h->a0, alpha0, n_atoms);
    up(h->c60, c6_0, n_atoms);
    up(h->r0, r0, n_atoms);
    up(h->img_scs, ti.data(), ti.size());
    {
      // descriptor images: r = |x_i - x_j + L| >= |L| - span, with span the
      // diagonal of the atoms' bounding box, so |L| > cutoff + span never reaches
      double lo[3] = {1e300, 1e300, 1e300}, hi[3] = {-1e300, -1e300, -1e300};
      for (int i = 0; i < n_atoms; ++i)
        for (int c = 0; c < 3; ++c) {
          lo[c] = std::min(lo[c], xyz[3 * i + c]);
          hi[c] = std::max(hi[c], xyz[3 * i + c]);
        }
      const double span[3] = {hi[0] - lo[0], hi[1] - lo[1], hi[2] - lo[2]};
      const double diam = norm3(span);
      std::vector<double> tn;
      h->center_net = -1;
      for (size_t q = 0; q < ti.size() / 3; ++q) {
        const double L = norm3(&ti[3 * q]);
        if ((int)q == h->nimg_scs / 2) h->center_net = (int)(tn.size() / 3);
        if (L <= kNetCut + diam || (int)q == h->nimg_scs / 2)
          for (int c = 0; c < 3; ++c) tn.push_back(ti[3 * q + c]);
      }
      // sorted by |L| (stable), so that the neighbour scan can bound, per atom
      // pair, the images that can come within the cutoff
      {
        const int nt = (int)(tn.size() / 3);
        std::vector<int> ord(nt);
        for (int q = 0; q < nt; ++q) ord[q] = q;
        std::stable_sort(ord.begin(), ord.end(),
                         [&](int a, int b) { return norm3(&tn[3 * a]) < norm3(&tn[3 * b]); });
        std::vector<double> ts(tn.size());
        int cnew = -1;
        for (int q = 0; q < nt; ++q) {
          for (int c = 0; c < 3; ++c) ts[3 * q + c] = tn[3 * ord[q] + c];
          if (ord[q] == h->center_net) cnew = q;
        }
        tn.swap(ts);
        h->center_net = cnew;
      }
      h->nimg_net = (int)(tn.size() / 3);
      up(h->img_net, tn.data(), tn.size());
    }
    up(h->img_cfdm, tc.data(), tc.size());
    up(h->lat_d, h->lat, 9);
    h->xyz_h.assign(xyz, xyz + 3L * n_atoms);
    h->hirsh_h.assign(hirshfeld, hirshfeld + n_atoms);
    h->a0_h.assign(alpha0, alpha0 + n_atoms);
    h->r0_h.assign(r0, r0 + n_atoms);
    h->cl_ready = false;
    h->cell.ensure(cells.size());
    MBD_HIP(hipMemcpyAsync(h->cell.p, cells.data(), sizeof(int) * cells.size(),
                           hipMemcpyHostToDevice, h->stream));
    MBD_HIP(hipStreamSynchronize(h->stream));
    h->has_sys = true;
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_scs(mbd_handle *h, int mode, double *alpha_eff, double *coupled_pol,
            double *molpol_eig, double *c6_eff, double *c6_mol, mbd_diag *d) {
  if (!h) return -1;
  if (!valid_mode(mode)) return -2;
  if (!h->has_sys) return MBD_ERR_NOSYS;
  try {
    ProfGuard pg(h);
    MBD_HIP(hipSetDevice(h->device));
    Timer tm;
    tm.start(h->stream);
    run_scs(h, mode, d);
    tm.stop(h->stream);
    const double ms = tm.ms();
    fetch_scs_outputs(h, alpha_eff, coupled_pol, molpol_eig, c6_eff, c6_mol);
    if (d) {
      d->t_scs_ms = ms;
      d->t_total_ms = ms;
    }
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_energy(mbd_handle *h, const double *alpha_eff, const double *c6_eff, double *e_mbd,
               double *omega, double *reff, mbd_diag *d) {
  if (!h) return -1;
  if (!alpha_eff) return -2;
  if (!c6_eff) return -3;
  if (!e_mbd) return -4;
  if (!h->has_sys) return MBD_ERR_NOSYS;
  try {
    ProfGuard pg(h);
    MBD_HIP(hipSetDevice(h->device));
    const int N = h->N;
    h->ext_alpha.ensure(N);
    h->ext_c6.ensure(N);
    MBD_HIP(hipMemcpyAsync(h->ext_alpha.p, alpha_eff, sizeof(double) * N, hipMemcpyHostToDevice, h->stream));
    MBD_HIP(hipMemcpyAsync(h->ext_c6.p, c6_eff, sizeof(double) * N, hipMemcpyHostToDevice, h->stream));
    Timer tm;
    tm.start(h->stream);
    run_energy(h, h->ext_alpha.p, h->ext_c6.p, d);
    tm.stop(h->stream);
    const double ms = tm.ms();
    fetch(h, omega, h->om_at.p, N);
    fetch(h, reff, h->reff.p, N);
    MBD_HIP(hipStreamSynchronize(h->stream));
    *e_mbd = h->e_val;
    if (h->eig_flag) {
      if (d) d->info_eig = 1;
      return MBD_ERR_EIG;
    }
    if (d) {
      d->n_negative = h->n_neg;
      d->t_mbd_ms = ms;
      d->t_total_ms = ms;
    }
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_run(mbd_handle *h, int mode, double *e_mbd, double *alpha_eff, double *coupled_pol,
            double *molpol_eig, double *c6_eff, double *c6_mol, mbd_diag *d) {
  if (!h) return -1;
  if (!valid_mode(mode)) return -2;
  if (!e_mbd) return -3;
  if (!h->has_sys) return MBD_ERR_NOSYS;
  try {
    ProfGuard pg(h);
    MBD_HIP(hipSetDevice(h->device));
    Timer t_all, t_mbd;
    t_all.start(h->stream);
    run_scs(h, mode, d);
    t_mbd.start(h->stream);
    run_energy(h, h->alpha.p, h->c6.p, d);
    t_mbd.stop(h->stream);
    t_all.stop(h->stream);
    const double ms_all = t_all.ms(), ms_mbd = t_mbd.ms();
    fetch_scs_outputs(h, alpha_eff, coupled_pol, molpol_eig, c6_eff, c6_mol);
    *e_mbd = h->e_val;
    if (h->eig_flag) {
      if (d) d->info_eig = 1;
      return MBD_ERR_EIG;
    }
    if (d) {
      d->n_negative = h->n_neg;
      d->t_total_ms = ms_all;
      d->t_mbd_ms = ms_mbd;
      d->t_scs_ms = ms_all - ms_mbd;
    }
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_profile_enable(mbd_handle *h, int enable) {
  if (!h) return -1;
  try {
    MBD_HIP(hipSetDevice(h->device));
    MBD_HIP(hipStreamSynchronize(h->stream));
    h->prof.reset();
    h->prof_on = enable != 0;
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_profile_read(mbd_handle *h, int cls, double *out, const char **name) {
  if (!h) return -1;
  if (cls < 0 || cls >= K_NUM_CLASSES) return -2;
  try {
    MBD_HIP(hipSetDevice(h->device));
    h->prof.resolve();
  } catch (const HipError &e) {
    return fail(h, e);
  }
  if (out) {
    out[0] = h->prof.count[cls];
    out[1] = h->prof.ms[cls];
    out[2] = h->prof.bytes[cls];
    out[3] = h->prof.flops[cls];
  }
  if (name) *name = kernel_class_name(cls);
  return 0;
}

// ---- learned form: network ------------------------------------------------


void mbd_net_layout(int *n_in, int *hidden, long *blob) {
  if (n_in) *n_in = kNetIn;
  if (hidden) *hidden = kNetHidden;
  if (blob) *blob = blob_floats();
}

int mbd_net_set_weights(mbd_handle *h, const float *blob, long n) {
  if (!h) return -1;
  if (!blob) {
    h->have_net = false;
    return 0;
  }
  if (n != blob_floats()) return -3;
  try {
    MBD_HIP(hipSetDevice(h->device));
    h->net_blob.ensure((size_t)n);
    MBD_HIP(hipMemcpy(h->net_blob.p, blob, sizeof(float) * n, hipMemcpyHostToDevice));
    h->have_net = true;
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_net_descriptors(mbd_handle *h, float *X, double *alpha_w) {
  if (!h) return -1;
  if (!X) return -2;
  if (!h->has_sys) return MBD_ERR_NOSYS;
  try {
    MBD_HIP(hipSetDevice(h->device));
    const int N = h->N;
    const long S = (long)kNumFreq * N;
    hipStream_t s = h->stream;
    h->alpha_w.ensure((size_t)S);
    h->sgm.ensure((size_t)S);
    h->rvdw.ensure(N);
    atom_params(s, N, kNumFreq, h->omega.p, h->hirsh.p, h->a0.p, h->c60.p, h->r0.p,
                h->alpha_w.p, h->sgm.p, h->rvdw.p);
    h->net_X.ensure((size_t)kNetIn * S);
    h->net_nbl.ensure((size_t)N * kNetCap);
    h->net_cnt.ensure((size_t)N);
    net_descriptors(s, N, kNumFreq, h->xyz.p, h->nimg_net, h->center_net, h->img_net.p, h->beta,
                    h->alpha_w.p, h->hirsh.p, h->rvdw.p, h->omega.p, h->net_nbl.p, h->net_cnt.p,
                    h->net_X.p);
    MBD_HIP(hipMemcpyAsync(X, h->net_X.p, sizeof(float) * kNetIn * S, hipMemcpyDeviceToHost, s));
    if (alpha_w)
      MBD_HIP(hipMemcpyAsync(alpha_w, h->alpha_w.p, sizeof(double) * S, hipMemcpyDeviceToHost, s));
    MBD_HIP(hipStreamSynchronize(s));
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_net_forward(int device, const float *blob, int B, const float *X, float *y) {
  if (!blob) return -2;
  if (B <= 0) return -3;
  if (!X) return -4;
  if (!y) return -5;
  try {
    MBD_HIP(hipSetDevice(device));
    DevScratch sc;
    float *db = sc.get<float>(blob_floats());
    float *dX = sc.get<float>((size_t)kNetIn * B);
    float *dXn = sc.get<float>((size_t)kNetIn * B);
    float *act0 = sc.get<float>((size_t)B * (3 * kNetHidden + 1));
    MBD_HIP(hipMemcpy(db, blob, sizeof(float) * blob_floats(), hipMemcpyHostToDevice));
    MBD_HIP(hipMemcpy(dX, X, sizeof(float) * kNetIn * B, hipMemcpyHostToDevice));
    float *act[4] = {act0, act0 + (long)B * kNetHidden, act0 + 2L * B * kNetHidden,
                     act0 + 3L * B * kNetHidden};
    mlp_gather(nullptr, B, nullptr, dX, B, db, dXn);
    mlp_forward(nullptr, B, db + 2 * kNetIn, dXn, act);
    MBD_HIP(hipDeviceSynchronize());
    MBD_HIP(hipMemcpy(y, act[3], sizeof(float) * B, hipMemcpyDeviceToHost));
  } catch (const HipError &e) {
    return fail(nullptr, e);
  }
  return 0;
}

int mbd_net_grad(int device, const float *blob, int B, const float *X, const float *t,
                 float *grad, float *loss) {
  if (!blob) return -2;
  if (B <= 0) return -3;
  if (!X || !t) return -4;
  if (!grad) return -6;
  try {
    MBD_HIP(hipSetDevice(device));
    DevScratch sc;
    const long np = net_param_count();
    float *db = sc.get<float>(blob_floats());
    float *dX = sc.get<float>((size_t)kNetIn * B);
    float *dXn = sc.get<float>((size_t)kNetIn * B);
    float *dt = sc.get<float>(B);
    float *g = sc.get<float>(B);
    float *G = sc.get<float>(np);
    float *lp = sc.get<float>(ceil_div(B, 256));
    float *act0 = sc.get<float>((size_t)B * (3 * kNetHidden + 1));
    float *del0 = sc.get<float>((size_t)B * (3 * kNetHidden + 1));
    MBD_HIP(hipMemcpy(db, blob, sizeof(float) * blob_floats(), hipMemcpyHostToDevice));
    MBD_HIP(hipMemcpy(dX, X, sizeof(float) * kNetIn * B, hipMemcpyHostToDevice));
    MBD_HIP(hipMemcpy(dt, t, sizeof(float) * B, hipMemcpyHostToDevice));
    float *act[4] = {act0, act0 + (long)B * kNetHidden, act0 + 2L * B * kNetHidden,
                     act0 + 3L * B * kNetHidden};
    float *del[4] = {del0, del0 + (long)B * kNetHidden, del0 + 2L * B * kNetHidden,
                     del0 + 3L * B * kNetHidden};
    mlp_gather(nullptr, B, nullptr, dX, B, db, dXn);
    mlp_forward(nullptr, B, db + 2 * kNetIn, dXn, act);
    mlp_loss(nullptr, B, act[3], nullptr, dt, g, lp);
    mlp_backward(nullptr, B, db + 2 * kNetIn, dXn, act, del, g, G);
    MBD_HIP(hipDeviceSynchronize());
    MBD_HIP(hipMemcpy(grad, G, sizeof(float) * np, hipMemcpyDeviceToHost));
    if (loss) {
      std::vector<float> l(ceil_div(B, 256));
      MBD_HIP(hipMemcpy(l.data(), lp, sizeof(float) * l.size(), hipMemcpyDeviceToHost));
      double acc = 0.0;
      for (float v : l) acc += v;
      *loss = (float)(acc / B);
    }
  } catch (const HipError &e) {
    return fail(nullptr, e);
  }
  return 0;
}

int mbd_net_train(int device, int S, const float *X, const float *t, int epochs, int batch,
                  float lr, unsigned seed, float *blob, float *loss_hist) {
  if (S <= 0) return -2;
  if (!X) return -3;
  if (!t) return -4;
  if (epochs <= 0) return -5;
  if (batch <= 0) return -6;
  if (!blob) return -9;
  try {
    MBD_HIP(hipSetDevice(device));
    DevScratch sc;
    const long np = net_param_count();
    const int B = std::min(batch, S);
    float *db = sc.get<float>(blob_floats());
    float *dX = sc.get<float>((size_t)kNetIn * S);
    float *dt = sc.get<float>(S);
    int *didx = sc.get<int>(S);
    float *dXn = sc.get<float>((size_t)kNetIn * B);
    float *g = sc.get<float>(B);
    float *G = sc.get<float>(np);
    float *m = sc.get<float>(np);
    float *v = sc.get<float>(np);
    const int nlp = ceil_div(B, 256);
    const int nbatch = ceil_div(S, B);
    float *lp = sc.get<float>((size_t)nlp * nbatch);
    float *act0 = sc.get<float>((size_t)B * (3 * kNetHidden + 1));
    float *del0 = sc.get<float>((size_t)B * (3 * kNetHidden + 1));
    MBD_HIP(hipMemcpy(db, blob, sizeof(float) * blob_floats(), hipMemcpyHostToDevice));
    MBD_HIP(hipMemcpy(dX, X, sizeof(float) * kNetIn * S, hipMemcpyHostToDevice));
    MBD_HIP(hipMemcpy(dt, t, sizeof(float) * S, hipMemcpyHostToDevice));
    MBD_HIP(hipMemset(m, 0, sizeof(float) * np));
    MBD_HIP(hipMemset(v, 0, sizeof(float) * np));
    float *act[4] = {act0, act0 + (long)B * kNetHidden, act0 + 2L * B * kNetHidden,
                     act0 + 3L * B * kNetHidden};
    float *del[4] = {del0, del0 + (long)B * kNetHidden, del0 + 2L * B * kNetHidden,
                     del0 + 3L * B * kNetHidden};
    std::vector<int> perm(S);
    for (int q = 0; q < S; ++q) perm[q] = q;
    unsigned long long st = seed ? seed : 1;
    int step = 0;
    std::vector<float> lh((size_t)nlp * nbatch);
    for (int ep = 0; ep < epochs; ++ep) {
      for (int q = S - 1; q > 0; --q) {  // Fisher-Yates with xorshift64
        st ^= st << 13;
        st ^= st >> 7;
        st ^= st << 17;
        std::swap(perm[q], perm[st % (unsigned long long)(q + 1)]);
      }
      MBD_HIP(hipMemcpy(didx, perm.data(), sizeof(int) * S, hipMemcpyHostToDevice));
      MBD_HIP(hipMemset(lp, 0, sizeof(float) * lh.size()));
      for (int bi = 0; bi < nbatch; ++bi) {
        const int b0 = bi * B, bb = std::min(B, S - b0);
        mlp_gather(nullptr, bb, didx + b0, dX, S, db, dXn);
        mlp_forward(nullptr, bb, db + 2 * kNetIn, dXn, act);
        mlp_loss(nullptr, bb, act[3], didx + b0, dt, g, lp + (long)bi * nlp);
        mlp_backward(nullptr, bb, db + 2 * kNetIn, dXn, act, del, g, G);
        adam_step(nullptr, (int)np, db + 2 * kNetIn, G, m, v, lr, ++step);
      }
      MBD_HIP(hipDeviceSynchronize());
      MBD_HIP(hipMemcpy(lh.data(), lp, sizeof(float) * lh.size(), hipMemcpyDeviceToHost));
      double acc = 0.0;
      for (float x : lh) acc += x;
      if (loss_hist) loss_hist[ep] = (float)(acc / S);
    }
    MBD_HIP(hipMemcpy(blob + 2 * kNetIn, db + 2 * kNetIn, sizeof(float) * np,
                      hipMemcpyDeviceToHost));
  } catch (const HipError &e) {
    return fail(nullptr, e);
  }
  return 0;
}

// ---- test hooks ----------------------------------------------------------

int mbd_debug_relay_matrix(mbd_handle *h, int mode, int k, double *A) {
  if (!h) return -1;
  if (!valid_mode(mode)) return -2;
  if (k < 0 || k >= kNumFreq) return -3;
  if (!A) return -4;
  if (!h->has_sys) return MBD_ERR_NOSYS;
  try {
    MBD_HIP(hipSetDevice(h->device));
    const int N = h->N, n = h->n();
    hipStream_t s = h->stream;
    h->alpha_w.ensure((size_t)kNumFreq * N);
    h->sgm.ensure((size_t)kNumFreq * N);
    h->rvdw.ensure(N);
    atom_params(s, N, kNumFreq, h->omega.p, h->hirsh.p, h->a0.p, h->c60.p, h->r0.p,
                h->alpha_w.p, h->sgm.p, h->rvdw.p);
    const double rc = h->rc_scs / kBohr;
    const size_t cnt = (size_t)n * n;
    if (mode == MBD_MODE_FP64) {
      h->A64.ensure(cnt);
      scs_build<double>(s, N, h->xyz.p, h->nimg_scs, h->nimg_scs / 2, h->img_scs.p, rc,
                        h->beta, h->alpha_w.p + (long)k * N, h->sgm.p + (long)k * N,
                        h->rvdw.p, h->A64.p, n, (long)cnt, 1, true);
      fetch(h, A, h->A64.p, cnt);
      MBD_HIP(hipStreamSynchronize(s));
    } else {
      h->A32.ensure(cnt);
      scs_build<float>(s, N, h->xyz.p, h->nimg_scs, h->nimg_scs / 2, h->img_scs.p, rc,
                       h->beta, h->alpha_w.p + (long)k * N, h->sgm.p + (long)k * N,
                       h->rvdw.p, h->A32.p, n, (long)cnt, 1, true);
      std::vector<float> tmp(cnt);
      MBD_HIP(hipMemcpyAsync(tmp.data(), h->A32.p, sizeof(float) * cnt, hipMemcpyDeviceToHost, s));
      MBD_HIP(hipStreamSynchronize(s));
      for (size_t q = 0; q < cnt; ++q) A[q] = tmp[q];
    }
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_debug_cfdm_matrix(mbd_handle *h, const double *alpha_eff, const double *omega,
                          const double *reff, double *C) {
  if (!h) return -1;
  if (!alpha_eff || !omega || !reff || !C) return -2;
  if (!h->has_sys) return MBD_ERR_NOSYS;
  try {
    MBD_HIP(hipSetDevice(h->device));
    const int N = h->N;
    hipStream_t s = h->stream;
    h->ext_alpha.ensure(N);
    h->om_at.ensure(N);
    h->reff.ensure(N);
    MBD_HIP(hipMemcpyAsync(h->ext_alpha.p, alpha_eff, sizeof(double) * N, hipMemcpyHostToDevice, s));
    MBD_HIP(hipMemcpyAsync(h->om_at.p, omega, sizeof(double) * N, hipMemcpyHostToDevice, s));
    MBD_HIP(hipMemcpyAsync(h->reff.p, reff, sizeof(double) * N, hipMemcpyHostToDevice, s));
    const long nm = 3L * N * h->ncell;
    h->C.ensure((size_t)nm * nm);
    cfdm_build(s, N, h->ncell, h->xyz.p, h->cell.p, h->lat_d.p, h->nimg_cfdm, h->nimg_cfdm / 2,
               h->img_cfdm.p, h->rc_cfdm / kBohr, h->beta, h->ext_alpha.p, h->om_at.p,
               h->reff.p, h->C.p, nm, true);
    fetch(h, C, h->C.p, (size_t)nm * nm);
    MBD_HIP(hipStreamSynchronize(s));
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_debug_cholesky(int device, int n, int batch, const double *A, double *L, int *info) {
  return debug_cholesky<double>(device, n, batch, A, L, info);
}

int mbd_debug_cholesky_fp32(int device, int n, int batch, const float *A, float *L, int *info) {
  return debug_cholesky<float>(device, n, batch, A, L, info);
}

int mbd_debug_sym_eigvals(int device, int n, const double *A, double *w) {
  if (n <= 0) return -2;
  if (!A) return -3;
  if (!w) return -4;
  std::vector<double *> bufs;
  hipStream_t s2 = nullptr;
  hipEvent_t ev[2] = {nullptr, nullptr};
  auto alloc = [&](size_t cnt) {
    double *p = nullptr;
    MBD_HIP(hipMalloc(&p, sizeof(double) * std::max<size_t>(cnt, 1)));
    bufs.push_back(p);
    return p;
  };
  auto release = [&]() {
    (void)hipDeviceSynchronize();
    for (auto *p : bufs) (void)hipFree(p);
    for (auto e : ev)
      if (e) (void)hipEventDestroy(e);
    if (s2) (void)hipStreamDestroy(s2);
  };
  try {
    MBD_HIP(hipSetDevice(device));
    // full symmetric copy from the lower triangle
    std::vector<double> full((size_t)n * n);
    for (int c = 0; c < n; ++c)
      for (int r = c; r < n; ++r) full[r + (size_t)c * n] = full[c + (size_t)r * n] = A[r + (size_t)c * n];
    double *dA = alloc((size_t)n * n);
    MBD_HIP(hipMemcpy(dA, full.data(), sizeof(double) * full.size(), hipMemcpyHostToDevice));
    TrdWork wk;
    wk.VW = alloc((size_t)n * 3 * kTrdNB);
    wk.ldv = n;
    wk.tau = alloc(n);
    wk.d = alloc(n);
    wk.e = alloc(n);
    wk.alpha = alloc(kTrdNB);
    wk.pald = n / 64 + 2;
    wk.pa = alloc((size_t)wk.pald * kTrdQuant);
    wk.pb = alloc((size_t)wk.pald);
    const size_t nbt = (size_t)ceil_div(n, kTrdTile);
    wk.py = alloc(nbt * nbt * kTrdTile);
    wk.qred = alloc(kTrdQred);
    wk.ps = alloc(nbt + 1);
    int abandoned = 0;
    if (eig_method(n) == 2) {
      const SbrSizes z = sbr_sizes(n);
      auto ialloc = [&](size_t cnt) {
        int *p = reinterpret_cast<int *>(alloc((cnt + 1) / 2));
        return p;
      };
      SbrWork sw{alloc(z.V), alloc(z.TR), alloc(z.TR), ialloc(z.cnt), alloc(z.X), alloc(z.Yp),
                 alloc(z.Mp), alloc((size_t)3 * kSbrB * kSbrB), ialloc(z.mcnt), alloc(z.AB),
                 ialloc(z.prog), ialloc(4), reinterpret_cast<unsigned long long *>(alloc(z.mail)),
                 ialloc(z.cq), alloc(z.cqR), wk.VW, wk.ldv, wk.d, wk.e};
      if (sbr_lookahead()) {
        sw.VW2 = alloc((size_t)n * 6 * kSbrB);
        MBD_HIP(hipStreamCreateWithFlags(&s2, hipStreamNonBlocking));
        MBD_HIP(hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
        MBD_HIP(hipEventCreateWithFlags(&ev[1], hipEventDisableTiming));
        sw.s2 = s2;
        sw.fork = ev[0];
        sw.join = ev[1];
      }
      sbr_tridiagonalize(nullptr, n, dA, n, sw);
      MBD_HIP(hipMemcpy(&abandoned, sw.flag, sizeof(int), hipMemcpyDeviceToHost));
    } else {
      tridiagonalize(nullptr, n, dA, n, wk);
    }
    double *e2 = alloc(n), *bounds = alloc(kBisectBounds), *lam = alloc(n);
    tridiag_eigvals(nullptr, n, wk.d, wk.e, e2, bounds, lam);
    MBD_HIP(hipDeviceSynchronize());
    MBD_HIP(hipMemcpy(w, lam, sizeof(double) * n, hipMemcpyDeviceToHost));
    if (abandoned) {
      release();
      return MBD_ERR_EIG;
    }
  } catch (const HipError &e) {
    release();
    return fail(nullptr, e);
  }
  release();
  return 0;
}

int mbd_debug_lu_solve(int device, int n, int batch, const double *A, double *X, int *info) {
  if (n <= 0) return -2;
  if (batch <= 0) return -3;
  if (!A) return -4;
  if (!X) return -5;
  if (!info) return -6;
  try {
    MBD_HIP(hipSetDevice(device));
    DevScratch sc;
    const long sA = (long)n * n, sX = 3L * n, sUt = (long)std::max(1, n - kLuNB) * kLuNB;
    double *dA = sc.get<double>((size_t)batch * sA);
    double *dX = sc.get<double>((size_t)batch * sX);
    double *dUt = sc.get<double>((size_t)batch * sUt);
    int *piv = sc.get<int>((size_t)batch * n);
    int *inf = sc.get<int>((size_t)batch);
    MBD_HIP(hipMemcpy(dA, A, sizeof(double) * batch * sA, hipMemcpyHostToDevice));
    MBD_HIP(hipMemset(inf, 0, sizeof(int) * batch));
    getrf_batched(nullptr, n, dA, n, sA, batch, piv, dUt, sUt, inf);
    set_rhs(nullptr, n, dX, n, sX, batch);
    getrs3_batched(nullptr, n, dA, n, sA, batch, piv, dX, n, sX);
    MBD_HIP(hipDeviceSynchronize());
    MBD_HIP(hipMemcpy(X, dX, sizeof(double) * batch * sX, hipMemcpyDeviceToHost));
    MBD_HIP(hipMemcpy(info, inf, sizeof(int) * batch, hipMemcpyDeviceToHost));
  } catch (const HipError &e) {
    return fail(nullptr, e);
  }
  return 0;
}

int mbd_debug_gemm_nt(int device, int fp32, int m, int n, int k, double alpha, const double *A,
                      const double *B, double beta, double *C) {
  if (m <= 0 || n <= 0 || k <= 0) return -3;
  if (!A || !B || !C) return -7;
  void *dA = nullptr, *dB = nullptr, *dC = nullptr;
  try {
    MBD_HIP(hipSetDevice(device));
    const size_t es = fp32 ? 4 : 8;
    MBD_HIP(hipMalloc(&dA, es * m * k));
    MBD_HIP(hipMalloc(&dB, es * n * k));
    MBD_HIP(hipMalloc(&dC, es * m * n));
    if (fp32) {
      std::vector<float> a(A, A + (size_t)m * k), b(B, B + (size_t)n * k), c(C, C + (size_t)m * n);
      MBD_HIP(hipMemcpy(dA, a.data(), 4 * a.size(), hipMemcpyHostToDevice));
      MBD_HIP(hipMemcpy(dB, b.data(), 4 * b.size(), hipMemcpyHostToDevice));
      MBD_HIP(hipMemcpy(dC, c.data(), 4 * c.size(), hipMemcpyHostToDevice));
      gemm_nt(nullptr, false, m, n, k, (float)alpha, (const float *)dA, m, 0, (const float *)dB,
              n, 0, (float)beta, (float *)dC, m, 0, 1);
      MBD_HIP(hipDeviceSynchronize());
      MBD_HIP(hipMemcpy(c.data(), dC, 4 * c.size(), hipMemcpyDeviceToHost));
      for (size_t q = 0; q < c.size(); ++q) C[q] = c[q];
    } else {
      MBD_HIP(hipMemcpy(dA, A, 8 * (size_t)m * k, hipMemcpyHostToDevice));
      MBD_HIP(hipMemcpy(dB, B, 8 * (size_t)n * k, hipMemcpyHostToDevice));
      MBD_HIP(hipMemcpy(dC, C, 8 * (size_t)m * n, hipMemcpyHostToDevice));
      gemm_nt(nullptr, false, m, n, k, alpha, (const double *)dA, m, 0, (const double *)dB, n, 0,
              beta, (double *)dC, m, 0, 1);
      MBD_HIP(hipDeviceSynchronize());
      MBD_HIP(hipMemcpy(C, dC, 8 * (size_t)m * n, hipMemcpyDeviceToHost));
    }
  } catch (const HipError &e) {
    if (dA) (void)hipFree(dA);
    if (dB) (void)hipFree(dB);
    if (dC) (void)hipFree(dC);
    return fail(nullptr, e);
  }
  (void)hipFree(dA);
  (void)hipFree(dB);
  (void)hipFree(dC);
  return 0;
}

}  // extern "C"

namespace {
__global__ __launch_bounds__(256) void k_copy_probe(const float4 *__restrict__ src,
                                                     float4 *__restrict__ dst, long n) {
  for (long q = (long)blockIdx.x * blockDim.x + threadIdx.x; q < n; q += (long)gridDim.x * blockDim.x)
    dst[q] = src[q];
}
}  // namespace

extern "C" int mbd_debug_copy(int device, long n_bytes, double *ms) {
  if (n_bytes <= 0 || n_bytes % 16) return -2;
  void *src = nullptr, *dst = nullptr;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  int rc = 0;
  try {
    MBD_HIP(hipSetDevice(device));
    MBD_HIP(hipMalloc(&src, n_bytes));
    MBD_HIP(hipMalloc(&dst, n_bytes));
    MBD_HIP(hipMemset(src, 0, n_bytes));
    MBD_HIP(hipEventCreate(&e0));
    MBD_HIP(hipEventCreate(&e1));
    const long n = n_bytes / 16;
    MBD_HIP(hipEventRecord(e0, nullptr));
    hipLaunchKernelGGL(k_copy_probe, dim3(8192), dim3(256), 0, nullptr, (const float4 *)src,
                       (float4 *)dst, n);
    MBD_LAUNCH_CHECK();
    MBD_HIP(hipEventRecord(e1, nullptr));
    MBD_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    MBD_HIP(hipEventElapsedTime(&t, e0, e1));
    if (ms) *ms = t;
  } catch (const HipError &e) {
    rc = fail(nullptr, e);
  }
  if (e0) (void)hipEventDestroy(e0);
  if (e1) (void)hipEventDestroy(e1);
  if (src) (void)hipFree(src);
  if (dst) (void)hipFree(dst);
  return rc;
}

// ---------------------------------------------------------------------------
// Batched molecules.
namespace {

int batch_default_config(int nmax) {
  const int pref[] = {2, 0};  // {32,256,1}, {16,256,1}
  for (int c : pref)
    if (batch_lds_bytes(kBatchConfigs[c], nmax)) return c;
  return -1;
}

// The persistent kernel over the molecules of b.ord[first ...].
BatchArgs batch_args(mbd_handle *h, int mode, int first) {
  auto &b = h->bt;
  BatchArgs a;
  a.nmol = b.nmol;
  a.ntask = (b.nmol - first) * kNumFreq;
  a.nmax = b.size[first];
  a.S = batch_lds_stride(a.nmax);
  a.natoms = b.natoms;
  a.mode = mode == MBD_MODE_FP64 ? 0 : 1;
  a.off = b.off.p;
  a.order = b.order.p + first;
  a.xyz = b.xyz.p;
  a.hirsh = b.hirsh.p;
  a.a0 = b.a0.p;
  a.c60 = b.c60.p;
  a.r0 = b.r0.p;
  a.omega = h->omega.p;
  a.weight = h->weight.p;
  a.beta = b.beta;
  a.rc_scs = b.rc_scs;
  a.rc_cfdm = b.rc_cfdm;
  a.work = b.work.p;
  a.slot_bytes = (long)batch_slot_bytes(a.nmax);
  a.alpha = b.alpha.p;
  a.c6 = b.c6.p;
  a.energy = b.energy.p;
  a.c6_mol = b.c6_mol.p;
  a.stat = b.stat.p;
  a.resid = b.resid.p;
  a.counter = b.counter.p;
  a.phase = (unsigned long long *)b.phase.p;
  return a;
}

// Molecules that the launches over all of them take: the large ones, unless
// MBD_EIG_METHOD asks for eigenvalues.
int batch_first(const mbd_handle *h) { return use_logdet() ? h->bt.nlarge : 0; }
// The same, with room for the others in the persistent kernel's slots (a
// change of MBD_EIG_METHOD since mbd_batch_set can ask for more; the captured
// launches hold the old address).
int batch_room(mbd_handle *h) {
  auto &b = h->bt;
  const int first = batch_first(h);
  const size_t need = first < b.nmol ? 2 * (size_t)b.ncu * batch_slot_bytes(b.size[first]) : 0;
  if (need > b.work.n) {
    MBD_HIP(hipStreamSynchronize(h->stream));
    batch_drop_graphs(h);
    b.work.ensure(need);
  }
  return first;
}

// Counters and per-molecule statistics to zero.
void batch_clear(mbd_handle *h) {
  auto &b = h->bt;
  batch_zero(h->stream, b.counter.p, 1 + b.nmol);
  batch_zero(h->stream, b.stat.p, 4 * b.nmol);
  batch_zero(h->stream, (int *)b.resid.p, 2 * b.nmol);
  batch_zero(h->stream, b.phase.p, 2 * kBatchPhases);
}

// The persistent kernel over the molecules from `first` on.
void batch_small(mbd_handle *h, hipStream_t s, int mode, int cfg, int first) {
  const BatchConfig &c = kBatchConfigs[cfg];
  if (first < h->bt.nmol) batch_launch(s, c, batch_args(h, mode, first), h->bt.ncu * c.per_cu);
}

// The first `count` molecules of the order by launches over all of them, in
// chunks within the SCS stage's memory budget; energies into `e` (by
// molecule).  Appends to `redo` those that the persistent kernel has to take:
// a failed factor, a refinement that did not converge, eigenvalues that the
// log-determinants do not cover, or no memory.
template <typename T>
void batch_large_chunk(mbd_handle *h, int m0, int m1, double *e, std::vector<int> &redo) {
  auto &b = h->bt;
  hipStream_t s = h->stream;
  const int nm = m1 - m0, NA = b.natoms, nmax = b.size[m0];
  std::vector<MolInfo> info(nm);
  long na = 0, nc = 0, ni = 0;
  for (int q = 0; q < nm; ++q) {
    const int n = b.size[m0 + q], id = b.ord[m0 + q];
    MolInfo &mi = info[q];
    mi = MolInfo{n, mol_ld(n), b.first[id], id, na, nc, ni};
    na += (long)kNumFreq * n * mi.ld;
    nc += (long)n * mi.ld;
    ni += kNumFreq * mol_inv_size(n);
  }
  const int nmat = nm * kNumFreq, nhi = ceil_div(nmax, 64);
  b.wA.ensure(na);
  b.wL.ensure(sizeof(T) * na);
  b.wC.ensure(nc);
  b.wInv.ensure(ni);
  b.wFac.ensure(nmat);
  b.wRedo.ensure(b.nmol);
  b.wHi.ensure((size_t)nm * (nhi + 2));
  b.wG.ensure(nmat);
  b.wShift.ensure(nmat);
  b.wInfo.ensure(sizeof(MolInfo) * nm);
  b.wMat.ensure(sizeof(MolMat) * nmat);
  const MolInfo *mols = (const MolInfo *)b.wInfo.p;
  const MolMat *mats = (const MolMat *)b.wMat.p;
  double *aw = b.par.p, *sg = aw + (long)kNumFreq * NA, *rv = sg + (long)kNumFreq * NA, *om = rv + NA,
         *rf = om + NA, *w2 = b.wHi.p + (size_t)nm * nhi;
  MBD_HIP(hipMemcpyAsync(b.wInfo.p, info.data(), sizeof(MolInfo) * nm, hipMemcpyHostToDevice, s));
  batch_zero(s, b.wFac.p, nmat);
  batch_zero(s, b.wRedo.p, b.nmol);

  // SCS at every grid point
  auto above = [&](int k) {  // matrices of order above k
    return kNumFreq * (int)(std::partition_point(info.begin(), info.end(),
                                                 [&](const MolInfo &m) { return m.n > k; }) - info.begin());
  };
  T *L = (T *)b.wL.p, *inv = (T *)b.wInv.p;
  scs_build_mols<T>(s, nm, nmax, NA, mols, b.xyz.p, b.rc_scs, b.beta, aw, sg, rv, b.wA.p, L);
  potrf_mols<T>(s, nmax, mols, nullptr, above, L, inv, b.wFac.p);
  solve_mols<T>(s, nm, nmax, NA, mols, b.wA.p, L, inv, b.wFac.p, sizeof(T) == 4 ? kBatchTol : INFINITY,
                sizeof(T) == 4 ? kBatchMaxIter : 0, b.alpha.p, b.stat.p, b.resid.p, b.wRedo.p);

  // coupled matrices and their bounds
  params_mols(s, nm, NA, mols, h->weight.p, b.a0.p, b.r0.p, b.alpha.p, b.c6.p, om, rf, b.c6_mol.p, w2);
  cfdm_build_mols(s, nm, nmax, mols, b.xyz.p, b.rc_cfdm, b.beta, b.alpha.p, om, rf, b.wC.p);
  ld_bounds_mols(s, nm, nmax, mols, b.wC.p, b.wHi.p);
  std::vector<double> hi((size_t)nm * (nhi + 2));
  std::vector<int> bad(b.nmol);
  MBD_HIP(hipMemcpyAsync(hi.data(), b.wHi.p, 8 * hi.size(), hipMemcpyDeviceToHost, s));
  MBD_HIP(hipMemcpyAsync(bad.data(), b.wRedo.p, 4 * bad.size(), hipMemcpyDeviceToHost, s));
  MBD_HIP(hipStreamSynchronize(s));
  std::vector<int> todo;  // molecules of the chunk without an energy
  for (int q = 0; q < nm; ++q) {
    if (bad[info[q].id])
      redo.push_back(info[q].id);
    else
      todo.push_back(q);
  }
  // energies, as in energy_by_logdet: two guesses of the lowest eigenvalue
  for (double frac : {0.3, 0.03}) {
    std::vector<MolMat> mat;
    std::vector<double> shift, wt;
    std::vector<int> order, left;
    for (int q : todo) {
      double top = hi[(size_t)nm * nhi + 2 * q + 1];
      bool ok = std::isfinite(top);
      for (int k = 0; k < ceil_div(info[q].n, 64); ++k) {
        const double v = hi[(size_t)q * nhi + k];
        ok = ok && std::isfinite(v);
        top = std::max(top, v);
      }
      LdNodes nd;
      if (!ok || !ld_nodes(frac * hi[(size_t)nm * nhi + 2 * q], top, nd)) {
        left.push_back(q);
        continue;
      }
      for (int k = 0; k <= nd.n; ++k) {
        mat.push_back(MolMat{q, k});
        shift.push_back(nd.t[k]);
        wt.push_back(nd.w[k]);
        order.push_back(info[q].n);
      }
    }
    const int cnt = (int)mat.size();
    if (cnt) {
      MBD_HIP(hipMemcpyAsync(b.wMat.p, mat.data(), sizeof(MolMat) * cnt, hipMemcpyHostToDevice, s));
      MBD_HIP(hipMemcpyAsync(b.wShift.p, shift.data(), 8 * cnt, hipMemcpyHostToDevice, s));
      batch_zero(s, b.wFac.p, nmat);
      ld_shift_mols(s, cnt, order[0], mols, mats, b.wShift.p, b.wC.p, b.wA.p);
      potrf_mols<double>(s, order[0], mols, mats,
                         [&](int k) {
                           return (int)(std::partition_point(order.begin(), order.end(),
                                                             [&](int n) { return n > k; }) - order.begin());
                         },
                         b.wA.p, b.wInv.p, b.wFac.p);
      ld_sums_mols(s, cnt, mols, mats, b.wShift.p, b.wA.p, om, b.wG.p);
      std::vector<double> g(cnt);
      std::vector<int> fac(cnt);
      MBD_HIP(hipMemcpyAsync(g.data(), b.wG.p, 8 * cnt, hipMemcpyDeviceToHost, s));
      MBD_HIP(hipMemcpyAsync(fac.data(), b.wFac.p, 4 * cnt, hipMemcpyDeviceToHost, s));
      MBD_HIP(hipStreamSynchronize(s));
      for (int k = 0; k < cnt;) {
        const int q = mat[k].mol;
        double sum = 0.0;
        bool ok = true;
        for (; k < cnt && mat[k].mol == q; ++k) {
          sum += wt[k] != 0.0 ? wt[k] * g[k] : 0.0;
          ok = ok && fac[k] == 0;
        }
        if (ok && std::isfinite(sum))
          e[info[q].id] = sum;
        else
          left.push_back(q);
      }
    }
    todo.swap(left);
    std::sort(todo.begin(), todo.end());
    if (todo.empty()) break;
  }
  for (int q : todo) redo.push_back(info[q].id);
}

void batch_large(mbd_handle *h, int mode, int count, double *e, std::vector<int> &redo) {
  auto &b = h->bt;
  const int NA = b.natoms;
  const size_t es = mode == MBD_MODE_FP64 ? 8 : 4, budget = mem_budget();
  int m0 = 0;
  try {
    b.par.ensure((size_t)(2 * kNumFreq + 3) * NA);
    double *aw = b.par.p, *sg = aw + (long)kNumFreq * NA, *rv = sg + (long)kNumFreq * NA;
    atom_params(h->stream, NA, kNumFreq, h->omega.p, b.hirsh.p, b.a0.p, b.c60.p, b.r0.p, aw, sg, rv);
    while (m0 < count) {
      int m1 = m0;
      for (size_t bytes = 0; m1 < count; ++m1) {
        const int n = b.size[m1];
        bytes += (size_t)n * mol_ld(n) * (kNumFreq * (8 + es) + 8) + 8 * (size_t)kNumFreq * mol_inv_size(n);
        if (bytes > budget && m1 > m0) break;
      }
      if (mode == MBD_MODE_FP64)
        batch_large_chunk<double>(h, m0, m1, e, redo);
      else
        batch_large_chunk<float>(h, m0, m1, e, redo);
      m0 = m1;
    }
  } catch (const HipError &x) {
    if (x.err != hipErrorOutOfMemory) throw;
    (void)hipGetLastError();
    for (; m0 < count; ++m0) redo.push_back(b.ord[m0]);
  }
}

// Molecules of `redo` by the persistent kernel, their statistics anew.
void batch_again(mbd_handle *h, int mode, std::vector<int> &redo) {
  auto &b = h->bt;
  hipStream_t s = h->stream;
  std::vector<int> rank(b.nmol);
  for (int k = 0; k < b.nmol; ++k) rank[b.ord[k]] = k;
  std::sort(redo.begin(), redo.end(), [&](int x, int y) { return rank[x] < rank[y]; });
  redo.erase(std::unique(redo.begin(), redo.end()), redo.end());
  const int first = rank[redo[0]];
  BatchArgs a = batch_args(h, mode, first);
  a.ntask = (int)redo.size() * kNumFreq;
  const int cfg = batch_default_config(a.nmax), grid = std::min(b.ncu * kBatchConfigs[cfg].per_cu, a.ntask);
  b.again.ensure((size_t)grid * a.slot_bytes);
  b.wList.ensure(redo.size());
  MBD_HIP(hipMemcpyAsync(b.wList.p, redo.data(), sizeof(int) * redo.size(), hipMemcpyHostToDevice, s));
  reset_mols(s, (int)redo.size(), b.wList.p, b.counter.p, b.stat.p, b.resid.p);
  a.work = b.again.p;
  a.order = b.wList.p;
  batch_prepare(kBatchConfigs[cfg], a.nmax);
  batch_launch(s, kBatchConfigs[cfg], a, grid);
  MBD_HIP(hipStreamSynchronize(s));  // the list is the caller's
  std::sort(redo.begin(), redo.end());
}

// One pass over the batch, `small(stream)` launching the persistent kernel:
// energies of the first `first` molecules into e, those of `redo` (sorted)
// and of the others left to the device array.  With molecules of both kinds
// the persistent kernel runs on a stream of its own beside the launches for
// the large ones: they share no results, and it leaves half of each CU idle.
template <typename F>
void batch_pass(mbd_handle *h, int mode, int first, F small, std::vector<double> &e, std::vector<int> &redo) {
  auto &b = h->bt;
  batch_clear(h);
  if (!first || first == b.nmol) {
    if (!first) small(h->stream);
  } else {
    if (!b.side) {
      MBD_HIP(hipStreamCreateWithFlags(&b.side, hipStreamNonBlocking));
      MBD_HIP(hipEventCreateWithFlags(&b.fork, hipEventDisableTiming));
      MBD_HIP(hipEventCreateWithFlags(&b.join, hipEventDisableTiming));
    }
    MBD_HIP(hipEventRecord(b.fork, h->stream));
    MBD_HIP(hipStreamWaitEvent(b.side, b.fork, 0));
    small(b.side);
    MBD_HIP(hipEventRecord(b.join, b.side));
  }
  if (!first) return;
  e.assign(b.nmol, 0.0);
  try {
    batch_large(h, mode, first, e.data(), redo);
  } catch (...) {
    if (b.side) (void)hipStreamSynchronize(b.side);
    throw;
  }
  if (first < b.nmol) MBD_HIP(hipStreamWaitEvent(h->stream, b.join, 0));
  if (!redo.empty()) batch_again(h, mode, redo);
}

}  // namespace

extern "C" {

int mbd_batch_config(int index, int *nb, int *nt, int *per_cu) {
  if (index < 0 || index >= kBatchNumConfigs) return -1;
  if (nb) *nb = kBatchConfigs[index].nb;
  if (nt) *nt = kBatchConfigs[index].nt;
  if (per_cu) *per_cu = kBatchConfigs[index].per_cu;
  return 0;
}

int mbd_batch_set(mbd_handle *h, int nmol, const int *offsets, const double *xyz,
                  const double *hirshfeld, const double *alpha0, const double *c6_0,
                  const double *r0, double beta, double rc_scs, double rc_cfdm) {
  if (!h) return -1;
  if (nmol <= 0) return -2;
  if (!offsets) return -3;
  if (!xyz) return -4;
  if (!hirshfeld) return -5;
  if (!alpha0) return -6;
  if (!c6_0) return -7;
  if (!r0) return -8;
  if (offsets[0] != 0) return -3;
  int nmax = 0;
  for (int m = 0; m < nmol; ++m) {
    const int na = offsets[m + 1] - offsets[m];
    if (na <= 0) return -3;
    nmax = std::max(nmax, 3 * na);
  }
  if (batch_default_config(nmax) < 0) {
    char buf[160];
    snprintf(buf, sizeof buf,
             "batched kernel holds molecules up to 3N = %d in LDS; largest here is 3N = %d",
             [] {
               int lo = 3;
               while (batch_default_config(lo + 3) >= 0) lo += 3;
               return lo;
             }(),
             nmax);
    h->err = buf;
    return MBD_ERR_TOOBIG;
  }
  try {
    MBD_HIP(hipSetDevice(h->device));
    MBD_HIP(hipStreamSynchronize(h->stream));
    batch_drop_graphs(h);
    auto &b = h->bt;
    b.nmol = nmol;
    b.natoms = offsets[nmol];
    b.nmax = nmax;
    b.beta = beta;
    b.rc_scs = rc_scs / kBohr;
    b.rc_cfdm = rc_cfdm / kBohr;
    MBD_HIP(hipDeviceGetAttribute(&b.ncu, hipDeviceAttributeMultiprocessorCount, h->device));
    std::vector<int> order(nmol);
    for (int m = 0; m < nmol; ++m) order[m] = m;
    std::stable_sort(order.begin(), order.end(), [&](int x, int y) {
      return offsets[x + 1] - offsets[x] > offsets[y + 1] - offsets[y];
    });
    const int NA = b.natoms;
    auto upd = [&](DevBuf<double> &d, const double *src, size_t cnt) {
      d.ensure(cnt);
      MBD_HIP(hipMemcpyAsync(d.p, src, sizeof(double) * cnt, hipMemcpyHostToDevice, h->stream));
    };
    auto upi = [&](DevBuf<int> &d, const int *src, size_t cnt) {
      d.ensure(cnt);
      MBD_HIP(hipMemcpyAsync(d.p, src, sizeof(int) * cnt, hipMemcpyHostToDevice, h->stream));
    };
    upi(b.off, offsets, nmol + 1);
    upi(b.order, order.data(), nmol);
    upd(b.xyz, xyz, 3L * NA);
    upd(b.hirsh, hirshfeld, NA);
    upd(b.a0, alpha0, NA);
    upd(b.c60, c6_0, NA);
    upd(b.r0, r0, NA);
    b.alpha.ensure((size_t)kNumFreq * NA);
    b.c6.ensure(NA);
    b.energy.ensure(nmol);
    b.c6_mol.ensure(nmol);
    b.resid.ensure(nmol);
    b.counter.ensure(1 + nmol);
    b.stat.ensure(4 * nmol);
    b.phase.ensure(2 * kBatchPhases);
    b.ord = order;
    b.first.assign(offsets, offsets + nmol);
    b.size.resize(nmol);
    for (int k = 0; k < nmol; ++k) b.size[k] = 3 * (offsets[order[k] + 1] - offsets[order[k]]);
    b.nlarge = (int)(std::partition_point(b.size.begin(), b.size.end(),
                                          [](int n) { return n > kMolMinOrder; }) - b.size.begin());
    batch_room(h);
    MBD_HIP(hipStreamSynchronize(h->stream));
    if (b.cfg >= 0 && !batch_lds_bytes(kBatchConfigs[b.cfg], nmax)) b.cfg = -1;
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_batch_set_config(mbd_handle *h, int index) {
  if (!h) return -1;
  if (index < -1 || index >= kBatchNumConfigs) return -2;
  if (!h->bt.nmol) return MBD_ERR_NOSYS;
  if (index >= 0 && !batch_lds_bytes(kBatchConfigs[index], h->bt.nmax)) return MBD_ERR_TOOBIG;
  h->bt.cfg = index;
  return 0;
}

int mbd_batch_tune(mbd_handle *h, int mode, int reps, double *times_ms, int *best) {
  if (!h) return -1;
  if (mode != MBD_MODE_FP64 && mode != MBD_MODE_MIXED) return -2;
  if (reps <= 0) return -3;
  if (!h->bt.nmol) return MBD_ERR_NOSYS;
  try {
    MBD_HIP(hipSetDevice(h->device));
    int arg = -1;
    double tbest = 0.0;
    const int first = batch_room(h);
    for (int c = 0; c < kBatchNumConfigs; ++c) {
      double t = -1.0;
      if (batch_lds_bytes(kBatchConfigs[c], h->bt.nmax)) {
        batch_prepare(kBatchConfigs[c], h->bt.nmax);
        auto go = [&] {
          std::vector<double> e;
          std::vector<int> redo;
          batch_pass(h, mode, first, [&](hipStream_t s) { batch_small(h, s, mode, c, first); }, e, redo);
        };
        go();  // warm-up
        Timer tm;
        tm.start(h->stream);
        for (int r = 0; r < reps; ++r) go();
        tm.stop(h->stream);
        t = tm.ms() / reps;
        if (arg < 0 || t < tbest) {
          arg = c;
          tbest = t;
        }
      }
      if (times_ms) times_ms[c] = t;
    }
    h->bt.cfg = arg;
    if (best) *best = arg;
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_batch_run(mbd_handle *h, int mode, double *energy, double *alpha_eff, double *c6_eff,
                  double *c6_mol, double *alpha_all, int *stat, mbd_batch_diag *d) {
  if (!h) return -1;
  if (mode != MBD_MODE_FP64 && mode != MBD_MODE_MIXED) return -2;
  if (!energy) return -3;
  auto &b = h->bt;
  if (!b.nmol) return MBD_ERR_NOSYS;
  try {
    MBD_HIP(hipSetDevice(h->device));
    const int cfg = b.cfg >= 0 ? b.cfg : batch_default_config(b.nmax);
    const int mi = mode == MBD_MODE_FP64 ? 0 : 1, first = batch_room(h);
    if (first < b.nmol && (!b.exec[mi] || b.exec_cfg[mi] != cfg || b.exec_first[mi] != first)) {
      if (b.exec[mi]) (void)hipGraphExecDestroy(b.exec[mi]);
      b.exec[mi] = nullptr;
      batch_prepare(kBatchConfigs[cfg], b.nmax);
      hipGraph_t g = nullptr;
      MBD_HIP(hipStreamBeginCapture(h->stream, hipStreamCaptureModeRelaxed));
      try {
        batch_small(h, h->stream, mode, cfg, first);
      } catch (const HipError &) {
        (void)hipStreamEndCapture(h->stream, &g);
        if (g) (void)hipGraphDestroy(g);
        throw;
      }
      MBD_HIP(hipStreamEndCapture(h->stream, &g));
      const hipError_t ie = hipGraphInstantiate(&b.exec[mi], g, nullptr, nullptr, 0);
      (void)hipGraphDestroy(g);
      MBD_HIP(ie);
      b.exec_cfg[mi] = cfg;
      b.exec_first[mi] = first;
    }
    std::vector<double> el;
    std::vector<int> redo;
    Timer tm;
    tm.start(h->stream);
    batch_pass(h, mode, first, [&](hipStream_t s) { MBD_HIP(hipGraphLaunch(b.exec[mi], s)); }, el, redo);
    tm.stop(h->stream);
    const double ms = tm.ms();
    const int NA = b.natoms, nm = b.nmol;
    std::vector<int> st(4 * (size_t)nm);
    std::vector<double> res(nm);
    auto get = [&](void *dst, const void *src, size_t bytes) {
      MBD_HIP(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, h->stream));
    };
    get(energy, b.energy.p, sizeof(double) * nm);
    get(st.data(), b.stat.p, sizeof(int) * 4 * nm);
    get(res.data(), b.resid.p, sizeof(double) * nm);
    if (alpha_eff) get(alpha_eff, b.alpha.p, sizeof(double) * NA);
    if (alpha_all) get(alpha_all, b.alpha.p, sizeof(double) * kNumFreq * NA);
    if (c6_eff) get(c6_eff, b.c6.p, sizeof(double) * NA);
    if (c6_mol) get(c6_mol, b.c6_mol.p, sizeof(double) * nm);
    MBD_HIP(hipStreamSynchronize(h->stream));
    for (int k = 0; k < first; ++k)
      if (!std::binary_search(redo.begin(), redo.end(), b.ord[k])) energy[b.ord[k]] = el[b.ord[k]];
    if (stat) std::copy(st.begin(), st.end(), stat);
    if (d) {
      const BatchConfig &c = kBatchConfigs[cfg];
      d->config = cfg;
      d->nb = c.nb;
      d->nt = c.nt;
      d->grid = b.ncu * c.per_cu;
      d->fallbacks = d->max_iters = d->n_failed = d->n_negative = 0;
      d->max_residual = 0.0;
      for (int m = 0; m < nm; ++m) {
        d->n_failed += st[4 * m] != 0;
        d->n_negative += st[4 * m + 1];
        d->max_iters = std::max(d->max_iters, st[4 * m + 2]);
        d->fallbacks += st[4 * m + 3];
        d->max_residual = std::max(d->max_residual, res[m]);
      }
      d->t_ms = ms;
      unsigned long long ph[kBatchPhases];
      MBD_HIP(hipMemcpy(ph, b.phase.p, sizeof ph, hipMemcpyDeviceToHost));
      int khz = 0;
      MBD_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, h->device));
      for (int k = 0; k < kBatchPhases; ++k) d->phase_ms[k] = khz > 0 ? (double)ph[k] / khz : 0.0;
    }
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

int mbd_batch_run_noalloc(mbd_handle *h, void *stream, int mode, int nmol, int natoms,
                          int max_atoms, const int *offsets, const double *xyz,
                          const double *hirshfeld, const double *alpha0, const double *c6_0,
                          const double *r0, double beta, double rc_scs, double rc_cfdm,
                          double *energy, double *alpha_all, double *c6_eff, double *c6_mol,
                          int *stat) {
  if (!h) return -1;
  if (mode != MBD_MODE_FP64 && mode != MBD_MODE_MIXED) return -3;
  if (nmol <= 0) return -4;
  if (natoms < nmol) return -5;
  if (max_atoms <= 0) return -6;
  if (!offsets || !xyz || !hirshfeld || !alpha0 || !c6_0 || !r0) return -7;
  if (!energy || !alpha_all || !c6_eff || !c6_mol || !stat) return -15;
  if (max_atoms > kNaMaxAtoms || nmol > kNaMaxMol) {
    char buf[160];
    snprintf(buf, sizeof buf,
             "mbd_batch_run_noalloc holds molecules of up to %d atoms and %d molecules per call "
             "(asked: %d atoms, %d molecules)",
             kNaMaxAtoms, kNaMaxMol, max_atoms, nmol);
    h->err = buf;
    return MBD_ERR_TOOBIG;
  }
  try {
    MBD_HIP(hipSetDevice(h->device));
    char *sc = h->device >= 0 && h->device < kNaMaxDevices ? (char *)na_ptr[h->device] : nullptr;
    if (!sc) {
      h->err = "mbd_batch_run_noalloc: no scratch address for this device";
      return MBD_ERR_HIP;
    }
    hipStream_t s = stream ? (hipStream_t)stream : h->stream;
    const int nmax = 3 * max_atoms;
    const int cfg = batch_default_config(nmax);
    const BatchConfig &c = kBatchConfigs[cfg];
    if (batch_slot_bytes(nmax) > kNaSlotBytes) return MBD_ERR_TOOBIG;
    int ncu = 0;
    MBD_HIP(hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, h->device));
    const int grid = std::max(1, std::min(ncu, kNaSlots));
    BatchArgs a;
    a.nmol = nmol;
    a.ntask = nmol * kNumFreq;
    a.nmax = nmax;
    a.S = batch_lds_stride(nmax);
    a.natoms = natoms;
    a.mode = mode == MBD_MODE_FP64 ? 0 : 1;
    a.off = offsets;
    a.order = nullptr;
    a.xyz = xyz;
    a.hirsh = hirshfeld;
    a.a0 = alpha0;
    a.c60 = c6_0;
    a.r0 = r0;
    a.omega = h->omega.p;
    a.weight = h->weight.p;
    a.beta = beta;
    a.rc_scs = rc_scs / kBohr;
    a.rc_cfdm = rc_cfdm / kBohr;
    a.work = sc;
    a.slot_bytes = (long)kNaSlotBytes;
    a.alpha = alpha_all;
    a.c6 = c6_eff;
    a.energy = energy;
    a.c6_mol = c6_mol;
    a.stat = stat;
    a.resid = (double *)(sc + kNaResidOff);
    a.counter = (int *)(sc + kNaCountOff);
    a.phase = (unsigned long long *)(sc + kNaPhaseOff);
    // counters, statistics and residual maxima start at zero (fill kernels)
    batch_zero(s, a.counter, 1 + nmol);
    batch_zero(s, stat, 4 * nmol);
    batch_zero(s, (int *)a.resid, 2 * nmol);
    batch_zero(s, (int *)a.phase, 2 * kBatchPhases);
    batch_prepare(c, nmax);
    batch_launch(s, c, a, grid);
  } catch (const HipError &e) {
    return fail(h, e);
  }
  return 0;
}

}  // extern "C"
