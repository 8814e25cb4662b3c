// Device-side data structures and kernel launchers of the TDVP path.
#pragma once

#include "qca_common.hpp"

#include <vector>

namespace qca {

// Maximum Krylov dimension (one wave holds the tridiagonal matrix).
constexpr int LZ_MAXK = 64;
// LanczosCtrl::hit_limit: the last vector's error estimate was above the tolerance,
// or the start or a matvec was not finite.
constexpr int LZ_NON_FINITE = 2;

// Lanczos control block, device resident.  Written by the reduction kernels,
// read back by the host only once per exponential.
struct LanczosCtrl {
  double beta0;
  double err;
  int done;
  int m;
  int zero;
  int hit_limit;
  double alpha[LZ_MAXK];
  double beta[LZ_MAXK];
  c128 z[LZ_MAXK];
};

// Workspace of one Lanczos exponential (vectors of length <= max_n).
struct LanczosWork {
  LanczosCtrl* ctrl = nullptr;
  c128* V = nullptr;      // [LZ_MAXK][max_n] Krylov basis
  c128* w64 = nullptr;    // [max_n] orthogonalised residual
  c128* part = nullptr;   // [max_blocks] partial sums of <V_j, w>
  c128* part2 = nullptr;  // [LZ_MAXK][max_blocks] partial projections on the basis, and the norm's
  double* part_norm = nullptr;
  c128* coef = nullptr;   // [LZ_MAXK] <V_j, w> of each iteration
  long max_n = 0;
  int max_blocks = 0;
  int max_m = LZ_MAXK;    // Krylov dimension limit of this workspace (<= LZ_MAXK)
};

// MPO tensor in compressed sparse rows over output channels: a channel is
// (physical, MPO bond) and the value of each stored entry is a W element.
template <typename T>
struct WSparseDev {
  int* rowptr = nullptr;
  int* col = nullptr;
  int* outv = nullptr;   // MPO bond index of each nonzero's row (row % group_rows)
  cplx<T>* val = nullptr;
  int nout = 0, nin = 0, nnz = 0;
  int group_rows = 0;    // rows per output physical index (the output MPO dimension)
  int group_max = 0;     // most nonzeros in any group of group_rows rows
  int ngroups = 0;       // nout / group_rows when at most SEG_STARTS_MAX, else 0
  int group_start[SEG_STARTS_MAX + 1] = {};  // rowptr[g * group_rows], g <= ngroups
  unsigned long long used = 0;   // columns with an entry, as bits (0: more than 64 columns)
};
// Fills ngroups, group_start and used of w from the host row pointer and columns.
template <typename T>
inline void set_group_starts(WSparseDev<T>& w, const std::vector<int>& rowptr, const std::vector<int>& col, int nin,
                             int group_rows) {
  w.used = 0;
  if (nin <= 64)
    for (int c : col) w.used |= 1ull << c;
  const int nout = (int)rowptr.size() - 1;
  w.ngroups = 0;
  if (group_rows <= 0 || nout % group_rows != 0 || nout / group_rows > SEG_STARTS_MAX) return;
  w.ngroups = nout / group_rows;
  for (int g = 0; g <= w.ngroups; ++g) w.group_start[g] = rowptr[(size_t)g * group_rows];
}

template <typename T>
void launch_wmix(const cplx<T>* Tin, long in_stride, long nxc, int nin, cplx<T>* U, int nq,
                 int Dout, const WSparseDev<T>& w, hipStream_t s, const int* skip = nullptr);

void launch_convert_c128_c64(const c128* in, c64* out, long n, hipStream_t s,
                             const int* skip = nullptr);
void launch_convert_c64_c128(const c64* in, c128* out, long n, hipStream_t s,
                             const int* skip = nullptr);
void launch_to_colmajor(const c128* in, c128* out, int rows, int cols, hipStream_t s);
void launch_site_to_rightqr(const c128* A, c128* X, int chil, int chir, hipStream_t s);
void launch_qr_gather_left(const c128* Q, const c128* X, c128* Anew, c128* C, int rows, int cols,
                           int qcols, int target, hipStream_t s);
void launch_qr_gather_right(const c128* Q, const c128* X, c128* Anew, c128* C, int chir, int cols,
                            int qcols, int target, hipStream_t s);
void launch_theta_to_svd(const c128* th, c128* X, int chil, int chir, int mode, hipStream_t s);
void launch_gather_isometry(const c128* X, const int* perm, const double* sigma, c128* A, int rows,
                            int chi_bond, int k, int mode, hipStream_t s);

int lanczos_nblk(long n);
const int* lanczos_done_flag(const LanczosWork& lw);
// v32 (optional): also write each new basis vector as complex64 there, the
// operand of the mixed path's next matvec.
void lanczos_begin(const c128* x, long n, LanczosWork& lw, hipStream_t s, c64* v32 = nullptr);
template <typename TW>
void lanczos_iteration_tail(const cplx<TW>* w, long n, int j, double tau, double tol,
                            LanczosWork& lw, hipStream_t s, c64* v32 = nullptr);
void lanczos_finish(long n, c128* y, LanczosWork& lw, hipStream_t s);

// ---------------------------------------------------------------- one-launch Krylov
// Longest vector of the one-workgroup exponential (8 residual elements per
// thread of 512).
constexpr long FUSED_KRYLOV_MAX_N = 4096;

// Device-side running totals of the one-launch exponentials of one engine.
struct KrylovTally {
  long matvecs[3];          // by kind: 2-site, 1-site, bond
  long limit_hits;
  long calls;
  unsigned long long ticks; // summed kernel time in wall-clock ticks
  double flops;
};

// x <- exp(-i tau H_eff) x, H_eff of `kind` (0: 2-site x[q][a][c], q = (p1,p2);
// 1: 1-site x[p][a][c]; 2: bond x[a][c]) with environments L[a][w][a*] and
// R[c][v][c*] of element type TE and the sparse MPO (forward form of the
// merged pair for kind 0, of the site for kind 1; unused for kind 2).  The
// contractions run in TE, the recurrence in FP64 whatever TE is.
template <typename TE>
struct FusedKrylovArgs {
  int kind = 0;
  int chil = 1, chir = 1;
  int Din = 1, Dout = 1;
  long n = 0;
  const cplx<TE>* L = nullptr;
  const cplx<TE>* R = nullptr;
  const int* rowptr = nullptr;
  const int* col = nullptr;
  const cplx<TE>* val = nullptr;
  int nnz = 0;                 // entries of the sparse MPO
  int group_max = 0;           // the most entries of any q' (0: not known)
  c128* x = nullptr;           // in/out, n elements
  c128* V = nullptr;           // basis, (max_m - 1) * n elements
  cplx<TE>* T1 = nullptr;      // dq * Din * chil * chir elements
  LanczosCtrl* ctrl = nullptr; // optional: m, error, limit flag of this call
  KrylovTally* tally = nullptr;// optional running totals
  double tau = 0, tol = 0;
  double flops_per_matvec = 0;
  int max_m = LZ_MAXK;
  // Filled by fused_krylov_place: byte offsets into the workgroup's LDS, whether T1
  // and the MPO, and the environments, lie there, the number of leading basis
  // vectors held there, the waves that share a tile of H_eff x (a power of two),
  // whether the result goes over T1, and for blocks whose H_eff x is taken element
  // by element the lanes that share one (a power of two; else 0).
  long offW = 0, offRow = 0, offCol = 0, offVal = 0, offL = 0, offR = 0, offV = 0;
  int t1_lds = 0, env_lds = 0, vcap = 0, parts = 1, overlay = 0, lanes = 0;
};

template <typename TE>
void launch_fused_krylov(const FusedKrylovArgs<TE>& a, hipStream_t s);

// population, rounded population and single-site entropy of n sites from their
// 2x2 density matrices; out holds 3n doubles.
void launch_observables(const c128* rho, int n, double* out, hipStream_t s);
void launch_rho(const c128* A, const c128* T, long nxb, c128* rho, hipStream_t s);

int exact_rho_blocks(int ncells);
void launch_exact_rho(const c128* psi, int ncells, double* part, c128* rho, hipStream_t s);

template <typename T>
void launch_exact_apply(const cplx<T>* psi, cplx<T>* out, int ncells, int distance, int lo, int hi,
                        hipStream_t s);
// psi <- exp(-i tau H) psi by Chebyshev series of at most CHEB_MAX_Z in tau*N
// each (a longer step is cut into equal parts).  Their tails together are below
// CHEB_TAIL * tol * |psi|: at the default tolerance below the rounding of the terms
// (cut at tol itself, the tail was most of the error: 12 to 15 cells, 2.0e-15
// relative to |psi| on average, against 2.4e-16; one or two terms more);
// returns the number of H applications.  bufa, bufb, acc: 2^ncells elements
// each; report: pinned host memory.  psi not finite: an error, psi is left as
// it was.  Returns with the stream drained.
constexpr double CHEB_MAX_Z = 512, CHEB_TAIL = 0.03;
// Basis states up to which the support of psi is told to the host, and up to which a
// set of them that H maps to itself is evolved there.
constexpr int EXACT_SUPPORT = 64;
struct ExactAmplitude {
  unsigned long long x;
  double re, im;
};
struct ExactProbe {      // device; the first two words are cleared for each call
  int bad;               // psi is not finite
  int count;             // nonzero amplitudes (some of them, where there are more than EXACT_SUPPORT)
  ExactAmplitude e[EXACT_SUPPORT];
};
struct ExactReport {     // pinned host memory, written by the device
  int word;
  ExactAmplitude e[EXACT_SUPPORT];   // the amplitudes, where word says that they fit
};
int launch_exact_expm(c128* psi, int ncells, int distance, int lo, int hi, double tau, double tol, c128* bufa,
                      c128* bufb, c128* acc, ExactProbe* probe, ExactReport* report, hipStream_t s);

// ---------------------------------------------------------------- SVD / QR
struct SvdResult {
  int k;              // truncation rank
  int nsweeps;        // Jacobi sweeps used
  int converged;
  int nsteps;         // closing steps used
  double norm_kept;   // ||s[:k]||
  double tail;        // ||s[k:]||
};

// Workspace of the Jacobi SVD (a matrix for which small_svd holds needs none of
// it but a non-null ws): device memory of at least
// jacobi_workspace_bytes(rows, cols) (control block, partial Grams, block
// rotations, matrices of the closing phase), 16 bytes of pinned host memory, and
// the sweep and closing-step counts of the previous call (the number launched
// before the first look at the device's state).
struct JacobiWork {
  void* ws = nullptr;
  size_t ws_bytes = 0;
  void* host = nullptr;
  int pred_sweeps = 4;
  int pred_newton = 3;
  // QR preconditioning: at least jacobi_precond_elems(rows, cols) complex128
  c128* pre = nullptr;
  size_t pre_elems = 0;
  // rotation threshold relative to the column norms; 0: eps * sqrt(rows)
  double tol = 0;
};

struct JacobiLayout {
  int nb = 2, kspl = 1;
  long gpart_elems = 0, j_elems = 0;
  size_t bytes = 0;
};
JacobiLayout jacobi_layout(int rows, int cols);
size_t jacobi_workspace_bytes(int max_rows, int max_cols);
size_t jacobi_precond_elems(int max_rows, int max_cols);
// One workgroup takes the whole SVD, or that of the triangle of a QR.
bool small_svd(int rows, int cols);
bool tall_svd(int rows, int cols);

// One-sided (block) Jacobi SVD of the column-major matrix X (rows x cols,
// FP64), in place.  On exit the columns are orthogonal; sigma (sorted
// descending), perm (column index of each sorted value) and the truncation
// result are written to device memory.
void launch_jacobi_svd(c128* X, int rows, int cols, double* sigma, int* perm, SvdResult* res,
                       int chi_max, double eps, int rank_cap, hipStream_t s, JacobiWork& w);

// Householder QR with LAPACK's zgeqr2/zung2r conventions (real beta, beta =
// -sign(Re alpha)*norm) of the column-major matrix M (rows x cols), in place:
// R on and above the diagonal, reflectors below it, tau[min(rows, cols)].
// Q's first qcols columns are written column-major to Q (skipped when null).
void launch_householder_qr(c128* M, int rows, int cols, c128* tau, c128* Q, int qcols,
                           hipStream_t s);
// Blocked Householder QR with LAPACK zgeqrf/zungqr semantics (same reflectors
// and signs as launch_householder_qr): M (rows <= 512 x cols, column-major) ->
// R on/above the diagonal, reflectors below; Q (rows x qcols) when Q != null.
// ws holds at least qr_workspace_elems(rows, cols) complex128.
constexpr int QR_MAX_ROWS = 512;
size_t qr_workspace_elems(int max_rows, int max_cols);
void launch_blocked_qr(c128* M, int rows, int cols, c128* Q, int qcols, c128* ws, size_t ws_elems, hipStream_t s);
// QR dispatch: the blocked version for rows <= QR_MAX_ROWS and more than one or two
// reflectors when ws is large enough, else the single-workgroup one.
void launch_qr(c128* M, int rows, int cols, c128* tau, c128* Q, int qcols, c128* ws,
               size_t ws_elems, hipStream_t s);

}  // namespace qca
