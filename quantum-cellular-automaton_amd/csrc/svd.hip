// FP64 SVD of the TDVP split (gfx950).
//
// jacobi_svd: block one-sided (Hestenes) Jacobi on the columns of a
// column-major matrix X, with the rotations of each block pair computed on its
// Gram matrix.  The columns are cut into blocks of 16; the blocks meet in
// the round-robin tournament, one outer round per kernel triple:
//   jac_gram   G_p = X_p^H X_p for every block pair p (2bs columns), each
//              workgroup one chunk of 64 rows on the FP64 matrix cores,
//              partial Grams to a workspace;
//   jac_inner  one workgroup per pair sums its partial Grams and runs one
//              cyclic sweep of two-sided Jacobi rotations on G_p in registers
//              (G <- R^H G R), accumulating J_p = product of the rotations;
//              two rounds of a sweep sweep all pairs of the 2bs columns,
//              the others only those across the two blocks;
//   jac_apply  X_p <- X_p J_p, each workgroup one chunk of rows, on the
//              FP64 matrix cores.
// The last sweeps of a preconditioned matrix are replaced by simultaneous
// rotations of all pairs as matrix products (closing phase below).
// Stream order separates the rounds.  The Gram is rebuilt from the columns in
// every round, so the test for a converged pair, |x_i^H x_j| <=
// tol*|x_i||x_j|, and the singular values (final column norms) carry the
// accuracy of the one-sided method: working precision relative to the largest
// singular value, which the 1e-10 truncation tail test needs.  A sweep without
// rotations above the convergence margin (jac_conv_tol) sets a device flag that
// turns the remaining launches into no-ops.
// A pair whose smaller column is below 16 eps of the matrix norm is left alone
// (JAC_NOISE2): such columns are rounding noise of the rotations, their
// contribution to any tail is < 4e-15, and rotating them against the signal
// columns of a matrix with more columns than rows would go on indefinitely.
// jac_finalize sorts the singular values and evaluates the truncation rank (first
// i with ||s[i:]|| < eps, capped; reference algorithms/tdvp.py:289-292).
#include "grouped.hpp"
#include "larfg.hpp"
#include "wave.hpp"

#include <algorithm>

namespace qca {
namespace {

constexpr int JAC_NT = 1024;         // threads of every Jacobi kernel
constexpr int JAC_MAXCOLS = 512;
constexpr int JAC_BS = 16;           // block size: pairs of 32 columns
constexpr int JAC_LMAX = 2 * JAC_BS;
constexpr int JAC_RC = 64;           // rows per Gram / apply chunk
constexpr int JAC_INNER_NT = 256;    // jac_inner: one 2x2 block of the Gram per thread
constexpr int JAC_GRAM_NT = 256;     // jac_gram: one wave per 16x16 block of the 32x32 Gram
constexpr int JAC_APPLY_NT = 512;    // jac_apply: one wave per 16x16 block of the 32x64 product
constexpr int JAC_MAX_SWEEPS = 60;
constexpr int JAC_MAXKSPL = 8;       // row chunks of a Gram: rows <= 512
constexpr size_t JAC_CTRL_BYTES = 512;   // slot of the control block
// Noise floor of a column, squared and relative to ||X||_F^2: (16 eps)^2.
// Columns below 16 eps ||X|| (3.6e-15 ||X||) are not orthogonalised further;
// their singular values are at the accuracy floor of the method, far below any
// truncation cutoff the engine is used with (1e-10).
constexpr double JAC_NOISE2 = 256.0 * 1.1102230246251565e-16 * 1.1102230246251565e-16;
// A pair is rotated when |g_ij| > tol sqrt(g_ii g_jj); a sweep counts as
// converged when no rotation had |g_ij| > conv sqrt(g_ii g_jj), conv =
// max(tol, 4 eps sqrt(rows)).  At the working-precision tolerance eps sqrt(rows)
// the inner products of freshly rotated columns carry rounding noise of about
// that size, so without the margin a pair can sit just above the threshold
// sweep after sweep; its last rotations are still applied.
__device__ __forceinline__ double jac_conv_tol(double tol, int rows) {
  return fmax(tol, 4.0 * 1.1102230246251565e-16 * sqrt((double)rows));
}

__device__ __forceinline__ double wsum(double v) { return wave_sum64(v); }

// Sum over rows r = lane, lane + 64, ... < rows (rows <= 512) of |col[r]|^2 in
// row order, with all of the lane's loads issued before the first add.
__device__ __forceinline__ double lane_norm2(const c128* __restrict__ col, int rows, int lane) {
  c128 v[8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (lane + 64 * i < rows) v[i] = col[lane + 64 * i];
  double a = 0;
#pragma unroll
  for (int i = 0; i < 8; ++i)
    if (lane + 64 * i < rows) a += v[i].re * v[i].re + v[i].im * v[i].im;
  return a;
}

// Sum of |x[e]|^2 over e = t, t + stride, ... < n in that order, eight loads
// in flight at a time.
__device__ __forceinline__ double strided_norm2(const c128* __restrict__ x, long n, long t, long stride) {
  double part = 0;
  for (long e0 = t; e0 < n; e0 += 8 * stride) {
    c128 v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (e0 + i * stride < n) v[i] = x[e0 + i * stride];
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (e0 + i * stride < n) part += v[i].re * v[i].re + v[i].im * v[i].im;
  }
  return part;
}

// Position t of round r in the round-robin tournament over n (even) players.
__device__ __forceinline__ int rr_player(int t, int r, int n) {
  return (t == 0) ? 0 : ((t - 1 + r) % (n - 1)) + 1;
}

struct JacobiCtrl {
  double fro;                  // ||X||_F^2
  int done;                    // converged
  int sweeps;                  // sweeps executed
  int phase;                   // 0: sweeps, 1: closing phase
  int newton;                  // closing steps executed
  int schulz;                  // Newton-Schulz steps of the next closing step
  int rot[JAC_MAX_SWEEPS];     // rotations above jac_conv_tol per sweep
};

struct JacobiGeom {
  int rows, cols, nb, kspl;
};

// Column of the matrix that is column c of block pair (bi, bj).
__device__ __forceinline__ int pair_column(int bi, int bj, int c) {
  return c < JAC_BS ? bi * JAC_BS + c : bj * JAC_BS + (c - JAC_BS);
}

// Stages rows [r0, r0+nr) of the 32 columns of pair p into a row-major LDS
// tile with a padded row stride (JAC_LMAX + 1) that spreads the banks; rows
// beyond nr and columns beyond the matrix are zero.  Lane bits give
// the row, the wave index walks the columns: no divisions, and each wave reads
// one contiguous 64-row run of a column.  NT is the workgroup size: all of a
// thread's loads are issued before its first LDS store, so the tile costs one
// memory latency, not one per column it holds.
template <int NT>
__device__ __forceinline__ void stage_tile(const c128* __restrict__ X, const JacobiGeom& g, int p,
                                           int round, int r0, int nr, c128* tile) {
  static_assert(JAC_RC == 64, "one row per lane");
  static_assert(NT % 64 == 0 && JAC_LMAX % (NT / 64) == 0, "whole columns per wave");
  constexpr int NW = NT / 64, IT = JAC_LMAX / NW;
  const int bi = rr_player(p, round, g.nb), bj = rr_player(g.nb - 1 - p, round, g.nb);
  const int r = threadIdx.x & 63, w = threadIdx.x >> 6;
  c128 v[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int gc = pair_column(bi, bj, w + i * NW);
    v[i] = (gc < g.cols && r < nr) ? X[(long)gc * g.rows + r0 + r] : c128{0.0, 0.0};
  }
#pragma unroll
  for (int i = 0; i < IT; ++i) tile[r * (JAC_LMAX + 1) + w + i * NW] = v[i];
}

// The pair products of a round on the FP64 matrix cores: v_mfma_f64_16x16x4f64
// takes A[m][k] from lane m + 16k and B[k][n] from lane n + 16k, and register
// r of lane l holds D[(l / 16) + 4r][l % 16].  A complex product is four real
// MFMAs.  One wave per 16x16 output tile, the whole K range in that wave, in
// order: the sums are deterministic.
typedef double jac_f64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ jac_f64x4 jac_mfma(double a, double b, jac_f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// ||X||_F^2 and reset of the control block (one workgroup).
__device__ __forceinline__ void jac_init_body(const c128* __restrict__ X, long n,
                                              JacobiCtrl* __restrict__ ctrl) {
  __shared__ double red[JAC_NT / 64];
  double part = 0;
  part = strided_norm2(X, n, threadIdx.x, JAC_NT);
  part = wsum(part);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = part;
  __syncthreads();
  if (threadIdx.x == 0) {
    double s = 0;
    for (int w = 0; w < JAC_NT / 64; ++w) s += red[w];
    ctrl->fro = s;
    ctrl->done = 0;
    ctrl->sweeps = 0;
    ctrl->phase = ctrl->newton = ctrl->schulz = 0;
  }
  if (threadIdx.x < JAC_MAX_SWEEPS) ctrl->rot[threadIdx.x] = 0;
}
__global__ __launch_bounds__(JAC_NT) void jac_init(const c128* __restrict__ X, long n,
                                                   JacobiCtrl* __restrict__ ctrl) {
  jac_init_body(X, n, ctrl);
}

// Partial Gram of pair blockIdx.x over row chunk blockIdx.y:
// Gpart[p][kc](i, j) = sum_r conj(X(r, c_i)) X(r, c_j), stored column-major.
// Four waves, wave w computing the 16x16 block (j in 16(w/2).., i in 16(w%2)..)
// as D[j][i] = sum_r X(r, c_j) conj(X(r, c_i)) over the chunk's 64 rows.
__device__ __forceinline__ void jac_gram_body(const c128* __restrict__ X, const JacobiGeom& g, int round,
                                              c128* __restrict__ Gpart,
                                              const JacobiCtrl* __restrict__ ctrl, int p, int kc) {
  // the control word is read alongside the tile, not before it: the round
  // kernels are latency bound, and a no-op round only stages a tile
  const int done = ctrl->done | ctrl->phase;
  constexpr int L = JAC_LMAX;
  __shared__ c128 tile[JAC_RC * (L + 1)];
  const int r0 = kc * JAC_RC, nr = min(JAC_RC, g.rows - r0);
  stage_tile<JAC_GRAM_NT>(X, g, p, round, r0, nr, tile);
  __syncthreads();
  if (done) return;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tj = (wave >> 1) * 16, ti = (wave & 1) * 16;
  const int q = lane >> 4, c = lane & 15;
  jac_f64x4 gre = {0, 0, 0, 0}, gim = {0, 0, 0, 0};
  const int kmax = (nr + 3) & ~3;
  for (int k0 = 0; k0 < kmax; k0 += 4) {
    const c128 a = tile[(k0 + q) * (L + 1) + tj + c];   // X(r, c_j)
    const c128 b = tile[(k0 + q) * (L + 1) + ti + c];   // X(r, c_i), conjugated below
    gre = jac_mfma(a.re, b.re, gre);
    gre = jac_mfma(a.im, b.im, gre);
    gim = jac_mfma(a.im, b.re, gim);
    gim = jac_mfma(-a.re, b.im, gim);
  }
  c128* out = Gpart + ((long)p * g.kspl + kc) * L * L;
#pragma unroll
  for (int rr = 0; rr < 4; ++rr) {
    const int j = tj + q + 4 * rr, i = ti + c;
    out[i + j * L] = c128{gre[rr], gim[rr]};
  }
}
__global__ __launch_bounds__(JAC_GRAM_NT) void jac_gram(const c128* __restrict__ X, JacobiGeom g,
                                                   int round, c128* __restrict__ Gpart,
                                                   const JacobiCtrl* __restrict__ ctrl) {
  jac_gram_body(X, g, round, Gpart, ctrl, blockIdx.x, blockIdx.y);
}

// Rotations of one Jacobi sweep on the Gram G of 2 x 16 columns held in
// registers by 256 threads (four waves: a barrier of four waves takes 44
// cycles, of sixteen 815).  Thread (P, Q), P = 4 wave + lane / 16 and Q =
// (lane + P) % 16, holds the 2x2 block of G of column pairs P and Q and two rows of J:
//   g = G(iP,iQ), G(iP,jQ), G(jP,iQ), G(jP,jQ);  j = J(P,iQ), J(P,jQ), J(P+16,iQ), J(P+16,jQ).
// Rotation of columns (i, j), with g = G(i, j) = x_i^H x_j, d = |x_j|^2 - |x_i|^2,
// h = sqrt(d^2 + 4|g|^2), w = h + |d|:
//   x_i' = c x_i - conj(s e) x_j,   x_j' = (s e) x_i + c x_j,
//   c = sqrt(w / (2h)),  s e = sign(d) g sqrt(2 / (h w)),
// the Rutishauser rotation t = sign(d)/(|zeta| + sqrt(1 + zeta^2)), zeta = d/(2|g|),
// c = 1/sqrt(1 + t^2), s = t c.  It is evaluated as c = w y, s e = 2 sign(d) g y
// with y = 1/sqrt(w^2 + 4|g|^2), so that c^2 + |s e|^2 = 1 whatever w is: the
// accuracy of the angle only sets how far the pair is from zero afterwards, and
// h comes from the hardware's reciprocal square root as it is (~1e-8).
// G <- R^H G R and J <- J R.  Every wave computes the rotations of all 16 pairs
// for itself (of pair Q in each row of lanes; lane 0 of a row has pair P), and
// carries their squared norms along, so a round costs one barrier and, of LDS,
// the way of the blocks that change rows and of the next pairs' inner products.
// What bounds a round is instruction issue: 1740 cycles, of which 114 FP64
// instructions at 9 cycles each (one wave per SIMD).  16 rounds with loads and
// stores take 13.7 us; with the Gram in LDS under 1024 threads and two barriers
// a round they took 16.7.  Squared norms and inner products read from LDS and
// the row rotation by lane permutes: 14.7.
struct InnerShared {
  c128 blk[2][3][256];    // G(iP,jQ), G(jP,iQ), G(jP,jQ) on their way to the next round
  c128 off[2][16];        // G(i,j) of the pairs of a round
  double diag[2][16];     // G(i,i), G(j,j) of the first round's pairs
};
struct JacRot {
  double c, sr, si;   // c, s e
};
struct InnerThresholds {
  double tol2, conv2, negl;
};

// Lane (l + 1) % 16, and lane 0, of each row of 16 lanes.
__device__ __forceinline__ double row_next(double v) { return dpp_f64<0x12F>(v); }    // row_ror:15
__device__ __forceinline__ double row_first(double v) { return dpp_f64<0x150>(v); }   // row_newbcast:0

// Rotation of one pair of squared norms a, b (updated) and inner product g;
// act: it is rotated, sig: above the convergence margin.
__device__ __forceinline__ JacRot pair_rotation(double& a, double& b, const c128& g, const InnerThresholds& th,
                                                bool& act, bool& sig) {
  const double ag2 = g.re * g.re + g.im * g.im;
  const double d = b - a;
  const double f = 4.0 * ag2;
  const double x = fma(d, d, f);
  const double w = fma(x, __builtin_amdgcn_rsq(x), fabs(d));
  // y = 1/sqrt(t): a third-order step on the hardware estimate, then one whose
  // residual 1 - t y^2 includes the exact error of t y, so that y carries no
  // bias (c and s share y: a biased y drifts the column norms)
  const double t = fma(w, w, f);
  double y = __builtin_amdgcn_rsq(t);
  const double e0 = fma(-t * y, y, 1.0);
  y = fma(y, e0 * fma(0.375, e0, 0.5), y);
  const double ty = t * y;
  const double e = fma(-ty, y, 1.0) - fma(t, y, -ty) * y;
  y = fma(0.5 * y, e, y);
  // a pair with a column at the noise floor is done: rotating noise against a
  // signal column only re-creates noise, and for matrices with more columns
  // than rows such pairs can rotate indefinitely
  const double ab = a * b;
  act = !(ag2 <= th.tol2 * ab || ag2 < 1e-300 || fmin(a, b) < th.negl);
  sig = act && ag2 > th.conv2 * ab;
  const double s = d >= 0 ? 2.0 * y : -2.0 * y;
  // |x_i|^2 and |x_j|^2 change by tan |g| = 2 |g|^2 / w
  double iw = __builtin_amdgcn_rcp(w);
  iw = fma(iw, fma(-w, iw, 1.0), iw);
  const double delta = act ? (d >= 0 ? 0.5 : -0.5) * f * iw : 0.0;
  a -= delta;
  b += delta;
  return act ? JacRot{w * y, s * g.re, s * g.im} : JacRot{1.0, 0.0, 0.0};
}

// x_i, x_j <- the rotated pair (columns).
__device__ __forceinline__ void rotate_cols(const JacRot& q, c128& x, c128& y) {
  const c128 a = x, b = y;
  x = c128{q.c * a.re - (q.sr * b.re + q.si * b.im), q.c * a.im - (q.sr * b.im - q.si * b.re)};
  y = c128{(q.sr * a.re - q.si * a.im) + q.c * b.re, (q.sr * a.im + q.si * a.re) + q.c * b.im};
}
// The conjugate rotation, for the rows of R^H G.
__device__ __forceinline__ void rotate_rows(const JacRot& p, c128& x, c128& y) {
  const c128 a = x, b = y;
  x = c128{p.c * a.re - (p.sr * b.re - p.si * b.im), p.c * a.im - (p.sr * b.im + p.si * b.re)};
  y = c128{(p.sr * a.re + p.si * a.im) + p.c * b.re, (p.sr * a.im - p.si * a.re) + p.c * b.im};
}

// H rounds: pair t of group m (2H columns from 2H m) joins column t of the
// group's first half and column H + (t + r) mod H of it in round r, so the
// blocks of the second columns move to the next pair's thread after each
// round (across lanes of a row by DPP moves or a lane read, across rows
// through LDS) and are back in place after the last.
template <int H>
__device__ __forceinline__ void inner_rounds(c128 (&g)[4], c128 (&j)[4], InnerShared& sh, const InnerThresholds& th,
                                             int& rotated, int& above) {
  const int lane = threadIdx.x & 15, P = threadIdx.x >> 4, Q = (lane + P) & 15;
  const int nP = (P & ~(H - 1)) | ((P + 1) & (H - 1)), nQ = (Q & ~(H - 1)) | ((Q + 1) & (H - 1));
  const int nl = (nQ - P) & 15;   // the lane of pair nQ
  const int at = P * 16 + Q, at_i = nP * 16 + Q, at_j = nP * 16 + nQ;
  int buf = 0;
  if (lane == 0) {
    sh.off[0][P] = g[1];
    sh.diag[0][P] = g[0].re;
    sh.diag[1][P] = g[3].re;
  }
  __syncthreads();
  double a = sh.diag[0][Q], b = sh.diag[1][Q];
  c128 off = sh.off[0][Q];
#pragma unroll 1
  for (int r = 0; r < H; ++r) {
    bool act, sig;
    const JacRot q = pair_rotation(a, b, off, th, act, sig);
    rotated += __popcll(__ballot(act) & 0xffff);
    above += __popcll(__ballot(sig) & 0xffff);
    const JacRot p{row_first(q.c), row_first(q.sr), row_first(q.si)};
    rotate_cols(q, g[0], g[1]);
    rotate_cols(q, g[2], g[3]);
    rotate_rows(p, g[0], g[2]);
    rotate_rows(p, g[1], g[3]);
    buf ^= 1;
    if (Q == nP) sh.off[buf][P] = g[1];
    sh.blk[buf][1][at] = g[2];
    sh.blk[buf][2][at] = g[3];
    if constexpr (H == 16) {
      g[1] = c128{row_next(g[1].re), row_next(g[1].im)};
      b = row_next(b);
    } else {
      sh.blk[buf][0][at] = g[1];
      b = __shfl(b, nl, 16);
    }
    rotate_cols(q, j[0], j[1]);
    rotate_cols(q, j[2], j[3]);
#pragma unroll
    for (int k = 1; k < 4; k += 2) {
      if constexpr (H == 16) j[k] = c128{row_next(j[k].re), row_next(j[k].im)};
      else j[k] = c128{__shfl(j[k].re, nl, 16), __shfl(j[k].im, nl, 16)};
    }
    __syncthreads();
    off = sh.off[buf][Q];
    g[2] = sh.blk[buf][1][at_i];
    g[3] = sh.blk[buf][2][at_j];
    if constexpr (H < 16) g[1] = sh.blk[buf][0][P * 16 + nQ];
  }
}

// From the pairs of groups of 2H columns to those of groups of H.
template <int H>
__device__ __forceinline__ void inner_regroup(c128 (&g)[4], c128 (&j)[4], InnerShared& sh) {
  c128* m = &sh.blk[0][0][0];   // 32 x 32
  const int P = threadIdx.x >> 4, Q = (threadIdx.x + P) & 15;
  const int iP = (P / H) * 2 * H + P % H, iQ = (Q / H) * 2 * H + Q % H;
  constexpr int K = H / 2;
  const int kP = (P / K) * H + P % K, kQ = (Q / K) * H + Q % K;
  __syncthreads();
  m[iP * 32 + iQ] = g[0];
  m[iP * 32 + iQ + H] = g[1];
  m[(iP + H) * 32 + iQ] = g[2];
  m[(iP + H) * 32 + iQ + H] = g[3];
  __syncthreads();
  g[0] = m[kP * 32 + kQ];
  g[1] = m[kP * 32 + kQ + K];
  g[2] = m[(kP + K) * 32 + kQ];
  g[3] = m[(kP + K) * 32 + kQ + K];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) m[(P + 16 * (k / 2)) * 32 + iQ + (k & 1) * H] = j[k];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) j[k] = m[(P + 16 * (k / 2)) * 32 + kQ + (k & 1) * K];
  __syncthreads();
}

// Outer rounds 0 and (nb - 1) / 2 of a sweep also visit the pairs inside each
// block (every block takes part in every outer round), by halves: the pairs
// across two groups of 16 columns, then of 8, 4, 2, 1 (31 rounds); the others
// visit only the pairs across their two blocks (16 rounds).  A sweep thus meets
// every column pair at least once, in 2 * 31 + 13 * 16 inner rounds for 16
// blocks of 16 instead of 15 * 31.  Inside pairs once per sweep (round 0 only)
// cost about one sweep more; twice keeps the sweep count of a full ordering
// within a fraction of a sweep.
__device__ __forceinline__ void jac_inner_body(const JacobiGeom& g, int round, int sweep,
                                               const c128* __restrict__ Gpart,
                                               c128* __restrict__ Jout, int* __restrict__ rotated,
                                               double tol, JacobiCtrl* __restrict__ ctrl, int p) {
  const int done = ctrl->done | ctrl->phase;  // read alongside the partial Grams
  constexpr int L = JAC_LMAX;
  __shared__ InnerShared sh;
  const int P = threadIdx.x >> 4, Q = (threadIdx.x + P) & 15;
  const double conv = jac_conv_tol(tol, g.rows);
  const InnerThresholds th{tol * tol, conv * conv, JAC_NOISE2 * ctrl->fro};
  // all chunk partials are loaded before the first add (one memory latency),
  // then summed in chunk order; G(P, Q) is read as conj(G(Q, P)), contiguous
  // over the lanes
  c128 v[JAC_MAXKSPL][4];
#pragma unroll
  for (int kc = 0; kc < JAC_MAXKSPL; ++kc)
    if (kc < g.kspl)
#pragma unroll
      for (int k = 0; k < 4; ++k)
        v[kc][k] = Gpart[((long)p * g.kspl + kc) * L * L + (P + 16 * (k / 2)) * L + Q + 16 * (k & 1)];
  c128 G[4], J[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    double re = 0, im = 0;
#pragma unroll
    for (int kc = 0; kc < JAC_MAXKSPL; ++kc)
      if (kc < g.kspl) {
        re += v[kc][k].re;
        im += v[kc][k].im;
      }
    G[k] = c128{re, -im};
    J[k] = c128{(k == 0 || k == 3) && P == Q ? 1.0 : 0.0, 0.0};
  }
  if (done) return;
  int total = 0, above = 0, h = 16;
  inner_rounds<16>(G, J, sh, th, total, above);
  if (round == 0 || round == (g.nb - 1) / 2) {
    inner_regroup<16>(G, J, sh);
    inner_rounds<8>(G, J, sh, th, total, above);
    inner_regroup<8>(G, J, sh);
    inner_rounds<4>(G, J, sh, th, total, above);
    inner_regroup<4>(G, J, sh);
    inner_rounds<2>(G, J, sh, th, total, above);
    inner_regroup<2>(G, J, sh);
    inner_rounds<1>(G, J, sh, th, total, above);
    h = 1;
  }
  // J(k, c) at c * L + k
  c128* jo = Jout + (long)p * L * L;
  const int iQ = h == 16 ? Q : 2 * Q;
#pragma unroll
  for (int k = 0; k < 4; ++k) jo[(iQ + (k & 1) * h) * L + P + 16 * (k / 2)] = J[k];
  if (threadIdx.x == 0) {
    rotated[p] = total;
    if (above) atomicAdd(&ctrl->rot[sweep], above);
  }
}
__global__ __launch_bounds__(JAC_INNER_NT) void jac_inner(JacobiGeom g, int round, int sweep,
                                                    const c128* __restrict__ Gpart,
                                                    c128* __restrict__ Jout,
                                                    int* __restrict__ rotated, double tol,
                                                    JacobiCtrl* __restrict__ ctrl) {
  jac_inner_body(g, round, sweep, Gpart, Jout, rotated, tol, ctrl, blockIdx.x);
}

// X_p <- X_p J_p on row chunk blockIdx.y of pair blockIdx.x; chunks from
// g.kspl on belong to the second matrix Z (geometry gz), which receives the
// same rotations (gz.kspl == 0 when there is none).
__device__ __forceinline__ void jac_apply_body(c128* __restrict__ Xa, const JacobiGeom& ga,
                                               c128* __restrict__ Za, const JacobiGeom& gz, int round,
                                               const c128* __restrict__ Jin,
                                               const int* __restrict__ rotated,
                                               const JacobiCtrl* __restrict__ ctrl, int p, int by) {
  // the control words are read alongside the tile and J, not before them
  const int skip = ctrl->done | ctrl->phase | (rotated[p] == 0);
  const bool second = by >= ga.kspl;
  c128* __restrict__ X = second ? Za : Xa;
  const JacobiGeom g = second ? gz : ga;
  const int kc = second ? by - ga.kspl : by;
  __shared__ c128 tile[JAC_RC * (JAC_LMAX + 1)];
  constexpr int L = JAC_LMAX;
  __shared__ c128 J[L * (L + 1)];   // J(k, c) at c * (L + 1) + k
  const int r0 = kc * JAC_RC, nr = min(JAC_RC, g.rows - r0);
  stage_tile<JAC_APPLY_NT>(X, g, p, round, r0, nr, tile);
  const c128* jp = Jin + (long)p * L * L;
  constexpr int JIT = L * L / JAC_APPLY_NT;
  c128 jv[JIT];
#pragma unroll
  for (int i = 0; i < JIT; ++i) jv[i] = jp[threadIdx.x + i * JAC_APPLY_NT];
#pragma unroll
  for (int i = 0; i < JIT; ++i) {
    const int e = threadIdx.x + i * JAC_APPLY_NT, k = e % L, c = e / L;
    J[c * (L + 1) + k] = jv[i];
  }
  __syncthreads();
  if (skip) return;
  // Eight waves: wave w computes the 16x16 block (columns c in 16(w%2)..,
  // rows r in 16(w/2)..) of the transposed product D[c][r] = sum_k J(k, c) X(r, k),
  // so that consecutive lanes store consecutive rows of a column.
  const int bi = rr_player(p, round, g.nb), bj = rr_player(g.nb - 1 - p, round, g.nb);
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int tc = (wave & 1) * 16, tr = (wave >> 1) * 16;
  if (tr >= nr) return;
  const int q = lane >> 4, cl = lane & 15;
  jac_f64x4 dre = {0, 0, 0, 0}, dim = {0, 0, 0, 0};
  for (int k0 = 0; k0 < L; k0 += 4) {
    const c128 a = J[(tc + cl) * (L + 1) + k0 + q];      // J(k, c)
    const c128 b = tile[(tr + cl) * (L + 1) + k0 + q];   // X(r, k)
    dre = jac_mfma(a.re, b.re, dre);
    dre = jac_mfma(-a.im, b.im, dre);
    dim = jac_mfma(a.re, b.im, dim);
    dim = jac_mfma(a.im, b.re, dim);
  }
  const int r = tr + cl;
  if (r < nr)
#pragma unroll
    for (int rr = 0; rr < 4; ++rr) {
      const int gc = pair_column(bi, bj, tc + q + 4 * rr);
      if (gc < g.cols) X[(long)gc * g.rows + r0 + r] = c128{dre[rr], dim[rr]};
    }
}
__global__ __launch_bounds__(JAC_APPLY_NT) void jac_apply(c128* __restrict__ Xa, JacobiGeom ga,
                                                    c128* __restrict__ Za, JacobiGeom gz, int round,
                                                    const c128* __restrict__ Jin,
                                                    const int* __restrict__ rotated,
                                                    const JacobiCtrl* __restrict__ ctrl) {
  jac_apply_body(Xa, ga, Za, gz, round, Jin, rotated, ctrl, blockIdx.x, blockIdx.y);
}

// Closes a sweep: converged when it made no rotation.
__device__ __forceinline__ void jac_check_body(JacobiCtrl* __restrict__ ctrl) {
  if (threadIdx.x != 0 || ctrl->done) return;
  ctrl->sweeps = 1;
  if (ctrl->rot[0] == 0) ctrl->done = 1;
}
// After sweep 0.
__global__ void jac_check(JacobiCtrl* __restrict__ ctrl) { jac_check_body(ctrl); }

// ------------------------------------------------------------------ closing phase
// Once the columns of Y are nearly orthogonal, all pairs are rotated at once:
// with the small rotations of the cyclic sweeps collected in an anti-Hermitian
// K, K_ij = sign(d) 2 g_ij / w for every pair (d, w as in the sweeps), Y <- Y J
// with a unitary J = I + K + O(K^2) squares the scaled off-diagonals just as a
// sweep does, but as products on the matrix cores instead of a chain of n
// rotation rounds: J starts as I + K + K^2 / 2 and is made unitary by
// Newton-Schulz steps J <- J (3 I - J^H J) / 2.  Each product keeps the relative
// accuracy of graded columns: K_ij, K^2 and J^H J - I carry the factor
// |y_j| / |y_i| of a pair with |y_j| << |y_i|.
// A matrix enters the phase after a sweep (the second or a later one) that
// leaves |K|_F <= NEWTON_KF, and goes back to sweeps if |K|_F should exceed it
// again (clusters of singular values keep K large: those are left to the
// sweeps).  It has converged when no pair is above the margin of jac_conv_tol.
// All of this is decided on the device from Y alone, so that a matrix takes the
// same steps alone and in a group.
// A step is bound by its eleven dependent launches: 50 us for 256 columns, of
// which the products (16x16 tiles, one workgroup each, k split over four waves)
// take 3-11 us each, against 380 us for a sweep's 15 rounds.  A 256x256 random
// two-site tensor takes 4 sweeps and 3 steps instead of 7 sweeps (split 3.36 ->
// 2.43 ms), a 154x90 one 2 and 3 instead of 6 (1.22 -> 0.81 ms).  NEWTON_KF: as
// far as three Newton-Schulz steps reach rounding; at 0.1 the 154x90 split takes
// a sweep more (0.91 ms).
constexpr int NEWTON_NT = 256;
constexpr int NEWTON_SCHULZ_MAX = 3;
constexpr double NEWTON_KF = 0.4;     // |K|_F up to which a matrix is in the closing phase
constexpr int NEWTON_MAX = 12;        // steps after which a matrix stays with the sweeps

struct NewtonArgs {
  c128* Y;            // yrows x n
  c128* Q;            // qrows x n, same rotations
  int yrows, qrows, n, ytiles, qtiles, ntiles;   // 16-row and 16-column tiles
  c128 *K, *W, *J0, *J1;   // K and W also take the new Y and Q (yrows x n, qrows x n)
  double* kf2;        // per tile: sum of |K|^2
  int* above;         // per tile: pairs above the convergence margin
  JacobiCtrl* ctrl;
  double tol;
};

struct NewtonShared {
  c128 part[4][16 * 17];
  double nrm[2][16][16];
  double red[4];
  int cnt[4];
};

// One 16x16 tile of a product over k < kdim, the four waves taking 16 of every
// 64 k each; the sum over the waves is left to tile_sum.  a(k, lane16) and
// b(k, lane16) give the operands' elements (k = row of the lane group).
template <typename FA, typename FB>
__device__ __forceinline__ void tile_product(int kdim, NewtonShared& sh, FA&& a, FB&& b) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  jac_f64x4 re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
  for (int k0 = 16 * wave; k0 < kdim; k0 += 128) {
    // two of the wave's blocks of 16 k: 16 loads in flight
    c128 x[8], y[8];
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      const int k = k0 + (s / 4) * 64 + 4 * (s & 3) + hi;
      x[s] = a(k, lo);
      y[s] = b(k, lo);
    }
#pragma unroll
    for (int s = 0; s < 8; ++s) {
      re = jac_mfma(x[s].re, y[s].re, re);
      im = jac_mfma(x[s].re, y[s].im, im);
      re = jac_mfma(-x[s].im, y[s].im, re);
      im = jac_mfma(x[s].im, y[s].re, im);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) sh.part[wave][(hi + 4 * r) * 17 + lo] = c128{re[r], im[r]};
}
// Element (i, j) of the tile for thread i + 16 j (after a barrier).
__device__ __forceinline__ c128 tile_sum(const NewtonShared& sh) {
  const int e = (threadIdx.x & 15) * 17 + (threadIdx.x >> 4);
  c128 s{0.0, 0.0};
#pragma unroll
  for (int w = 0; w < 4; ++w) {
    s.re += sh.part[w][e].re;
    s.im += sh.part[w][e].im;
  }
  return s;
}
// X(k, c) of a column-major matrix, zero outside rows x cols.
__device__ __forceinline__ c128 col_elem(const c128* __restrict__ X, int rows, int cols, int k, int c) {
  const c128 v = X[(unsigned)min(c, cols - 1) * rows + min(k, rows - 1)];
  return k < rows && c < cols ? v : c128{0.0, 0.0};
}
__device__ __forceinline__ c128 conj_of(c128 v) { return c128{v.re, -v.im}; }

// Phase words: a matrix is in sweeps (0) or in the closing phase (1).
__device__ __forceinline__ bool newton_off(const JacobiCtrl* ctrl) { return ctrl->done || ctrl->phase == 0; }

// K of column tiles (bi, bj), bi <= bj, and its mirror; after a sweep (closing
// = 0) for matrices in sweeps, after a closing step for those in the phase.
__device__ __forceinline__ void newton_corr_body(const NewtonArgs& a, const c128* __restrict__ Y,
                                                 c128* __restrict__ K, int closing, int bi, int bj, NewtonShared& sh) {
  if (bi > bj || a.ctrl->done || a.ctrl->phase != closing) return;
  const int n = a.n, rows = a.yrows, i0 = 16 * bi, j0 = 16 * bj;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double na = 0, nb = 0;
  tile_product(
      rows, sh,
      [&](int k, int c) {
        const c128 v = col_elem(Y, rows, n, k, i0 + c);
        na += v.re * v.re + v.im * v.im;
        return conj_of(v);
      },
      [&](int k, int c) {
        const c128 v = col_elem(Y, rows, n, k, j0 + c);
        nb += v.re * v.re + v.im * v.im;
        return v;
      });
  sh.nrm[0][4 * wave + (lane >> 4)][lane & 15] = na;
  sh.nrm[1][4 * wave + (lane >> 4)][lane & 15] = nb;
  __syncthreads();
  const c128 g = tile_sum(sh);
  const int i = threadIdx.x & 15, j = threadIdx.x >> 4;
  double pa = 0, pb = 0;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    pa += sh.nrm[0][s][i];
    pb += sh.nrm[1][s][j];
  }
  const int gi = i0 + i, gj = j0 + j;
  const double conv = jac_conv_tol(a.tol, rows);
  const double ag2 = g.re * g.re + g.im * g.im, ab = pa * pb;
  const bool pair = gi < gj && gj < n;
  const bool act = pair && !(ag2 <= a.tol * a.tol * ab || ag2 < 1e-300 || fmin(pa, pb) < JAC_NOISE2 * a.ctrl->fro);
  const bool sig = act && ag2 > conv * conv * ab;
  double t = 0;
  if (act) {
    const double d = pb - pa;
    t = (d >= 0 ? 2.0 : -2.0) / (sqrt(fma(d, d, 4.0 * ag2)) + fabs(d));
  }
  const c128 kij{t * g.re, t * g.im};
  if (pair) {
    K[(unsigned)gj * n + gi] = kij;
    K[(unsigned)gi * n + gj] = c128{-kij.re, kij.im};
  } else if (gi == gj && gi < n) {
    K[(unsigned)gj * n + gi] = c128{0.0, 0.0};
  }
  const double kf = wave_sum64(2.0 * (kij.re * kij.re + kij.im * kij.im));
  const int cnt = __popcll(__ballot(sig));
  if (lane == 0) {
    sh.red[wave] = kf;
    sh.cnt[wave] = cnt;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const int tile = bi * a.ntiles + bj;
    a.kf2[tile] = (sh.red[0] + sh.red[1]) + (sh.red[2] + sh.red[3]);
    a.above[tile] = sh.cnt[0] + sh.cnt[1] + sh.cnt[2] + sh.cnt[3];
  }
}

// After sweep `sweep` (>= 0) or a closing step (-1): converged, closing phase
// or sweeps.
__device__ __forceinline__ void newton_decide_body(const NewtonArgs& a, JacobiCtrl* __restrict__ ctrl, int sweep) {
  const int closing = sweep < 0 ? 1 : 0;
  if (ctrl->done || ctrl->phase != closing) return;
  __shared__ double red[NEWTON_NT / 64];
  __shared__ int cnt[NEWTON_NT / 64];
  double kf = 0;
  int above = 0;
  for (int t = threadIdx.x; t < a.ntiles * a.ntiles; t += NEWTON_NT)
    if (t / a.ntiles <= t % a.ntiles) {
      kf += a.kf2[t];
      above += a.above[t];
    }
  kf = wave_sum64(kf);
  for (int o = 32; o > 0; o >>= 1) above += __shfl_xor(above, o, 64);
  if ((threadIdx.x & 63) == 0) {
    red[threadIdx.x >> 6] = kf;
    cnt[threadIdx.x >> 6] = above;
  }
  __syncthreads();
  if (threadIdx.x != 0) return;
  kf = (red[0] + red[1]) + (red[2] + red[3]);
  above = cnt[0] + cnt[1] + cnt[2] + cnt[3];
  if (closing) ctrl->newton += 1;
  else ctrl->sweeps += 1;   // sweeps launched during the closing phase are no-ops
  if (closing ? above == 0 : ctrl->rot[sweep] == 0) {
    ctrl->done = 1;
    return;
  }
  const bool in = kf <= NEWTON_KF * NEWTON_KF && ctrl->newton < NEWTON_MAX;
  ctrl->phase = in ? 1 : 0;
  // Newton-Schulz steps until |J^H J - I| <= 1e-17: it is |K|^4 / 4 at first and
  // 3/4 of its square after a step (4e-19 after three from NEWTON_KF)
  int schulz = 0;
  for (double e = 0.25 * kf * kf; e > 1e-17 && schulz < NEWTON_SCHULZ_MAX; e = 0.75 * e * e) ++schulz;
  ctrl->schulz = schulz;
}

// J0 = I + K + K^2 / 2, K^2 = -K^H K.
__device__ __forceinline__ void newton_start_body(const NewtonArgs& a, const c128* __restrict__ K,
                                                  c128* __restrict__ J, int bi, int bj, NewtonShared& sh) {
  if (newton_off(a.ctrl)) return;
  const int n = a.n, i0 = 16 * bi, j0 = 16 * bj;
  tile_product(n, sh, [&](int k, int c) { return conj_of(col_elem(K, n, n, k, i0 + c)); },
               [&](int k, int c) { return col_elem(K, n, n, k, j0 + c); });
  __syncthreads();
  const c128 s = tile_sum(sh);
  const int gi = i0 + (threadIdx.x & 15), gj = j0 + (threadIdx.x >> 4);
  if (gi < n && gj < n) {
    const c128 k = K[(unsigned)gj * n + gi];
    J[(unsigned)gj * n + gi] = c128{(gi == gj ? 1.0 : 0.0) + k.re - 0.5 * s.re, k.im - 0.5 * s.im};
  }
}
// W = J^H J (`step`-th Newton-Schulz step, if there is one).
__device__ __forceinline__ void newton_gram_body(const NewtonArgs& a, const c128* __restrict__ J,
                                                 c128* __restrict__ W, int step, int bi, int bj, NewtonShared& sh) {
  if (newton_off(a.ctrl) || a.ctrl->schulz < step) return;
  const int n = a.n, i0 = 16 * bi, j0 = 16 * bj;
  tile_product(n, sh, [&](int k, int c) { return conj_of(col_elem(J, n, n, k, i0 + c)); },
               [&](int k, int c) { return col_elem(J, n, n, k, j0 + c); });
  __syncthreads();
  const c128 s = tile_sum(sh);
  const int gi = i0 + (threadIdx.x & 15), gj = j0 + (threadIdx.x >> 4);
  if (gi < n && gj < n) W[(unsigned)gj * n + gi] = s;
}
// Jn = 1.5 J - 0.5 J W, W Hermitian (W(l, j) read as conj(W(j, l))).
__device__ __forceinline__ void newton_schulz_body(const NewtonArgs& a, const c128* __restrict__ J,
                                                   const c128* __restrict__ W, c128* __restrict__ Jn, int step,
                                                   int bi, int bj, NewtonShared& sh) {
  if (newton_off(a.ctrl) || a.ctrl->schulz < step) return;
  const int n = a.n, i0 = 16 * bi, j0 = 16 * bj;
  tile_product(n, sh, [&](int k, int c) { return col_elem(J, n, n, i0 + c, k); },
               [&](int k, int c) { return conj_of(col_elem(W, n, n, j0 + c, k)); });
  __syncthreads();
  const c128 s = tile_sum(sh);
  const int gi = i0 + (threadIdx.x & 15), gj = j0 + (threadIdx.x >> 4);
  if (gi < n && gj < n) {
    const c128 z = J[(unsigned)gj * n + gi];
    Jn[(unsigned)gj * n + gi] = c128{1.5 * z.re - 0.5 * s.re, 1.5 * z.im - 0.5 * s.im};
  }
}
// Row tile br of (Y; Q), column tile bj: the new Y to K's buffer, the new Q to
// W's.
__device__ __forceinline__ void newton_apply_body(const NewtonArgs& a, const c128* __restrict__ Y,
                                                  const c128* __restrict__ Q, const c128* __restrict__ J0,
                                                  const c128* __restrict__ J1, c128* __restrict__ Yn,
                                                  c128* __restrict__ Qn, int br, int bj, NewtonShared& sh) {
  if (newton_off(a.ctrl)) return;
  const c128* __restrict__ J = a.ctrl->schulz & 1 ? J1 : J0;
  const bool second = br >= a.ytiles;
  const c128* __restrict__ X = second ? Q : Y;
  c128* __restrict__ out = second ? Qn : Yn;
  const int rows = second ? a.qrows : a.yrows, n = a.n;
  const int i0 = 16 * (second ? br - a.ytiles : br), j0 = 16 * bj;
  tile_product(n, sh, [&](int k, int c) { return col_elem(X, rows, n, i0 + c, k); },
               [&](int k, int c) { return col_elem(J, n, n, k, j0 + c); });
  __syncthreads();
  const c128 s = tile_sum(sh);
  const int gi = i0 + (threadIdx.x & 15), gj = j0 + (threadIdx.x >> 4);
  if (gi < rows && gj < n) out[(unsigned)gj * rows + gi] = s;
}
__device__ __forceinline__ void newton_copy_body(const NewtonArgs& a, c128* __restrict__ Y, c128* __restrict__ Q,
                                                 const c128* __restrict__ Yn, const c128* __restrict__ Qn,
                                                 unsigned blk, unsigned nblk) {
  if (newton_off(a.ctrl)) return;
  const int ny = a.yrows * a.n, nq = a.qrows * a.n;
  for (int e = blk * NEWTON_NT + threadIdx.x; e < ny + nq; e += nblk * NEWTON_NT) {
    if (e < ny) Y[e] = Yn[e];
    else Q[e - ny] = Qn[e - ny];
  }
}

// The kernels of the phase, one for a single matrix and one for a group.
enum NewtonOp { NEWTON_CORR, NEWTON_START, NEWTON_GRAM, NEWTON_SCHULZ, NEWTON_APPLY, NEWTON_COPY };
template <int OP>
__device__ __forceinline__ void newton_body(const NewtonArgs& a, int arg, unsigned bx, unsigned by, unsigned nx) {
  __shared__ NewtonShared sh;
  c128 *Y = gbl(a.Y), *Q = gbl(a.Q), *K = gbl(a.K), *W = gbl(a.W), *J0 = gbl(a.J0), *J1 = gbl(a.J1);
  // arg: closing (corr); Newton-Schulz step 1 or 3 (J0 -> J1) or 2 (J1 -> J0)
  if constexpr (OP == NEWTON_CORR) newton_corr_body(a, Y, K, arg, bx, by, sh);
  if constexpr (OP == NEWTON_START) newton_start_body(a, K, J0, bx, by, sh);
  if constexpr (OP == NEWTON_GRAM) newton_gram_body(a, arg & 1 ? J0 : J1, W, arg, bx, by, sh);
  if constexpr (OP == NEWTON_SCHULZ) newton_schulz_body(a, arg & 1 ? J0 : J1, W, arg & 1 ? J1 : J0, arg, bx, by, sh);
  if constexpr (OP == NEWTON_APPLY) newton_apply_body(a, Y, Q, J0, J1, K, W, bx, by, sh);
  if constexpr (OP == NEWTON_COPY) newton_copy_body(a, Y, Q, K, W, bx, nx);
}
template <int OP>
__global__ __launch_bounds__(NEWTON_NT) void newton_kernel(NewtonArgs a, int arg) {
  newton_body<OP>(a, arg, blockIdx.x, blockIdx.y, gridDim.x);
}
template <int OP>
__global__ __launch_bounds__(NEWTON_NT) void newton_grouped(const GRec<NewtonArgs>* __restrict__ recs, int n, int arg) {
  unsigned bx, by, bz;
  const GRec<NewtonArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const NewtonArgs a = r.a;
  newton_body<OP>(a, arg, bx, by, r.grid.x);
}
__global__ __launch_bounds__(NEWTON_NT) void newton_decide(NewtonArgs a, int sweep) {
  newton_decide_body(a, a.ctrl, sweep);
}
__global__ __launch_bounds__(NEWTON_NT) void newton_decide_grouped(const GRec<NewtonArgs>* __restrict__ recs, int sweep) {
  const NewtonArgs a = recs[blockIdx.x].a;
  newton_decide_body(a, gbl(a.ctrl), sweep);
}

// Position of keys[c] among the first n keys, largest first, equal keys in column
// order; keys are compared as bit patterns (they are not negative), so that the
// positions are a permutation with NaN among them too.  8 threads per column
// count a share each (a group of 8 lanes, the count the same in each).
__device__ __forceinline__ int key_rank(const double* keys, int n, int c) {
  const unsigned long long mine = __builtin_bit_cast(unsigned long long, keys[min(c, n - 1)]);
  int rank = 0;
#pragma unroll 4
  for (int o = threadIdx.x & 7; o < n; o += 8) {
    const unsigned long long other = __builtin_bit_cast(unsigned long long, keys[o]);
    rank += other > mine || (other == mine && o < c) ? 1 : 0;
  }
  for (int d = 4; d > 0; d >>= 1) rank += __shfl_xor(rank, d, 64);
  return rank;
}

// Column norms, descending sort and truncation rank (one workgroup of JAC_NT).
// Bound by latency: 16 columns at a time, a rank by counting (no barriers; a
// bitonic sort's 36 of sixteen waves take 12 us at 256 columns) and suffix sums
// over one wave (a serial pass over LDS took 25 us).  256 columns: 50 -> 18.5 us.
__device__ void finalize_body(const c128* __restrict__ X, int rows, int cols,
                              double* __restrict__ sigma, int* __restrict__ perm,
                              SvdResult* __restrict__ res, int chi_max, double eps, int rank_cap,
                              const JacobiCtrl* __restrict__ ctrl) {
  __shared__ double skey[JAC_MAXCOLS], sorted[JAC_MAXCOLS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = JAC_NT / 64;
  for (int c = wave; c < cols; c += nw) {
    const double a = wsum(lane_norm2(X + (long)c * rows, rows, lane));
    if (lane == 0) skey[c] = sqrt(a);
  }
  __syncthreads();
  for (int c0 = 0; c0 < cols; c0 += JAC_NT / 8) {
    const int c = c0 + (tid >> 3);
    const int rank = key_rank(skey, cols, c);
    if (c < cols && (tid & 7) == 0) {
      sorted[rank] = skey[c];
      sigma[rank] = skey[c];
      perm[rank] = c;
    }
  }
  __syncthreads();
  if (tid >= 64) return;
  // first i (< cap) with ||s[i:]|| < eps over the min(rows, cols) values a
  // reduced SVD returns; the tail norms form a non-increasing sequence.  Lane l
  // holds values 8 l .. 8 l + 7.
  constexpr int PER = JAC_MAXCOLS / 64;
  const int ns = min(rank_cap, cols), cap = min(chi_max, ns);
  double v[PER], total = 0;
#pragma unroll
  for (int q = PER - 1; q >= 0; --q) {
    const int e = PER * lane + q;
    const double s = e < ns ? sorted[e] : 0.0;
    v[q] = s * s;
    total += v[q];
  }
  double after = total;   // of this lane and the ones after it, then of the latter
  for (int d = 1; d < 64; d <<= 1) {
    const double t = __shfl_down(after, d, 64);
    after += lane + d < 64 ? t : 0.0;
  }
  const double t1 = __shfl_down(after, 1, 64);
  after = lane < 63 ? t1 : 0.0;
  int k = cap;
#pragma unroll
  for (int q = PER - 1; q >= 0; --q) {
    after += v[q];
    if (PER * lane + q < cap && sqrt(after) < eps) k = PER * lane + q;
  }
  for (int d = 32; d > 0; d >>= 1) k = min(k, __shfl_xor(k, d, 64));
  double kept = 0, tail = 0;
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    if (PER * lane + q < k) kept += v[q];
    else tail += v[q];
  }
  kept = wsum(kept);
  tail = wsum(tail);
  if (tid == 0) {
    res->k = k;
    res->nsweeps = ctrl->sweeps;
    res->converged = ctrl->done;
    res->nsteps = ctrl->newton;
    res->norm_kept = sqrt(kept);
    res->tail = sqrt(tail);
  }
}

__global__ __launch_bounds__(JAC_NT) void jac_finalize(const c128* __restrict__ X, int rows, int cols,
                                                       double* __restrict__ sigma,
                                                       int* __restrict__ perm,
                                                       SvdResult* __restrict__ res, int chi_max,
                                                       double eps, int rank_cap,
                                                       const JacobiCtrl* __restrict__ ctrl) {
  finalize_body(X, rows, cols, sigma, perm, res, chi_max, eps, rank_cap, ctrl);
}

// ------------------------------------------------------------------ small matrices
// The whole SVD of a matrix with min(rows, cols) <= 32 and max(rows, cols) <= 128
// in one workgroup of four waves.  One-sided Jacobi on the columns of X takes 6
// to 19 sweeps on the graded spectra of a TDVP split; on the triangle of a
// QR with the columns sorted by norm it takes one to four, so:
//   rows >= cols:  X P1 = Q1 R1,  R1^H P2 = Q2 R2,  Y = R2^H,  X <- Q1 P2 (Y J)
//   rows <  cols:  X^H P1 = Q1 R1,  Y = R1^H,  X <- P1 (Y J)
// (P: columns by descending norm; Y is at most 32x32).  Y J has orthogonal
// columns U S, so neither J nor Q2 is needed.  A sweep is that of jac_inner on
// the Gram of Y; from |K|_F <= NEWTON_KF on, closing steps as above follow.
// A QR keeps the matrix in registers, column c in the 8 lanes of its group and
// its rows c' = lane, lane + 8, ...: a reduction is three DPP moves and a
// column one barrier (0.6 us at 32 rows).  What bounds the kernel is the chain
// of rounds and reflectors.  32x32, graded over eight decades: load and order 1
// us, QR 19 + 20, two sweeps 42 + 10 (rounds, products), four closing steps 34, Q1
// 5, norms and rank 3; a split of that size in all 721 -> 256 us, 24x32 647 ->
// 246, 60x30 531 -> 265.  Without the second QR 54 us more sweeps, for 25 of QR
// and Q1.  Rows beyond 128 (register columns): the triangle of a QR when there are at
// most 32 columns (tall_svd), else the launches below.
constexpr int SMALL_NT = 256;
constexpr int SMALL_ROWS = 128;
constexpr int SMALL_LDV = SMALL_ROWS + 1;
constexpr int SMALL_LD = JAC_LMAX + 1;
constexpr int SMALL_M = JAC_LMAX * SMALL_LD;   // element (r, c) at c * SMALL_LD + r

struct SmallShared {
  c128 V[JAC_LMAX * SMALL_LDV];   // columns on their way into order, then the reflectors of Q1
  c128 Y[SMALL_M], G[SMALL_M], J0[SMALL_M];
  union {
    c128 m[2][SMALL_M];           // J1 and W of a closing step; reflectors of Q2
    InnerShared inner;
  };
  c128 tau[JAC_LMAX], tau2[JAC_LMAX];
  double key[JAC_LMAX], sorted[JAC_LMAX];
  int rank[JAC_LMAX];
  double red[SMALL_NT / 64];
  int cnt[SMALL_NT / 64];
};

// Sum over the 8 lanes of a group, the same value in each.
__device__ __forceinline__ double sum8(double v) {
  v += dpp_f64<0xB1>(v);    // quad_perm(1,0,3,2)
  v += dpp_f64<0x4E>(v);    // quad_perm(2,3,0,1)
  v += dpp_f64<0x141>(v);   // row_half_mirror
  return v;
}

// Position of key[c] (c = thread / 8) among the 32 keys, largest first.  Keys are
// compared as bit patterns (they are not negative), which orders NaN too: the
// positions are a permutation whatever the keys are.
__device__ __forceinline__ int small_rank(const double* key) {
  const int c = threadIdx.x >> 3, rl = threadIdx.x & 7;
  const unsigned long long mine = __builtin_bit_cast(unsigned long long, key[c]);
  int rank = 0;
#pragma unroll
  for (int i = 0; i < JAC_LMAX / 8; ++i) {
    const int o = rl + 8 * i;
    const unsigned long long other = __builtin_bit_cast(unsigned long long, key[o]);
    const unsigned long long b = __ballot(other > mine || (other == mine && o < c));
    rank += __popc((unsigned)(b >> (threadIdx.x & 56)) & 0xffu);
  }
  return rank;
}

template <int IT>
__device__ __forceinline__ double small_norm2(const c128 (&x)[IT]) {
  double s = 0;
#pragma unroll
  for (int i = 0; i < IT; ++i) s += x[i].re * x[i].re + x[i].im * x[i].im;
  return sum8(s);
}

// Sorts the columns (by `stage`, stride ld) by descending norm; rank[c] is where
// column c went.
template <int IT>
__device__ __forceinline__ void small_sort(c128 (&x)[IT], SmallShared& sh, c128* stage, int ld) {
  const int c = threadIdx.x >> 3, rl = threadIdx.x & 7;
  const double n2 = small_norm2(x);
  if (rl == 0) sh.key[c] = n2;
  __syncthreads();
  const int rank = small_rank(sh.key);
  if (rl == 0) sh.rank[c] = rank;
#pragma unroll
  for (int i = 0; i < IT; ++i) stage[rank * ld + rl + 8 * i] = x[i];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < IT; ++i) x[i] = stage[c * ld + rl + 8 * i];
}

// Householder QR of the columns in x: kq reflectors, to V (column k at k * ld,
// valid from row 8 (k / 8) on) and tau; x becomes (R, v).  The slot of a
// reflector is written by the lanes that read that column of the stage, so V may
// be the stage of small_sort.
template <int IT>
__device__ __forceinline__ void small_qr(c128 (&x)[IT], int kq, c128* V, int ld, c128* tau) {
  const int c = threadIdx.x >> 3, rl = threadIdx.x & 7;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
#pragma unroll
  for (int i0 = 0; i0 < JAC_LMAX / 8; ++i0) {
#pragma unroll 1
    for (int k8 = 0; k8 < 8; ++k8) {
      const int k = 8 * i0 + k8;
      if (k >= kq) return;
      if (wave == i0) {   // columns 8 i0 .. 8 i0 + 7
        double n2 = rl > k8 ? x[i0].re * x[i0].re + x[i0].im * x[i0].im : 0.0;
#pragma unroll
        for (int i = i0 + 1; i < IT; ++i) n2 += x[i].re * x[i].re + x[i].im * x[i].im;
        n2 = sum8(n2);
        c128 alpha{sum8(rl == k8 ? x[i0].re : 0.0), sum8(rl == k8 ? x[i0].im : 0.0)};
        int ex = 0;
        if (c == k && !larfg_in_range(alpha.re * alpha.re + alpha.im * alpha.im + n2)) {
          // squares over- or underflow (all zero in most cases): the reflector of the
          // scaled column is the same
          double top = 0;
#pragma unroll
          for (int i = i0; i < IT; ++i)
            if (i > i0 || rl >= k8) top = fmax(top, fmax(fabs(x[i].re), fabs(x[i].im)));
          for (int o = 4; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o, 8));
          ex = larfg_exponent(top);
          n2 = 0;
#pragma unroll
          for (int i = i0; i < IT; ++i)
            if (i > i0 || rl >= k8) {
              x[i] = c128{ldexp(x[i].re, -ex), ldexp(x[i].im, -ex)};
              if (i > i0 || rl > k8) n2 += x[i].re * x[i].re + x[i].im * x[i].im;
            }
          n2 = sum8(n2);
          alpha = c128{ldexp(alpha.re, -ex), ldexp(alpha.im, -ex)};
        }
        Larfg h = larfg(alpha, n2);
        if (ex) h.beta = ldexp(h.beta, ex);
        if (c == k) {
#pragma unroll
          for (int i = i0; i < IT; ++i) {
            const c128 s{x[i].re * h.scale.re - x[i].im * h.scale.im, x[i].re * h.scale.im + x[i].im * h.scale.re};
            if (i > i0) {
              x[i] = s;
              V[k * ld + rl + 8 * i] = s;
            } else {
              V[k * ld + rl + 8 * i] = rl > k8 ? s : c128{rl == k8 ? 1.0 : 0.0, 0.0};
              if (rl > k8) x[i] = s;
              if (rl == k8) x[i] = c128{h.beta, 0.0};
            }
          }
          if (rl == 0) tau[k] = h.tau;
        }
      }
      __syncthreads();
      if (c > k) {
        c128 v[IT];
        double dr = 0, di = 0;
        const c128 t = tau[k];
#pragma unroll
        for (int i = i0; i < IT; ++i) v[i] = V[k * ld + rl + 8 * i];
#pragma unroll
        for (int i = i0; i < IT; ++i) {
          dr += v[i].re * x[i].re + v[i].im * x[i].im;
          di += v[i].re * x[i].im - v[i].im * x[i].re;
        }
        dr = sum8(dr);
        di = sum8(di);
        const double fr = t.re * dr + t.im * di, fi = t.re * di - t.im * dr;
#pragma unroll
        for (int i = i0; i < IT; ++i) {
          x[i].re -= v[i].re * fr - v[i].im * fi;
          x[i].im -= v[i].re * fi + v[i].im * fr;
        }
      }
    }
  }
}

// z <- H_0 ... H_{kq-1} z for the columns in z.
template <int IT>
__device__ __forceinline__ void small_apply_q(c128 (&z)[IT], int kq, const c128* V, int ld, const c128* tau) {
  const int rl = threadIdx.x & 7;
#pragma unroll
  for (int i0 = JAC_LMAX / 8 - 1; i0 >= 0; --i0) {
#pragma unroll 1
    for (int k = min(8 * i0 + 7, kq - 1); k >= 8 * i0; --k) {
      c128 v[IT];
      double dr = 0, di = 0;
      const c128 t = tau[k];
#pragma unroll
      for (int i = i0; i < IT; ++i) v[i] = V[k * ld + rl + 8 * i];
#pragma unroll
      for (int i = i0; i < IT; ++i) {
        dr += v[i].re * z[i].re + v[i].im * z[i].im;
        di += v[i].re * z[i].im - v[i].im * z[i].re;
      }
      dr = sum8(dr);
      di = sum8(di);
      const double fr = t.re * dr - t.im * di, fi = t.re * di + t.im * dr;
#pragma unroll
      for (int i = i0; i < IT; ++i) {
        z[i].re -= v[i].re * fr - v[i].im * fi;
        z[i].im -= v[i].re * fi + v[i].im * fr;
      }
    }
  }
}

// This wave's 16x16 tile (wave & 1, wave / 2) of op(A) B of matrices in LDS,
// inner dimension kd (16 or 32), handed to out(row, col, value).
template <bool ADJOINT, typename Out>
__device__ __forceinline__ void small_mm(const c128* A, const c128* B, int kd, Out&& out) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i0 = 16 * (wave & 1), j0 = 16 * (wave >> 1);
  if (i0 >= kd || j0 >= kd) return;
  jac_f64x4 re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
  for (int k0 = 0; k0 < kd; k0 += 16) {
    c128 a[4], b[4];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int k = k0 + 4 * s + hi;
      a[s] = ADJOINT ? conj_of(A[(i0 + lo) * SMALL_LD + k]) : A[k * SMALL_LD + i0 + lo];
      b[s] = B[(j0 + lo) * SMALL_LD + k];
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      re = jac_mfma(a[s].re, b[s].re, re);
      im = jac_mfma(a[s].re, b[s].im, im);
      re = jac_mfma(-a[s].im, b[s].im, re);
      im = jac_mfma(a[s].im, b[s].re, im);
    }
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) out(i0 + hi + 4 * r, j0 + lo, c128{re[r], im[r]});
}

// Y <- Y J, G <- Y^H Y.
__device__ __forceinline__ void small_update(SmallShared& sh, const c128* J, int kd) {
  c128 y[4];
  int n = 0, at[4] = {-1, -1, -1, -1};
  small_mm<false>(sh.Y, J, kd, [&](int r, int c, const c128& v) {
    y[n] = v;
    at[n++] = c * SMALL_LD + r;
  });
  __syncthreads();
#pragma unroll
  for (int q = 0; q < 4; ++q)
    if (at[q] >= 0) sh.Y[at[q]] = y[q];
  __syncthreads();
}
__device__ __forceinline__ void small_gram(SmallShared& sh, int kd) {
  small_mm<true>(sh.Y, sh.Y, kd, [&](int r, int c, const c128& v) { sh.G[c * SMALL_LD + r] = v; });
  __syncthreads();
}

// K of the Gram (to m[0]); |K|_F^2 and the pairs above the convergence margin.
__device__ __forceinline__ void small_corr(SmallShared& sh, int kq, const InnerThresholds& th, double& kf, int& above) {
  c128* K = sh.m[0];
  double part = 0;
  int sig = 0;
#pragma unroll
  for (int q = 0; q < JAC_LMAX * JAC_LMAX / SMALL_NT; ++q) {
    const int i = threadIdx.x & 31, j = (threadIdx.x >> 5) + 8 * q;
    const int a = min(i, j), b = max(i, j);
    const c128 g = sh.G[b * SMALL_LD + a];
    const double pa = sh.G[a * SMALL_LD + a].re, pb = sh.G[b * SMALL_LD + b].re;
    const double ag2 = g.re * g.re + g.im * g.im, ab = pa * pb, d = pb - pa;
    const bool act = a < b && b < kq && !(ag2 <= th.tol2 * ab || ag2 < 1e-300 || fmin(pa, pb) < th.negl);
    const double t = act ? (d >= 0 ? 2.0 : -2.0) / (sqrt(fma(d, d, 4.0 * ag2)) + fabs(d)) : 0.0;
    const c128 k = act ? c128{i < j ? t * g.re : -t * g.re, t * g.im} : c128{0.0, 0.0};
    K[j * SMALL_LD + i] = k;
    part += k.re * k.re + k.im * k.im;
    sig += __popcll(__ballot(act && i < j && ag2 > th.conv2 * ab));
  }
  part = wave_sum64(part);
  if ((threadIdx.x & 63) == 0) {
    sh.red[threadIdx.x >> 6] = part;
    sh.cnt[threadIdx.x >> 6] = sig;
  }
  __syncthreads();
  kf = (sh.red[0] + sh.red[1]) + (sh.red[2] + sh.red[3]);
  above = (sh.cnt[0] + sh.cnt[1]) + (sh.cnt[2] + sh.cnt[3]);
}

// One-sided Jacobi on the columns of Y (kq of them, zero elsewhere); returns
// whether they are orthogonal, and the sweeps it took.
__device__ __forceinline__ bool small_jacobi(SmallShared& sh, int kq, const InnerThresholds& th, int& sweeps) {
  const int P = threadIdx.x >> 4, Q = (threadIdx.x + P) & 15;
  const int kd = kq > 16 ? 32 : 16;
  int h0 = 16;   // pairs of the first rounds: half the columns
  while (h0 > 1 && kq <= h0) h0 >>= 1;
  const int iP = (P / h0) * 2 * h0 + P % h0, iQ = (Q / h0) * 2 * h0 + Q % h0;
  int steps = 0;
  small_gram(sh, kd);
  for (sweeps = 0; sweeps < JAC_MAX_SWEEPS;) {
    c128 g[4], j[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int r = iP + h0 * (q / 2), c = iQ + h0 * (q & 1);
      g[q] = r < kd && c < kd ? sh.G[c * SMALL_LD + r] : c128{0.0, 0.0};
      j[q] = c128{P + 16 * (q / 2) == c ? 1.0 : 0.0, 0.0};
    }
    int total = 0, above = 0;
    if (h0 == 16) {
      inner_rounds<16>(g, j, sh.inner, th, total, above);
      inner_regroup<16>(g, j, sh.inner);
    }
    if (h0 >= 8) {
      inner_rounds<8>(g, j, sh.inner, th, total, above);
      inner_regroup<8>(g, j, sh.inner);
    }
    if (h0 >= 4) {
      inner_rounds<4>(g, j, sh.inner, th, total, above);
      inner_regroup<4>(g, j, sh.inner);
    }
    if (h0 >= 2) {
      inner_rounds<2>(g, j, sh.inner, th, total, above);
      inner_regroup<2>(g, j, sh.inner);
    }
    inner_rounds<1>(g, j, sh.inner, th, total, above);
    ++sweeps;
    // the counts of one wave decide for all
    if (threadIdx.x == 0) {
      sh.cnt[0] = total;
      sh.cnt[1] = above;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) sh.J0[(2 * Q + (q & 1)) * SMALL_LD + P + 16 * (q / 2)] = j[q];
    __syncthreads();
    total = sh.cnt[0];
    above = sh.cnt[1];
    if (total == 0) return true;
    small_update(sh, sh.J0, kd);
    if (above == 0) return true;
    small_gram(sh, kd);
    double kf;
    small_corr(sh, kq, th, kf, above);
    for (; kf <= NEWTON_KF * NEWTON_KF && steps < NEWTON_MAX; ++steps) {
      c128 *K = sh.m[0], *W = sh.m[1];
      small_mm<true>(K, K, kd, [&](int r, int c, const c128& v) {
        const c128 k = K[c * SMALL_LD + r];
        sh.J0[c * SMALL_LD + r] = c128{(r == c ? 1.0 : 0.0) + k.re - 0.5 * v.re, k.im - 0.5 * v.im};
      });
      __syncthreads();
      c128 *A = sh.J0, *B = K;
      int schulz = 0;
      for (double e = 0.25 * kf * kf; e > 1e-17 && schulz < NEWTON_SCHULZ_MAX; e = 0.75 * e * e, ++schulz) {
        small_mm<true>(A, A, kd, [&](int r, int c, const c128& v) { W[c * SMALL_LD + r] = v; });
        __syncthreads();
        small_mm<false>(A, W, kd, [&](int r, int c, const c128& v) {
          const c128 z = A[c * SMALL_LD + r];
          B[c * SMALL_LD + r] = c128{1.5 * z.re - 0.5 * v.re, 1.5 * z.im - 0.5 * v.im};
        });
        __syncthreads();
        c128* t = A;
        A = B;
        B = t;
      }
      small_update(sh, A, kd);
      small_gram(sh, kd);
      small_corr(sh, kq, th, kf, above);
      if (above == 0) return true;
    }
  }
  return false;
}

template <int IT>
__device__ __forceinline__ void jac_small_body(const c128* __restrict__ in, int ld, c128* __restrict__ X, int rows,
                                               int cols, double* __restrict__ sigma, int* __restrict__ perm,
                                               SvdResult* __restrict__ res, int chi_max, double eps, int rank_cap,
                                               double tol, SmallShared& sh) {
  const int tid = threadIdx.x, c = tid >> 3, rl = tid & 7;
  const bool wide = rows < cols;
  const int kq = min(rows, cols), nr = max(rows, cols);
  c128 x[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int r = rl + 8 * i, cc = min(c, kq - 1), rr = min(r, nr - 1);
    x[i] = wide ? conj_of(in[rr * ld + cc]) : in[cc * ld + rr];
    if (c >= kq || r >= nr || (ld > rows && r > c)) x[i] = c128{0.0, 0.0};
  }
  small_sort(x, sh, sh.V, SMALL_LDV);
  double fro = 0;
  for (int q = 0; q < JAC_LMAX; ++q) fro += sh.key[q];
  const double conv = jac_conv_tol(tol, kq);
  const InnerThresholds th{tol * tol, conv * conv, JAC_NOISE2 * fro};
  small_qr(x, kq, sh.V, SMALL_LDV, sh.tau);
  // R^H: column r is the conjugate of row r of R
  auto adjoint = [&](c128* out, const c128* r4) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = rl + 8 * i;
      out[r * SMALL_LD + c] = r <= c ? conj_of(r4[i]) : c128{0.0, 0.0};
    }
    __syncthreads();
  };
  if (wide) {
    adjoint(sh.Y, x);
  } else {
    adjoint(sh.G, x);
    c128 b[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) b[i] = sh.G[c * SMALL_LD + rl + 8 * i];
    small_sort(b, sh, sh.m[0], SMALL_LD);
    small_qr(b, kq, sh.m[0], SMALL_LD, sh.tau2);
    adjoint(sh.Y, b);
  }
  int sweeps;
  const bool converged = small_jacobi(sh, kq, th, sweeps);
  // left singular vectors times singular values, and their norms: those of the
  // columns as they leave, so that the isometry's columns are normalised to the last
  // bits (from the norms before Q1, up to 16x16 cells: 3.0e-16 against 1.6e-16)
  c128 z[IT];
  const int me = c < kq ? c : 0;
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const int r = rl + 8 * i;
    z[i] = i < 4 && r < kq ? sh.Y[me * SMALL_LD + sh.rank[r & 31]] : c128{0.0, 0.0};
  }
  if (!wide) small_apply_q(z, kq, sh.V, SMALL_LDV, sh.tau);
  const double n2 = small_norm2(z);
  if (rl == 0) sh.key[c] = c < kq ? sqrt(n2) : 0.0;
  if (c < kq)
#pragma unroll
    for (int i = 0; i < IT; ++i)
      if (rl + 8 * i < rows) X[c * rows + rl + 8 * i] = z[i];
  __syncthreads();
  const int rank = small_rank(sh.key);
  if (rl == 0) {
    sh.sorted[rank] = sh.key[c];
    if (c < kq) {   // padding sorts behind
      sigma[rank] = sh.key[c];
      perm[rank] = c;
    }
  }
  __syncthreads();
  if (tid >= 64) return;
  // first i (< cap) with ||s[i:]|| < eps over the values a reduced SVD returns:
  // lane e sums s[e:] from the smallest value up
  const int ns = min(rank_cap, kq), cap = min(chi_max, ns);
  const double s = tid < ns ? sh.sorted[tid] : 0.0, s2 = s * s;
  double suffix = 0;
  for (int e = ns - 1; e >= 0; --e) {
    const double v = readlane_f64(s2, e);
    if (e >= tid) suffix += v;
  }
  const unsigned long long below = __ballot(tid < cap && sqrt(suffix) < eps);
  const int k = below ? __ffsll((unsigned long long)below) - 1 : cap;
  double kept = 0, tail = 0;
  for (int e = 0; e < ns; ++e) {
    const double v = readlane_f64(s2, e);
    if (e < k) kept += v;
    else tail += v;
  }
  if (tid == 0) {
    res->k = k;
    res->nsweeps = sweeps;
    res->converged = converged;
    res->nsteps = 0;
    res->norm_kept = sqrt(kept);
    res->tail = sqrt(tail);
  }
}
// Rows of the tall orientation in registers: 32, 64 or 128.  `in` is X itself (ld =
// rows), or the square matrix is the triangle of a QR above the diagonal of a taller
// matrix (ld > rows).
__device__ __forceinline__ void jac_small_rows(const c128* in, int ld, c128* X, int rows, int cols, double* sigma,
                                               int* perm, SvdResult* res, int chi_max, double eps, int rank_cap,
                                               double tol) {
  __shared__ SmallShared sh;
  const int nr = max(rows, cols);
  if (nr <= 32) jac_small_body<4>(in, ld, X, rows, cols, sigma, perm, res, chi_max, eps, rank_cap, tol, sh);
  else if (nr <= 64) jac_small_body<8>(in, ld, X, rows, cols, sigma, perm, res, chi_max, eps, rank_cap, tol, sh);
  else jac_small_body<16>(in, ld, X, rows, cols, sigma, perm, res, chi_max, eps, rank_cap, tol, sh);
}
__global__ __launch_bounds__(SMALL_NT) void jac_small(const c128* in, int ld, c128* X, int rows, int cols,
                                                      double* __restrict__ sigma, int* __restrict__ perm,
                                                      SvdResult* __restrict__ res, int chi_max, double eps,
                                                      int rank_cap, double tol) {
  jac_small_rows(in, ld, X, rows, cols, sigma, perm, res, chi_max, eps, rank_cap, tol);
}

// ---------------------------------------------------------- QR preconditioning
// order[c]: columns of X (rows x cols) by descending norm (ties by index).  Ranks
// by counting instead of a bitonic sort: 256 columns 25 -> 16.4 us.
__device__ __forceinline__ void col_norm_order_body(const c128* __restrict__ X, int rows, int cols,
                                                    int* __restrict__ order) {
  __shared__ double skey[JAC_MAXCOLS];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nw = JAC_NT / 64;
  for (int c = wave; c < cols; c += nw) {
    const double a = wsum(lane_norm2(X + (long)c * rows, rows, lane));
    if (lane == 0) skey[c] = a;
  }
  __syncthreads();
  for (int c0 = 0; c0 < cols; c0 += JAC_NT / 8) {
    const int c = c0 + (tid >> 3);
    const int rank = key_rank(skey, cols, c);
    if (c < cols && (tid & 7) == 0) order[rank] = c;
  }
}
__global__ __launch_bounds__(JAC_NT) void col_norm_order(const c128* __restrict__ X, int rows, int cols,
                                                         int* __restrict__ order) {
  col_norm_order_body(X, rows, cols, order);
}

// Xp[:, c] = X[:, order[c]], or a copy (order null)
__device__ __forceinline__ void permute_cols_body(const c128* __restrict__ X, int rows, int cols,
                                                  const int* __restrict__ order, c128* __restrict__ Xp,
                                                  unsigned blk, unsigned nblk) {
  for (long e = blk * (long)blockDim.x + threadIdx.x; e < (long)rows * cols;
       e += (long)nblk * blockDim.x) {
    const int c = (int)(e / rows), r = (int)(e - (long)c * rows);
    Xp[e] = X[(long)(order ? order[c] : c) * rows + r];
  }
}
__global__ void permute_cols(const c128* __restrict__ X, int rows, int cols,
                             const int* __restrict__ order, c128* __restrict__ Xp) {
  permute_cols_body(X, rows, cols, order, Xp, blockIdx.x, gridDim.x);
}

// Y = R^H (cols x kq, column-major) from the R on/above the diagonal of the
// QR-factored M (rows x cols): Y(c, k) = conj(R(k, c)), zero for k > c.
__device__ __forceinline__ void rh_from_qr_body(const c128* __restrict__ M, int rows, int cols, int kq,
                                                c128* __restrict__ Y, unsigned blk, unsigned nblk) {
  for (long e = blk * (long)blockDim.x + threadIdx.x; e < (long)cols * kq;
       e += (long)nblk * blockDim.x) {
    const int k = (int)(e / cols), c = (int)(e - (long)k * cols);
    const c128 v = (k <= c) ? M[(long)c * rows + k] : c128{0.0, 0.0};
    Y[e] = c128{v.re, -v.im};
  }
}
__global__ void rh_from_qr(const c128* __restrict__ M, int rows, int cols, int kq,
                           c128* __restrict__ Y) {
  rh_from_qr_body(M, rows, cols, kq, Y, blockIdx.x, gridDim.x);
}

// X[:, j] = |Y[:, j]| * Z[:, j], j < kq: the left singular vectors (columns of
// Z = Q J, orthonormal) scaled by the singular values, the form X J = U S the
// callers gather from.
__device__ __forceinline__ void scale_by_norms_body(const c128* __restrict__ Y, int yrows,
                                                    const c128* __restrict__ Z, int rows, int kq,
                                                    c128* __restrict__ X, unsigned blk, unsigned nblk) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  for (int j = blk * (JAC_NT / 64) + wave; j < kq; j += nblk * (JAC_NT / 64)) {
    const double sg = sqrt(wsum(lane_norm2(Y + (long)j * yrows, yrows, lane)));
    for (int r = lane; r < rows; r += 64) {
      const c128 z = Z[(long)j * rows + r];
      X[(long)j * rows + r] = c128{sg * z.re, sg * z.im};
    }
  }
}
__global__ __launch_bounds__(JAC_NT) void scale_by_norms(const c128* __restrict__ Y, int yrows,
                                                         const c128* __restrict__ Z, int rows, int kq,
                                                         c128* __restrict__ X) {
  scale_by_norms_body(Y, yrows, Z, rows, kq, X, blockIdx.x, gridDim.x);
}

// ------------------------------------------------------------------ grouped kernels
struct JacSmallArgs {
  const c128* in;
  int ld;
  c128* X;
  int rows, cols;
  double* sigma;
  int* perm;
  SvdResult* res;
  int chi_max;
  double eps;
  int rank_cap;
  double tol;
};
struct ColOrderArgs {
  const c128* X;
  int rows, cols;
  int* order;
  c128* Xp;          // permute_cols output
};
struct RhArgs {
  const c128* M;
  int rows, cols, kq;
  c128* Y;
};
struct ScaleArgs {
  const c128* Y;
  int yrows;
  const c128* Z;
  int rows, kq;
  c128* X;
};
// The block Jacobi of one matrix (gram_jacobi's launch arguments).
struct JacArgs {
  c128* Y;
  JacobiGeom g;
  c128* Z;
  JacobiGeom gz;
  JacobiCtrl* ctrl;
  int* rotated;
  c128* Gpart;
  c128* Jbuf;
  double tol;
};
struct FinArgs {
  const c128* X;
  int rows, cols;
  double* sigma;
  int* perm;
  SvdResult* res;
  int chi_max;
  double eps;
  int rank_cap;
  const JacobiCtrl* ctrl;
};

__global__ __launch_bounds__(SMALL_NT) void jac_small_grouped(const GRec<JacSmallArgs>* __restrict__ recs, int n) {
  const JacSmallArgs a = recs[blockIdx.x].a;
  jac_small_rows(gbl(a.in), a.ld, gbl(a.X), a.rows, a.cols, gbl(a.sigma), gbl(a.perm), gbl(a.res), a.chi_max, a.eps, a.rank_cap,
                 a.tol);
}
__global__ __launch_bounds__(JAC_NT) void col_norm_order_grouped(const GRec<ColOrderArgs>* __restrict__ recs,
                                                                 int n) {
  const ColOrderArgs a = recs[blockIdx.x].a;
  col_norm_order_body(gbl(a.X), a.rows, a.cols, gbl(a.order));
}
__global__ void permute_cols_grouped(const GRec<ColOrderArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<ColOrderArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  permute_cols_body(gbl(r.a.X), r.a.rows, r.a.cols, r.a.order ? gbl(r.a.order) : nullptr, gbl(r.a.Xp), bx, r.grid.x);
}
__global__ void rh_from_qr_grouped(const GRec<RhArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<RhArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  rh_from_qr_body(gbl(r.a.M), r.a.rows, r.a.cols, r.a.kq, gbl(r.a.Y), bx, r.grid.x);
}
__global__ __launch_bounds__(JAC_NT) void scale_by_norms_grouped(const GRec<ScaleArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<ScaleArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  scale_by_norms_body(gbl(r.a.Y), r.a.yrows, gbl(r.a.Z), r.a.rows, r.a.kq, gbl(r.a.X), bx, r.grid.x);
}
__global__ __launch_bounds__(JAC_NT) void jac_init_grouped(const GRec<JacArgs>* __restrict__ recs, int n) {
  const JacArgs& a = recs[blockIdx.x].a;
  jac_init_body(gbl(a.Y), (long)a.g.rows * a.g.cols, gbl(a.ctrl));
}
// Rounds beyond a matrix's own tournament (nb - 1 rounds) are no-ops for it.
__global__ __launch_bounds__(JAC_GRAM_NT) void jac_gram_grouped(const GRec<JacArgs>* __restrict__ recs, int n,
                                                           int round) {
  unsigned bx, by, bz;
  const GRec<JacArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const JacobiGeom g = r.a.g;
  if (round >= g.nb - 1) return;
  jac_gram_body(gbl(r.a.Y), g, round, gbl(r.a.Gpart), gbl(r.a.ctrl), bx, by);
}
__global__ __launch_bounds__(JAC_INNER_NT) void jac_inner_grouped(const GRec<JacArgs>* __restrict__ recs, int n,
                                                            int round, int sweep) {
  unsigned bx, by, bz;
  const GRec<JacArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const JacobiGeom g = r.a.g;
  if (round >= g.nb - 1) return;
  jac_inner_body(g, round, sweep, gbl(r.a.Gpart), gbl(r.a.Jbuf), gbl(r.a.rotated), r.a.tol, gbl(r.a.ctrl), bx);
}
__global__ __launch_bounds__(JAC_APPLY_NT) void jac_apply_grouped(const GRec<JacArgs>* __restrict__ recs, int n,
                                                            int round) {
  unsigned bx, by, bz;
  const GRec<JacArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const JacobiGeom g = r.a.g, gz = r.a.gz;
  if (round >= g.nb - 1) return;
  jac_apply_body(gbl(r.a.Y), g, gbl(r.a.Z), gz, round, gbl(r.a.Jbuf), gbl(r.a.rotated), gbl(r.a.ctrl), bx, by);
}
__global__ void jac_check_grouped(const GRec<JacArgs>* __restrict__ recs) {
  jac_check_body(gbl(recs[blockIdx.x].a.ctrl));
}
// out[i] = 0: matrix i sweeps, 1: closing phase, 2: converged (one thread per record)
__global__ void jac_state_gather(const GRec<JacArgs>* __restrict__ recs, int n, int* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = recs[i].a.ctrl->done ? 2 : recs[i].a.ctrl->phase;
}
__global__ __launch_bounds__(JAC_NT) void jac_finalize_grouped(const GRec<FinArgs>* __restrict__ recs, int n) {
  const FinArgs a = recs[blockIdx.x].a;
  finalize_body(gbl(a.X), a.rows, a.cols, gbl(a.sigma), gbl(a.perm), gbl(a.res), a.chi_max, a.eps, a.rank_cap,
                gbl(a.ctrl));
}

}  // namespace

JacobiLayout jacobi_layout(int rows, int cols) {
  JacobiLayout l;
  l.nb = std::max(2, ceil_div(cols, JAC_BS));
  if (l.nb & 1) ++l.nb;
  l.kspl = ceil_div(rows, JAC_RC);
  QCA_CHECK(l.kspl <= JAC_MAXKSPL, "Jacobi rows out of range (1..512)");
  const long L = JAC_LMAX, np = l.nb / 2;
  l.gpart_elems = np * l.kspl * L * L;
  l.j_elems = np * L * L;
  l.bytes = JAC_CTRL_BYTES + (sizeof(int) * np + 15) / 16 * 16 + sizeof(c128) * (l.gpart_elems + l.j_elems);
  return l;
}

// Closing phase of an n-column matrix: K, W, J0 and J1, K and W large enough for
// the new Y and Q, and the per-tile sums.
size_t newton_bytes(int rows, int n) {
  const size_t t = ceil_div(n, 16);
  return 4 * sizeof(c128) * (size_t)rows * n + 16 * t * t;
}

// Blocks and closing phase of the min(rows, cols) columns of R^H, in either
// orientation.
size_t jacobi_workspace_bytes(int max_rows, int max_cols) {
  const int n = std::min(max_rows, max_cols), m = std::max(max_rows, max_cols);
  return jacobi_layout(m, n).bytes + newton_bytes(m, n) + 1024;
}

bool small_svd(int rows, int cols) {
  return std::min(rows, cols) <= JAC_LMAX && std::max(rows, cols) <= SMALL_ROWS;
}
// Longer than the one workgroup's registers hold, but no wider: the workgroup takes
// the triangle of a QR.  130 x 2 151 us for the whole split (sweeps in one workgroup
// 143, the launches 307), 130 x 16 214 (286, 350), 512 x 32 346 (897, 454): at every
// size ahead of the launches.
bool tall_svd(int rows, int cols) { return rows > SMALL_ROWS && cols <= JAC_LMAX; }

namespace {

NewtonArgs newton_args(c128* Y, int yrows, c128* Q, int qrows, int n, unsigned char* at, const unsigned char* base,
                       size_t ws_bytes, JacobiCtrl* ctrl, double tol) {
  NewtonArgs a{};
  a.Y = Y;
  a.Q = Q;
  a.yrows = yrows;
  a.qrows = qrows;
  a.n = n;
  a.ytiles = ceil_div(yrows, 16);
  a.qtiles = ceil_div(qrows, 16);
  a.ntiles = ceil_div(n, 16);
  const long m = (long)std::max(yrows, qrows) * n;
  a.K = reinterpret_cast<c128*>(at);
  a.W = a.K + m;
  a.J0 = a.W + m;
  a.J1 = a.J0 + m;
  a.kf2 = reinterpret_cast<double*>(a.J1 + m);
  a.above = reinterpret_cast<int*>(a.kf2 + (long)a.ntiles * a.ntiles);
  QCA_CHECK(reinterpret_cast<unsigned char*>(a.above + (long)a.ntiles * a.ntiles) - base <= (long)ws_bytes,
            "Jacobi workspace too small");
  a.ctrl = ctrl;
  a.tol = tol;
  return a;
}

// One closing step of one matrix, and the state it leaves.
void newton_step(const NewtonArgs& a, hipStream_t s) {
  const dim3 nn(a.ntiles, a.ntiles), t(NEWTON_NT);
  hipLaunchKernelGGL(newton_kernel<NEWTON_START>, nn, t, 0, s, a, 0);
  for (int step = 1; step <= NEWTON_SCHULZ_MAX; ++step) {
    hipLaunchKernelGGL(newton_kernel<NEWTON_GRAM>, nn, t, 0, s, a, step);
    hipLaunchKernelGGL(newton_kernel<NEWTON_SCHULZ>, nn, t, 0, s, a, step);
  }
  hipLaunchKernelGGL(newton_kernel<NEWTON_APPLY>, dim3(a.ytiles + a.qtiles, a.ntiles), t, 0, s, a, 0);
  hipLaunchKernelGGL(newton_kernel<NEWTON_COPY>, dim3(256), t, 0, s, a, 0);
  hipLaunchKernelGGL(newton_kernel<NEWTON_CORR>, nn, t, 0, s, a, 1);
  hipLaunchKernelGGL(newton_decide, dim3(1), t, 0, s, a, -1);
}

// Gram-based block Jacobi on the columns of Y (rows x cols) and its closing
// phase, the same rotations applied to the columns of Z (zrows x cols); leaves
// the control block in the workspace for the finalize.
JacobiCtrl* gram_jacobi(c128* Y, int rows, int cols, c128* Z, int zrows, hipStream_t s,
                        JacobiWork& w) {
  const JacobiLayout l = jacobi_layout(rows, cols);
  QCA_CHECK(l.bytes <= w.ws_bytes, "Jacobi workspace too small");
  static_assert(sizeof(JacobiCtrl) <= JAC_CTRL_BYTES, "control block exceeds its slot");
  unsigned char* base = reinterpret_cast<unsigned char*>(w.ws);
  JacobiCtrl* ctrl = reinterpret_cast<JacobiCtrl*>(base);
  int* rotated = reinterpret_cast<int*>(base + JAC_CTRL_BYTES);
  c128* Gpart = reinterpret_cast<c128*>(base + JAC_CTRL_BYTES + ((sizeof(int) * (l.nb / 2) + 15) / 16) * 16);
  c128* Jbuf = Gpart + l.gpart_elems;
  const JacobiGeom g{rows, cols, l.nb, l.kspl};
  const JacobiGeom gz{zrows, cols, l.nb, ceil_div(zrows, JAC_RC)};
  const int np = l.nb / 2;
  const double tol = w.tol > 0 ? w.tol : 1.1102230246251565e-16 * sqrt((double)rows);
  const NewtonArgs na = newton_args(Y, rows, Z, zrows, cols, reinterpret_cast<unsigned char*>(Jbuf + l.j_elems),
                                    base, w.ws_bytes, ctrl, tol);
  const dim3 nn(na.ntiles, na.ntiles);
  hipLaunchKernelGGL(jac_init, dim3(1), dim3(JAC_NT), 0, s, Y, (long)rows * cols, ctrl);
  // Launch the sweeps and closing steps of the previous call, then read the
  // device's state once per chunk (what is launched beyond it does nothing).
  int sweep = 0, chunk = std::max(2, w.pred_sweeps), steps = std::max(1, w.pred_newton);
  while (sweep < JAC_MAX_SWEEPS || steps > 0) {
    for (int c = 0; c < chunk && sweep < JAC_MAX_SWEEPS; ++c, ++sweep) {
      for (int r = 0; r < l.nb - 1; ++r) {
        hipLaunchKernelGGL(jac_gram, dim3(np, l.kspl), dim3(JAC_GRAM_NT), 0, s, (const c128*)Y, g, r,
                           Gpart, (const JacobiCtrl*)ctrl);
        hipLaunchKernelGGL(jac_inner, dim3(np), dim3(JAC_INNER_NT), 0, s, g, r, sweep, (const c128*)Gpart,
                           Jbuf, rotated, tol, ctrl);
        hipLaunchKernelGGL(jac_apply, dim3(np, l.kspl + gz.kspl), dim3(JAC_APPLY_NT), 0, s, Y, g, Z, gz, r,
                           (const c128*)Jbuf, (const int*)rotated, (const JacobiCtrl*)ctrl);
      }
      if (sweep == 0) {   // never enters the closing phase
        hipLaunchKernelGGL(jac_check, dim3(1), dim3(64), 0, s, ctrl);
      } else {
        hipLaunchKernelGGL(newton_kernel<NEWTON_CORR>, nn, dim3(NEWTON_NT), 0, s, na, 0);
        hipLaunchKernelGGL(newton_decide, dim3(1), dim3(NEWTON_NT), 0, s, na, sweep);
      }
    }
    for (int q = 0; q < steps; ++q) newton_step(na, s);
    QCA_HIP(hipGetLastError());
    QCA_HIP(hipMemcpyAsync(w.host, &ctrl->done, 4 * sizeof(int), hipMemcpyDeviceToHost, s));
    QCA_HIP(hipStreamSynchronize(s));
    const int* hc = reinterpret_cast<const int*>(w.host);   // done, sweeps, phase, newton
    if (hc[0]) {
      w.pred_sweeps = hc[1];
      w.pred_newton = hc[3];
      break;
    }
    // in the closing phase: more steps; else a sweep and the steps after it
    chunk = hc[2] ? 0 : 1;
    steps = hc[2] ? 1 : (hc[3] < NEWTON_MAX && sweep < JAC_MAX_SWEEPS ? 2 : 0);
  }
  return ctrl;
}

}  // namespace

size_t jacobi_precond_elems(int max_rows, int max_cols) {
  const long kq = std::min(max_rows, max_cols);
  return (size_t)max_rows * max_cols       // column-permuted copy, then R / reflectors
         + (size_t)max_rows * kq           // Q, then Q J
         + (size_t)max_cols * kq           // Y = R^H
         + qr_workspace_elems(max_rows, max_cols);
}

namespace {
// X = Q R, R = U' S V^H in one workgroup, X <- Q (U' S): the copy that becomes V and
// R, U' S, and T, in the preconditioning workspace.
struct TallSvd {
  c128 *Xp, *Z, *T;
  size_t t_elems;
  TallSvd(c128* pre, size_t elems, int rows, int cols)
      : Xp(pre), Z(Xp + (long)rows * cols), T(Z + (long)cols * cols), t_elems(elems - (size_t)(T - pre)) {}
};
}  // namespace

void launch_jacobi_svd(c128* X, int rows, int cols, double* sigma, int* perm, SvdResult* res,
                       int chi_max, double eps, int rank_cap, hipStream_t s, JacobiWork& w) {
  QCA_CHECK(rows >= 1 && rows <= 512, "SVD rows out of range (1..512)");
  QCA_CHECK(cols >= 1 && cols <= JAC_MAXCOLS, "SVD cols out of range (1..512)");
  QCA_CHECK(w.ws != nullptr && w.host != nullptr, "Jacobi workspace not set");
  const int kq = std::min(rows, cols);
  if (small_svd(rows, cols)) {
    const double tol = w.tol > 0 ? w.tol : 1.1102230246251565e-16 * sqrt((double)kq);
    hipLaunchKernelGGL(jac_small, dim3(1), dim3(SMALL_NT), 0, s, (const c128*)X, rows, X, rows, cols, sigma, perm,
                       res, chi_max, eps, rank_cap, tol);
    QCA_HIP(hipGetLastError());
    return;
  }
  QCA_CHECK(w.pre != nullptr && w.pre_elems >= jacobi_precond_elems(rows, cols), "Jacobi workspace too small");
  if (tall_svd(rows, cols)) {
    const TallSvd t(w.pre, w.pre_elems, rows, cols);
    hipLaunchKernelGGL(permute_cols, dim3(256), dim3(256), 0, s, (const c128*)X, rows, cols, (const int*)nullptr, t.Xp);
    launch_blocked_qr(t.Xp, rows, cols, nullptr, 0, t.T, t.t_elems, s);
    const double tol = w.tol > 0 ? w.tol : 1.1102230246251565e-16 * sqrt((double)kq);
    hipLaunchKernelGGL(jac_small, dim3(1), dim3(SMALL_NT), 0, s, (const c128*)t.Xp, rows, t.Z, cols, cols, sigma, perm,
                       res, chi_max, eps, rank_cap, tol);
    launch_form_q(form_q_step(t.Xp, rows, cols, t.T, X, cols, t.Z), s);
    return;
  }
  // Preconditioned: X P = Q R with the columns by descending norm, one-sided
  // Jacobi on Y = R^H with the same rotations applied to Q.  Y J = U' S and
  // Q J = U, the left singular vectors of X, orthonormal by construction.
  c128* Xp = w.pre;
  c128* Q = Xp + (long)rows * cols;
  c128* Y = Q + (long)rows * kq;
  c128* qws = Y + (long)cols * kq;
  const size_t qws_elems = w.pre_elems - (size_t)(qws - w.pre);
  int* order = perm;  // scratch until the finalize writes the permutation
  hipLaunchKernelGGL(col_norm_order, dim3(1), dim3(JAC_NT), 0, s, (const c128*)X, rows, cols, order);
  hipLaunchKernelGGL(permute_cols, dim3(256), dim3(256), 0, s, (const c128*)X, rows, cols,
                     (const int*)order, Xp);
  launch_blocked_qr(Xp, rows, cols, Q, kq, qws, qws_elems, s);
  hipLaunchKernelGGL(rh_from_qr, dim3(256), dim3(256), 0, s, (const c128*)Xp, rows, cols, kq, Y);
  JacobiCtrl* ctrl = gram_jacobi(Y, cols, kq, Q, rows, s, w);
  hipLaunchKernelGGL(jac_finalize, dim3(1), dim3(JAC_NT), 0, s, (const c128*)Y, cols, kq, sigma,
                     perm, res, chi_max, eps, rank_cap, (const JacobiCtrl*)ctrl);
  hipLaunchKernelGGL(scale_by_norms, dim3(ceil_div(kq, JAC_NT / 64)), dim3(JAC_NT), 0, s,
                     (const c128*)Y, cols, (const c128*)Q, rows, kq, X);
  QCA_HIP(hipGetLastError());
}

void grouped_jacobi_svd(const std::vector<SvdJob>& jobs, RecordArena& arena, GroupFlags& flags,
                        hipStream_t s) {
  std::vector<GRec<JacSmallArgs>> small, triangle;
  std::vector<GRec<QrFormArgs>> back;
  int back_rows = 0;
  size_t back_lds = 0;
  std::vector<GRec<ColOrderArgs>> order1, perm;
  std::vector<GRec<RhArgs>> rh;
  std::vector<GRec<ScaleArgs>> scale;
  std::vector<GRec<JacArgs>> jac_one, jac_gram_r, jac_inner_r, jac_apply_r;
  std::vector<GRec<FinArgs>> fin;
  std::vector<QrStep> steps;
  std::vector<GRec<NewtonArgs>> newton_one, newton_nn, newton_app, newton_cp;
  int max_rounds = 0, pred = 2, steps_pred = 1;
  for (const SvdJob& j : jobs) {
    QCA_CHECK(j.rows >= 1 && j.rows <= 512, "SVD rows out of range (1..512)");
    QCA_CHECK(j.cols >= 1 && j.cols <= JAC_MAXCOLS, "SVD cols out of range (1..512)");
    JacobiWork& w = *j.w;
    QCA_CHECK(w.ws != nullptr, "Jacobi workspace not set");
    const int kq = std::min(j.rows, j.cols);
    if (small_svd(j.rows, j.cols)) {
      const double tol = w.tol > 0 ? w.tol : 1.1102230246251565e-16 * sqrt((double)kq);
      small.push_back(grec(JacSmallArgs{j.X, j.rows, j.X, j.rows, j.cols, j.sigma, j.perm, j.res, j.chi_max, j.eps,
                                        j.rank_cap, tol}, 1));
      continue;
    }
    QCA_CHECK(w.pre != nullptr && w.pre_elems >= jacobi_precond_elems(j.rows, j.cols), "Jacobi workspace too small");
    if (tall_svd(j.rows, j.cols)) {
      const TallSvd t(w.pre, w.pre_elems, j.rows, j.cols);
      const double tol = w.tol > 0 ? w.tol : 1.1102230246251565e-16 * sqrt((double)kq);
      perm.push_back(grec(ColOrderArgs{j.X, j.rows, j.cols, nullptr, t.Xp}, 256));
      for (QrStep& st : blocked_qr_steps(t.Xp, j.rows, j.cols, nullptr, 0, t.T, t.t_elems)) steps.push_back(st);
      triangle.push_back(grec(JacSmallArgs{t.Xp, j.rows, t.Z, j.cols, j.cols, j.sigma, j.perm, j.res, j.chi_max, j.eps,
                                           j.rank_cap, tol}, 1));
      const QrStep f = form_q_step(t.Xp, j.rows, j.cols, t.T, j.X, j.cols, t.Z);
      back.push_back(grec(f.form, f.blocks));
      back_rows = std::max(back_rows, j.rows);
      back_lds = std::max(back_lds, f.lds);
      continue;
    }
    c128* Xp = w.pre;
    c128* Z = Xp + (long)j.rows * j.cols;
    c128* Y = Z + (long)j.rows * kq;
    c128* qws = Y + (long)j.cols * kq;
    const size_t qws_elems = w.pre_elems - (size_t)(qws - w.pre);
    const ColOrderArgs co{j.X, j.rows, j.cols, j.perm, Xp};
    order1.push_back(grec(co, 1));
    perm.push_back(grec(co, 256));
    for (QrStep& st : blocked_qr_steps(Xp, j.rows, j.cols, Z, kq, qws, qws_elems)) steps.push_back(st);
    rh.push_back(grec(RhArgs{Xp, j.rows, j.cols, kq, Y}, 256));
    scale.push_back(grec(ScaleArgs{Y, j.cols, Z, j.rows, kq, j.X}, ceil_div(kq, JAC_NT / 64)));
    const JacobiLayout l = jacobi_layout(j.cols, kq);
    QCA_CHECK(l.bytes <= w.ws_bytes, "Jacobi workspace too small");
    unsigned char* base = reinterpret_cast<unsigned char*>(w.ws);
    JacArgs a{};
    a.ctrl = reinterpret_cast<JacobiCtrl*>(base);
    a.rotated = reinterpret_cast<int*>(base + JAC_CTRL_BYTES);
    a.Gpart = reinterpret_cast<c128*>(base + JAC_CTRL_BYTES + ((sizeof(int) * (l.nb / 2) + 15) / 16) * 16);
    a.Jbuf = a.Gpart + l.gpart_elems;
    a.Y = Y;
    a.g = JacobiGeom{j.cols, kq, l.nb, l.kspl};
    a.Z = Z;
    a.gz = JacobiGeom{j.rows, kq, l.nb, ceil_div(j.rows, JAC_RC)};
    a.tol = w.tol > 0 ? w.tol : 1.1102230246251565e-16 * sqrt((double)j.cols);
    const int np = l.nb / 2;
    jac_one.push_back(grec(a, 1));
    const NewtonArgs na = newton_args(Y, j.cols, Z, j.rows, kq, reinterpret_cast<unsigned char*>(a.Jbuf + l.j_elems),
                                      base, w.ws_bytes, a.ctrl, a.tol);
    newton_one.push_back(grec(na, 1));
    newton_nn.push_back(grec(na, na.ntiles, na.ntiles));
    newton_app.push_back(grec(na, na.ytiles + na.qtiles, na.ntiles));
    newton_cp.push_back(grec(na, 256));
    jac_gram_r.push_back(grec(a, np, l.kspl));
    jac_inner_r.push_back(grec(a, np));
    jac_apply_r.push_back(grec(a, np, l.kspl + a.gz.kspl));
    fin.push_back(grec(FinArgs{Y, j.cols, kq, j.sigma, j.perm, j.res, j.chi_max, j.eps, j.rank_cap, a.ctrl}, 1));
    max_rounds = std::max(max_rounds, l.nb - 1);
    pred = std::max(pred, w.pred_sweeps);
    steps_pred = std::max(steps_pred, w.pred_newton);
  }
  KGroup<JacSmallArgs> g_small, g_triangle;
  KGroup<QrFormArgs> g_back;
  KGroup<ColOrderArgs> g_order, g_perm;
  KGroup<RhArgs> g_rh;
  KGroup<ScaleArgs> g_scale;
  KGroup<JacArgs> g_one, g_gram, g_inner, g_apply;
  KGroup<NewtonArgs> n_one, n_nn, n_app, n_cp;
  KGroup<FinArgs> g_fin;
  g_small.prepare(small, arena);
  g_triangle.prepare(triangle, arena);
  g_back.prepare(back, arena);
  g_order.prepare(order1, arena);
  g_perm.prepare(perm, arena);
  g_rh.prepare(rh, arena);
  g_scale.prepare(scale, arena);
  g_one.prepare(jac_one, arena);
  n_one.prepare(newton_one, arena);
  n_nn.prepare(newton_nn, arena);
  n_app.prepare(newton_app, arena);
  n_cp.prepare(newton_cp, arena);
  g_gram.prepare(jac_gram_r, arena);
  g_inner.prepare(jac_inner_r, arena);
  g_apply.prepare(jac_apply_r, arena);
  g_fin.prepare(fin, arena);
  // blocked QR steps of every preconditioned matrix, slot by slot
  std::sort(steps.begin(), steps.end(), [](const QrStep& x, const QrStep& y) { return x.slot < y.slot; });
  struct Slot {
    int kind;
    size_t lds;
    int rows;
    KGroup<QrStepArgs> step;
    KGroup<QrFormArgs> form;
  };
  std::vector<Slot> slots;
  for (size_t i = 0; i < steps.size();) {
    size_t e = i;
    while (e < steps.size() && steps[e].slot == steps[i].slot) ++e;
    Slot sl{};
    sl.kind = steps[i].kind;
    std::vector<GRec<QrStepArgs>> v;
    std::vector<GRec<QrFormArgs>> f;
    for (size_t k = i; k < e; ++k) {
      sl.lds = std::max(sl.lds, steps[k].lds);
      sl.rows = std::max(sl.rows, sl.kind == 0 ? steps[k].step.rows : steps[k].form.rows);
      if (sl.kind == 0) v.push_back(grec(steps[k].step, steps[k].blocks));
      else f.push_back(grec(steps[k].form, steps[k].blocks));
    }
    sl.step.prepare(v, arena);
    sl.form.prepare(f, arena);
    slots.push_back(sl);
    i = e;
  }
  QCA_CHECK((int)jac_one.size() <= flags.cap, "convergence flag buffer too small");
  arena.upload(s);

  if (!g_small.empty())
    hipLaunchKernelGGL(jac_small_grouped, dim3(g_small.l.blocks), dim3(SMALL_NT), 0, s, g_small.l.recs, g_small.l.n);
  if (!g_order.empty())
    hipLaunchKernelGGL(col_norm_order_grouped, dim3(g_order.l.blocks), dim3(JAC_NT), 0, s, g_order.l.recs,
                       g_order.l.n);
  if (!g_perm.empty())
    hipLaunchKernelGGL(permute_cols_grouped, dim3(g_perm.l.blocks), dim3(256), 0, s, g_perm.l.recs, g_perm.l.n);
  for (const Slot& sl : slots) {
    launch_qr_step_grouped(sl.step, sl.rows, sl.lds, s);
    launch_form_q_grouped(sl.form, sl.rows, sl.lds, s);
  }
  if (!g_triangle.empty()) {
    hipLaunchKernelGGL(jac_small_grouped, dim3(g_triangle.l.blocks), dim3(SMALL_NT), 0, s, g_triangle.l.recs,
                       g_triangle.l.n);
    launch_form_q_grouped(g_back, back_rows, back_lds, s);
  }
  if (!g_rh.empty())
    hipLaunchKernelGGL(rh_from_qr_grouped, dim3(g_rh.l.blocks), dim3(256), 0, s, g_rh.l.recs, g_rh.l.n);
  QCA_HIP(hipGetLastError());
  if (!g_one.empty()) {
    hipLaunchKernelGGL(jac_init_grouped, dim3(g_one.l.blocks), dim3(JAC_NT), 0, s, g_one.l.recs, g_one.l.n);
    const int nj = g_one.l.n;
    const dim3 nt(NEWTON_NT);
    auto check = [&](int sweep) {
      if (sweep == 0) {
        hipLaunchKernelGGL(jac_check_grouped, dim3(g_one.l.n), dim3(64), 0, s, g_one.l.recs);
        return;
      }
      hipLaunchKernelGGL(newton_grouped<NEWTON_CORR>, dim3(n_nn.l.blocks), nt, 0, s, n_nn.l.recs, n_nn.l.n, 0);
      hipLaunchKernelGGL(newton_decide_grouped, dim3(n_one.l.n), nt, 0, s, n_one.l.recs, sweep);
    };
    auto step = [&] {
      hipLaunchKernelGGL(newton_grouped<NEWTON_START>, dim3(n_nn.l.blocks), nt, 0, s, n_nn.l.recs, n_nn.l.n, 0);
      for (int q = 1; q <= NEWTON_SCHULZ_MAX; ++q) {
        hipLaunchKernelGGL(newton_grouped<NEWTON_GRAM>, dim3(n_nn.l.blocks), nt, 0, s, n_nn.l.recs, n_nn.l.n, q);
        hipLaunchKernelGGL(newton_grouped<NEWTON_SCHULZ>, dim3(n_nn.l.blocks), nt, 0, s, n_nn.l.recs, n_nn.l.n, q);
      }
      hipLaunchKernelGGL(newton_grouped<NEWTON_APPLY>, dim3(n_app.l.blocks), nt, 0, s, n_app.l.recs, n_app.l.n, 0);
      hipLaunchKernelGGL(newton_grouped<NEWTON_COPY>, dim3(n_cp.l.blocks), nt, 0, s, n_cp.l.recs, n_cp.l.n, 0);
      hipLaunchKernelGGL(newton_grouped<NEWTON_CORR>, dim3(n_nn.l.blocks), nt, 0, s, n_nn.l.recs, n_nn.l.n, 1);
      hipLaunchKernelGGL(newton_decide_grouped, dim3(n_one.l.n), nt, 0, s, n_one.l.recs, -1);
    };
    int sweep = 0, chunk = std::max(2, pred), steps = steps_pred, steps_done = 0;
    while (sweep < JAC_MAX_SWEEPS || steps > 0) {
      for (int c = 0; c < chunk && sweep < JAC_MAX_SWEEPS; ++c, ++sweep) {
        for (int r = 0; r < max_rounds; ++r) {
          hipLaunchKernelGGL(jac_gram_grouped, dim3(g_gram.l.blocks), dim3(JAC_GRAM_NT), 0, s, g_gram.l.recs,
                             g_gram.l.n, r);
          hipLaunchKernelGGL(jac_inner_grouped, dim3(g_inner.l.blocks), dim3(JAC_INNER_NT), 0, s, g_inner.l.recs,
                             g_inner.l.n, r, sweep);
          hipLaunchKernelGGL(jac_apply_grouped, dim3(g_apply.l.blocks), dim3(JAC_APPLY_NT), 0, s, g_apply.l.recs,
                             g_apply.l.n, r);
        }
        check(sweep);
      }
      for (int q = 0; q < steps; ++q, ++steps_done) step();
      hipLaunchKernelGGL(jac_state_gather, dim3(ceil_div(nj, 256)), dim3(256), 0, s, g_one.l.recs, nj, flags.dev);
      QCA_HIP(hipGetLastError());
      QCA_HIP(hipMemcpyAsync(flags.host, flags.dev, sizeof(int) * nj, hipMemcpyDeviceToHost, s));
      QCA_HIP(hipStreamSynchronize(s));
      bool sweeping = false, closing = false;
      for (int i = 0; i < nj; ++i) {
        sweeping = sweeping || flags.host[i] == 0;
        closing = closing || flags.host[i] == 1;
      }
      if (!sweeping && !closing) break;
      // a matrix takes at most NEWTON_MAX closing steps, wherever its sweeps end
      chunk = sweeping ? 1 : 0;
      steps = closing ? 1 : (steps_done < 2 * NEWTON_MAX ? 2 : 0);
    }
    hipLaunchKernelGGL(jac_finalize_grouped, dim3(g_fin.l.blocks), dim3(JAC_NT), 0, s, g_fin.l.recs, g_fin.l.n);
    if (!g_scale.empty())
      hipLaunchKernelGGL(scale_by_norms_grouped, dim3(g_scale.l.blocks), dim3(JAC_NT), 0, s, g_scale.l.recs,
                         g_scale.l.n);
  }
  QCA_HIP(hipGetLastError());
}

}  // namespace qca
