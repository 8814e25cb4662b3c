// Non-GEMM device kernels of the TDVP path (gfx950).
//
//  * wmix      -- sparse MPO mixing between the two GEMMs of every contraction
//  * permute   -- Theta <-> SVD matrix layouts, gathers of singular vectors
//  * lanczos   -- FP64 Krylov exp(-i tau H) v: the three-term step and one classical
//                 Gram-Schmidt pass against the whole basis;
//                 the tridiagonal exponential runs on one wave (Taylor with
//                 scaling) so no host round trip is needed per iteration
//  * measure   -- <n_i> and the single-site density matrix from the transfer
#include "grouped.hpp"
#include "wave.hpp"

#include <cstring>

namespace qca {
namespace {

// ------------------------------------------------------------------ helpers
template <typename T>
__device__ __forceinline__ cplx<T> cmul(cplx<T> a, cplx<T> b) {
  return cplx<T>{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
}
template <typename T>
__device__ __forceinline__ cplx<T> cmulc(cplx<T> a, cplx<T> b) {  // conj(a) * b
  return cplx<T>{a.re * b.re + a.im * b.im, a.re * b.im - a.im * b.re};
}

__device__ __forceinline__ double wave_sum(double v) { return wave_sum64(v); }

// Block-wide sum of a double; blockDim.x must be a multiple of 64, <= 1024.
__device__ double block_sum(double v, double* sh) {
  v = wave_sum(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  const int nw = blockDim.x >> 6;
  double r = 0;
  if (threadIdx.x < 64) {
    r = (l < nw) ? sh[l] : 0.0;
    r = wave_sum(r);
    if (l == 0) sh[0] = r;
  }
  __syncthreads();
  r = sh[0];
  __syncthreads();
  return r;
}

// ------------------------------------------------------------------ wmix
// U[q][xc][v] = sum_{i} Wsp[(q,v), i] * Tin[i][xc]
// A block owns WMIX_XC consecutive xc and runs WMIX_WAVES groups of WMIX_XC
// threads: the input channels of those xc are staged through LDS once (each
// element read from memory once), the groups share the nq*Dout output
// channels, and the output rows [q][xc0..xc0+WMIX_XC)[0..Dout) are written as
// contiguous runs.  32 xc per block (two groups per wave, two blocks' worth of
// LDS per CU at chi = 128) beat 64: 51.5 vs 52.5 us per 2-site H_eff.
constexpr int WMIX_XC = 32;
constexpr int WMIX_WAVES = 16;
constexpr int WMIX_DMAX = 16;

template <typename T>
__device__ __forceinline__ void wmix_body(const cplx<T>* __restrict__ Tin, long in_stride, long nxc,
                                          int nin, cplx<T>* __restrict__ U, int nq, int Dout,
                                          const int* __restrict__ rowptr, const int* __restrict__ col,
                                          const cplx<T>* __restrict__ val, const int* __restrict__ skip,
                                          unsigned blk, unsigned char* smem_raw) {
  if (skip && *skip) return;
  cplx<T>* sin = reinterpret_cast<cplx<T>*>(smem_raw);        // [nin][64]
  cplx<T>* sout = sin + (long)nin * WMIX_XC;                   // [nq][WMIX_XC][Dout]
  const int t = threadIdx.x & (WMIX_XC - 1), wv = threadIdx.x / WMIX_XC;
  const long xc0 = (long)blk * WMIX_XC;
  const long xc = xc0 + t;
  const bool live = xc < nxc;
  for (int i = wv; i < nin; i += WMIX_WAVES)
    sin[i * WMIX_XC + t] = live ? Tin[(long)i * in_stride + xc] : cplx<T>{T(0), T(0)};
  __syncthreads();
  for (int o = wv; o < nq * Dout; o += WMIX_WAVES) {
    const int q = o / Dout, v = o - q * Dout;
    T ar = 0, ai = 0;
    for (int z = rowptr[o]; z < rowptr[o + 1]; ++z) {
      const cplx<T> x = sin[col[z] * WMIX_XC + t];
      const cplx<T> w = val[z];
      ar += w.re * x.re - w.im * x.im;
      ai += w.re * x.im + w.im * x.re;
    }
    sout[((long)q * WMIX_XC + t) * Dout + v] = cplx<T>{ar, ai};
  }
  __syncthreads();
  const int nrun = (int)min<long>(WMIX_XC, nxc - xc0);
  for (int q = 0; q < nq; ++q) {
    cplx<T>* dst = U + ((long)q * nxc + xc0) * Dout;
    const cplx<T>* src = sout + (long)q * WMIX_XC * Dout;
    for (int e = threadIdx.x; e < nrun * Dout; e += WMIX_XC * WMIX_WAVES) dst[e] = src[e];
  }
}

template <typename T>
__global__ __launch_bounds__(WMIX_XC * WMIX_WAVES) void wmix_kernel(
    const cplx<T>* __restrict__ Tin, long in_stride, long nxc, int nin, cplx<T>* __restrict__ U,
    int nq, int Dout, const int* __restrict__ rowptr, const int* __restrict__ col,
    const cplx<T>* __restrict__ val, const int* __restrict__ skip) {
  extern __shared__ unsigned char smem_raw[];
  wmix_body<T>(Tin, in_stride, nxc, nin, U, nq, Dout, rowptr, col, val, skip, blockIdx.x, smem_raw);
}

template <typename T>
__global__ __launch_bounds__(WMIX_XC * WMIX_WAVES) void wmix_grouped(const GRec<WmixArgs<T>>* __restrict__ recs,
                                                                     int n) {
  extern __shared__ unsigned char smem_raw[];
  unsigned bx, by, bz;
  const GRec<WmixArgs<T>>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const WmixArgs<T> a = r.a;
  wmix_body<T>(gbl(a.Tin), a.in_stride, a.nxc, a.nin, gbl(a.U), a.nq, a.Dout, gbl(a.rowptr), gbl(a.col),
               gbl(a.val), gbl(a.skip), bx, smem_raw);
}

// ------------------------------------------------------------------ conversions
template <typename S, typename D>
__device__ __forceinline__ void convert_body(const cplx<S>* __restrict__ in, cplx<D>* __restrict__ out,
                                             long n, const int* __restrict__ skip, unsigned blk,
                                             unsigned nblk) {
  if (skip && *skip) return;
  for (long i = blk * (long)blockDim.x + threadIdx.x; i < n; i += (long)nblk * blockDim.x)
    out[i] = cplx<D>{D(in[i].re), D(in[i].im)};
}
template <typename S, typename D>
__global__ void convert_kernel(const cplx<S>* __restrict__ in, cplx<D>* __restrict__ out, long n,
                               const int* __restrict__ skip) {
  convert_body<S, D>(in, out, n, skip, blockIdx.x, gridDim.x);
}
__global__ void convert_grouped(const GRec<ConvArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<ConvArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  convert_body<double, float>(gbl(r.a.in), gbl(r.a.out), r.a.n, gbl(r.a.skip), bx, r.grid.x);
}

// ------------------------------------------------------------------ permutes
// Theta[p1][p2][a][c] -> column-major X of the SVD matrix M[(p1,a),(p2,c)].
// mode 0: X[j][r] = M[r][j] (columns of M); mode 1: X[r][j] = conj(M[r][j])
// (columns of M^dagger).
__device__ __forceinline__ void theta_to_svd_body(const c128* __restrict__ th, c128* __restrict__ X,
                                                  int chil, int chir, int mode, unsigned blk,
                                                  unsigned nblk) {
  const long m = 2L * chil, n = 2L * chir;
  for (long idx = blk * (long)blockDim.x + threadIdx.x; idx < m * n;
       idx += (long)nblk * blockDim.x) {
    // idx enumerates Theta in memory order: p1, p2, a, c
    const long c = idx % chir;
    long t = idx / chir;
    const long a = t % chil;
    t /= chil;
    const long p2 = t % 2, p1 = t / 2;
    const long r = p1 * chil + a, j = p2 * chir + c;
    c128 v = th[idx];
    if (mode == 0) {
      X[j * m + r] = v;
    } else {
      v.im = -v.im;
      X[r * n + j] = v;
    }
  }
}
__global__ void theta_to_svd(const c128* __restrict__ th, c128* __restrict__ X, int chil, int chir,
                             int mode) {
  theta_to_svd_body(th, X, chil, chir, mode, blockIdx.x, gridDim.x);
}
__global__ void theta_to_svd_grouped(const GRec<ThetaSvdArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<ThetaSvdArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  theta_to_svd_body(gbl(r.a.th), gbl(r.a.X), r.a.chil, r.a.chir, r.a.mode, bx, r.grid.x);
}

// A[p][a][k] = X[perm[k]][(p,a)] / sigma[k]   (mode 0, left isometry from U)
// A[p][k][c] = conj(X[perm[k]][(p,c)]) / sigma[k]  (mode 1, right isometry from V)
__device__ __forceinline__ void gather_isometry_body(const c128* __restrict__ X, const int* __restrict__ perm,
                                                     const double* __restrict__ sigma, c128* __restrict__ A,
                                                     int rows, int chi_bond, int k, int mode, unsigned blk,
                                                     unsigned nblk) {
  // rows = 2*chi_bond (length of each singular vector)
  const long total = (long)rows * k;
  for (long idx = blk * (long)blockDim.x + threadIdx.x; idx < total;
       idx += (long)nblk * blockDim.x) {
    const int kk = (int)(idx % k);
    const int r = (int)(idx / k);
    const double s = sigma[kk];
    const double inv = s > 0 ? 1.0 / s : 0.0;
    c128 v = X[(long)perm[kk] * rows + r];
    const int p = r / chi_bond, a = r - p * chi_bond;
    if (mode == 0) {
      A[((long)p * chi_bond + a) * k + kk] = c128{v.re * inv, v.im * inv};
    } else {
      A[((long)p * k + kk) * chi_bond + a] = c128{v.re * inv, -v.im * inv};
    }
  }
}
__global__ void gather_isometry(const c128* __restrict__ X, const int* __restrict__ perm,
                                const double* __restrict__ sigma, c128* __restrict__ A, int rows,
                                int chi_bond, int k, int mode) {
  gather_isometry_body(X, perm, sigma, A, rows, chi_bond, k, mode, blockIdx.x, gridDim.x);
}
__global__ void gather_isometry_grouped(const GRec<GatherIsoArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<GatherIsoArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const GatherIsoArgs a = r.a;
  gather_isometry_body(gbl(a.X), gbl(a.perm), gbl(a.sigma), gbl(a.A), a.rows, a.chi_bond, a.k, a.mode, bx,
                       r.grid.x);
}

// Row-major (rows x cols) -> column-major copy: out[c*rows + r] = in[r*cols + c]
__global__ void to_colmajor(const c128* __restrict__ in, c128* __restrict__ out, int rows, int cols) {
  const long n = (long)rows * cols;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const long r = e / cols, c = e - r * cols;
    out[c * rows + r] = in[e];
  }
}

// A[p][a][b] -> column-major X of A^T reshaped: X[a][(p,b)], rows = 2*chir
__global__ void site_to_rightqr(const c128* __restrict__ A, c128* __restrict__ X, int chil, int chir) {
  const long n = 2L * chil * chir;
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < n; e += (long)gridDim.x * blockDim.x) {
    const long b = e % chir, t = e / chir;
    const long a = t % chil, p = t / chil;
    X[a * (2L * chir) + p * chir + b] = A[e];
  }
}

// Left QR results: Anew[(p,a)][k] = Q[k][(p,a)] (k < qcols, else 0) for k < target;
// C[k][b] = R[k][b] (upper triangle of X, zero below / beyond min(rows, cols)).
__global__ void qr_gather_left(const c128* __restrict__ Q, const c128* __restrict__ X, c128* __restrict__ Anew,
                               c128* __restrict__ C, int rows, int cols, int qcols, int target) {
  const long na = (long)rows * target, nc = (long)target * cols;
  const int kmin = min(rows, cols);
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < na + nc; e += (long)gridDim.x * blockDim.x) {
    if (e < na) {
      const long r = e / target, k = e - r * target;
      Anew[e] = (k < qcols) ? Q[k * rows + r] : c128{0.0, 0.0};
    } else {
      const long f = e - na;
      const long k = f / cols, b = f - k * cols;
      C[f] = (k <= b && k < kmin) ? X[b * rows + k] : c128{0.0, 0.0};
    }
  }
}

// Right QR results: Anew[p][k][b] = Q[k][(p,b)] (k < qcols, else 0), rows = 2*chir;
// C[a][k] = R[k][a] for k < target.
__global__ void qr_gather_right(const c128* __restrict__ Q, const c128* __restrict__ X, c128* __restrict__ Anew,
                                c128* __restrict__ C, int chir, int cols, int qcols, int target) {
  const int rows = 2 * chir;
  const long na = 2L * target * chir, nc = (long)cols * target;
  const int kmin = min(rows, cols);
  for (long e = blockIdx.x * (long)blockDim.x + threadIdx.x; e < na + nc; e += (long)gridDim.x * blockDim.x) {
    if (e < na) {
      const long b = e % chir, t = e / chir;
      const long k = t % target, p = t / target;
      Anew[e] = (k < qcols) ? Q[k * rows + p * chir + b] : c128{0.0, 0.0};
    } else {
      const long f = e - na;
      const long a = f / target, k = f - a * target;
      C[f] = (k <= a && k < kmin) ? X[a * rows + k] : c128{0.0, 0.0};
    }
  }
}

// ------------------------------------------------------------------ lanczos
// Per iteration three launches after the matvec: lz_dot, <V_j, w>; lz_three_term,
// w <- w - c V_j - beta_{j-1} V_{j-1} with the partial projections of the result
// on the whole basis and its partial norm; lz_next, the Gram-Schmidt pass with
// those, normalisation and the stopping test.  What the three-term step leaves
// along the older vectors is rounding (of the matvec's precision), so one pass
// restores orthogonality, and beta^2 = |w|^2 - sum |c_i|^2 loses nothing.  Two
// full Gram-Schmidt passes with the norm between launches took four launches and
// twice the basis traffic: 22.8 us an iteration at 65536 elements (12 vectors), 3.4 +
// 5.4 + 6.1 us here; what bounds these is launch and memory latency, not traffic.
// Sums over the blocks are taken by every block that needs them, in one fixed
// order: no reduction launch.
constexpr int LZ_BLOCK = 256;   // one vector element per thread
constexpr int LZ_NORM = LZ_MAXK - 1;   // row of the partial sums that holds |w|^2 (j < LZ_NORM)

__device__ __forceinline__ void lz_norm_partials_body(const c128* __restrict__ x, long n,
                                                      double* __restrict__ part, unsigned blk) {
  __shared__ double sh[16];
  double acc = 0;
  const long i = (long)blk * LZ_BLOCK + threadIdx.x;
  if (i < n) acc = x[i].re * x[i].re + x[i].im * x[i].im;
  acc = block_sum(acc, sh);
  if (threadIdx.x == 0) part[blk] = acc;
}
__global__ void lz_norm_partials(const c128* __restrict__ x, long n, double* __restrict__ part) {
  lz_norm_partials_body(x, n, part, blockIdx.x);
}

// V_0 = x / |x|, and its complex64 copy when v32 is given; block 0 opens the
// control block.
__device__ __forceinline__ void lz_scale_first_body(const c128* __restrict__ x, c128* __restrict__ v0,
                                                    long n, const double* __restrict__ part, int nblk,
                                                    LanczosCtrl* ctrl, c64* __restrict__ v32, unsigned blk) {
  __shared__ double sum;
  if (threadIdx.x < 64) {
    double s = 0;
    for (int b = threadIdx.x; b < nblk; b += 64) s += part[b];
    s = wave_sum(s);
    if (threadIdx.x == 0) sum = s;
  }
  __syncthreads();
  const double b = sqrt(sum), inv = b > 0 ? 1.0 / b : 0.0;
  const long i = (long)blk * LZ_BLOCK + threadIdx.x;
  if (i < n) {
    const c128 v{x[i].re * inv, x[i].im * inv};
    v0[i] = v;
    if (v32) v32[i] = c64{float(v.re), float(v.im)};
  }
  if (blk == 0 && threadIdx.x == 0) {
    ctrl->beta0 = b;
    const bool finite = b < __builtin_inf();
    ctrl->zero = (sum == 0.0) ? 1 : 0;
    ctrl->done = sum == 0.0 || !finite ? 1 : 0;
    ctrl->m = 0;
    ctrl->err = 0;
    ctrl->hit_limit = finite ? 0 : LZ_NON_FINITE;
  }
}
__global__ __launch_bounds__(LZ_BLOCK) void lz_scale_first(const c128* __restrict__ x, c128* __restrict__ v0, long n,
                                                           const double* __restrict__ part, int nblk,
                                                           LanczosCtrl* ctrl, c64* __restrict__ v32) {
  lz_scale_first_body(x, v0, n, part, nblk, ctrl, v32, blockIdx.x);
}

// part[blk] = this block's share of <V_j, w>.
template <typename TW>
__device__ __forceinline__ void lz_dot_body(const LanczosCtrl* ctrl, const cplx<TW>* __restrict__ w,
                                            const c128* __restrict__ vj, long n, c128* __restrict__ part,
                                            unsigned blk) {
  const int done = ctrl->done;  // tested once the loads are in flight
  __shared__ c128 sh[LZ_BLOCK / 64];
  const long e = (long)blk * LZ_BLOCK + threadIdx.x;
  double ar = 0, ai = 0;
  if (e < n) {
    const c128 a = vj[e];
    const cplx<TW> x = w[e];
    ar = a.re * double(x.re) + a.im * double(x.im);
    ai = a.re * double(x.im) - a.im * double(x.re);
  }
  if (done) return;
  ar = wave_sum(ar);
  ai = wave_sum(ai);
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = c128{ar, ai};
  __syncthreads();
  if (threadIdx.x == 0) part[blk] = c128{(sh[0].re + sh[1].re) + (sh[2].re + sh[3].re),
                                         (sh[0].im + sh[1].im) + (sh[2].im + sh[3].im)};
}
template <typename TW>
__global__ __launch_bounds__(LZ_BLOCK) void lz_dot(const LanczosCtrl* ctrl, const cplx<TW>* __restrict__ w,
                                                   const c128* __restrict__ vj, long n, c128* __restrict__ part) {
  lz_dot_body<TW>(ctrl, w, vj, n, part, blockIdx.x);
}

// One wave: the sum of part[0..nblk), in every lane.
__device__ __forceinline__ c128 lz_sum(const c128* __restrict__ part, int nblk) {
  double ar = 0, ai = 0;
  for (int b = threadIdx.x & 63; b < nblk; b += 64) {
    const c128 p = part[b];
    ar += p.re;
    ai += p.im;
  }
  return c128{wave_sum(ar), wave_sum(ai)};
}

// w64 = w - c V_j - beta_{j-1} V_{j-1} (promoting w to FP64), c = <V_j, w> from
// lz_dot's shares; this block's shares of <V_i, w64>, i <= j, go to
// part_out[i * nblk + blk], its share of |w64|^2 to row LZ_NORM.
template <typename TW>
__device__ __forceinline__ void lz_three_term_body(const LanczosCtrl* ctrl, const cplx<TW>* __restrict__ w,
                                                   c128* __restrict__ w64, const c128* __restrict__ V, long n,
                                                   int j, const c128* __restrict__ part_in, int nblk,
                                                   c128* __restrict__ coef, c128* __restrict__ part_out,
                                                   unsigned blk) {
  const int done = ctrl->done;  // tested after the loads
  constexpr int NW = LZ_BLOCK / 64;
  __shared__ double sh[NW][LZ_MAXK][2];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const c128 c = lz_sum(part_in, nblk);   // every wave for itself
  const double bp = j > 0 ? ctrl->beta[j - 1] : 0.0;
  const long e = (long)blk * LZ_BLOCK + threadIdx.x;
  const bool in = e < n;
  const long ec = in ? e : n - 1;
  const c128 vj = V[(long)j * n + ec], vp = V[(long)(j > 0 ? j - 1 : 0) * n + ec];
  const cplx<TW> y = w[ec];
  if (done) return;
  const double xr = in ? double(y.re) - (c.re * vj.re - c.im * vj.im + bp * vp.re) : 0.0;
  const double xi = in ? double(y.im) - (c.re * vj.im + c.im * vj.re + bp * vp.im) : 0.0;
  if (in) w64[e] = c128{xr, xi};
  if (blk == 0 && threadIdx.x == 0) coef[j] = c;
  const double nrm = wave_sum(xr * xr + xi * xi);
  if (lane == 0) {
    sh[wv][LZ_NORM][0] = nrm;
    sh[wv][LZ_NORM][1] = 0.0;
  }
#pragma unroll 4
  for (int i = 0; i <= j; ++i) {
    const c128 a = V[(long)i * n + ec];
    const double pr = wave_sum(a.re * xr + a.im * xi), pi = wave_sum(a.re * xi - a.im * xr);
    if (lane == 0) {
      sh[wv][i][0] = pr;
      sh[wv][i][1] = pi;
    }
  }
  __syncthreads();
  const int t = threadIdx.x;
  if (t <= j || t == LZ_NORM) {
    double ar = 0, ai = 0;
    for (int k = 0; k < NW; ++k) {
      ar += sh[k][t][0];
      ai += sh[k][t][1];
    }
    part_out[(long)t * nblk + blk] = c128{ar, ai};
  }
}
template <typename TW>
__global__ __launch_bounds__(LZ_BLOCK) void lz_three_term(const LanczosCtrl* ctrl, const cplx<TW>* __restrict__ w,
                                                          c128* __restrict__ w64, const c128* __restrict__ V, long n,
                                                          int j, const c128* __restrict__ part_in, int nblk,
                                                          c128* __restrict__ coef, c128* __restrict__ part_out) {
  lz_three_term_body<TW>(ctrl, w, w64, V, n, j, part_in, nblk, coef, part_out, blockIdx.x);
}

// One wave: close iteration j.  alpha_j = Re(c_j + c'_j), beta_j = |w|;
// z = exp(-i tau T_{j+1}) e_0 by scaled Taylor steps on the tridiagonal
// (lane = row); converged when beta0*beta_j*|z_j| < tol*beta0.
__device__ void lz_close_iteration(LanczosCtrl* ctrl, double beta, double alpha_j, int j, double tau, double tol,
                                   int max_m) {
  const int l = threadIdx.x & 63;
  if (l == 0) {
    ctrl->alpha[j] = alpha_j;
    ctrl->beta[j] = beta;
  }
  const int m = j + 1;
  if (!(beta < __builtin_inf())) {   // a non-finite start or matvec: the host reports it
    if (l == 0) {
      ctrl->m = m;
      ctrl->done = 1;
      ctrl->hit_limit = LZ_NON_FINITE;
    }
    return;
  }
  // alpha[0..j-1] and beta[0..j-1] were written by earlier launches
  const double al = (l < j) ? ctrl->alpha[l] : ((l == j) ? alpha_j : 0.0);
  const double bup = (l + 1 < m) ? ctrl->beta[l] : 0.0;     // T[l][l+1]
  const double bdn = (l >= 1 && l < m) ? ctrl->beta[l - 1] : 0.0;  // T[l][l-1]
  const bool breakdown = beta <= 1e-13 * fmax(1.0, fabs(alpha_j));
  // The estimate is at least 2 tol by a lower bound of |z_j| (the product of the
  // betas and |tau|^j / j! times the cosine of half the spectrum's phase width,
  // from the divided-difference form of z_j as a mean of exp(-i tau s) over s
  // between Gershgorin's bounds): not converged, without the exponential (2.5 us).
  if (!breakdown && m < max_m - 1) {
    const double r = fabs(bdn) + (l == j ? beta : fabs(bup));
    double prod = l < j ? bup * fabs(tau) / (l + 1) : 1.0;
    double high = l < m ? al + r : -1e300, low = l < m ? r - al : -1e300;   // low: minus the lower bound
    for (int o = 32; o > 0; o >>= 1) {
      prod *= __shfl_xor(prod, o, 64);
      high = fmax(high, __shfl_xor(high, o, 64));
      low = fmax(low, __shfl_xor(low, o, 64));
    }
    const double half = 0.5 * fabs(tau) * (high + low);
    if (half < 1.4 && beta * prod * (1.0 - 0.5 * half * half) >= 2.0 * tol) return;   // cos x >= 1 - x^2 / 2
  }
  double rown = fabs(al) + fabs(bup) + fabs(bdn);
  for (int o = 32; o > 0; o >>= 1) rown = fmax(rown, __shfl_xor(rown, o, 64));
  const double h = fabs(tau) * rown;
  const int nsub = (h < 2048.0) ? max(1, (int)ceil(h / 0.5)) : 1;
  const double dt = tau / nsub;
  // z <- exp(-i dt T) z, nsub times;  multiplying by -i dt: (x+iy)*(-i dt) = dt*y - i dt*x
  double zr = (l == 0) ? 1.0 : 0.0, zi = 0.0;
  for (int sstep = 0; sstep < nsub; ++sstep) {
    double ar = zr, ai = zi, tr = zr, ti = zi;
    for (int k = 1; k < 60; ++k) {
      const double upr = __shfl_down(tr, 1, 64), upi = __shfl_down(ti, 1, 64);
      const double dnr = __shfl_up(tr, 1, 64), dni = __shfl_up(ti, 1, 64);
      double yr = al * tr + bup * upr + bdn * dnr;
      double yi = al * ti + bup * upi + bdn * dni;
      if (l >= m) { yr = 0; yi = 0; }
      const double nr = dt * yi / k, ni = -dt * yr / k;
      tr = nr;
      ti = ni;
      ar += tr;
      ai += ti;
      // stop once every row's term is below 1e-18 (a NaN keeps going, bounded)
      if (__ballot(!(fabs(tr) + fabs(ti) < 1e-18)) == 0) break;
    }
    zr = ar;
    zi = ai;
  }
  const double zlr = __shfl(zr, j, 64), zli = __shfl(zi, j, 64);
  const double err = beta * sqrt(zlr * zlr + zli * zli);
  const bool conv = breakdown || err < tol || m >= max_m - 1;
  if (l < m) {
    ctrl->z[l] = c128{zr, zi};
  }
  if (l == 0) {
    ctrl->err = err;
    if (conv) {
      ctrl->m = m;
      ctrl->done = 1;
      ctrl->hit_limit = (!breakdown && err >= tol) ? 1 : 0;
    }
  }
}

// Closes iteration j: every block sums the projections c_i and the norm, the
// first wave of block 0 takes alpha_j, beta_j and the stopping test, and all
// blocks write V_{j+1} = (w - sum_i c_i V_i) / beta_j, plus its complex64 copy for
// the mixed path's next matvec when v32 is given.  Blocks that start after
// convergence skip the write; V_{j+1} is not read then.
__device__ __forceinline__ void lz_next_body(LanczosCtrl* ctrl, const c128* __restrict__ part, int nblk,
                                             const c128* __restrict__ coef, int j, double tau, double tol, int max_m,
                                             const c128* __restrict__ w, c128* V, c64* __restrict__ v32, long n,
                                             unsigned blk) {
  const int done = ctrl->done;  // tested after the loads
  __shared__ c128 cs[LZ_MAXK];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int i = wv; i <= j + 1; i += LZ_BLOCK / 64) {
    const int row = i <= j ? i : LZ_NORM;
    const c128 c = lz_sum(part + (long)row * nblk, nblk);
    if (lane == 0) cs[row] = c;
  }
  const long e = (long)blk * LZ_BLOCK + threadIdx.x, ec = e < n ? e : n - 1;
  c128 x = w[ec];
  __syncthreads();
  if (done) return;
  double b2 = cs[LZ_NORM].re;
  for (int i = 0; i <= j; ++i) b2 -= cs[i].re * cs[i].re + cs[i].im * cs[i].im;
  const double beta = sqrt(b2 < 0.0 ? 0.0 : b2), inv = 1.0 / beta;   // a NaN stays one
  if (blk == 0 && threadIdx.x < 64) lz_close_iteration(ctrl, beta, coef[j].re + cs[j].re, j, tau, tol, max_m);
#pragma unroll 4
  for (int i = 0; i <= j; ++i) {
    const c128 a = V[(long)i * n + ec], c = cs[i];
    x.re -= c.re * a.re - c.im * a.im;
    x.im -= c.re * a.im + c.im * a.re;
  }
  if (e >= n) return;
  const c128 v{x.re * inv, x.im * inv};
  V[(long)(j + 1) * n + e] = v;
  if (v32) v32[e] = c64{float(v.re), float(v.im)};
}
__global__ __launch_bounds__(LZ_BLOCK) void lz_next(LanczosCtrl* ctrl, const c128* __restrict__ part, int nblk,
                                                    const c128* __restrict__ coef, int j, double tau, double tol,
                                                    int max_m, const c128* __restrict__ w, c128* V,
                                                    c64* __restrict__ v32, long n) {
  lz_next_body(ctrl, part, nblk, coef, j, tau, tol, max_m, w, V, v32, n, blockIdx.x);
}

// y = beta0 * sum_{i<m} z_i V_i   (a zero input stays zero)
__device__ __forceinline__ void lz_combine_body(const LanczosCtrl* ctrl, const c128* __restrict__ V,
                                                long n, c128* __restrict__ y, unsigned blk,
                                                unsigned ngrid) {
  __shared__ c128 zs[LZ_MAXK];
  const int m = ctrl->m;
  const double b0 = ctrl->beta0;
  if (threadIdx.x < m) zs[threadIdx.x] = ctrl->z[threadIdx.x];
  __syncthreads();
  for (long e = blk * (long)blockDim.x + threadIdx.x; e < n; e += (long)ngrid * blockDim.x) {
    double r = 0, im = 0;
    for (int i = 0; i < m; ++i) {
      const c128 a = V[(long)i * n + e];
      r += zs[i].re * a.re - zs[i].im * a.im;
      im += zs[i].re * a.im + zs[i].im * a.re;
    }
    y[e] = c128{b0 * r, b0 * im};
  }
}
__global__ void lz_combine(const LanczosCtrl* ctrl, const c128* __restrict__ V, long n,
                           c128* __restrict__ y) {
  lz_combine_body(ctrl, V, n, y, blockIdx.x, gridDim.x);
}

// ---- grouped Lanczos: one record per instance (LzArgs), the iteration index
// j shared by all instances of the launch (they iterate in lockstep; an
// instance that has converged skips every kernel through its done flag).
__global__ void lz_norm_partials_grouped(const GRec<LzArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<LzArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  lz_norm_partials_body(gbl(r.a.x), r.a.n, gbl(r.a.part_norm), bx);
}
__global__ __launch_bounds__(LZ_BLOCK) void lz_scale_first_grouped(const GRec<LzArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<LzArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  lz_scale_first_body(gbl(r.a.x), gbl(r.a.V), r.a.n, gbl(r.a.part_norm), r.a.nblk, gbl(r.a.ctrl), gbl(r.a.v32), bx);
}
template <typename TW>
__global__ __launch_bounds__(LZ_BLOCK) void lz_dot_grouped(const GRec<LzArgs>* __restrict__ recs, int n, int j) {
  unsigned bx, by, bz;
  const GRec<LzArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  lz_dot_body<TW>(gbl(r.a.ctrl), gbl(reinterpret_cast<const cplx<TW>*>(r.a.w)), gbl(r.a.V + (long)j * r.a.n), r.a.n,
                  gbl(r.a.part), bx);
}
template <typename TW>
__global__ __launch_bounds__(LZ_BLOCK) void lz_three_term_grouped(const GRec<LzArgs>* __restrict__ recs, int n,
                                                                  int j) {
  unsigned bx, by, bz;
  const GRec<LzArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const LzArgs a = r.a;
  lz_three_term_body<TW>(gbl(a.ctrl), gbl(reinterpret_cast<const cplx<TW>*>(a.w)), gbl(a.w64), gbl(a.V), a.n, j,
                         gbl(a.part), a.nblk, gbl(a.coef), gbl(a.part2), bx);
}
__global__ __launch_bounds__(LZ_BLOCK) void lz_next_grouped(const GRec<LzArgs>* __restrict__ recs, int n, int j) {
  unsigned bx, by, bz;
  const GRec<LzArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  const LzArgs a = r.a;
  lz_next_body(gbl(a.ctrl), gbl(a.part2), a.nblk, gbl(a.coef), j, a.tau, a.tol, a.max_m, gbl(a.w64), gbl(a.V),
               gbl(a.v32), a.n, bx);
}
__global__ void lz_combine_grouped(const GRec<LzArgs>* __restrict__ recs, int n) {
  unsigned bx, by, bz;
  const GRec<LzArgs>& r = grec_find(recs, n, blockIdx.x, bx, by, bz);
  lz_combine_body(gbl(r.a.ctrl), gbl(r.a.V), r.a.n, gbl(r.a.y), bx, r.grid.x);
}

// ------------------------------------------------------------------ measurement
// rho[p][q] = sum_{x,b} A[p][x][b] * T[q][x][b], T[q][x][b] = sum_y E[x][y] conj(A[q][y][b])
// One block; writes rho (2x2 complex) for one site.
__global__ void rho_kernel(const c128* __restrict__ A, const c128* __restrict__ T, long nxb,
                           c128* __restrict__ rho) {
  __shared__ double sh[16];
  for (int p = 0; p < 2; ++p)
    for (int q = 0; q < 2; ++q) {
      double ar = 0, ai = 0;
      for (long e = threadIdx.x; e < nxb; e += blockDim.x) {
        const c128 a = A[(long)p * nxb + e], t = T[(long)q * nxb + e];
        ar += a.re * t.re - a.im * t.im;
        ai += a.re * t.im + a.im * t.re;
      }
      ar = block_sum(ar, sh);
      ai = block_sum(ai, sh);
      if (threadIdx.x == 0) rho[p * 2 + q] = c128{ar, ai};
    }
}

// Observables of the reference's MPS.measure (mps.py:122-140) from per-site
// 2x2 density matrices: <n_i> = Re rho[1][1] (not normalised), its rounding
// (half to even, as numpy.round), and -Tr rho log2 rho from the eigenvalues of
// the Hermitian part, (a+d)/2 +- sqrt(((a-d)/2)^2 + |b|^2), with 0 log 0 = 0.
// out = [population(n) | d_population(n) | single_site_entropy(n)].
__global__ void observables_kernel(const c128* __restrict__ rho, int n, double* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const c128 r00 = rho[4 * i], r01 = rho[4 * i + 1], r10 = rho[4 * i + 2], r11 = rho[4 * i + 3];
  const double a = r00.re, d = r11.re;
  const double br = 0.5 * (r01.re + r10.re), bi = 0.5 * (r01.im - r10.im);
  const double mean = 0.5 * (a + d), half = 0.5 * (a - d);
  const double rad = sqrt(half * half + br * br + bi * bi);
  const double lam[2] = {mean + rad, mean - rad};
  double sse = 0.0;
  for (int k = 0; k < 2; ++k)
    if (lam[k] > 0.0) sse -= lam[k] * log2(lam[k]);
  out[i] = d;
  out[n + i] = rint(d);
  out[2 * n + i] = sse;
}

int grid_for(long n, int block = 256, int maxb = 8192) {
  return (int)std::max<long>(1, std::min<long>((n + block - 1) / block, maxb));
}

}  // namespace

// ------------------------------------------------------------------ word gather
__global__ void gather_words_kernel(const void* const* __restrict__ src, int words, int n,
                                    unsigned long long* __restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned long long* p = reinterpret_cast<const unsigned long long*>(src[i]);
  for (int w = 0; w < words; ++w) out[(long)i * words + w] = p[w];
}

void launch_gather_words(const void* const* src, int words, int n, unsigned long long* out, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(gather_words_kernel, dim3(ceil_div(n, 64)), dim3(64), 0, s, src, words, n, out);
  QCA_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ record arena
void RecordArena::reserve(size_t bytes) {
  if (bytes <= cap_) return;
  QCA_CHECK(used_ == 0, "record arena grown while holding records");
  release();
  QCA_HIP(hipHostMalloc((void**)&host_, bytes));
  QCA_HIP(hipMalloc((void**)&dev_, bytes));
  cap_ = bytes;
}

void RecordArena::release() {
  if (host_) (void)hipHostFree(host_);
  if (dev_) (void)hipFree(dev_);
  host_ = dev_ = nullptr;
  cap_ = used_ = uploaded_ = 0;
}

const void* RecordArena::push_bytes(const void* src, size_t bytes) {
  const size_t off = (used_ + 63) / 64 * 64;
  QCA_CHECK(off + bytes <= cap_, "record arena full");
  std::memcpy(host_ + off, src, bytes);
  used_ = off + bytes;
  return dev_ + off;
}

void RecordArena::upload(hipStream_t s) {
  if (used_ > uploaded_) {
    QCA_HIP(hipMemcpyAsync(dev_ + uploaded_, host_ + uploaded_, used_ - uploaded_, hipMemcpyHostToDevice, s));
    uploaded_ = used_;
  }
}

// ------------------------------------------------------------------ grouped launchers
GRec<ConvArgs> conv_rec(const c128* in, c64* out, long n, const int* skip) {
  return grec(ConvArgs{in, out, n, skip}, grid_for(n));
}
GRec<ThetaSvdArgs> theta_svd_rec(const c128* th, c128* X, int chil, int chir, int mode) {
  return grec(ThetaSvdArgs{th, X, chil, chir, mode}, grid_for(4L * chil * chir));
}
GRec<GatherIsoArgs> gather_iso_rec(const c128* X, const int* perm, const double* sigma, c128* A,
                                   int rows, int chi_bond, int k, int mode) {
  return grec(GatherIsoArgs{X, perm, sigma, A, rows, chi_bond, k, mode}, grid_for((long)rows * k));
}
template <typename T>
size_t wmix_lds_bytes(int nin, int nq, int Dout) {
  return ((size_t)nin * WMIX_XC + (size_t)nq * WMIX_XC * Dout) * sizeof(cplx<T>);
}
template <typename T>
GRec<WmixArgs<T>> wmix_rec(const cplx<T>* Tin, long in_stride, long nxc, int nin, cplx<T>* U, int nq,
                           int Dout, const WSparseDev<T>& w, const int* skip) {
  QCA_CHECK(Dout <= WMIX_DMAX, "MPO bond dimension above 16");
  QCA_CHECK(nin <= 64, "too many input channels in MPO mixing");
  QCA_CHECK(wmix_lds_bytes<T>(nin, nq, Dout) <= 150 * 1024, "MPO mixing stage exceeds LDS");
  return grec(WmixArgs<T>{Tin, in_stride, nxc, nin, U, nq, Dout, w.rowptr, w.col, w.val, skip},
              (unsigned)ceil_div(nxc, WMIX_XC));
}
template GRec<WmixArgs<double>> wmix_rec<double>(const c128*, long, long, int, c128*, int, int,
                                                 const WSparseDev<double>&, const int*);
template GRec<WmixArgs<float>> wmix_rec<float>(const c64*, long, long, int, c64*, int, int,
                                               const WSparseDev<float>&, const int*);
template size_t wmix_lds_bytes<double>(int, int, int);
template size_t wmix_lds_bytes<float>(int, int, int);

void launch_conv_grouped(const KGroup<ConvArgs>& g, hipStream_t s) {
  if (g.empty()) return;
  hipLaunchKernelGGL(convert_grouped, dim3(g.l.blocks), dim3(256), 0, s, g.l.recs, g.l.n);
  QCA_HIP(hipGetLastError());
}
void launch_theta_svd_grouped(const KGroup<ThetaSvdArgs>& g, hipStream_t s) {
  if (g.empty()) return;
  hipLaunchKernelGGL(theta_to_svd_grouped, dim3(g.l.blocks), dim3(256), 0, s, g.l.recs, g.l.n);
  QCA_HIP(hipGetLastError());
}
void launch_gather_iso_grouped(const KGroup<GatherIsoArgs>& g, hipStream_t s) {
  if (g.empty()) return;
  hipLaunchKernelGGL(gather_isometry_grouped, dim3(g.l.blocks), dim3(256), 0, s, g.l.recs, g.l.n);
  QCA_HIP(hipGetLastError());
}
template <typename T>
void launch_wmix_grouped(const KGroup<WmixArgs<T>>& g, size_t lds, hipStream_t s) {
  if (g.empty()) return;
  ensure_dynamic_lds((const void*)wmix_grouped<T>, lds);
  hipLaunchKernelGGL(wmix_grouped<T>, dim3(g.l.blocks), dim3(WMIX_XC * WMIX_WAVES), lds, s, g.l.recs, g.l.n);
  QCA_HIP(hipGetLastError());
}
template void launch_wmix_grouped<double>(const KGroup<WmixArgs<double>>&, size_t, hipStream_t);
template void launch_wmix_grouped<float>(const KGroup<WmixArgs<float>>&, size_t, hipStream_t);

void LzGroup::prepare(const std::vector<LzArgs>& jobs, RecordArena& arena) {
  std::vector<GRec<LzArgs>> a, b;
  for (const LzArgs& j : jobs) {
    QCA_CHECK(j.nblk == lanczos_nblk(j.n), "Lanczos block count does not match the vector");
    a.push_back(grec(j, j.nblk));
    b.push_back(grec(j, grid_for(j.n)));
  }
  nb.prepare(a, arena);
  gf.prepare(b, arena);
}
void LzGroup::begin(hipStream_t s) const {
  if (empty()) return;
  hipLaunchKernelGGL(lz_norm_partials_grouped, dim3(nb.l.blocks), dim3(LZ_BLOCK), 0, s, nb.l.recs, nb.l.n);
  hipLaunchKernelGGL(lz_scale_first_grouped, dim3(nb.l.blocks), dim3(LZ_BLOCK), 0, s, nb.l.recs, nb.l.n);
  QCA_HIP(hipGetLastError());
}
template <typename TW>
void LzGroup::tail(int j, hipStream_t s) const {
  if (empty()) return;
  QCA_CHECK(j + 1 < LZ_MAXK, "Krylov dimension limit");
  hipLaunchKernelGGL(lz_dot_grouped<TW>, dim3(nb.l.blocks), dim3(LZ_BLOCK), 0, s, nb.l.recs, nb.l.n, j);
  hipLaunchKernelGGL(lz_three_term_grouped<TW>, dim3(nb.l.blocks), dim3(LZ_BLOCK), 0, s, nb.l.recs, nb.l.n, j);
  hipLaunchKernelGGL(lz_next_grouped, dim3(nb.l.blocks), dim3(LZ_BLOCK), 0, s, nb.l.recs, nb.l.n, j);
  QCA_HIP(hipGetLastError());
}
template void LzGroup::tail<double>(int, hipStream_t) const;
template void LzGroup::tail<float>(int, hipStream_t) const;
void LzGroup::finish(hipStream_t s) const {
  if (empty()) return;
  hipLaunchKernelGGL(lz_combine_grouped, dim3(gf.l.blocks), dim3(256), 0, s, gf.l.recs, gf.l.n);
  QCA_HIP(hipGetLastError());
}

// ------------------------------------------------------------------ launchers
template <typename T>
void launch_wmix(const cplx<T>* Tin, long in_stride, long nxc, int nin, cplx<T>* U, int nq,
                 int Dout, const WSparseDev<T>& w, hipStream_t s, const int* skip) {
  QCA_CHECK(Dout <= WMIX_DMAX, "MPO bond dimension above 16");
  QCA_CHECK(nin <= 64, "too many input channels in MPO mixing");
  if (nxc == 0) return;
  const size_t shm = ((size_t)nin * WMIX_XC + (size_t)nq * WMIX_XC * Dout) * sizeof(cplx<T>);
  QCA_CHECK(shm <= 150 * 1024, "MPO mixing stage exceeds LDS");
  ensure_dynamic_lds((const void*)wmix_kernel<T>, shm);
  hipLaunchKernelGGL(wmix_kernel<T>, dim3(ceil_div(nxc, WMIX_XC)), dim3(WMIX_XC * WMIX_WAVES), shm, s, Tin,
                     in_stride, nxc, nin, U, nq, Dout, w.rowptr, w.col, w.val, skip);
  QCA_HIP(hipGetLastError());
}
template void launch_wmix<double>(const c128*, long, long, int, c128*, int, int,
                                  const WSparseDev<double>&, hipStream_t, const int*);
template void launch_wmix<float>(const c64*, long, long, int, c64*, int, int,
                                 const WSparseDev<float>&, hipStream_t, const int*);

void launch_convert_c128_c64(const c128* in, c64* out, long n, hipStream_t s, const int* skip) {
  if (n == 0) return;
  hipLaunchKernelGGL((convert_kernel<double, float>), dim3(grid_for(n)), dim3(256), 0, s, in, out, n, skip);
  QCA_HIP(hipGetLastError());
}
void launch_convert_c64_c128(const c64* in, c128* out, long n, hipStream_t s, const int* skip) {
  if (n == 0) return;
  hipLaunchKernelGGL((convert_kernel<float, double>), dim3(grid_for(n)), dim3(256), 0, s, in, out, n, skip);
  QCA_HIP(hipGetLastError());
}

void launch_to_colmajor(const c128* in, c128* out, int rows, int cols, hipStream_t s) {
  hipLaunchKernelGGL(to_colmajor, dim3(grid_for((long)rows * cols)), dim3(256), 0, s, in, out, rows, cols);
  QCA_HIP(hipGetLastError());
}
void launch_site_to_rightqr(const c128* A, c128* X, int chil, int chir, hipStream_t s) {
  hipLaunchKernelGGL(site_to_rightqr, dim3(grid_for(2L * chil * chir)), dim3(256), 0, s, A, X, chil, chir);
  QCA_HIP(hipGetLastError());
}
void launch_qr_gather_left(const c128* Q, const c128* X, c128* Anew, c128* C, int rows, int cols,
                           int qcols, int target, hipStream_t s) {
  const long n = (long)rows * target + (long)target * cols;
  hipLaunchKernelGGL(qr_gather_left, dim3(grid_for(n)), dim3(256), 0, s, Q, X, Anew, C, rows, cols, qcols, target);
  QCA_HIP(hipGetLastError());
}
void launch_qr_gather_right(const c128* Q, const c128* X, c128* Anew, c128* C, int chir, int cols,
                            int qcols, int target, hipStream_t s) {
  const long n = 2L * target * chir + (long)cols * target;
  hipLaunchKernelGGL(qr_gather_right, dim3(grid_for(n)), dim3(256), 0, s, Q, X, Anew, C, chir, cols, qcols, target);
  QCA_HIP(hipGetLastError());
}

void launch_theta_to_svd(const c128* th, c128* X, int chil, int chir, int mode, hipStream_t s) {
  const long n = 4L * chil * chir;
  hipLaunchKernelGGL(theta_to_svd, dim3(grid_for(n)), dim3(256), 0, s, th, X, chil, chir, mode);
  QCA_HIP(hipGetLastError());
}

void launch_gather_isometry(const c128* X, const int* perm, const double* sigma, c128* A, int rows,
                            int chi_bond, int k, int mode, hipStream_t s) {
  const long n = (long)rows * k;
  if (n == 0) return;
  hipLaunchKernelGGL(gather_isometry, dim3(grid_for(n)), dim3(256), 0, s, X, perm, sigma, A, rows,
                     chi_bond, k, mode);
  QCA_HIP(hipGetLastError());
}

int lanczos_nblk(long n) { return (int)std::max<long>(1, (n + LZ_BLOCK - 1) / LZ_BLOCK); }

const int* lanczos_done_flag(const LanczosWork& lw) { return &lw.ctrl->done; }

void lanczos_begin(const c128* x, long n, LanczosWork& lw, hipStream_t s, c64* v32) {
  const int nb = lanczos_nblk(n);
  QCA_CHECK(nb <= lw.max_blocks, "Lanczos vector longer than the workspace");
  hipLaunchKernelGGL(lz_norm_partials, dim3(nb), dim3(LZ_BLOCK), 0, s, x, n, lw.part_norm);
  hipLaunchKernelGGL(lz_scale_first, dim3(nb), dim3(LZ_BLOCK), 0, s, x, lw.V, n, (const double*)lw.part_norm, nb,
                     lw.ctrl, v32);
  QCA_HIP(hipGetLastError());
}

template <typename TW>
void lanczos_iteration_tail(const cplx<TW>* w, long n, int j, double tau, double tol,
                            LanczosWork& lw, hipStream_t s, c64* v32) {
  QCA_CHECK(j + 1 < lw.max_m && lw.max_m <= LZ_MAXK, "Krylov dimension limit");
  const int nb = lanczos_nblk(n);
  const LanczosCtrl* cc = lw.ctrl;
  hipLaunchKernelGGL(lz_dot<TW>, dim3(nb), dim3(LZ_BLOCK), 0, s, cc, w, (const c128*)(lw.V + (long)j * n), n,
                     lw.part);
  hipLaunchKernelGGL(lz_three_term<TW>, dim3(nb), dim3(LZ_BLOCK), 0, s, cc, w, lw.w64, (const c128*)lw.V, n, j,
                     (const c128*)lw.part, nb, lw.coef, lw.part2);
  hipLaunchKernelGGL(lz_next, dim3(nb), dim3(LZ_BLOCK), 0, s, lw.ctrl, (const c128*)lw.part2, nb,
                     (const c128*)lw.coef, j, tau, tol, lw.max_m, (const c128*)lw.w64, lw.V, v32, n);
  QCA_HIP(hipGetLastError());
}
template void lanczos_iteration_tail<double>(const c128*, long, int, double, double, LanczosWork&,
                                             hipStream_t, c64*);
template void lanczos_iteration_tail<float>(const c64*, long, int, double, double, LanczosWork&,
                                            hipStream_t, c64*);

void lanczos_finish(long n, c128* y, LanczosWork& lw, hipStream_t s) {
  hipLaunchKernelGGL(lz_combine, dim3(grid_for(n)), dim3(256), 0, s, (const LanczosCtrl*)lw.ctrl,
                     lw.V, n, y);
  QCA_HIP(hipGetLastError());
}

void launch_observables(const c128* rho, int n, double* out, hipStream_t s) {
  hipLaunchKernelGGL(observables_kernel, dim3(ceil_div(n, 64)), dim3(64), 0, s, rho, n, out);
  QCA_HIP(hipGetLastError());
}

void launch_rho(const c128* A, const c128* T, long nxb, c128* rho, hipStream_t s) {
  hipLaunchKernelGGL(rho_kernel, dim3(1), dim3(256), 0, s, A, T, nxb, rho);
  QCA_HIP(hipGetLastError());
}

}  // namespace qca
