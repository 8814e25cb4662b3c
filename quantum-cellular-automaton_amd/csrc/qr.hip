// Householder QR with LAPACK's conventions (gfx950).
//
// zgeqrf + zungqr semantics (reference tensor_networks/mps.py:86 calls
// numpy.linalg.qr -> LAPACK), including zlarfg's sign beta = -sign(Re alpha)
// |x|, so R has a real diagonal and Q matches LAPACK's complete-QR complement
// columns.  Two forms:
//   * blocked (rows <= 512): panels of 16 columns, one launch per panel and one
//     that forms Q.  The launch of panel p applies the block reflector of panel
//     p-1 to all remaining columns, 16 per workgroup, and its first workgroup
//     goes on to factor the columns it has just updated;
//   * one workgroup (householder_qr_kernel), for longer rows and for one or two
//     reflectors.
//
// What bounds the blocked form is the chain of 16 dependent columns of a panel,
// so a panel lives in registers (wave w holds columns w and w + 8, lane l their rows
// l, l + 64, ...), a reflector goes from wave to wave through LDS under a flag,
// without a barrier, and T is built along the way.
// The block reflectors run on the FP64 matrix cores with the updated columns in
// accumulator registers: the accumulator layout (row (l / 16) + 4 r in register
// r) is the B operand layout of four consecutive rows, so V^H A and A -= V W
// both use them in place.  512 x 256 with 256 columns of Q: 2.07 -> 0.78 ms
// (a panel launch 36 us where panel, two GEMMs and a reduce took 102; Q 165 us);
// 256 x 256 within a split: 1.6 -> 0.55 ms; 16 x 32: 73 -> 39 us.
#include "grouped.hpp"
#include "larfg.hpp"
#include "wave.hpp"

#include <algorithm>

namespace qca {
namespace {

constexpr int QR_THREADS = 512;
constexpr int QR_WAVES = QR_THREADS / 64;
constexpr int QR_PB = 16;

typedef double f64x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ f64x4 mfma(double a, double b, f64x4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// LDS of the blocked kernels.  `big` is the partial products of the waves
// (8 x 256) and, for the panel, the 16 columns on their way from the
// accumulator layout to whole columns per wave, then the published reflectors.
struct QrShared {
  c128 W[4][QR_PB * QR_PB];     // op(T) V^H A by quarters of its inner index, at k * 16 + n
  c128 T[QR_PB * QR_PB];        // panel: T(k, i) at i * 16 + k
  c128 vv[QR_PB * QR_PB];       // panel: v_k^H v_i at k * 16 + i, k < i
  c128 tau[QR_PB];
  int flag[QR_PB];              // reflector published
  int done;                     // waves that have visited every reflector
};
// 64-row chunks of a panel of nr rows: the register blocks that factor_panel has
__host__ __device__ constexpr int panel_chunks(int nr) {
  return nr <= 64 ? 1 : nr <= 128 ? 2 : nr <= 192 ? 3 : nr <= 256 ? 4 : nr <= 384 ? 6 : 8;
}
__host__ __device__ constexpr int panel_stride(int nr) { return 64 * panel_chunks(nr) + 1; }
__host__ __device__ constexpr long big_elems(int rows) {
  const long part = (long)QR_WAVES * QR_PB * QR_PB, cols = (long)QR_PB * panel_stride(rows);
  return part > cols ? part : cols;
}

// p[i] with a 32-bit byte offset from a uniform base (a factored matrix is below
// 4 MB): one address register per load.
__device__ __forceinline__ c128 at(const c128* __restrict__ p, unsigned i) {
  return *reinterpret_cast<const c128*>(reinterpret_cast<const char*>(p) + (i << 4));
}

// V of one panel and T, as the matrix-core operands of this wave's tiles.
template <int QR_TILES>
struct QrOperands {
  c128 va[QR_TILES][4];   // V(16 tile + 4 r + lane / 16, lane % 16): for V^H A
  c128 vb[QR_TILES][4];   // V(16 tile + lane % 16, 4 r + lane / 16): for A -= V W
  c128 t;                 // op(T)(lane % 16, 4 wave + lane / 16), waves 0..3
};
template <int QR_TILES>
__device__ __forceinline__ void load_operands(const c128* __restrict__ M, int rows, int j0, int pb,
                                              const c128* __restrict__ Tg, bool conj_t, QrOperands<QR_TILES>& o) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = j0 >> 4, last = (rows + 15) >> 4;   // tiles with a nonzero V
  // V is unit lower trapezoidal: (r, k) is M's entry below row j0 + k, 1 on it
  // and 0 above; columns from pb on are 0
  const unsigned ca = (unsigned)(j0 + min(lo, pb - 1)) * rows;
  const int da = lo < pb ? j0 + lo : 1 << 20;
  unsigned cb[4];
  int db[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int k = 4 * r + hi;
    cb[r] = (unsigned)(j0 + min(k, pb - 1)) * rows;
    db[r] = k < pb ? j0 + k : 1 << 20;
  }
  auto unit = [](c128 m, int r, int d) {
    return c128{r > d ? m.re : (r == d ? 1.0 : 0.0), r > d ? m.im : 0.0};
  };
#pragma unroll
  for (int t = 0; t < QR_TILES; ++t) {
    const int tile = wave + QR_WAVES * t;
    if (tile < first || tile >= last) continue;
    const int rb = 16 * tile + lo;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ra = 16 * tile + 4 * r + hi;
      o.va[t][r] = at(M, ca + min(ra, rows - 1));
      o.vb[t][r] = at(M, cb[r] + min(rb, rows - 1));
    }
  }
#pragma unroll
  for (int t = 0; t < QR_TILES; ++t) {
    const int tile = wave + QR_WAVES * t;
    if (tile < first || tile >= last) continue;
    const int rb = 16 * tile + lo;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int ra = 16 * tile + 4 * r + hi;
      o.va[t][r] = unit(o.va[t][r], ra < rows ? ra : -1, da);
      o.vb[t][r] = unit(o.vb[t][r], rb < rows ? rb : -1, db[r]);
    }
  }
  // T(k, i) is stored at i * 16 + k, zero below the diagonal
  const int k = lo, l = 4 * (wave & 3) + hi;
  o.t = conj_t ? Tg[k * QR_PB + l] : Tg[l * QR_PB + k];
  if (conj_t) o.t.im = -o.t.im;
  if (k >= pb || l >= pb) o.t = c128{0.0, 0.0};
}

// q <- (I - V op(T) V^H) q for the 16 columns whose 16-row tiles wave w holds in
// accumulator layout (tile w + 8 t in q*[t]).  Sums run over the waves in order.
template <int QR_TILES>
__device__ __forceinline__ void block_reflect(const QrOperands<QR_TILES>& o, int rows, int j0, f64x4 (&qre)[QR_TILES],
                                              f64x4 (&qim)[QR_TILES], c128* part, QrShared& sh) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int first = j0 >> 4, last = (rows + 15) >> 4;
  // the two halves of each complex sum apart: half the chain of roundings
  f64x4 wre = {0, 0, 0, 0}, wim = {0, 0, 0, 0}, xre = {0, 0, 0, 0}, xim = {0, 0, 0, 0};
#pragma unroll
  for (int t = 0; t < QR_TILES; ++t) {
    const int tile = wave + QR_WAVES * t;
    if (tile < first || tile >= last) continue;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const c128 v = o.va[t][r];
      wre = mfma(v.re, qre[t][r], wre);
      wim = mfma(v.re, qim[t][r], wim);
      xre = mfma(v.im, qim[t][r], xre);
      xim = mfma(-v.im, qre[t][r], xim);
    }
  }
  {
    wre += xre;
    wim += xim;
    c128* p = part + wave * (QR_PB * QR_PB);
#pragma unroll
    for (int r = 0; r < 4; ++r) p[(hi + 4 * r) * QR_PB + lo] = c128{wre[r], wim[r]};
  }
  __syncthreads();
  if (wave < 4) {
    // wave s sums rows 4s.. of V^H A, the B operand of step s of op(T) (V^H A)
    double re = 0, im = 0;
#pragma unroll
    for (int w = 0; w < QR_WAVES; ++w) {
      const c128 x = part[w * (QR_PB * QR_PB) + (4 * wave + hi) * QR_PB + lo];
      re += x.re;
      im += x.im;
    }
    f64x4 pre = {0, 0, 0, 0}, pim = {0, 0, 0, 0};
    pre = mfma(o.t.re, re, pre);
    pim = mfma(o.t.re, im, pim);
    pre = mfma(-o.t.im, im, pre);
    pim = mfma(o.t.im, re, pim);
#pragma unroll
    for (int r = 0; r < 4; ++r) sh.W[wave][(hi + 4 * r) * QR_PB + lo] = c128{pre[r], pim[r]};
  }
  __syncthreads();
  c128 wt[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    c128 x[4];
#pragma unroll
    for (int q = 0; q < 4; ++q) x[q] = sh.W[q][(4 * s + hi) * QR_PB + lo];
    wt[s] = c128{(x[0].re + x[1].re) + (x[2].re + x[3].re), (x[0].im + x[1].im) + (x[2].im + x[3].im)};
  }
#pragma unroll
  for (int t = 0; t < QR_TILES; ++t) {
    const int tile = wave + QR_WAVES * t;
    if (tile < first || tile >= last) continue;
    f64x4 ure = {0, 0, 0, 0}, uim = {0, 0, 0, 0}, xr = {0, 0, 0, 0}, xi = {0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const c128 v = o.vb[t][s];
      ure = mfma(v.re, wt[s].re, ure);
      uim = mfma(v.re, wt[s].im, uim);
      xr = mfma(-v.im, wt[s].im, xr);
      xi = mfma(v.im, wt[s].re, xi);
    }
    ure += xr;
    uim += xi;
    // one rounding at the size of q, not 32: Q of 512 x 256 to 6.0e-16 in the 2-norm
    // against 1.33e-15 with the products added to q itself and a reciprocal square
    // root without its last step in larfg, in less time (829 -> 780 us)
    qre[t] -= ure;
    qim[t] -= uim;
  }
}

// Factors pb reflectors of the panel (ncols columns at src, stride ldsrc; columns
// pb.. only receive the reflectors) and writes the columns (R, v) to M and T to
// Tg.  Wave w holds columns w and w + 8, lane l their rows l, l + 64, ....
//
// Column c+1 needs nothing but reflector c, so there is no barrier in the loop:
// the owner of c+1 waits for flag c, updates that column first, publishes its
// reflector in slot c+1 of `vs` and raises flag c+1, and only then turns to its
// other column; the other waves follow at their own pace.  A wave waits only
// for reflectors of lower columns, whose owners never wait for it, so every
// wait ends.  (With a barrier of eight waves per column, 268 cycles, and the
// owner's other column in its way a column took 2500 cycles at 100 rows, here
// 1850: wait and read 400, update 550, norm 300, scalars 400, publish 200.)
template <int IT>
__device__ __forceinline__ void factor_panel(const c128* __restrict__ src, int ldsrc, c128* vs, c128* __restrict__ M,
                                             int rows, int j0, int pb, int ncols, c128* __restrict__ Tg,
                                             QrShared& sh) {
  constexpr int LDV = 64 * IT + 1;
  const int lane = threadIdx.x & 63, lo = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int nr = rows - j0;
  c128 x[2][IT];
#pragma unroll
  for (int q = 0; q < 2; ++q)
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const int r = lane + 64 * i;
      x[q][i] = src[(long)min(wave + QR_WAVES * q, ncols - 1) * ldsrc + min(r, nr - 1)];
      if (r >= nr) x[q][i] = c128{0.0, 0.0};
    }
  if (threadIdx.x < QR_PB) sh.flag[threadIdx.x] = 0;
  if (threadIdx.x == 0) sh.done = 0;
  if (threadIdx.x < QR_PB * QR_PB) sh.T[threadIdx.x] = sh.vv[threadIdx.x] = c128{0.0, 0.0};
  __syncthreads();   // every column is in registers: the slots may be written
  auto raise = [&](int* word) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    if (lane == 0) __hip_atomic_fetch_add(word, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
  };
  auto wait = [&](int* word, int n) {
    while (__hip_atomic_load(word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < n) {
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  };
  auto publish = [&](int c, c128 (&y)[IT]) {
    double part = 0;
#pragma unroll
    for (int i = 0; i < IT; ++i)
      if (i > 0 || lane > c) part += y[i].re * y[i].re + y[i].im * y[i].im;
    double xnorm2 = wave_sum64(part);
    c128 alpha{readlane_f64(y[0].re, c), readlane_f64(y[0].im, c)};
    int ex = 0;
    if (!larfg_in_range(alpha.re * alpha.re + alpha.im * alpha.im + xnorm2)) {
      // a column whose squares over- or underflow (all zero in most cases): the
      // reflector of the scaled column is the same
      double top = 0;
#pragma unroll
      for (int i = 0; i < IT; ++i)
        if (i > 0 || lane >= c) top = fmax(top, fmax(fabs(y[i].re), fabs(y[i].im)));
      for (int o = 32; o > 0; o >>= 1) top = fmax(top, __shfl_xor(top, o, 64));
      ex = larfg_exponent(top);
      part = 0;
#pragma unroll
      for (int i = 0; i < IT; ++i)
        if (i > 0 || lane >= c) {
          y[i] = c128{ldexp(y[i].re, -ex), ldexp(y[i].im, -ex)};
          if (i > 0 || lane > c) part += y[i].re * y[i].re + y[i].im * y[i].im;
        }
      xnorm2 = wave_sum64(part);
      alpha = c128{ldexp(alpha.re, -ex), ldexp(alpha.im, -ex)};
    }
    Larfg h = larfg(alpha, xnorm2);
    if (ex) h.beta = ldexp(h.beta, ex);
    c128* v = vs + c * LDV;
#pragma unroll
    for (int i = 0; i < IT; ++i) {
      const c128 s{y[i].re * h.scale.re - y[i].im * h.scale.im, y[i].re * h.scale.im + y[i].im * h.scale.re};
      if (i > 0) {
        y[i] = s;
        v[lane + 64 * i] = s;
      } else {
        v[lane] = lane > c ? s : c128{lane == c ? 1.0 : 0.0, 0.0};
        if (lane > c) y[0] = s;
        if (lane == c) y[0] = c128{h.beta, 0.0};
      }
    }
    if (lane == 0) sh.tau[c] = h.tau;
    raise(&sh.flag[c]);
  };
  if (wave == 0) publish(0, x[0]);
  for (int c = 0; c < pb; ++c) {
    wait(&sh.flag[c], 1);
    c128 v[IT];
#pragma unroll
    for (int i = 0; i < IT; ++i) v[i] = vs[c * LDV + lane + 64 * i];
    const c128 tau = sh.tau[c];
    // column `col` in registers y: y <- (I - conj(tau) v v^H) y when it is right
    // of c, its inner product with v when it is left of c
    auto visit = [&](int col, c128 (&y)[IT]) {
      if (col == c || col >= ncols) return;
      double dr = 0, di = 0;
#pragma unroll
      for (int i = 0; i < IT; ++i) {
        dr += v[i].re * y[i].re + v[i].im * y[i].im;
        di += v[i].re * y[i].im - v[i].im * y[i].re;
      }
      dr = wave_sum64(dr);
      di = wave_sum64(di);
      if (col > c) {
        const double fr = tau.re * dr + tau.im * di, fi = tau.re * di - tau.im * dr;
#pragma unroll
        for (int i = 0; i < IT; ++i) {
          y[i].re -= v[i].re * fr - v[i].im * fi;
          y[i].im -= v[i].re * fi + v[i].im * fr;
        }
      } else if (lane == 0) {
        sh.vv[col * QR_PB + c] = c128{dr, -di};   // v_col^H v_c: v_c is zero above row c
      }
    };
    const bool next = c + 1 < pb && wave == ((c + 1) & (QR_WAVES - 1));
    if (next) {
      __builtin_amdgcn_s_setprio(3);
      if (c + 1 < QR_WAVES) {
        visit(c + 1, x[0]);
        publish(c + 1, x[0]);
      } else {
        visit(c + 1, x[1]);
        publish(c + 1, x[1]);
      }
      __builtin_amdgcn_s_setprio(0);
    }
    if (!(next && c + 1 < QR_WAVES)) visit(wave, x[0]);
    if (!(next && c + 1 >= QR_WAVES)) visit(wave + QR_WAVES, x[1]);
  }
  raise(&sh.done);
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int col = wave + QR_WAVES * q;
    c128* out = M + (long)(j0 + min(col, ncols - 1)) * rows + j0;
#pragma unroll
    for (int i = 0; i < IT; ++i)
      if (col < ncols && lane + 64 * i < nr) out[lane + 64 * i] = x[q][i];
  }
  if (wave != QR_WAVES - 1) return;
  // T with I - V T V^H = H_0 H_1 ... (zlarft, forward columnwise) by merging
  // blocks of width b = 1, 2, 4, 8: T12 = -T11 (V1^H V2) T22, one new entry per
  // lane (a column at a time took twice as long)
  wait(&sh.done, QR_WAVES);
  if (lane < pb) sh.T[lane * QR_PB + lane] = sh.tau[lane];
#pragma unroll
  for (int b = 1; b < QR_PB; b *= 2) {
    const int base = lane / (b * b) * 2 * b, r = lane & (b - 1), sidx = lane / b & (b - 1);
    const int k = (base + r) & 15, i2 = (base + b + sidx) & 15;
    __builtin_amdgcn_wave_barrier();
    double ar = 0, ai = 0;
#pragma unroll
    for (int l = 0; l < b; ++l) {
      const int m = (base + b + l) & 15;
      const c128 g = sh.vv[k * QR_PB + m], t = sh.T[i2 * QR_PB + m];
      ar += g.re * t.re - g.im * t.im;
      ai += g.re * t.im + g.im * t.re;
    }
    if (lane < 8 * b) sh.W[0][lane] = c128{ar, ai};
    __builtin_amdgcn_wave_barrier();
    ar = ai = 0;
#pragma unroll
    for (int l = 0; l < b; ++l) {
      const c128 t = sh.T[((base + l) & 15) * QR_PB + k], g = sh.W[0][(lane & ~(b - 1)) + l];
      ar += t.re * g.re - t.im * g.im;
      ai += t.re * g.im + t.im * g.re;
    }
    __builtin_amdgcn_wave_barrier();
    if (lane < 8 * b) sh.T[i2 * QR_PB + k] = c128{-ar, -ai};
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int e = 0; e < QR_PB * QR_PB; e += 64) Tg[e + lane] = sh.T[e + lane];
}

// Launch p of the factorisation, column block blk (columns 16 (p + blk)..).
template <int QR_TILES>
__device__ __forceinline__ void qr_step_body(const QrStepArgs& a, c128* __restrict__ M, c128* __restrict__ T, int blk,
                                             c128* big, QrShared& sh) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rows = a.rows, p = a.p;
  const int kmax = min(rows, a.cols);
  const int c0 = QR_PB * (p + blk), ncols = min(QR_PB, a.cols - c0);
  const bool panel = blk == 0 && c0 < kmax;
  const int nr = rows - c0;                 // rows of the panel
  const int pb = min(QR_PB, kmax - c0);
  c128* Tg = T + (long)p * QR_PB * QR_PB;
  const c128* src = M + (long)c0 * rows + c0;   // the panel's columns
  int lds = rows;
  if (p > 0) {
    const int j0 = QR_PB * (p - 1);
    const int ldp = panel_stride(max(nr, 1));
    QrOperands<QR_TILES> o;
    load_operands(M, rows, j0, min(QR_PB, kmax - j0), T + (long)(p - 1) * QR_PB * QR_PB, true, o);
    f64x4 qre[QR_TILES], qim[QR_TILES];
    const unsigned ca = (unsigned)(c0 + min(lo, ncols - 1)) * rows;
#pragma unroll
    for (int t = 0; t < QR_TILES; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * (wave + QR_WAVES * t) + 4 * r + hi;
        const c128 m = at(M, ca + min(row, rows - 1));
        const bool in = row < rows && row >= j0 && lo < ncols;
        qre[t][r] = in ? m.re : 0.0;
        qim[t][r] = in ? m.im : 0.0;
      }
    block_reflect(o, rows, j0, qre, qim, big, sh);
    // (the partial products in `big` were last read before block_reflect's
    // second barrier)
#pragma unroll
    for (int t = 0; t < QR_TILES; ++t)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = 16 * (wave + QR_WAVES * t) + 4 * r + hi;
        if (row >= rows || row < j0) continue;
        const c128 m{qre[t][r], qim[t][r]};
        if (panel && row >= c0) big[lo * ldp + row - c0] = m;
        else if (lo < ncols) M[(long)(c0 + lo) * rows + row] = m;
      }
    if (!panel) return;
    __syncthreads();
    src = big;
    lds = ldp;
  }
  switch (panel_chunks(nr)) {
    case 1: factor_panel<1>(src, lds, big, M, rows, c0, pb, ncols, Tg, sh); break;
    case 2: factor_panel<2>(src, lds, big, M, rows, c0, pb, ncols, Tg, sh); break;
    case 3: factor_panel<3>(src, lds, big, M, rows, c0, pb, ncols, Tg, sh); break;
    case 4: factor_panel<4>(src, lds, big, M, rows, c0, pb, ncols, Tg, sh); break;
    case 6: if constexpr (QR_TILES > 2) factor_panel<6>(src, lds, big, M, rows, c0, pb, ncols, Tg, sh); break;
    default: if constexpr (QR_TILES > 2) factor_panel<8>(src, lds, big, M, rows, c0, pb, ncols, Tg, sh); break;
  }
}

// Columns 16 blk.. of Q = H_0 ... H_{kk-1} [e_0 .. e_{qcols-1}], or of H_0 ...
// H_{kk-1} (Z; 0): the block reflectors from the last panel back, on columns that
// stay in registers.  A panel right of the block's columns of [e_0 ..] leaves them as
// they are.
template <int QR_TILES>
__device__ __forceinline__ void form_q_body(const QrFormArgs& a, const c128* __restrict__ M,
                                            const c128* __restrict__ T, c128* __restrict__ Q,
                                            const c128* __restrict__ Z, int blk, c128* big, QrShared& sh) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int rows = a.rows, kk = a.kk, c0 = QR_PB * blk;
  f64x4 qre[QR_TILES], qim[QR_TILES];
#pragma unroll
  for (int t = 0; t < QR_TILES; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (wave + QR_WAVES * t) + 4 * r + hi, col = c0 + lo;
      c128 z{row == col ? 1.0 : 0.0, 0.0};
      if (Z) z = row < kk && col < a.qcols ? Z[(long)col * kk + row] : c128{0.0, 0.0};
      qre[t][r] = z.re;
      qim[t][r] = z.im;
    }
  const int last = (kk + QR_PB - 1) / QR_PB - 1;
  for (int p = Z ? last : min(last, blk); p >= 0; --p) {
    const int j0 = p * QR_PB, pb = min(QR_PB, kk - j0);
    QrOperands<QR_TILES> o;
    load_operands(M, rows, j0, pb, T + (long)p * QR_PB * QR_PB, false, o);
    block_reflect(o, rows, j0, qre, qim, big, sh);
  }
#pragma unroll
  for (int t = 0; t < QR_TILES; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * (wave + QR_WAVES * t) + 4 * r + hi;
      if (row < rows && c0 + lo < a.qcols) Q[(long)(c0 + lo) * rows + row] = c128{qre[t][r], qim[t][r]};
    }
}

// 256 VGPRs: two waves per SIMD.  TILES: 16-row tiles per wave, 2 up to 256
// rows and 4 up to 512; sums do not depend on it.
#define QCA_QR_BOUNDS __launch_bounds__(QR_THREADS) __attribute__((amdgpu_waves_per_eu(2, 2)))

template <int TILES>
__global__ QCA_QR_BOUNDS void qr_step_kernel(QrStepArgs a) {
  extern __shared__ __align__(16) unsigned char qr_lds[];
  __shared__ QrShared sh;
  qr_step_body<TILES>(a, a.M, a.T, blockIdx.x, reinterpret_cast<c128*>(qr_lds), sh);
}
template <int TILES>
__global__ QCA_QR_BOUNDS void qr_step_grouped(const GRec<QrStepArgs>* __restrict__ recs, int n) {
  extern __shared__ __align__(16) unsigned char qr_lds[];
  __shared__ QrShared sh;
  unsigned bx, by, bz;
  const QrStepArgs a = grec_find(recs, n, blockIdx.x, bx, by, bz).a;
  qr_step_body<TILES>(a, gbl(a.M), gbl(a.T), bx, reinterpret_cast<c128*>(qr_lds), sh);
}
template <int TILES>
__global__ QCA_QR_BOUNDS void form_q_kernel(QrFormArgs a) {
  extern __shared__ __align__(16) unsigned char qr_lds[];
  __shared__ QrShared sh;
  form_q_body<TILES>(a, a.M, a.T, a.Q, a.Z, blockIdx.x, reinterpret_cast<c128*>(qr_lds), sh);
}
template <int TILES>
__global__ QCA_QR_BOUNDS void form_q_grouped(const GRec<QrFormArgs>* __restrict__ recs, int n) {
  extern __shared__ __align__(16) unsigned char qr_lds[];
  __shared__ QrShared sh;
  unsigned bx, by, bz;
  const QrFormArgs a = grec_find(recs, n, blockIdx.x, bx, by, bz).a;
  form_q_body<TILES>(a, gbl(a.M), gbl(a.T), gbl(a.Q), a.Z ? gbl(a.Z) : nullptr, bx, reinterpret_cast<c128*>(qr_lds), sh);
}

constexpr int HH_THREADS = 1024;
constexpr int HH_WAVES = HH_THREADS / 64;

__device__ double qr_block_sum(double v, double* sh) {
  v = wave_sum64(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  double r = (l < HH_WAVES) ? sh[l] : 0.0;
  r = wave_sum64(r);
  __syncthreads();
  return r;
}

__device__ double qr_block_max(double v, double* sh) {
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) sh[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0;
  for (int w = 0; w < HH_WAVES; ++w) r = fmax(r, sh[w]);
  __syncthreads();
  return r;
}

// M (rows x cols, column-major) -> reflectors below the diagonal, R on and
// above it (zgeqr2), then Q's first qcols columns (zung2r) into Q.
__global__ __launch_bounds__(HH_THREADS) void householder_qr_kernel(c128* __restrict__ M, int rows,
                                                                    int cols, c128* __restrict__ tau,
                                                                    c128* __restrict__ Q, int qcols) {
  __shared__ double sh[HH_WAVES];
  __shared__ c128 s_tau;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int kmax = min(rows, cols);
  for (int j = 0; j < kmax; ++j) {
    c128* x = M + (long)j * rows;
    double part = 0;
    for (int r = j + 1 + tid; r < rows; r += HH_THREADS) part += x[r].re * x[r].re + x[r].im * x[r].im;
    double xnorm2 = qr_block_sum(part, sh);
    c128 alpha = x[j];
    int ex = 0;
    if (!larfg_in_range(alpha.re * alpha.re + alpha.im * alpha.im + xnorm2)) {
      // squares over- or underflow: the reflector of the scaled column is the same
      double top = 0;
      for (int r = j + tid; r < rows; r += HH_THREADS) top = fmax(top, fmax(fabs(x[r].re), fabs(x[r].im)));
      ex = larfg_exponent(qr_block_max(top, sh));
      part = 0;
      for (int r = j + 1 + tid; r < rows; r += HH_THREADS) {
        x[r] = c128{ldexp(x[r].re, -ex), ldexp(x[r].im, -ex)};
        part += x[r].re * x[r].re + x[r].im * x[r].im;
      }
      xnorm2 = qr_block_sum(part, sh);
      alpha = c128{ldexp(alpha.re, -ex), ldexp(alpha.im, -ex)};
    }
    const bool identity = xnorm2 == 0.0 && alpha.im == 0.0;
    const Larfg h = larfg(alpha, xnorm2);
    const c128 scale = h.scale, tj = h.tau;
    const double beta = ex ? ldexp(h.beta, ex) : h.beta;
    __syncthreads();
    if (!identity) {
      for (int r = j + 1 + tid; r < rows; r += HH_THREADS) {
        const c128 v = x[r];
        x[r] = c128{v.re * scale.re - v.im * scale.im, v.re * scale.im + v.im * scale.re};
      }
    }
    __syncthreads();
    if (tid == 0) {
      if (!identity) x[j] = c128{beta, 0.0};
      tau[j] = tj;
      s_tau = tj;
    }
    __syncthreads();
    if (!identity) {
      // C <- (I - conj(tau) v v^H) C on columns j+1..cols-1, v_j = 1
      const c128 ct{s_tau.re, -s_tau.im};
      for (int c = j + 1 + wave; c < cols; c += HH_WAVES) {
        c128* y = M + (long)c * rows;
        double wr = 0, wi = 0;  // w = v^H y
        for (int r = j + lane; r < rows; r += 64) {
          const c128 v = (r == j) ? c128{1.0, 0.0} : x[r];
          wr += v.re * y[r].re + v.im * y[r].im;
          wi += v.re * y[r].im - v.im * y[r].re;
        }
        wr = wave_sum64(wr);
        wi = wave_sum64(wi);
        // f = conj(tau) * w
        const double fr = ct.re * wr - ct.im * wi, fi = ct.re * wi + ct.im * wr;
        for (int r = j + lane; r < rows; r += 64) {
          const c128 v = (r == j) ? c128{1.0, 0.0} : x[r];
          y[r].re -= v.re * fr - v.im * fi;
          y[r].im -= v.re * fi + v.im * fr;
        }
      }
    }
    __syncthreads();
  }
  if (Q == nullptr || qcols == 0) return;
  // Q = H_0 ... H_{kk-1} [e_0 .. e_{qcols-1}]; reflectors with index >= qcols
  // leave those columns unchanged.
  const int kk = min(kmax, qcols);
  for (long e = tid; e < (long)rows * qcols; e += HH_THREADS) {
    const int c = (int)(e / rows), r = (int)(e - (long)c * rows);
    Q[e] = c128{(r == c) ? 1.0 : 0.0, 0.0};
  }
  __syncthreads();
  for (int i = kk - 1; i >= 0; --i) {
    const c128* v = M + (long)i * rows;
    const c128 ti = tau[i];
    for (int c = i + wave; c < qcols; c += HH_WAVES) {
      c128* y = Q + (long)c * rows;
      double wr = 0, wi = 0;
      for (int r = i + lane; r < rows; r += 64) {
        const c128 vv = (r == i) ? c128{1.0, 0.0} : v[r];
        wr += vv.re * y[r].re + vv.im * y[r].im;
        wi += vv.re * y[r].im - vv.im * y[r].re;
      }
      wr = wave_sum64(wr);
      wi = wave_sum64(wi);
      const double fr = ti.re * wr - ti.im * wi, fi = ti.re * wi + ti.im * wr;
      for (int r = i + lane; r < rows; r += 64) {
        const c128 vv = (r == i) ? c128{1.0, 0.0} : v[r];
        y[r].re -= vv.re * fr - vv.im * fi;
        y[r].im -= vv.re * fi + vv.im * fr;
      }
    }
    __syncthreads();
  }
}

}  // namespace

size_t qr_workspace_elems(int max_rows, int max_cols) {
  return (size_t)ceil_div(std::max(1, std::min(max_rows, max_cols)), QR_PB) * QR_PB * QR_PB;   // T per panel
}

QrStep form_q_step(const c128* M, int rows, int kk, const c128* T, c128* Q, int qcols, const c128* Z) {
  QrStep st{};
  st.slot = QR_SLOT_Q;
  st.kind = 1;
  st.blocks = ceil_div(qcols, QR_PB);
  st.lds = sizeof(c128) * (size_t)QR_WAVES * QR_PB * QR_PB;
  st.form = QrFormArgs{M, rows, kk, T, Q, qcols, Z};
  return st;
}

// The blocked QR as a list of launches, each with a slot number that orders
// it among those of any other matrix: the single-matrix launcher runs them in
// order, the grouped one runs every slot for all matrices that have it.
std::vector<QrStep> blocked_qr_steps(c128* M, int rows, int cols, c128* Q, int qcols, c128* ws, size_t ws_elems) {
  QCA_CHECK(rows >= 1 && cols >= 1, "empty QR");
  QCA_CHECK(rows <= QR_MAX_ROWS, "blocked QR rows above 512");
  QCA_CHECK(ws_elems >= qr_workspace_elems(rows, cols), "QR workspace too small");
  QCA_CHECK(qcols <= rows, "more columns of Q than rows");
  const int kmax = std::min(rows, cols), panels = ceil_div(kmax, QR_PB);
  std::vector<QrStep> out;
  for (int p = 0; p <= panels; ++p) {
    const int blocks = p == 0 ? 1 : ceil_div(cols - QR_PB * p, QR_PB);
    if (blocks <= 0) continue;   // no column right of the last panel
    QrStep st{};
    st.slot = p;
    st.kind = 0;
    st.blocks = blocks;
    st.lds = sizeof(c128) * (size_t)big_elems(rows);
    st.step = QrStepArgs{M, rows, cols, p, ws};
    out.push_back(st);
  }
  if (Q != nullptr && qcols > 0) out.push_back(form_q_step(M, rows, std::min(kmax, qcols), ws, Q, qcols, nullptr));
  return out;
}

namespace {
template <typename... A>
void launch_rows(void (*small)(A...), void (*large)(A...), int rows, unsigned blocks, size_t lds, hipStream_t s, A... a) {
  void (*k)(A...) = rows <= 256 ? small : large;
  ensure_dynamic_lds((const void*)k, lds);
  hipLaunchKernelGGL(k, dim3(blocks), dim3(QR_THREADS), lds, s, a...);
}
}  // namespace

void launch_qr_step_grouped(const KGroup<QrStepArgs>& g, int rows, size_t lds, hipStream_t s) {
  if (g.empty()) return;
  launch_rows(qr_step_grouped<2>, qr_step_grouped<4>, rows, g.l.blocks, lds, s, g.l.recs, g.l.n);
  QCA_HIP(hipGetLastError());
}
void launch_form_q_grouped(const KGroup<QrFormArgs>& g, int rows, size_t lds, hipStream_t s) {
  if (g.empty()) return;
  launch_rows(form_q_grouped<2>, form_q_grouped<4>, rows, g.l.blocks, lds, s, g.l.recs, g.l.n);
  QCA_HIP(hipGetLastError());
}

void launch_form_q(const QrStep& st, hipStream_t s) {
  launch_rows(form_q_kernel<2>, form_q_kernel<4>, st.form.rows, st.blocks, st.lds, s, st.form);
  QCA_HIP(hipGetLastError());
}

void launch_blocked_qr(c128* M, int rows, int cols, c128* Q, int qcols, c128* ws, size_t ws_elems, hipStream_t s) {
  for (const QrStep& st : blocked_qr_steps(M, rows, cols, Q, qcols, ws, ws_elems)) {
    if (st.kind == 0) launch_rows(qr_step_kernel<2>, qr_step_kernel<4>, rows, st.blocks, st.lds, s, st.step);
    else launch_form_q(st, s);
  }
  QCA_HIP(hipGetLastError());
}

void launch_qr(c128* M, int rows, int cols, c128* tau, c128* Q, int qcols, c128* ws, size_t ws_elems,
               hipStream_t s) {
  // one or two reflectors are quicker without the second launch: 2 x 2 27.8 us against
  // 30.2, 512 x 1 27.4 against 40.2, 512 x 2 36.7 against 42.2, 2 x 64 33.2 against
  // 35.2; with three the forms are equal (4 x 3 30.6 us, 512 x 3 44.6 against 44.2),
  // with more, or beside many columns, the blocked one is ahead (2 x 256 54 against 36,
  // 8 x 4 33.5 against 31.3, 64 x 32 147 against 63)
  const bool few = std::min(rows, cols) <= 2 && cols <= 64;
  if (!few && ws != nullptr && rows <= QR_MAX_ROWS && ws_elems >= qr_workspace_elems(rows, cols))
    launch_blocked_qr(M, rows, cols, Q, qcols, ws, ws_elems, s);
  else
    launch_householder_qr(M, rows, cols, tau, Q, qcols, s);
}

void launch_householder_qr(c128* M, int rows, int cols, c128* tau, c128* Q, int qcols, hipStream_t s) {
  QCA_CHECK(rows >= 1 && cols >= 1, "empty QR");
  hipLaunchKernelGGL(householder_qr_kernel, dim3(1), dim3(HH_THREADS), 0, s, M, rows, cols, tau, Q, qcols);
  QCA_HIP(hipGetLastError());
}

}  // namespace qca
