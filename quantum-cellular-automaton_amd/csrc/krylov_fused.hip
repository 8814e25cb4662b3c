// One-launch Krylov exponential for small blocks (gfx950).
//
// y = exp(-i tau H_eff) x for the 2-site, 1-site and bond effective
// Hamiltonians of reference algorithms/tdvp.py:298-326 (applied matrix-free)
// with the Lanczos scheme of lautils.py:44-81, entirely inside one workgroup:
//
//   * H_eff: T1 = L-contraction -> sparse MPO mixing -> R-contraction on the
//     matrix cores, in the environments' type (complex128, or complex64 on FP32
//     for the mixed path, as on the multi-launch path).  T1 lies in LDS with the
//     left index fastest, the layout of the second product's A operand, so the
//     mixing is a sparse sum of operands on their way into registers;
//   * recurrence: FP64, the three-term step and then one classical Gram-Schmidt
//     pass against the whole basis (a second pass: what the first leaves is
//     the non-Hermitian rounding of H_eff), the residual and the last two
//     basis vectors in registers (element e belongs to thread e % 512);
//   * tridiagonal exponential and the stopping test on wave 0, as in the
//     multi-launch path (Taylor with scaling, lane = row of T), from the
//     iteration on in which it can pass at all (fk_unconverged).
//
// The multi-launch path needs ~11 launches and a host round trip per Krylov
// iteration; at small bond dimension those dominate. This kernel needs one
// launch and no host round trip per exponential; it works on one CU, so it is
// used only below a size limit chosen by the engine.
// What bounds it: the two products (FP64 matrix rate of one CU: 2.6 us each for
// 4 x 16 x 16 with MPO bond 6) and the passes over the basis.  Eight waves: two
// per SIMD hide the operand loads, and a barrier takes 268 cycles where sixteen
// waves take 815.  Per iteration at bond 16 (averages over a 15-cell run, MPO bond 6): left
// product 3.1 us, mixing and right product 4.4, three-term step 1.1, projection
// 1.4, subtraction and norm 1.5, basis vector 0.5: 12 us, before 22 (sixteen
// waves, vector products from LDS and global memory, two full Gram-Schmidt
// passes, a tridiagonal exponential of 3.6 us every time).  The run: 155 -> 104
// ms, and 95 with the elements of small blocks on their own.  Above FUSED_KRYLOV_DEFAULT_N elements the whole chip is faster: bond 30,
// 82 ms with this limit and 86 with all blocks here.
#include "grouped.hpp"
#include "wave.hpp"

namespace qca {
namespace {

constexpr int FK_THREADS = 512;
constexpr int FK_WAVES = FK_THREADS / 64;
// Residual elements per thread: blocks up to FK_SMALL_N and up to the limit.
constexpr long FK_SMALL_N = 2 * FK_THREADS;
constexpr int FK_EPT_MAX = FUSED_KRYLOV_MAX_N / FK_THREADS;
// Dynamic LDS of one launch (the static part, FkShared, adds ~3 KB; 160 KB per CU).
constexpr long FK_LDS_BYTES = 152 * 1024;

struct FkShared {
  c128 coef[LZ_MAXK];
  double alpha[LZ_MAXK];
  double beta[LZ_MAXK];
  c128 z[LZ_MAXK];
  c128 red[2][FK_WAVES];
  double err;
  int flag, limit;
  unsigned long long used;     // channels (q, w) that the MPO reads, as bits
  unsigned char channel[64];   // and as a list
};

// Matrix-core tile of the element type: A[i][k] from lane i + 16 k, B[k][j] from
// lane j + 16 k, k < 4; register r of lane l holds D[row(r, l / 16)][l % 16].
template <typename T> struct FkMfma;
template <> struct FkMfma<double> {
  typedef double acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mul(double a, double b, acc c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int r, int hi) { return hi + 4 * r; }
};
template <> struct FkMfma<float> {
  typedef float acc __attribute__((ext_vector_type(4)));
  static __device__ __forceinline__ acc mul(float a, float b, acc c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int r, int hi) { return 4 * hi + r; }
};
// The two halves of each complex sum have accumulators of their own, and every 16 c
// of the right product a tile of their own: a quarter of the chain of roundings at
// bond 24 (error of one exponential over 126 blocks of bonds 8..30 against extended
// precision, one chain for all -> this: FP32 2.9e-8 -> 2.0e-8, FP64 2.14e-16 ->
// 2.10e-16; a 15-cell run 101.9 -> 103.6 ms).  A branch in the loop over the entries
// that sets sums aside costs 4 to 8%.
template <typename T>
struct FkTile {
  typename FkMfma<T>::acc re = {0, 0, 0, 0}, im = {0, 0, 0, 0}, xre = {0, 0, 0, 0}, xim = {0, 0, 0, 0};
  __device__ __forceinline__ void add(const cplx<T>& a, const cplx<T>& b) {
    re = FkMfma<T>::mul(a.re, b.re, re);
    im = FkMfma<T>::mul(a.re, b.im, im);
    xre = FkMfma<T>::mul(-a.im, b.im, xre);
    xim = FkMfma<T>::mul(a.im, b.re, xim);
  }
};
// Sum of tiles.
template <typename T>
struct FkSum {
  typename FkMfma<T>::acc re = {0, 0, 0, 0}, im = {0, 0, 0, 0};
  __device__ __forceinline__ void add(const FkTile<T>& t) {
    re += t.re + t.xre;
    im += t.im + t.xim;
  }
};

__device__ __forceinline__ double lane_value(double v, int lane) { return readlane_f64(v, lane); }
__device__ __forceinline__ float lane_value(float v, int lane) {
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), lane));
}

// Sum of (re, im) over the workgroup, returned to every thread; calls alternate
// between the halves of sh.red, so one barrier per sum is enough.
__device__ __forceinline__ c128 fk_block_sum(double re, double im, int half, FkShared& sh) {
  re = wave_sum64(re);
  im = wave_sum64(im);
  if ((threadIdx.x & 63) == 0) sh.red[half][threadIdx.x >> 6] = c128{re, im};
  __syncthreads();
  c128 t{0.0, 0.0};
#pragma unroll
  for (int i = 0; i < FK_WAVES; ++i) {
    t.re += sh.red[half][i].re;
    t.im += sh.red[half][i].im;
  }
  return t;
}

// T1[q][w][c][x] = sum_a v[q][a][c] L[a][w][x] for the nch channels q * Din + w in
// `channel` (null: all): 16x16 tiles (c, x), one wave each, the operands of the
// next 16 a on their way while the products of these run.
template <typename TE>
__device__ __forceinline__ void fk_left(const FusedKrylovArgs<TE>& a, const c128* v, const cplx<TE>* L, cplx<TE>* T1,
                                        const unsigned char* channel, int nch) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chil = a.chil, chir = a.chir, Din = a.Din;
  const int xt = (chil + 15) >> 4, ct = (chir + 15) >> 4, tiles = nch * xt * ct;
  auto fetch = [&](int t, int k0, c128(&av)[4], cplx<TE>(&bv)[4]) {
    const int n = t % nch, r1 = t / nch, ci = r1 % ct, xi = r1 / ct;
    const int qw = channel ? __builtin_amdgcn_readfirstlane((int)channel[n]) : n;
    const int q = qw / Din, w = qw - q * Din;
    const c128* vp = v + (unsigned)(q * chil * chir + min(16 * ci + lo, chir - 1));
    const cplx<TE>* lp = L + (unsigned)(w * chil + min(16 * xi + lo, chil - 1));
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const unsigned k = min(k0 + 4 * s + hi, chil - 1);
      av[s] = vp[k * chir];
      bv[s] = lp[k * (unsigned)(Din * chil)];
    }
  };
  c128 av[4], an[4];
  cplx<TE> bv[4], bn[4];
  FkTile<TE> acc;
  if (wave < tiles) fetch(wave, 0, av, bv);
  for (int t = wave, k0 = 0; t < tiles;) {
    const int kn = k0 + 16 < chil ? k0 + 16 : 0, tn = kn ? t : t + FK_WAVES;
    if (tn < tiles) fetch(tn, kn, an, bn);
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const bool in = k0 + 4 * s + hi < chil;
      if (k0 + 4 * s < chil)
        acc.add(cplx<TE>{in ? TE(av[s].re) : TE(0), in ? TE(av[s].im) : TE(0)}, bv[s]);
    }
    if (kn == 0) {
      const int n = t % nch, r1 = t / nch, ci = r1 % ct, xi = r1 / ct;
      const int qw = channel ? __builtin_amdgcn_readfirstlane((int)channel[n]) : n;
      const int x = 16 * xi + lo;
      cplx<TE>* out = T1 + (unsigned)(qw * chir * chil);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int cc = 16 * ci + FkMfma<TE>::row(r, hi);
        if (cc < chir && x < chil)
          out[(unsigned)(cc * chil + x)] = cplx<TE>{acc.re[r] + acc.xre[r], acc.im[r] + acc.xim[r]};
      }
      acc = FkTile<TE>();
    }
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      av[s] = an[s];
      bv[s] = bn[s];
    }
    t = tn;
    k0 = kn;
  }
}

// Lane i holds entry z0 + i of the sparse MPO's rows (q', 0..Dout-1): its row v,
// column and value, so that a wave-uniform lookup is a lane read instead of a
// chain of three memory reads (kind 2: one entry per v).
template <typename TE>
struct FkEntries {
  int first, last;   // entries of q'
  int v, c;
  cplx<TE> x;
};
template <typename TE>
__device__ __forceinline__ void fk_entries(const FusedKrylovArgs<TE>& a, int q, int z0, const int* rowptr,
                                           const int* col, const cplx<TE>* val, FkEntries<TE>& e) {
  const int z = min(z0 + (int)(threadIdx.x & 63), e.last - 1);
  e.v = e.c = z;
  e.x = cplx<TE>{TE(1), TE(0)};
  if (a.kind == 2 || z < z0) return;
  e.v = 0;
  for (int r = 1; r < a.Dout; ++r) e.v += rowptr[q * a.Dout + r] <= z ? 1 : 0;
  e.c = col[z];
  e.x = val[z];
}
template <typename TE>
__device__ __forceinline__ FkEntries<TE> fk_rows(const FusedKrylovArgs<TE>& a, int q, const int* rowptr,
                                                 const int* col, const cplx<TE>* val) {
  FkEntries<TE> e;
  e.first = a.kind == 2 ? 0 : __builtin_amdgcn_readfirstlane(rowptr[q * a.Dout]);
  e.last = a.kind == 2 ? a.Dout : __builtin_amdgcn_readfirstlane(rowptr[(q + 1) * a.Dout]);
  fk_entries(a, q, e.first, rowptr, col, val, e);
  return e;
}
// q' of this wave's first tile of y.
template <typename TE>
__device__ __forceinline__ int fk_first_q(const FusedKrylovArgs<TE>& a, int dq) {
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  return min((wave / a.parts) / (((a.chil + 15) >> 4) * ((a.chir + 15) >> 4)), dq - 1);
}

// y[q'][x][yy] = sum_{v,c} U[q'][x][c][v] R[c][v][yy], U[q'][x][c][v] the sum of
// val * T1[col][c][x] over row (q', v) of the sparse MPO (kind 2: U = T1[v]).
// Tiles (x, yy) of q', the rows v of each dealt to `parts` waves; partial sums go
// to part[p][e].  `mine` holds the entries of the wave's first tile (they are the
// same in every iteration).  With one tile per wave `part` lies over T1, hence
// the barrier.
template <typename TE>
__device__ __forceinline__ void fk_right(const FusedKrylovArgs<TE>& a, const cplx<TE>* T1, const cplx<TE>* R,
                                         const int* rowptr, const int* col, const cplx<TE>* val,
                                         const FkEntries<TE>& mine, c128* part) {
  const int lane = threadIdx.x & 63, lo = lane & 15, hi = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int chil = a.chil, chir = a.chir, Dout = a.Dout, parts = a.parts;
  const int dq = a.kind == 0 ? 4 : (a.kind == 1 ? 2 : 1);
  const int xt = (chil + 15) >> 4, yt = (chir + 15) >> 4, lr = chil * chir;
  const int p = wave & (parts - 1), ntiles = dq * xt * yt;
  auto compute = [&](int t, FkEntries<TE> e, FkSum<TE>& sum) {
    const int yi = t % yt, r1 = t / yt, xi = r1 % xt, q = r1 / xt;
    const cplx<TE>* tp = T1 + min(16 * xi + lo, chil - 1);
    const cplx<TE>* rp = R + min(16 * yi + lo, chir - 1);
    for (int z0 = e.first; z0 < e.last; z0 += 64) {
      if (z0 > e.first) fk_entries(a, q, z0, rowptr, col, val, e);
      const int nz = min(64, e.last - z0);
      for (int k0 = 0; k0 < chir; k0 += 16) {
        unsigned at[4], ar[4];
#pragma unroll
        for (int s = 0; s < 4; ++s) {
          const unsigned c = min(k0 + 4 * s + hi, chir - 1);
          at[s] = c * chil;
          ar[s] = c * (unsigned)(Dout * chir);
        }
        // the wave's entries are i with row v = p, p + parts, ...
        auto next = [&](int i) {
          while (i < nz && (__builtin_amdgcn_readlane(e.v, i) & (parts - 1)) != p) ++i;
          return i;
        };
        auto fetch = [&](int i, cplx<TE>(&u)[4], cplx<TE>(&av)[4]) {
          const cplx<TE>* tz = tp + (unsigned)(__builtin_amdgcn_readlane(e.c, i) * lr);
          const cplx<TE>* rz = rp + (unsigned)(__builtin_amdgcn_readlane(e.v, i) * chir);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            u[s] = tz[at[s]];
            av[s] = rz[ar[s]];
          }
        };
        cplx<TE> u[4], av[4], un[4], an[4], bv[4];
        FkTile<TE> acc;   // of these 16 c: a chain over the entries, not over all c
        int i = next(0);
        if (i < nz) fetch(i, u, av);
        bool fresh = true;
        while (i < nz) {
          const int in = next(i + 1);
          const bool more = in < nz && __builtin_amdgcn_readlane(e.v, in) == __builtin_amdgcn_readlane(e.v, i);
          if (in < nz) fetch(in, un, an);
          const cplx<TE> wv{lane_value(e.x.re, i), lane_value(e.x.im, i)};
          if (wv.re != TE(1) || wv.im != TE(0))   // the rules' MPOs have ones only
#pragma unroll
            for (int s = 0; s < 4; ++s)
              u[s] = cplx<TE>{wv.re * u[s].re - wv.im * u[s].im, wv.re * u[s].im + wv.im * u[s].re};
#pragma unroll
          for (int s = 0; s < 4; ++s) bv[s] = fresh ? u[s] : cplx<TE>{bv[s].re + u[s].re, bv[s].im + u[s].im};
          fresh = !more;
          if (!more) {
#pragma unroll
            for (int s = 0; s < 4; ++s) {
              const bool inside = k0 + 4 * s + hi < chir;
              if (k0 + 4 * s < chir)
                acc.add(bv[s], cplx<TE>{inside ? av[s].re : TE(0), inside ? av[s].im : TE(0)});
            }
          }
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            u[s] = un[s];
            av[s] = an[s];
          }
          i = in;
        }
        sum.add(acc);
      }
    }
  };
  auto store = [&](int t, const FkSum<TE>& acc) {
    const int yi = t % yt, r1 = t / yt, xi = r1 % xt, q = r1 / xt;
    const int yy = 16 * yi + lo;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int x = 16 * xi + FkMfma<TE>::row(r, hi);
      if (yy < chir && x < chil)
        part[(unsigned)(p * dq * lr + (q * chil + x) * chir + yy)] = c128{double(acc.re[r]), double(acc.im[r])};
    }
  };
  int t = wave / parts;
  if (a.overlay) {
    FkSum<TE> acc;
    if (t < ntiles) compute(t, mine, acc);
    __syncthreads();
    if (t < ntiles) store(t, acc);
  } else {
    for (; t < ntiles; t += FK_WAVES / parts) {
      FkSum<TE> acc;
      compute(t, fk_rows(a, t / (xt * yt), rowptr, col, val), acc);
      store(t, acc);
    }
  }
}

// Small blocks, element by element: a 16x16 tile would be padding for the most part,
// and its wave would walk the entries one after another.  Thread t takes
// elements t, t + 512, ... of T1, and S lanes share an element of y, each with every
// S-th entry of its q'.  What a thread reads is the same in every iteration, so the
// offsets are kept in registers.
constexpr int FK_SMALL_LEFT = 8;      // elements of T1 per thread
constexpr int FK_SMALL_RIGHT = 8;     // entries per thread
template <typename TE>
struct FkSmall {
  int v[FK_SMALL_LEFT], l[FK_SMALL_LEFT], out[FK_SMALL_LEFT];   // out < 0: none
  int t[FK_SMALL_RIGHT], r[FK_SMALL_RIGHT], entries;
  cplx<TE> val[FK_SMALL_RIGHT];
};
template <typename TE>
__device__ __forceinline__ void fk_small_init(const FusedKrylovArgs<TE>& a, const unsigned char* channel, int nch,
                                              const int* rowptr, const int* col, const cplx<TE>* val,
                                              FkSmall<TE>& m) {
  const int lr = a.chil * a.chir, tid = threadIdx.x;
#pragma unroll
  for (int k = 0; k < FK_SMALL_LEFT; ++k) {
    const int i = tid + FK_THREADS * k, n = i / lr, rem = i - n * lr, c = rem / a.chil, x = rem - c * a.chil;
    const bool in = n < nch;
    const int qw = !in ? 0 : channel ? channel[n] : n, q = qw / a.Din, w = qw - q * a.Din;
    m.v[k] = q * lr + c;
    m.l[k] = w * a.chil + x;
    m.out[k] = in ? qw * lr + rem : -1;
  }
  const int e = tid / a.lanes, s = tid & (a.lanes - 1), q = e / lr, rem = e - q * lr, x = rem / a.chir,
            yy = rem - x * a.chir;
  m.entries = 0;
#pragma unroll
  for (int k = 0; k < FK_SMALL_RIGHT; ++k) {
    m.t[k] = m.r[k] = 0;
    m.val[k] = cplx<TE>{TE(1), TE(0)};
  }
  if (e >= (int)a.n) return;
  const int first = a.kind == 2 ? 0 : rowptr[q * a.Dout], last = a.kind == 2 ? a.Dout : rowptr[(q + 1) * a.Dout];
#pragma unroll
  for (int k = 0; k < FK_SMALL_RIGHT; ++k) {
    const int z = first + s + a.lanes * k;
    if (z >= last) break;
    int v = z, cz = z;
    if (a.kind != 2) {
      v = 0;
      for (int r = 1; r < a.Dout; ++r) v += rowptr[q * a.Dout + r] <= z ? 1 : 0;
      cz = col[z];
      m.val[k] = val[z];
    }
    m.t[k] = cz * lr + x;
    m.r[k] = v * a.chir + yy;
    m.entries = k + 1;
  }
}
template <typename TE>
__device__ __forceinline__ void fk_small_left(const FusedKrylovArgs<TE>& a, const c128* v, const cplx<TE>* L,
                                              cplx<TE>* T1, const FkSmall<TE>& m) {
  cplx<TE> acc[FK_SMALL_LEFT] = {};
  const int ls = a.Din * a.chil;
  for (int i = 0; i < a.chil; ++i) {
#pragma unroll
    for (int k = 0; k < FK_SMALL_LEFT; ++k) {
      if (m.out[k] < 0) continue;
      const c128 x = v[m.v[k] + i * a.chir];
      const cplx<TE> y = L[m.l[k] + i * ls], z{TE(x.re), TE(x.im)};
      acc[k].re += z.re * y.re - z.im * y.im;
      acc[k].im += z.re * y.im + z.im * y.re;
    }
  }
#pragma unroll
  for (int k = 0; k < FK_SMALL_LEFT; ++k)
    if (m.out[k] >= 0) T1[m.out[k]] = acc[k];
}
template <typename TE>
__device__ __forceinline__ void fk_small_right(const FusedKrylovArgs<TE>& a, const cplx<TE>* T1, const cplx<TE>* R,
                                               const FkSmall<TE>& m, c128* y) {
  double re = 0, im = 0;
  const int rs = a.Dout * a.chir;
#pragma unroll
  for (int k = 0; k < FK_SMALL_RIGHT; ++k) {
    if (k >= m.entries) continue;
    cplx<TE> acc{TE(0), TE(0)};
    for (int c = 0; c < a.chir; ++c) {
      const cplx<TE> t = T1[m.t[k] + c * a.chil], r = R[m.r[k] + c * rs];
      acc.re += t.re * r.re - t.im * r.im;
      acc.im += t.re * r.im + t.im * r.re;
    }
    re += double(m.val[k].re * acc.re - m.val[k].im * acc.im);
    im += double(m.val[k].re * acc.im + m.val[k].im * acc.re);
  }
  // over the lanes of an element (a row of 16 at most)
  if (a.lanes > 1) re += dpp_f64<0xB1>(re), im += dpp_f64<0xB1>(im);      // quad_perm(1,0,3,2)
  if (a.lanes > 2) re += dpp_f64<0x4E>(re), im += dpp_f64<0x4E>(im);      // quad_perm(2,3,0,1)
  if (a.lanes > 4) re += dpp_f64<0x141>(re), im += dpp_f64<0x141>(im);    // row_half_mirror
  if (a.lanes > 8) re += dpp_f64<0x140>(re), im += dpp_f64<0x140>(im);    // row_mirror
  const int e = threadIdx.x / a.lanes;
  if ((threadIdx.x & (a.lanes - 1)) == 0 && e < (int)a.n) y[e] = c128{re, im};
}

// Lane l + 1 and lane l - 1 of the wave, 0 beyond its ends.
template <int CTRL>
__device__ __forceinline__ double wave_shift(double v) {
  const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ double lane_above(double v) { return wave_shift<0x130>(v); }   // wave_shl:1
__device__ __forceinline__ double lane_below(double v) { return wave_shift<0x138>(v); }   // wave_shr:1

// Largest v of the wave, in every lane.
__device__ __forceinline__ double wave_max64(double v) {
  v = fmax(v, dpp_f64<0xB1>(v));    // quad_perm(1,0,3,2)
  v = fmax(v, dpp_f64<0x4E>(v));    // quad_perm(2,3,0,1)
  v = fmax(v, dpp_f64<0x141>(v));   // row_half_mirror
  v = fmax(v, dpp_f64<0x140>(v));   // row_mirror
  return fmax(fmax(readlane_f64(v, 0), readlane_f64(v, 16)), fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// Wave 0: z = exp(-i tau T_m) e_0 for the m = j+1 leading rows of the
// tridiagonal T (alpha on the diagonal, beta off it), by Taylor steps with
// scaling (lane = row); returns |beta_j z_j| on every lane.
__device__ double fk_tridiag_exp(const FkShared& sh, int j, double beta, double tau, double& zr,
                                 double& zi) {
  const int l = threadIdx.x & 63;
  const int m = j + 1;
  const double al = (l < m) ? sh.alpha[l] : 0.0;
  const double bup = (l + 1 < m) ? sh.beta[l] : 0.0;
  const double bdn = (l >= 1 && l < m) ? sh.beta[l - 1] : 0.0;
  const double rown = wave_max64(fabs(al) + fabs(bup) + fabs(bdn));
  const double h = fabs(tau) * rown;
  const int nsub = (h < 2048.0) ? max(1, (int)ceil(h / 0.5)) : 1;
  const double dt = tau / nsub;
  zr = (l == 0) ? 1.0 : 0.0;
  zi = 0.0;
  for (int sstep = 0; sstep < nsub; ++sstep) {
    double ar = zr, ai = zi, tr = zr, ti = zi;
    for (int k = 1; k < 60; ++k) {
      const double upr = lane_above(tr), upi = lane_above(ti);
      const double dnr = lane_below(tr), dni = lane_below(ti);
      double yr = al * tr + bup * upr + bdn * dnr;
      double yi = al * ti + bup * upi + bdn * dni;
      if (l >= m) {
        yr = 0;
        yi = 0;
      }
      const double ck = dt / k;
      const double nr = ck * yi, ni = -ck * yr;
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
  const double zlr = readlane_f64(zr, j), zli = readlane_f64(zi, j);
  return beta * sqrt(zlr * zlr + zli * zli);
}

// Whether the error estimate beta_j |z_j| of iteration j is certainly above 2 tol,
// from a lower bound: z_j is the product of the betas times a divided difference
// of exp(-i tau .) over the eigenvalues of T, (-i tau)^j times the mean of
// exp(-i tau s) / j! over a simplex of points s between them (Hermite-Genocchi),
// so |z_j| >= prod |tau|^j / j! cos(tau width / 2) with Gershgorin's width.  The
// tridiagonal exponential (1.6 us) is evaluated when this does not decide: one or
// two times per call instead of m.
struct FkBound {
  double prod = 1.0, low = 0.0, high = 0.0, last = 0.0;
  __device__ __forceinline__ bool unconverged(int j, double alpha, double beta, double tau, double tol) {
    tau = fabs(tau);
    if (j > 0) prod *= last * tau / j;
    const double r = last + beta;
    low = j > 0 ? fmin(low, alpha - r) : alpha - r;
    high = j > 0 ? fmax(high, alpha + r) : alpha + r;
    last = beta;
    const double h = 0.5 * tau * (high - low);
    return h < 1.4 && beta * prod * (1.0 - 0.5 * h * h) >= 2.0 * tol;   // cos h >= 1 - h^2 / 2
  }
};

template <typename TE, int EPT, bool SMALL>
__device__ __forceinline__ void fused_krylov_body(const FusedKrylovArgs<TE>& a, unsigned char* arena, FkShared& sh) {
  const int n = (int)a.n, tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const unsigned long long t0 = wall_clock64();
  // LDS: T1, the partial sums of y and then the residual (over T1 where that is
  // used up), the MPO; T1 and the MPO stay in global memory when they don't fit
  cplx<TE>* T1l = reinterpret_cast<cplx<TE>*>(arena);
  c128* wbuf = reinterpret_cast<c128*>(arena + a.offW);
  int* rowptr = reinterpret_cast<int*>(arena + a.offRow);
  int* col = reinterpret_cast<int*>(arena + a.offCol);
  cplx<TE>* val = reinterpret_cast<cplx<TE>*>(arena + a.offVal);
  cplx<TE>* Ll = reinterpret_cast<cplx<TE>*>(arena + a.offL);
  cplx<TE>* Rl = reinterpret_cast<cplx<TE>*>(arena + a.offR);
  c128* Vl = reinterpret_cast<c128*>(arena + a.offV);   // leading vcap basis vectors
  c128* __restrict__ Vg = a.V;                          // the others
  const int dq = a.kind == 0 ? 4 : (a.kind == 1 ? 2 : 1);
  if (a.t1_lds && a.kind != 2) {
    for (int i = tid; i <= dq * a.Dout; i += FK_THREADS) rowptr[i] = a.rowptr[i];
    for (int i = tid; i < a.nnz; i += FK_THREADS) {
      col[i] = a.col[i];
      val[i] = a.val[i];
    }
  }
  if (a.env_lds) {
    const int nL = a.chil * a.Din * a.chil, nR = a.chir * a.Dout * a.chir;
#pragma unroll 4
    for (int i = tid; i < nL; i += FK_THREADS) Ll[i] = a.L[i];
#pragma unroll 4
    for (int i = tid; i < nR; i += FK_THREADS) Rl[i] = a.R[i];
  }
  // channels of T1 that some row of the MPO reads
  const int ncol = dq * a.Din;
  const bool listed = a.kind != 2 && ncol <= 64;
  if (tid == 0) sh.used = 0;
  __syncthreads();
  if (listed)
    for (int i = tid; i < a.nnz; i += FK_THREADS) atomicOr(&sh.used, 1ull << a.col[i]);
  __syncthreads();
  const unsigned long long used = sh.used;
  if (listed && tid < 64 && (used >> tid & 1)) sh.channel[__popcll(used & ((1ull << tid) - 1))] = (unsigned char)tid;
  const unsigned char* channel = listed ? sh.channel : nullptr;
  const int nch = listed ? __popcll(used) : ncol;
  FkSmall<TE> sm;
  FkEntries<TE> mine;
  if constexpr (SMALL) {
    __syncthreads();
    fk_small_init(a, channel, nch, rowptr, col, val, sm);
  } else {
    const int q0 = fk_first_q(a, dq);
    mine = a.t1_lds ? fk_rows(a, q0, rowptr, col, val) : fk_rows(a, q0, a.rowptr, a.col, a.val);
  }
  // f(V_i) with the basis vector in its own address space
  auto with_basis = [&](int i, auto&& f) {
    if (i < a.vcap) f(Vl + (unsigned)(i * n));
    else f(Vg + (unsigned)(i * n));
  };
  c128 w[EPT], v0[EPT], v1[EPT];   // residual, V_j, V_{j-1}: elements tid, tid + 512, ...
  double nrm = 0;
#pragma unroll
  for (int r = 0; r < EPT; ++r) {
    const int e = tid + r * FK_THREADS;
    w[r] = e < n ? a.x[e] : c128{0.0, 0.0};
    v0[r] = c128{0.0, 0.0};
    nrm += w[r].re * w[r].re + w[r].im * w[r].im;
  }
  const double beta0 = sqrt(fk_block_sum(nrm, 0.0, 0, sh).re);
  int m = 0, hit_limit = 0;
  double err = 0;
  if (beta0 > 0.0) {
    FkBound bound;
    double beta = beta0;
    for (int j = 0;; ++j) {
      // V_j
      const double inv = 1.0 / beta;
#pragma unroll
      for (int r = 0; r < EPT; ++r) {
        v1[r] = v0[r];
        v0[r] = c128{w[r].re * inv, w[r].im * inv};
      }
      with_basis(j, [&](c128* vj) {
#pragma unroll
        for (int r = 0; r < EPT; ++r)
          if (tid + r * FK_THREADS < n) vj[tid + r * FK_THREADS] = v0[r];
      });
      __syncthreads();
      // w = H_eff V_j
      const c128* vj = j < a.vcap ? Vl + (unsigned)(j * n) : Vg + (unsigned)(j * n);
      if constexpr (SMALL) {
        fk_small_left(a, vj, Ll, T1l, sm);
        __syncthreads();
        fk_small_right(a, T1l, Rl, sm, wbuf);
      } else if (a.env_lds) {
        fk_left<TE>(a, vj, Ll, T1l, channel, nch);
        __syncthreads();
        fk_right<TE>(a, T1l, Rl, rowptr, col, val, mine, wbuf);
      } else if (a.t1_lds) {
        fk_left<TE>(a, vj, a.L, T1l, channel, nch);
        __syncthreads();
        fk_right<TE>(a, T1l, a.R, rowptr, col, val, mine, wbuf);
      } else {
        fk_left<TE>(a, vj, a.L, a.T1, channel, nch);
        __syncthreads();
        fk_right<TE>(a, a.T1, a.R, a.rowptr, a.col, a.val, mine, wbuf);
      }
      __syncthreads();
      double ar = 0, ai = 0;
#pragma unroll
      for (int r = 0; r < EPT; ++r) {
        const int e = tid + r * FK_THREADS;
        w[r] = c128{0.0, 0.0};
        if (e < n)
          for (int p = 0; p < a.parts; ++p) {
            const c128 y = wbuf[p * n + e];
            w[r].re += y.re;
            w[r].im += y.im;
          }
        ar += v0[r].re * w[r].re + v0[r].im * w[r].im;
        ai += v0[r].re * w[r].im - v0[r].im * w[r].re;
      }
      // three-term step
      const c128 c1 = fk_block_sum(ar, ai, 1, sh);
      const double bp = j > 0 ? beta : 0.0;
#pragma unroll
      for (int r = 0; r < EPT; ++r) {
        w[r].re -= c1.re * v0[r].re - c1.im * v0[r].im + bp * v1[r].re;
        w[r].im -= c1.re * v0[r].im + c1.im * v0[r].re + bp * v1[r].im;
        if (tid + r * FK_THREADS < n) wbuf[tid + r * FK_THREADS] = w[r];
      }
      __syncthreads();
      // coef_i = <V_i, w>: the residual is in LDS, wave k takes i = k, k + 8, ...
      for (int i = wave; i <= j; i += FK_WAVES) {
        double pr = 0, pi = 0;
        with_basis(i, [&](const c128* vi) {
#pragma unroll 8
          for (int e = lane; e < n; e += 64) {
            const c128 b = vi[e], x = wbuf[e];
            pr += b.re * x.re + b.im * x.im;
            pi += b.re * x.im - b.im * x.re;
          }
        });
        pr = wave_sum64(pr);
        pi = wave_sum64(pi);
        if (lane == 0) sh.coef[i] = c128{pr, pi};
      }
      __syncthreads();
      // w -= sum_i coef_i V_i
      auto subtract = [&](const c128* vi, const c128& c) {
#pragma unroll
        for (int r = 0; r < EPT; ++r) {
          const c128 b = vi[min(tid + r * FK_THREADS, n - 1)];
          w[r].re -= c.re * b.re - c.im * b.im;
          w[r].im -= c.re * b.im + c.im * b.re;
        }
      };
      const int nl = min(j, a.vcap);
#pragma unroll 2
      for (int i = 0; i < nl; ++i) subtract(Vl + (unsigned)(i * n), sh.coef[i]);
#pragma unroll 4
      for (int i = nl; i < j; ++i) subtract(Vg + (unsigned)(i * n), sh.coef[i]);
      const c128 c2 = sh.coef[j];
      double s = 0;
#pragma unroll
      for (int r = 0; r < EPT; ++r) {
        w[r].re -= c2.re * v0[r].re - c2.im * v0[r].im;
        w[r].im -= c2.re * v0[r].im + c2.im * v0[r].re;
        if (tid + r * FK_THREADS >= n) w[r] = c128{0.0, 0.0};
        s += w[r].re * w[r].re + w[r].im * w[r].im;
      }
      beta = sqrt(fk_block_sum(s, 0.0, 0, sh).re);
      const double alpha_j = c1.re + c2.re;
      if (tid == 0) {
        sh.alpha[j] = alpha_j;
        sh.beta[j] = beta;
      }
      const bool breakdown = beta <= 1e-13 * fmax(1.0, fabs(alpha_j));
      const bool unconverged = bound.unconverged(j, alpha_j, beta, a.tau, a.tol);
      if (unconverged && !breakdown && j + 1 < a.max_m - 1) continue;
      if (wave == 0) {
        // wave 0 reads its own writes: wave-local LDS order holds
        __builtin_amdgcn_wave_barrier();
        double zr, zi;
        const double e = fk_tridiag_exp(sh, j, beta, a.tau, zr, zi);
        const bool conv = breakdown || e < a.tol || j + 1 >= a.max_m - 1;
        if (lane <= j) sh.z[lane] = c128{zr, zi};
        if (lane == 0) {
          sh.flag = conv ? 1 : 0;
          sh.err = e;
          sh.limit = !breakdown && e >= a.tol;
        }
      }
      __syncthreads();
      err = sh.err;
      hit_limit = sh.limit;
      if (sh.flag) {
        m = j + 1;
        break;
      }
    }
  }
  // x = beta0 * sum_{i<m} z_i V_i  (a zero input stays zero)
#pragma unroll
  for (int r = 0; r < EPT; ++r) w[r] = c128{0.0, 0.0};
  auto add = [&](const c128* vi, const c128& z) {
#pragma unroll
    for (int r = 0; r < EPT; ++r) {
      const c128 b = vi[min(tid + r * FK_THREADS, n - 1)];
      w[r].re += z.re * b.re - z.im * b.im;
      w[r].im += z.re * b.im + z.im * b.re;
    }
  };
  const int nl = min(m, a.vcap);
#pragma unroll 2
  for (int i = 0; i < nl; ++i) add(Vl + (unsigned)(i * n), sh.z[i]);
#pragma unroll 4
  for (int i = nl; i < m; ++i) add(Vg + (unsigned)(i * n), sh.z[i]);
#pragma unroll
  for (int r = 0; r < EPT; ++r) {
    const int e = tid + r * FK_THREADS;
    if (e < n) a.x[e] = c128{beta0 * w[r].re, beta0 * w[r].im};
  }
  if (tid == 0) {
    if (a.ctrl) {
      a.ctrl->beta0 = beta0;
      a.ctrl->err = err;
      a.ctrl->m = m;
      a.ctrl->done = 1;
      a.ctrl->zero = beta0 == 0.0;
      a.ctrl->hit_limit = hit_limit;
    }
    if (a.tally) {
      // stream-ordered per engine: plain read-modify-write is race free
      a.tally->matvecs[a.kind] += m;
      a.tally->limit_hits += hit_limit;
      a.tally->flops += m * a.flops_per_matvec;
      a.tally->ticks += wall_clock64() - t0;
      a.tally->calls += 1;
    }
  }
}

template <typename TE, int EPT, bool SMALL>
__global__ __launch_bounds__(FK_THREADS) void fused_krylov_kernel(FusedKrylovArgs<TE> a) {
  extern __shared__ __align__(16) unsigned char arena[];
  __shared__ FkShared sh;
  fused_krylov_body<TE, EPT, SMALL>(a, arena, sh);
}

// One exponential per workgroup, each with its own arguments and LDS placement
// (the dynamic LDS of the launch is the largest placement).
template <typename TE, int EPT>
__global__ __launch_bounds__(FK_THREADS) void fused_krylov_grouped(const GRec<FusedKrylovArgs<TE>>* __restrict__ recs,
                                                                   int n) {
  extern __shared__ __align__(16) unsigned char arena[];
  FusedKrylovArgs<TE> a = recs[blockIdx.x].a;
  a.L = gbl(a.L);
  a.R = gbl(a.R);
  a.rowptr = gbl(a.rowptr);
  a.col = gbl(a.col);
  a.val = gbl(a.val);
  a.x = gbl(a.x);
  a.V = gbl(a.V);
  a.T1 = gbl(a.T1);
  a.ctrl = gbl(a.ctrl);
  a.tally = gbl(a.tally);
  __shared__ FkShared sh;
  if (a.lanes > 0) fused_krylov_body<TE, 1, true>(a, arena, sh);
  else fused_krylov_body<TE, EPT, false>(a, arena, sh);
}

}  // namespace

template <typename TE>
size_t fused_krylov_place(const FusedKrylovArgs<TE>& a, FusedKrylovArgs<TE>& b) {
  QCA_CHECK(a.n >= 1 && a.n <= FUSED_KRYLOV_MAX_N, "fused Krylov block above its size limit");
  QCA_CHECK(a.kind >= 0 && a.kind <= 2, "unknown effective-Hamiltonian kind");
  const int dq = a.kind == 0 ? 4 : (a.kind == 1 ? 2 : 1);
  QCA_CHECK(a.n == (long)dq * a.chil * a.chir, "Krylov vector length does not match the block");
  QCA_CHECK(a.max_m >= 2 && a.max_m <= LZ_MAXK, "Krylov dimension limit out of range");
  QCA_CHECK(a.kind == 2 || (a.rowptr && a.col && a.val), "sparse MPO missing");
  QCA_CHECK(a.kind != 2 || a.Din == a.Dout, "bond block needs equal MPO bonds");
  QCA_CHECK(a.kind == 2 || a.nnz >= 0, "negative MPO entry count");
  QCA_CHECK(a.kind == 2 || a.Dout <= 16, "MPO bond dimension above 16");
  b = a;
  const long lr = (long)a.chil * a.chir;
  const long t1 = (long)dq * a.Din * lr * sizeof(cplx<TE>);
  const long nnz = a.kind == 2 ? 0 : a.nnz, nrow = a.kind == 2 ? 0 : dq * a.Dout + 1;
  const long mpo = 48 + nrow * (long)sizeof(int) + nnz * (long)(sizeof(int) + sizeof(cplx<TE>));
  const long envL = (long)a.chil * a.Din * a.chil * sizeof(cplx<TE>), envR = (long)a.chir * a.Dout * a.chir * sizeof(cplx<TE>);
  // Up to 64 elements of chil x chir, element by element, by as many lanes per
  // element of y as there are (16 at most), if a thread's share fits its registers and
  // the operands LDS (MPO bond 13, FP64, tiles -> elements: two-site 1 x 1 64.7 -> 22.7
  // us, 4 x 4 146 -> 63, 4 x 8 210 -> 118, 8 x 8 221 -> 150, 16 x 4 203 -> 146; one-site 8 x 8
  // 148 -> 120; from 8 x 16 on tiles: 172 against 186 there).  A bond block has one
  // entry per row, so only its walk along c is left to shorten: up to 12 (4 x 12 101 ->
  // 82; 4 x 16 106 against 135).
  b.lanes = 16;
  while (b.lanes > 0 && b.lanes * a.n > FK_THREADS) b.lanes /= 2;
  const int group = a.kind == 2 ? a.Dout : (a.group_max > 0 ? a.group_max : a.nnz);
  if (b.lanes > 0 && (lr > 64 || (a.kind == 2 && a.chir > 12) ||
                      (long)dq * a.Din * lr > (long)FK_SMALL_LEFT * FK_THREADS ||
                      ceil_div(group, b.lanes) > FK_SMALL_RIGHT ||
                      t1 + 16 + a.n * (long)sizeof(c128) + mpo + envL + envR + 32 > FK_LDS_BYTES))
    b.lanes = 0;
  // tiles of y and the waves that share one, splitting its MPO rows
  const long tiles = (long)dq * ceil_div(a.chil, 16) * ceil_div(a.chir, 16);
  b.parts = 1;
  if (b.lanes == 0)
    while (2 * b.parts * tiles <= FK_WAVES && 2 * b.parts <= a.Dout) b.parts *= 2;
  // LDS: T1 and the MPO if both fit (else they stay in global memory), the partial
  // sums of y (over T1 if every wave has its tiles in registers by then), leading
  // basis vectors
  b.overlay = b.lanes == 0 && tiles * b.parts <= FK_WAVES;
  long off = 0;
  auto take = [&](long bytes) {
    const long o = off;
    off += (bytes + 15) / 16 * 16;
    return o;
  };
  const long py = b.parts * a.n * (long)sizeof(c128);
  const long work = b.overlay ? std::max(t1, py) : t1 + 16 + py;
  b.t1_lds = work + 16 + mpo <= FK_LDS_BYTES;
  if (b.t1_lds) {
    take(b.overlay ? std::max(t1, py) : t1);
    b.offW = b.overlay ? 0 : take(py);
    b.offVal = take(nnz * sizeof(cplx<TE>));
    b.offRow = take(nrow * sizeof(int));
    b.offCol = take(nnz * sizeof(int));
  } else {
    b.offW = take(py);
  }
  // environments: both, ahead of the basis (their latency is in the way of every
  // product; the basis is streamed)
  b.env_lds = b.t1_lds && off + envL + envR + 32 <= FK_LDS_BYTES;
  b.offL = b.env_lds ? take(envL) : 0;
  b.offR = b.env_lds ? take(envR) : 0;
  const long vbytes = a.n * (long)sizeof(c128);
  b.vcap = (int)std::min<long>(a.max_m - 1, (FK_LDS_BYTES - off) / vbytes);
  b.offV = take(b.vcap * vbytes);
  return (size_t)off;
}
template size_t fused_krylov_place<double>(const FusedKrylovArgs<double>&, FusedKrylovArgs<double>&);
template size_t fused_krylov_place<float>(const FusedKrylovArgs<float>&, FusedKrylovArgs<float>&);

template <typename TE>
void launch_fused_krylov(const FusedKrylovArgs<TE>& a, hipStream_t s) {
  FusedKrylovArgs<TE> b;
  const size_t off = fused_krylov_place(a, b);
  auto run = [&](auto kernel) {
    ensure_dynamic_lds((const void*)kernel, off);
    hipLaunchKernelGGL(kernel, dim3(1), dim3(FK_THREADS), off, s, b);
  };
  if (b.lanes > 0) run(fused_krylov_kernel<TE, 1, true>);
  else if (a.n <= FK_SMALL_N) run(fused_krylov_kernel<TE, 2, false>);
  else run(fused_krylov_kernel<TE, FK_EPT_MAX, false>);
  QCA_HIP(hipGetLastError());
}
template void launch_fused_krylov<double>(const FusedKrylovArgs<double>&, hipStream_t);
template void launch_fused_krylov<float>(const FusedKrylovArgs<float>&, hipStream_t);

template <typename TE>
void launch_fused_krylov_grouped(const KGroup<FusedKrylovArgs<TE>>& g, long max_n, size_t lds, hipStream_t s) {
  if (g.empty()) return;
  auto run = [&](auto kernel) {
    ensure_dynamic_lds((const void*)kernel, lds);
    hipLaunchKernelGGL(kernel, dim3(g.l.blocks), dim3(FK_THREADS), lds, s, g.l.recs, g.l.n);
  };
  if (max_n <= FK_SMALL_N) run(fused_krylov_grouped<TE, 2>);
  else run(fused_krylov_grouped<TE, FK_EPT_MAX>);
  QCA_HIP(hipGetLastError());
}
template void launch_fused_krylov_grouped<double>(const KGroup<FusedKrylovArgs<double>>&, long, size_t, hipStream_t);
template void launch_fused_krylov_grouped<float>(const KGroup<FusedKrylovArgs<float>>&, long, size_t, hipStream_t);

}  // namespace qca
