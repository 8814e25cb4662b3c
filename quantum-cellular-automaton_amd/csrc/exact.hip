// Exact state-vector path (gfx950): the rule Hamiltonian on 2^N amplitudes,
// its time evolution by a Chebyshev series, and the single-site density
// matrices.
//
//   (H psi)[x] = sum_i [number of alive cells within `distance` of cell i lies
//                       in [lo, hi)] psi[x ^ bit_i],  cell i is bit N-1-i.
//
// exp(-i tau H) psi = sum_k (2 - [k = 0]) (-i)^k J_k(tau R) T_k(H / R) psi with
// |H| <= R = N (a row of H has at most N unit entries).  The recurrence
// phi_{k+1} = (2/R) H phi_k - phi_{k-1} needs three vectors and no inner
// products, where the Krylov basis it replaced read every earlier vector
// several times per step.  One step of 2^23 amplitudes, tau = 0.785: 41 Krylov
// vectors 101 ms, 47 Chebyshev terms 7.8 ms; 2^12, tau = 0.31: 1.07 -> 0.15 ms.
#include "kernels.hpp"
#include "wave.hpp"

#include <algorithm>
#include <cmath>
#include <cstddef>
#include <vector>

namespace qca {
namespace {

__device__ double rho_block_sum(double v, double* sh) {
  v = wave_sum64(v);
  const int w = threadIdx.x >> 6, l = threadIdx.x & 63;
  __syncthreads();
  if (l == 0) sh[w] = v;
  __syncthreads();
  const int nw = blockDim.x >> 6;
  double r = 0;
  for (int i = 0; i < nw; ++i) r += sh[i];
  return r;
}

// Bit i of the result: the count of set bits of x within distance d of bit i
// (bit i itself excluded) lies in [lo, hi).  All cells at once: the counts are
// held as bit planes and the 2d shifted copies of x are added with carries.
// D > 0: the distance, known at compile time; D == 0: `d`.  Bits >= ncells of
// the result are meaningless.
template <typename I, int D>
__device__ __forceinline__ I active_cells(I x, int d, int lo, int hi) {
  constexpr int P = D == 1 ? 2 : (D == 2 ? 3 : 6);   // counts up to 2, 4, 63
  I pl[P];
#pragma unroll
  for (int k = 0; k < P; ++k) pl[k] = 0;
  auto add = [&](I s) {
#pragma unroll
    for (int k = 0; k < P; ++k) {
      const I t = pl[k] & s;
      pl[k] ^= s;
      s = t;
    }
  };
  if constexpr (D > 0) {
#pragma unroll
    for (int o = 1; o <= D; ++o) {
      add(x >> o);
      add(x << o);
    }
  } else {
    for (int o = 1; o <= d; ++o) {
      add(x >> o);
      add(x << o);
    }
  }
  auto at_least = [&](int v) -> I {
    if (v <= 0) return ~I(0);
    if (v >= (1 << P)) return I(0);
    I g = ~I(0);
#pragma unroll
    for (int k = 0; k < P; ++k) g = ((v >> k) & 1) ? (pl[k] & g) : (pl[k] | g);
    return g;
  };
  return at_least(lo) & ~at_least(hi);
}

// What becomes of h = H phi: out = h (apply), or one Chebyshev step
//   next = scale h - prev (prev may be null),
//   dst  = (init ? 0 : acc) + e0 phi + (e2 + i o1) next.
template <typename T>
struct ExactStep {
  cplx<T>* next = nullptr;         // null: not stored
  const cplx<T>* prev = nullptr;
  const cplx<T>* acc = nullptr;    // null: starts at zero
  cplx<T>* dst = nullptr;          // null: no sum in this step
  T scale = 1, e0 = 0, e2 = 0, o1 = 0;
  ExactProbe* probe = nullptr;     // first step: what phi is like; last step: phi not
  int first = 0, last = 0;         // finite leaves dst unwritten
};

// This wave's share of the probe (own[e] at x0 + stride e).
template <typename T>
__device__ __forceinline__ void probe_state(const ExactStep<T>& st, const cplx<T> (&own)[4], const bool (&live)[4],
                                            size_t x0, size_t stride) {
  ExactProbe* p = st.probe;
  bool fin = true;
#pragma unroll
  for (int e = 0; e < 4; ++e) fin = fin && isfinite(own[e].re) && isfinite(own[e].im);
  if (!fin) atomicOr(&p->bad, 1);
  if (__hip_atomic_load(&p->count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) <= EXACT_SUPPORT) {
    const int lane = threadIdx.x & 63;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const bool some = live[e] && (own[e].re != T(0) || own[e].im != T(0));
      const unsigned long long m = __ballot(some);
      if (!m) continue;
      int at = 0;
      if (lane == __ffsll(m) - 1) at = atomicAdd(&p->count, __popcll(m));
      at = __shfl(at, __ffsll(m) - 1, 64) + __popcll(m & ((1ull << lane) - 1));
      if (some && at < EXACT_SUPPORT)
        p->e[at] = ExactAmplitude{(unsigned long long)(x0 + stride * e), double(own[e].re), double(own[e].im)};
    }
  }
}

// The probe to the host: 1 + the nonzero amplitudes (more than EXACT_SUPPORT: just
// that), or EXACT_BAD; and the amplitudes where they are few, so that the host need not
// copy them, which drains the stream (a set that is not closed, 2^8: 135 -> 81 us).  A
// launch of its own: by the last workgroup of the first step, with the fence that takes
// in each of them, it cost 0.7 ms at 2^23.
constexpr int EXACT_BAD = 1 << 30;
__global__ __launch_bounds__(EXACT_SUPPORT) void tell_probe(const ExactProbe* p, ExactReport* report) {
  const int n = p->count, i = threadIdx.x;
  if (n <= EXACT_SUPPORT && i < n) {
    report->e[i] = p->e[i];
    __threadfence_system();
  }
  __syncthreads();
  if (i == 0)
    __hip_atomic_store(&report->word, p->bad ? EXACT_BAD : 1 + n, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// One workgroup owns a tile of 2^TB consecutive states (the whole vector when
// it is shorter), staged in LDS; partners across the low bits come from the
// tile.  Of the higher bits, those at least `distance` above the tile have the
// same activity for the whole tile: one scalar mask, and one contiguous tile
// read per active bit.  The sum runs from the highest bit down (the order of
// the cells).  What bounds it: memory and last-level cache, 167 us per step of
// 2^23 amplitudes against 109 us for reading phi, prev, half of acc and
// writing next and half of acc at the rate of a large copy; the rest is the
// tile reads (half of N - TB of them).  prev and acc are loaded with the tile,
// before the gathers (2^23: 7.9 -> 7.5 ms for 45 steps).  Giving each XCD a
// contiguous range of tiles cost 9%.
template <typename T, typename I, int D, int TB>
__global__ __launch_bounds__((1 << TB) / 4) void exact_kernel(const cplx<T>* __restrict__ phi, int ncells,
                                                              int distance, int lo, int hi, ExactStep<T> st) {
  constexpr int NT = (1 << TB) / 4;
  __shared__ cplx<T> tile[1 << TB];
  const int dist = D > 0 ? D : min(distance, ncells - 1);
  const I base = (I)blockIdx.x << TB;
  const unsigned tsize = ncells < TB ? 1u << ncells : 1u << TB;
  const unsigned t0 = threadIdx.x;
  cplx<T> own[4];
  bool live[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const unsigned t = t0 + NT * e;
    live[e] = t < tsize;
    own[e] = live[e] ? phi[(size_t)base + t] : cplx<T>{T(0), T(0)};
  }
  cplx<T> pv[4], av[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const size_t x = (size_t)base + t0 + NT * e;
    pv[e] = st.prev && live[e] ? st.prev[x] : cplx<T>{T(0), T(0)};
    av[e] = st.acc && live[e] ? st.acc[x] : cplx<T>{T(0), T(0)};
  }
  I act[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    tile[t0 + NT * e] = own[e];
    act[e] = active_cells<I, D>(base | (I)(t0 + NT * e), dist, lo, hi);
  }
  T ar[4] = {0, 0, 0, 0}, ai[4] = {0, 0, 0, 0};
  const int top = min(ncells, TB + dist);
  // bits top .. ncells-1: the same activity for every state of the tile
  I um = active_cells<I, D>(base, dist, lo, hi);
  um &= ncells >= (int)(8 * sizeof(I)) ? ~I(0) : (I(1) << ncells) - 1;
  um = top >= (int)(8 * sizeof(I)) ? I(0) : (um >> top) << top;
  while (um) {
    const int b = 8 * (int)sizeof(I) - 1 - (sizeof(I) == 4 ? __clz((int)(unsigned)um) : __clzll((long long)um));
    um ^= I(1) << b;
    const cplx<T>* src = phi + (size_t)(base ^ (I(1) << b)) + t0;
    cplx<T> v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = src[NT * e];   // a higher bit exists: the tile is full
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ar[e] += v[e].re;
      ai[e] += v[e].im;
    }
  }
  for (int b = top - 1; b >= TB; --b) {
    const cplx<T>* src = phi + (size_t)(base ^ (I(1) << b)) + t0;
    cplx<T> v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = cplx<T>{T(0), T(0)};
      if ((act[e] >> b) & 1) v[e] = src[NT * e];
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      ar[e] += v[e].re;
      ai[e] += v[e].im;
    }
  }
  __syncthreads();
#pragma unroll
  for (int b = TB - 1; b >= 0; --b) {
    if (b >= ncells) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const cplx<T> v = tile[(t0 + NT * e) ^ (1u << b)];
      const bool on = (act[e] >> b) & 1;
      ar[e] += on ? v.re : T(0);
      ai[e] += on ? v.im : T(0);
    }
  }
  bool off = false;
  if (st.probe) {
    if (st.first) probe_state(st, own, live, (size_t)base + t0, NT);
    if (st.last) off = st.probe->bad != 0;
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    if (!live[e]) continue;
    const size_t x = (size_t)base + t0 + NT * e;
    const cplx<T> nx{st.scale * ar[e] - pv[e].re, st.scale * ai[e] - pv[e].im};
    if (st.next) st.next[x] = nx;
    if (st.dst && !off) {
      cplx<T> a = av[e];
      a.re += st.e0 * own[e].re + (st.e2 * nx.re - st.o1 * nx.im);
      a.im += st.e0 * own[e].im + (st.e2 * nx.im + st.o1 * nx.re);
      st.dst[x] = a;
    }
  }
}

template <typename T, typename I, int D>
void launch_step_d(const cplx<T>* phi, int ncells, int distance, int lo, int hi, const ExactStep<T>& st,
                   hipStream_t s) {
  // Tiles of 1024 states from two workgroups per CU on, of 256 below, where
  // more and shorter workgroups count.  Tiles of 4096 read fewer partners from
  // memory and measured the same (2^23: 7.78 ms, 1024: 7.87, 256: 7.94 for 45
  // steps; 2^16: 0.253 against 0.197 and 0.200).
  auto tiles = [&](int tb) { return 1L << std::max(0, ncells - tb); };
#define QCA_EXACT_L(TB)                                                                          \
  hipLaunchKernelGGL((exact_kernel<T, I, D, TB>), dim3((unsigned)tiles(TB)), dim3((1 << TB) / 4), 0, s, phi, \
                     ncells, distance, lo, hi, st)
  if (tiles(10) >= 512) QCA_EXACT_L(10);
  else QCA_EXACT_L(8);
#undef QCA_EXACT_L
  QCA_HIP(hipGetLastError());
}

template <typename T>
void launch_step(const cplx<T>* phi, int ncells, int distance, int lo, int hi, const ExactStep<T>& st,
                 hipStream_t s) {
  QCA_CHECK(ncells >= 1 && ncells <= 34, "ncells out of range for the state vector");
  if (ncells > 32) launch_step_d<T, unsigned long long, 0>(phi, ncells, distance, lo, hi, st, s);
  else if (distance == 1) launch_step_d<T, unsigned, 1>(phi, ncells, distance, lo, hi, st, s);
  else if (distance == 2) launch_step_d<T, unsigned, 2>(phi, ncells, distance, lo, hi, st, s);
  else launch_step_d<T, unsigned, 0>(phi, ncells, distance, lo, hi, st, s);
}

// J_0(z) .. J_kmax(z), z >= 0, by Miller's downward recurrence normalised with
// J_0 + 2 (J_2 + J_4 + ...) = 1; for tiny z by the first two series terms.
std::vector<double> bessel_j(long double z, int kmax) {
  std::vector<double> f(kmax + 1, 0.0);
  if (z < 1e-3L) {
    double t = 1.0;   // (z/2)^k / k!
    for (int k = 0; k <= kmax; ++k) {
      const double q = (double)(z * z / 4);
      f[k] = t * (1.0 - q / (k + 1) * (1.0 - q / (2.0 * (k + 2))));
      t *= (double)z / 2 / (k + 1);
    }
    return f;
  }
  const int start = 2 * ((std::max(kmax, (int)z) + 40 + (int)(12 * std::cbrt((double)z))) / 2);
  long double up = 0, cur = 1e-300L, sum = 0;
  for (int k = start; k >= 0; --k) {
    // cur = J_k up to the common factor
    if (k <= kmax) f[k] = (double)cur;
    sum += k == 0 ? cur : ((k & 1) ? 0.0L : 2 * cur);
    const long double down = 2 * k / z * cur - up;
    up = cur;
    cur = down;
    if (std::fabs((double)cur) > 1e200) {
      up *= 1e-200L;
      cur *= 1e-200L;
      sum *= 1e-200L;
      for (int q = k; q <= kmax; ++q) f[q] *= 1e-200;
    }
  }
  for (double& v : f) v = (double)(v / sum);
  return f;
}

// Single-site reduced density matrices of a 2^N state, two-stage reduction.
// rho_i[p][q] = sum_{x: x_i = p} psi_x conj(psi_{x with x_i = q}); site i is bit N-1-i.
// Stage 1: block (bx, i) writes partial (rho00, rho11, Re rho01, Im rho01).
__global__ void exact_rho_partials(const c128* __restrict__ psi, int ncells, double* __restrict__ part) {
  __shared__ double sh[16];
  const int i = blockIdx.y;
  const long dim = 1L << ncells;
  const long bit = 1L << (ncells - 1 - i);
  double d0 = 0, d1 = 0, orr = 0, oi = 0;
  for (long x = blockIdx.x * (long)blockDim.x + threadIdx.x; x < dim; x += (long)gridDim.x * blockDim.x) {
    const c128 a = psi[x];
    const double n2 = a.re * a.re + a.im * a.im;
    if (x & bit) {
      d1 += n2;
    } else {
      d0 += n2;
      const c128 b = psi[x | bit];  // conj(b) * a summed into rho01 = sum a conj(b)
      orr += a.re * b.re + a.im * b.im;
      oi += a.im * b.re - a.re * b.im;
    }
  }
  d0 = rho_block_sum(d0, sh);
  d1 = rho_block_sum(d1, sh);
  orr = rho_block_sum(orr, sh);
  oi = rho_block_sum(oi, sh);
  if (threadIdx.x == 0) {
    double* p = part + ((long)i * gridDim.x + blockIdx.x) * 4;
    p[0] = d0; p[1] = d1; p[2] = orr; p[3] = oi;
  }
}

__global__ void exact_rho_finalize(const double* __restrict__ part, int nbx, int ncells, c128* __restrict__ rho) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= ncells) return;
  double d0 = 0, d1 = 0, orr = 0, oi = 0;
  for (int b = 0; b < nbx; ++b) {
    const double* p = part + ((long)i * nbx + b) * 4;
    d0 += p[0]; d1 += p[1]; orr += p[2]; oi += p[3];
  }
  rho[4L * i + 0] = c128{d0, 0.0};
  rho[4L * i + 1] = c128{orr, oi};
  rho[4L * i + 2] = c128{orr, -oi};
  rho[4L * i + 3] = c128{d1, 0.0};
}

}  // namespace

template <typename T>
void launch_exact_apply(const cplx<T>* psi, cplx<T>* out, int ncells, int distance, int lo, int hi,
                        hipStream_t s) {
  ExactStep<T> st;
  st.next = out;
  launch_step<T>(psi, ncells, distance, lo, hi, st, s);
}
template void launch_exact_apply<double>(const c128*, c128*, int, int, int, int, hipStream_t);
template void launch_exact_apply<float>(const c64*, c64*, int, int, int, int, hipStream_t);

std::vector<double> chebyshev_coefficients(long double z, double tol) {
  // the tail beyond k = z + 20 cbrt(z) + 40 is below 1e-40
  const int top = (int)z + (int)(20 * std::cbrt((double)z)) + 40;
  std::vector<double> j = bessel_j(z, top);
  // smallest K >= 2 with 2 sum_{k > K} |J_k| < tol
  int K = top;
  double tail = 0;
  while (K > 2 && tail + 2 * std::fabs(j[K]) < tol) tail += 2 * std::fabs(j[K--]);
  j.resize(K + 1);
  for (int k = 1; k <= K; ++k) j[k] *= 2;
  return j;
}

namespace {

// exp(-i tau H) psi as substeps of K terms each: their number, and the coefficient of
// T_k, c_k (-i sign(tau))^k, even k real, odd k imaginary.
struct ChebSeries {
  double scale;   // 2/R as the recurrence multiplies by it
  long substeps;
  std::vector<double> c;
  int K;          // >= 2
  // The series is that of the R that 2/R as rounded stands for (a relative error of
  // 1e-16 in R shifts every phase by z times as much).
  ChebSeries(double tau, int R, double tol) : scale(2.0 / R) {
    const long double total = 2.0L * std::fabs(tau) / scale;
    QCA_CHECK(total < 4e10, "time step too long for the state vector");
    substeps = std::max(1L, (long)std::ceil((double)total / CHEB_MAX_Z));
    c = chebyshev_coefficients(total / substeps, CHEB_TAIL * tol / substeps);
    K = (int)c.size() - 1;
    const double sg = tau < 0 ? -1.0 : 1.0;
    for (int k = 0; k <= K; ++k) c[k] *= (k & 3) == 0 ? 1.0 : (k & 3) == 1 ? -sg : (k & 3) == 2 ? -1.0 : sg;
  }
  double coef(int k) const { return k > K ? 0.0 : c[k]; }
  int applications() const { return (int)std::min<long>(substeps * K, 0x7fffffffL); }
};

// Basis states that H maps among themselves, from those of psi's support, and the
// amplitudes on them.
struct ClosedSet {
  int n = 0;
  unsigned long long x[EXACT_SUPPORT];
  double re[EXACT_SUPPORT], im[EXACT_SUPPORT];
};

__global__ void scatter_closed_set(ClosedSet c, c128* __restrict__ psi) {
  const int i = threadIdx.x;
  if (i < c.n) psi[c.x[i]] = c128{c.re[i], c.im[i]};
}

// Evolves psi on the smallest set of basis states with its support that H maps to
// itself, if that has at most EXACT_SUPPORT states; returns the H applications, or 0.
// (Still lifes, blinkers and the like: the Chebyshev series in the whole space takes
// as many terms for them as for any state, where H acts on a handful of numbers.)
int evolve_closed_set(c128* psi, const ExactAmplitude* support, int nsupport, int ncells, int distance, int lo,
                      int hi, double tau, double tol, hipStream_t s) {
  ClosedSet cs;
  unsigned char to[EXACT_SUPPORT][EXACT_SUPPORT];   // neighbours: at most one for each cell
  int nto[EXACT_SUPPORT];
  int slot[256];                       // open addressing over the states
  std::fill(slot, slot + 256, -1);
  auto find = [&](unsigned long long x) {
    unsigned h = (unsigned)((x * 0x9E3779B97F4A7C15ull) >> 56);
    while (slot[h] >= 0 && cs.x[slot[h]] != x) h = (h + 1) & 255;
    if (slot[h] < 0) {
      if (cs.n == EXACT_SUPPORT) return -1;
      cs.x[cs.n] = x;
      cs.re[cs.n] = cs.im[cs.n] = 0;
      nto[cs.n] = 0;
      slot[h] = cs.n++;
    }
    return slot[h];
  };
  for (int a = 0; a < nsupport; ++a) {
    const int i = find(support[a].x);
    cs.re[i] = support[a].re;
    cs.im[i] = support[a].im;
  }
  std::vector<unsigned long long> near(ncells);
  for (int b = 0; b < ncells; ++b)
    for (int o = std::max(0, b - distance); o <= std::min(ncells - 1, b + distance); ++o)
      if (o != b) near[b] |= 1ull << o;
  int R = 0;
  for (int i = 0; i < cs.n; ++i) {
    for (int b = 0; b < ncells; ++b) {
      const int alive = __builtin_popcountll(cs.x[i] & near[b]);
      if (alive < lo || alive >= hi) continue;
      const int j = find(cs.x[i] ^ (1ull << b));
      if (j < 0) return 0;
      to[i][nto[i]++] = (unsigned char)j;
    }
    R = std::max(R, nto[i]);
  }
  if (R == 0) return 1;   // H psi = 0
  const ChebSeries f(tau, R, tol);
  typedef std::vector<c128> Vec;
  Vec v(cs.n);
  for (int i = 0; i < cs.n; ++i) v[i] = c128{cs.re[i], cs.im[i]};
  Vec prev(cs.n), cur(cs.n), next(cs.n);
  auto step = [&](const Vec& p, double scale, const Vec* minus, Vec& out) {
    for (int i = 0; i < cs.n; ++i) {
      c128 h{0, 0};
      for (int t = 0; t < nto[i]; ++t) {
        h.re += p[to[i][t]].re;
        h.im += p[to[i][t]].im;
      }
      out[i] = minus ? c128{scale * h.re - (*minus)[i].re, scale * h.im - (*minus)[i].im}
                     : c128{scale * h.re, scale * h.im};
    }
  };
  for (long sub = 0; sub < f.substeps; ++sub) {
    prev = v;
    step(prev, 0.5 * f.scale, nullptr, cur);
    for (int i = 0; i < cs.n; ++i)
      v[i] = c128{f.coef(0) * prev[i].re - f.coef(1) * cur[i].im, f.coef(0) * prev[i].im + f.coef(1) * cur[i].re};
    for (int k = 2; k <= f.K; ++k) {
      step(cur, f.scale, &prev, next);
      const double ck = f.coef(k);
      for (int i = 0; i < cs.n; ++i) {
        v[i].re += k & 1 ? -ck * next[i].im : ck * next[i].re;
        v[i].im += k & 1 ? ck * next[i].re : ck * next[i].im;
      }
      prev.swap(cur);
      cur.swap(next);
    }
  }
  for (int i = 0; i < cs.n; ++i) {
    cs.re[i] = v[i].re;
    cs.im[i] = v[i].im;
  }
  hipLaunchKernelGGL(scatter_closed_set, dim3(1), dim3(EXACT_SUPPORT), 0, s, cs, psi);
  QCA_HIP(hipGetLastError());
  return f.applications();
}

}  // namespace

// The first step looks psi over (finite, and how many amplitudes are not zero) and
// tells the host through memory of its own while the next steps are on their
// way, so a general state pays no wait for it.  What it learns by the eighth step: a
// closed set of few states is evolved on the host (dead or blinking cells, dt 5, 12
// cells: 640 -> 46 us, 23 cells 28 -> 1.0 ms; with the Krylov evolution before the
// series 0.2 and 3.9 ms).
int launch_exact_expm(c128* psi, int ncells, int distance, int lo, int hi, double tau, double tol, c128* bufa,
                      c128* bufb, c128* acc, ExactProbe* probe, ExactReport* report, hipStream_t s) {
  const ChebSeries f(tau, ncells, tol);
  const int K = f.K;
  __atomic_store_n(&report->word, 0, __ATOMIC_RELAXED);
  QCA_HIP(hipMemsetAsync(probe, 0, offsetof(ExactProbe, e), s));
  auto look = [&](bool wait) {
    for (;;) {
      const int v = __atomic_load_n(&report->word, __ATOMIC_ACQUIRE);
      if (v != 0 || !wait) return v;
      const hipError_t e = hipStreamQuery(s);   // ends with the stream's work, if not before
      if (e == hipSuccess) return __atomic_load_n(&report->word, __ATOMIC_ACQUIRE);
      if (e != hipErrorNotReady) QCA_HIP(e);
      (void)hipGetLastError();   // "not ready" is no error of the launches below
    }
  };
  int seen = 0, launched = 0;
  for (long sub = 0; sub < f.substeps; ++sub) {
    // step k forms phi_{k+1}; odd phi join the sum together with the even one before
    for (int k = 0; k < K; ++k, ++launched) {
      if (seen == 0 && launched > 0 && launched <= 8) {
        seen = look(launched == 8);
        if (seen == EXACT_BAD) break;
        if (seen > 0 && seen - 1 <= EXACT_SUPPORT)   // psi is written by a substep's last step at the earliest
          if (const int m = evolve_closed_set(psi, report->e, seen - 1, ncells, distance, lo, hi, tau, tol, s)) {
            QCA_HIP(hipStreamSynchronize(s));
            return m;
          }
      }
      ExactStep<double> st;
      const c128* phi = k == 0 ? psi : (k & 1 ? bufb : bufa);
      c128* next = k & 1 ? bufa : bufb;
      st.prev = k == 0 ? nullptr : (k == 1 ? psi : next);
      st.scale = k == 0 ? 0.5 * f.scale : f.scale;
      st.last = k == K - 1;
      st.first = k == 0 && sub == 0;
      if (st.first || st.last) st.probe = probe;
      st.next = st.last ? nullptr : next;
      if (!(k & 1)) {               // phi_k even, phi_{k+1} odd
        st.acc = k == 0 ? nullptr : acc;
        st.dst = st.last ? psi : acc;
        st.e0 = f.coef(k);
        st.o1 = f.coef(k + 1);
      } else if (st.last) {         // K even: phi_K alone
        st.acc = acc;
        st.dst = psi;
        st.e2 = f.coef(k + 1);
      }
      launch_step<double>(phi, ncells, distance, lo, hi, st, s);
      if (st.first) 
        hipLaunchKernelGGL(tell_probe, dim3(1), dim3(EXACT_SUPPORT), 0, s, (const ExactProbe*)probe, report);
    }
    if (seen == EXACT_BAD) break;
  }
  QCA_HIP(hipStreamSynchronize(s));
  if (__atomic_load_n(&report->word, __ATOMIC_ACQUIRE) == EXACT_BAD)
    throw Error(QCA_ERR_NOT_CONVERGED_CODE, "exponential of a state vector with non-finite amplitudes");
  return f.applications();
}

int exact_rho_blocks(int ncells) {
  const long dim = 1L << ncells;
  return (int)std::max<long>(1, std::min<long>((dim + 255) / 256, 512));
}

void launch_exact_rho(const c128* psi, int ncells, double* part, c128* rho, hipStream_t s) {
  const int nbx = exact_rho_blocks(ncells);
  hipLaunchKernelGGL(exact_rho_partials, dim3(nbx, ncells), dim3(256), 0, s, psi, ncells, part);
  hipLaunchKernelGGL(exact_rho_finalize, dim3((ncells + 63) / 64), dim3(64), 0, s, part, nbx, ncells, rho);
  QCA_HIP(hipGetLastError());
}

}  // namespace qca
