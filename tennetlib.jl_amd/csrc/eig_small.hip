// Eigen-decomposition of symmetric / Hermitian blocks that one workgroup can
// hold, in FP64: Householder tridiagonalisation with the block in registers,
// divide and conquer on the tridiagonal with its eigenvectors in LDS, and the
// back-transformation one wavefront per one or two eigenvectors.  A launch takes
// one block (described by a kernel argument) or a list of blocks of one size
// class.  eig_dc.hip uses the same kernels for the last columns, the leaves
// and the back-transformation of larger matrices.
#include "tn_internal.h"

#include <algorithm>
#include <type_traits>

namespace tn {
namespace {

constexpr double EPS = 2.220446049250313e-16;
// A column whose entries below the subdiagonal are under 2^-450 of the block's
// largest entry (one, after scaling) is left as it is: dropping them is far
// below its rounding, and a reflector from squares that lost bits would not be
// orthogonal.
constexpr double TINY_SS = 0x1p-900;

__device__ __forceinline__ const SmallEig& pick(const SmallEig& one, const SmallEig* list, unsigned b) {
  return list ? list[b] : one;
}

// element arithmetic of real and complex matrices
template <bool CX> struct El;
template <> struct El<false> {
  typedef double T;
  static __device__ __forceinline__ T zero() { return 0.0; }
  static __device__ __forceinline__ T one() { return 1.0; }
  static __device__ __forceinline__ T mul(T a, T b) { return a * b; }
  static __device__ __forceinline__ T cmul(T a, T b) { return a * b; }  // conj(a) b
  static __device__ __forceinline__ T add(T a, T b) { return a + b; }
  static __device__ __forceinline__ T sub(T a, T b) { return a - b; }
  // a - x conj(y) - w conj(z)
  static __device__ __forceinline__ T sub2(T a, T x, T y, T w, T z) { return fma(-w, z, fma(-x, y, a)); }
  static __device__ __forceinline__ T scale(T a, double s) { return a * s; }
  static __device__ __forceinline__ double norm2(T a) { return a * a; }
  static __device__ __forceinline__ double re(T a) { return a; }
  static __device__ __forceinline__ int high_word(T a) { return __double2hiint(a) & 0x7fffffff; }
  static __device__ __forceinline__ bool is_zero(T a) { return a == 0.0; }
  static __device__ __forceinline__ T sel(bool f, T a, T b) { return f ? a : b; }
  template <class F> static __device__ __forceinline__ T each(T a, F f) { return f(a); }
  // reflector H = I - tau v v^T of x (x_0, sum of squares ss of the rest): H x = beta e_1
  static __device__ __forceinline__ void reflector(T x0, double ss, T& tau, double& beta, T& sc) {
    trd_reflector(x0, ss < TINY_SS ? 0.0 : ss, tau, beta, sc);
  }
};
template <> struct El<true> {
  typedef double2 T;
  static __device__ __forceinline__ T zero() { return make_double2(0.0, 0.0); }
  static __device__ __forceinline__ T one() { return make_double2(1.0, 0.0); }
  static __device__ __forceinline__ T mul(T a, T b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
  }
  static __device__ __forceinline__ T cmul(T a, T b) {
    return make_double2(a.x * b.x + a.y * b.y, a.x * b.y - a.y * b.x);
  }
  static __device__ __forceinline__ T add(T a, T b) { return make_double2(a.x + b.x, a.y + b.y); }
  static __device__ __forceinline__ T sub(T a, T b) { return make_double2(a.x - b.x, a.y - b.y); }
  static __device__ __forceinline__ T sub2(T a, T x, T y, T w, T z) {
    return make_double2(fma(-w.y, z.y, fma(-w.x, z.x, fma(-x.y, y.y, fma(-x.x, y.x, a.x)))),
                        fma(w.x, z.y, fma(-w.y, z.x, fma(x.x, y.y, fma(-x.y, y.x, a.y)))));
  }
  static __device__ __forceinline__ T scale(T a, double s) { return make_double2(a.x * s, a.y * s); }
  static __device__ __forceinline__ double norm2(T a) { return a.x * a.x + a.y * a.y; }
  static __device__ __forceinline__ double re(T a) { return a.x; }
  static __device__ __forceinline__ int high_word(T a) {
    return max(__double2hiint(a.x) & 0x7fffffff, __double2hiint(a.y) & 0x7fffffff);
  }
  static __device__ __forceinline__ bool is_zero(T a) { return a.x == 0.0 && a.y == 0.0; }
  static __device__ __forceinline__ T sel(bool f, T a, T b) { return make_double2(f ? a.x : b.x, f ? a.y : b.y); }
  template <class F> static __device__ __forceinline__ T each(T a, F f) { return make_double2(f(a.x), f(a.y)); }
  // the zlarfg convention: beta real
  static __device__ __forceinline__ void reflector(T x0, double ss, T& tau, double& beta, T& sc) {
    if (ss + x0.y * x0.y < TINY_SS) {
      tau = sc = zero();
      beta = x0.x;
      return;
    }
    const double nrm = sqrt(x0.x * x0.x + x0.y * x0.y + ss);
    beta = (x0.x >= 0.0) ? -nrm : nrm;
    tau = make_double2((beta - x0.x) / beta, -x0.y / beta);
    const double ar = x0.x - beta, ai = x0.y, d = ar * ar + ai * ai;
    sc = make_double2(ar / d, -ai / d);
  }
};

// sum over a quad of lanes (every lane gets the same bits; the quad's lanes
// must be active together)
__device__ __forceinline__ double sum4(double x) {
  x = dpp_add<0xB1>(x);
  return dpp_add<0x4E>(x);
}

// ---------------------------------------------------------------------------
// Householder tridiagonalisation, one workgroup per block, n <= GR * NR rows.
// Bound by the chain of one column: three barriers, two wavefront sums, a
// square root and a division, and by the instructions every wavefront spends
// on them.  The block therefore never leaves the registers, spread over as
// few wavefronts as hold it: thread (tr, tc) of a GR x GC grid has the
// elements (tr + GR i, tc + GC j), the rank-2 update needs no exchange, the
// product with the reflector one LDS reduction over the GR partial sums of a
// column (the block is Hermitian), and every wavefront forms the reflector
// and the dot product for itself.  Nothing is stored to global memory inside
// the loop (a barrier would wait for the stores): column j of the block is
// dead after step j and keeps the reflector, as does row j.
// SE_ROWS: row j of A receives the reflector right of the diagonal and
// zeros elsewhere.
// Measured: 32 rows 13 us, 64 rows 63 us, 192 rows 420 us (136 rows in LDS
// with 256 threads: 504 us; the same registers over 1024 threads: 910 us, the
// sums and divisions repeated by every wavefront then bound it).
// ---------------------------------------------------------------------------
template <bool CX, int GR, int GC, int NR, int NC>
__global__ __launch_bounds__(GR* GC) void trd_reg_kernel(SmallEig one, const SmallEig* __restrict__ list,
                                                         void* __restrict__ Abase, double* __restrict__ dbase,
                                                         double* __restrict__ ebase, void* __restrict__ taubase) {
  typedef El<CX> E;
  typedef typename E::T T;
  constexpr int NT = GR * GC, NM = GR * NR, NP = NM + 2, NW = (NM + 63) / 64, SEG = GC;
  static_assert(NM == GC * NC && GR % 4 == 0 && GC % GR == 0 && NC <= 8, "square block");
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  T* part = reinterpret_cast<T*>(smem);  // GR x NP
  T* xs = part + GR * NP;                // 2 x NM: the current column below the diagonal, zeros above
  T* ys = xs + 2 * NM;                   // NM
  T* ts = ys + NM;                       // NM
  double* ds = reinterpret_cast<double*>(ts + NM);
  double* es = ds + NM;
  const SmallEig S = pick(one, list, blockIdx.x);
  const int n = S.n;
  const int tid = threadIdx.x, lane = tid & 63, tr = tid / GC, tc = tid % GC;
  T* A = reinterpret_cast<T*>(Abase) + S.a;
  T a[NR][NC];
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int r = tr + GR * i, c = tc + GC * j;
      a[i][j] = (r < n && c < n) ? A[(long)r * S.lda + c] : E::zero();
    }
  // scaled by a power of two to a largest entry in [1/2, 1), so that no sum of
  // squares leaves the range (exponents: the high words of the absolute values)
  int hw = 0;
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) hw = max(hw, E::high_word(a[i][j]));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) hw = max(hw, __shfl_xor(hw, o, 64));
  int* hws = reinterpret_cast<int*>(part);
  if (lane == 0) hws[tid >> 6] = hw;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < NT / 64; ++k) hw = max(hw, hws[k]);
  const int ex = __builtin_amdgcn_readfirstlane((hw >> 20) < 2047 ? (hw >> 20) - 1022 : 0);
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) a[i][j] = E::each(a[i][j], [ex](double x) { return ldexp(x, -ex); });
  // column j, held in column chunk J0 or (J2 > J0 + 1) J0 + 1, to LDS; its diagonal element to ds
  auto publish = [&](int j, auto J0, auto J2) {
    constexpr int C0 = decltype(J0)::value, C1 = decltype(J2)::value - 1;
    if (tc != j % GC) return;
    T* x = xs + (j & 1) * NM;
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int r = tr + GR * i;
      const T v = E::sel(j / GC == C0, a[i][C0], a[i][C1]);
      x[r] = E::sel(r > j, v, E::zero());
      if (r == j) ds[j] = E::re(v);
    }
  };
  publish(0, std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{});
  __syncthreads();
  // columns [SEG s, SEG (s + 1)): rows and columns of earlier segments are done
  auto segment = [&](auto sg) {
    constexpr int SI = decltype(sg)::value * SEG, I0 = SI / GR, J0 = SI / GC;
    constexpr int I1 = I0 + SEG / GR, J1 = J0 + SEG / GC, J2 = J1 < NC ? J1 + 1 : NC;
    const int jend = min(SI + SEG, n - 1);
    for (int j = SI; j < jend; ++j) {
      const T* x = xs + (j & 1) * NM;
      // the reflector of column j, by every wavefront
      T xv[NW];
      double ss = 0.0;
#pragma unroll
      for (int q = 0; q < NW; ++q) {
        const int c = lane + 64 * q;
        xv[q] = x[NM % 64 == 0 ? c : min(c, NM - 1)];
        const double x2 = E::norm2(xv[q]);
        ss += (c < NM && c != j + 1) ? x2 : 0.0;
      }
      // this thread's entries of x: reads without branches, on their way during the sums
      T xr[NR], xc[NC];
#pragma unroll
      for (int i = I0; i < NR; ++i) xr[i] = x[tr + GR * i];
#pragma unroll
      for (int jj = J0; jj < NC; ++jj) xc[jj] = x[tc + GC * jj];
      const T x0 = x[j + 1];
      ss = wave_sum64(ss);
      T tau, sc;
      double beta;
      E::reflector(x0, ss, tau, beta, sc);
      if (tid == 0) {
        es[j] = beta;
        ts[j] = tau;
      }
#pragma unroll
      for (int i = I0; i < NR; ++i) xr[i] = E::sel(tr + GR * i == j + 1, E::one(), E::mul(xr[i], sc));  // v
#pragma unroll
      for (int jj = J0; jj < NC; ++jj) xc[jj] = E::sel(tc + GC * jj == j + 1, E::one(), E::mul(xc[jj], sc));
      if (!E::is_zero(tau)) {
        // A^H v through the columns this thread holds (A is Hermitian)
        T acc[NC];
#pragma unroll
        for (int jj = J0; jj < NC; ++jj) acc[jj] = E::zero();
#pragma unroll
        for (int i = I0; i < NR; ++i)
#pragma unroll
          for (int jj = J0; jj < NC; ++jj) acc[jj] = E::add(acc[jj], E::cmul(a[i][jj], xr[i]));
#pragma unroll
        for (int jj = J0; jj < NC; ++jj) part[tr * NP + tc + GC * jj] = acc[jj];
        __syncthreads();
        for (int c4 = tid + 4 * GC * J0; c4 < 4 * NM; c4 += NT) {  // four threads per column (whole wavefronts)
          const int c = c4 >> 2, s = c4 & 3;
          T sum = E::zero();
#pragma unroll
          for (int k = 0; k < GR / 4; ++k) sum = E::add(sum, part[(s * (GR / 4) + k) * NP + c]);
          sum = E::each(sum, [](double u) { return sum4(u); });
          const T yv = E::mul(tau, sum);
          if (s == 0) ys[c] = E::sel(c > j, yv, E::zero());
        }
        __syncthreads();
        T dt = E::zero();  // y^H v
        T yc[NC];
#pragma unroll
        for (int q = 0; q < NW; ++q) {
          const int c = lane + 64 * q;
          const T yq = ys[NM % 64 == 0 ? c : min(c, NM - 1)];
          const T t = E::cmul(yq, E::sel(c == j + 1, E::one(), E::mul(xv[q], sc)));
          if (64 * (q + 1) > GC * J0) dt = E::add(dt, E::sel(c < NM && c > j, t, E::zero()));
        }
#pragma unroll
        for (int jj = J0; jj < NC; ++jj) yc[jj] = ys[tc + GC * jj];
        dt = E::each(dt, [](double u) { return wave_sum64(u); });
        const T hs = E::scale(E::mul(tau, dt), 0.5);
        // w = y - (tau / 2) (y^H v) v; rows and columns up to j have v = 0 and y = 0
#pragma unroll
        for (int jj = J0; jj < NC; ++jj) yc[jj] = E::sub(yc[jj], E::mul(hs, xc[jj]));
#pragma unroll
        for (int i = I0; i < NR; ++i) {
          const T w = E::sub(ys[tr + GR * i], E::mul(hs, xr[i]));
#pragma unroll
          for (int jj = J0; jj < NC; ++jj) a[i][jj] = E::sub2(a[i][jj], xr[i], yc[jj], w, xc[jj]);
        }
      }
      // the reflector into column j (below the diagonal) and row j (right of it)
      static_assert(J1 == J0 + 1 && I1 <= I0 + 2, "a segment is one chunk of columns");
#pragma unroll
      for (int i = I0; i < NR; ++i) {
        const int r = tr + GR * i;
        a[i][J0] = E::sel(tc + GC * J0 == j && r > j, xr[i], a[i][J0]);
      }
#pragma unroll
      for (int i = I0; i < I1; ++i)
#pragma unroll
        for (int jj = J0; jj < NC; ++jj) a[i][jj] = E::sel(tr + GR * i == j && tc + GC * jj > j, xc[jj], a[i][jj]);
      publish(j + 1, std::integral_constant<int, J0>{}, std::integral_constant<int, J2>{});
      __syncthreads();
    }
  };
  segment(std::integral_constant<int, 0>{});
  if constexpr (NM > SEG) segment(std::integral_constant<int, 1>{});
  if constexpr (NM > 2 * SEG) segment(std::integral_constant<int, 2>{});
  if constexpr (NM > 3 * SEG) segment(std::integral_constant<int, 3>{});
  if constexpr (NM > 4 * SEG) segment(std::integral_constant<int, 4>{});
  if constexpr (NM > 5 * SEG) segment(std::integral_constant<int, 5>{});
  if constexpr (NM > 6 * SEG) segment(std::integral_constant<int, 6>{});
  if constexpr (NM > 7 * SEG) segment(std::integral_constant<int, 7>{});
#pragma unroll
  for (int i = 0; i < NR; ++i)
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      const int r = tr + GR * i, c = tc + GC * j;
      if (r < n && c < n) A[(long)r * S.lda + c] = ((S.flags & SE_ROWS) && c <= r) ? E::zero() : a[i][j];
    }
  T* tauv = reinterpret_cast<T*>(taubase) + S.de;
  for (int t = tid; t < n; t += NT) {
    dbase[S.de + t] = ldexp(ds[t], ex);
    tauv[t] = t < n - 1 ? ts[t] : E::zero();
    if (t < n - 1) ebase[S.de + t] = ldexp(es[t], ex);
  }
}

// ---------------------------------------------------------------------------
// Divide and conquer on a symmetric tridiagonal (d, e) of n <= NM rows, one
// workgroup of 4 NM threads per block.  Cuppen's tearing from leaves of one
// or two rows up; all merges of a level run together.  Per merge: deflation
// in ascending order of the poles (negligible z, Givens rotation for nearly
// equal poles, the LAPACK dlaed2 rule), four lanes per secular root (Li's
// middle-way iteration in tau = lambda - pole), the Gu-Eisenstat z, and
// Q <- Q U as FP64 MFMA tiles whose U entries are formed in registers from
// (z, pole, root): U is never stored, so Q alone fills the LDS.  Deflated
// columns are unit columns of U.  The last level writes Q to global memory.
// Eigenvalues come unsorted, in the order of Q's columns.
// Bound by serial chains, not by arithmetic: of 220 us at 124 rows (graded
// spectrum) 83 are the secular iterations, 54 the tiles, 46 the deflation;
// 20 rows take 24 us.  Parallel Jacobi on 32-row leaves took 323 us and left
// two more merge levels to the host.
// ---------------------------------------------------------------------------
typedef double d4 __attribute__((ext_vector_type(4)));

// Least deflation tolerance of a matrix scaled to entries of one: far below its
// rounding.  Kept columns then have rho |z| and pole distances above 2^-400 and
// (|z| being above rounding) rho z^2 above 2^-510, all with a normal square.
// Without it a block of entries near 2^-1030 has the tolerance zero and rcp2
// gets a denormal: NaN.
constexpr double TINY = 0x1p-400;

template <int NM>
constexpr size_t dc_small_lds() {
  return ((size_t)NM * (NM + 1) + 12 * NM) * sizeof(double) + (size_t)9 * NM * sizeof(int);
}

// 1 / x for normal x: hardware estimate and two Newton steps (within about
// one unit in the last place; a third of the instructions of a division)
__device__ __forceinline__ double rcp2(double x) {
  double y = __builtin_amdgcn_rcp(x);
  y = fma(fma(-x, y, 1.0), y, y);
  return fma(fma(-x, y, 1.0), y, y);
}

__device__ __forceinline__ double prod4(double x) {
  auto mul = [](double v, auto ctrl) {
    constexpr int C = decltype(ctrl)::value;
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(b & 0xffffffffLL), C, 0xF, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), C, 0xF, 0xF, false);
    return v * __longlong_as_double(((long long)hi << 32) | (long long)(unsigned int)lo);
  };
  x = mul(x, std::integral_constant<int, 0xB1>{});
  return mul(x, std::integral_constant<int, 0x4E>{});
}

// root i of 1 + sum_q rz_q / (dd_q - lambda) (k poles, increasing, rz > 0) by
// four lanes: the origin pole and tau = lambda - dd_origin
__device__ void secular_root4(const double* dd, const double* rz, int k, int i, int sub, int& org, double& tau) {
  int o;
  double lo, hi, df;  // bracket of tau, far pole relative to the origin (0: none)
  if (i < k - 1) {
    const double mid = 0.5 * (dd[i] + dd[i + 1]);
    double f = 0.0;
    for (int q = sub; q < k; q += 4) f += rz[q] * rcp2(dd[q] - mid);
    f = 1.0 + sum4(f);
    if (f >= 0.0) {
      o = i; lo = 0.0; hi = mid - dd[i]; df = dd[i + 1] - dd[i];
    } else {
      o = i + 1; lo = mid - dd[i + 1]; hi = 0.0; df = dd[i] - dd[i + 1];
    }
  } else {
    o = i;
    lo = 0.0;
    df = 0.0;
    double z2 = 0.0;
    for (int q = sub; q < k; q += 4) z2 += rz[q];
    hi = sum4(z2);
    for (int it = 0; it < 64; ++it) {  // make sure the bracket holds the root
      double gh = 0.0;
      for (int q = sub; q < k; q += 4) gh += rz[q] / ((dd[q] - dd[o]) - hi);
      if (1.0 + sum4(gh) >= 0.0) break;
      hi *= 2.0;
    }
  }
  const double dO = dd[o];
  double t = 0.5 * (lo + hi);
  for (int it = 0; it < 100; ++it) {
    // the poles up to i and those above: each sum has terms of one sign, so
    // their sizes also bound the rounding error of the whole
    double sl = 0.0, dl = 0.0, sr = 0.0, dr = 0.0;
    int q = sub;
#pragma unroll 4
    for (; q <= i; q += 4) {
      const double v = rcp2((dd[q] - dO) - t), r = rz[q] * v;
      sl += r;
      dl += r * v;
    }
#pragma unroll 4
    for (; q < k; q += 4) {
      const double v = rcp2((dd[q] - dO) - t), r = rz[q] * v;
      sr += r;
      dr += r * v;
    }
    sl = sum4(sl);
    dl = sum4(dl);
    sr = sum4(sr);
    dr = sum4(dr);
    const double gv = 1.0 + sl + sr;
    if (fabs(gv) <= 8.0 * EPS * (1.0 + fabs(sl) + fabs(sr))) break;  // within its own rounding error
    if (gv < 0.0) lo = t;
    else hi = t;
    const double so = (o == i) ? sl : sr, dso = (o == i) ? dl : dr;  // origin side
    const double sf = (o == i) ? sr : sl, dsf = (o == i) ? dr : dl;  // far side
    // model c + bo / (0 - x) + bf / (df - x), matching value and slope at t:
    // c x^2 - b x + bo df = 0, b = c df + bo + bf (df = 0, the last root: no
    // far side, and the roots are 0 and bo / c)
    const double g = df - t, bo = dso * t * t;
    const double bf = df != 0.0 ? dsf * g * g : 0.0;
    const double cc = 1.0 + (so + dso * t) + (df != 0.0 ? sf - dsf * g : sf);
    const double bq = cc * df + bo + bf, cq = bo * df;
    const double disc = fmax(bq * bq - 4.0 * cc * cq, 0.0);
    const double h = bq + copysign(sqrt(disc), bq);
    const double t1 = 0.5 * h * rcp2(cc), t2 = 2.0 * cq * rcp2(h);
    double tn = (t2 > lo && t2 < hi) ? t2 : t1;  // NaN from a zero divisor: bisected below
    if (!(tn > lo && tn < hi)) tn = 0.5 * (lo + hi);
    const bool done = fabs(tn - t) <= 4.0 * EPS * fabs(tn) || (hi - lo) <= 4.0 * EPS * fmax(fabs(lo), fabs(hi));
    t = tn;
    if (done) break;
  }
  org = o;
  tau = t;
}

// Deflation state of one merge: columns [a, en) come in ascending order of
// their poles; kept ones go to the front of the packed arrays, deflated ones
// (their eigenvalue is known) to the back.
struct Deflate {
  double* D;
  int* src;
  double *nD, *dK, *zK;
  int *ra, *rb;
  double *rc, *rs;
  int a, en;
  double rho, tol;
  int k = 0, nd = 0, nr = 0, pj = -1;
  double dp = 0.0, zp = 0.0;
  __device__ void drop(int c, double v) {
    ++nd;
    src[en - nd] = c;
    nD[en - nd] = v;
  }
  __device__ void keep() {
    src[a + k] = pj;
    dK[a + k] = dp;
    zK[a + k] = zp;
    ++k;
  }
  __device__ bool negligible(double zc) const { return rho * fabs(zc) <= tol; }
  __device__ bool close(double dc, double zc) const {
    return pj >= 0 && fabs((dc - dp) * zc * zp) <= tol * (zc * zc + zp * zp);
  }
  __device__ void rotate(int c, double& dc, double& zc) {  // the previous kept column deflates into this one
    const double h = sqrt(zc * zc + zp * zp);
    const double ct = zc / h, st = -zp / h;
    ra[a + nr] = pj;
    rb[a + nr] = c;
    rc[a + nr] = ct;
    rs[a + nr] = st;
    ++nr;
    drop(pj, dp * ct * ct + dc * st * st);
    dc = dp * st * st + dc * ct * ct;
    zc = h;
  }
  __device__ void advance(int c, double dc, double zc) {
    pj = c;
    dp = dc;
    zp = zc;
  }
  __device__ void column(int c, double dc, double zc) {
    if (negligible(zc)) {
      drop(c, dc);
      return;
    }
    if (close(dc, zc)) rotate(c, dc, zc);
    else if (pj >= 0) keep();
    advance(c, dc, zc);
  }
  // the same with every lane of a wavefront holding the same values: scalar branches
  __device__ __forceinline__ void column_wave(int c, double dc, double zc) {
    if (__ballot(negligible(zc))) {
      drop(c, dc);
      return;
    }
    if (__ballot(close(dc, zc))) rotate(c, dc, zc);
    else if (__builtin_amdgcn_readfirstlane(pj) >= 0) keep();
    advance(c, dc, zc);
  }
  __device__ void finish(int* kc, int* nrot) {
    if (pj >= 0) keep();
    kc[a] = k;
    nrot[a] = nr;
  }
};

template <int NM>
__global__ __launch_bounds__(4 * NM) void dc_small_kernel(SmallEig one, const SmallEig* __restrict__ list,
                                                          const double* __restrict__ dbase,
                                                          const double* __restrict__ ebase, double* __restrict__ Qbase,
                                                          double* __restrict__ lbase) {
  constexpr int LD = NM + 1, NT = 4 * NM, NRT = NM / 16;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  double* Q = reinterpret_cast<double*>(smem);  // NM x LD
  double* D = Q + NM * LD;                      // eigenvalues of the blocks, by column
  double* z = D + NM;
  double* dK = z + NM;   // poles, z and rho z^2 of the kept columns, packed per merge
  double* zK = dK + NM;
  double* rz = zK + NM;
  double* zh = rz + NM;    // also: z in pole order, before the deflation
  double* tau = zh + NM;   // also: D in pole order
  double* inv = tau + NM;  // 1 / |u| of a root's column; the merge's deflation tolerance before that
  double* nD = inv + NM;
  double* ee = nD + NM;
  double* rc = ee + NM;    // rotations, packed per merge
  double* rs = rc + NM;
  int* src = reinterpret_cast<int*>(rs + NM);  // new column -> old column (kept ones first)
  int* org = src + NM;
  int* perm = org + NM;
  int* kc = perm + NM;   // kept columns and rotations of the merge, at its first column
  int* nrot = kc + NM;
  int* ba = nrot + NM;   // first column of the merge, at every column
  int* be = ba + NM;     // its end
  int* ra = be + NM;
  int* rb = ra + NM;
  const SmallEig S = pick(one, list, blockIdx.x);
  const int n = S.n;
  const double* d = dbase + S.de;
  const double* e = ebase + S.de;
  double* Qg = Qbase + S.q;
  double* lam = lbase + S.de;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int L = 31 - __clz(n);  // leaves: 2^L of one or two rows
  auto bnd = [&](int i) { return (i * n) >> L; };
  auto leaf_of = [&](int t) { return (((t + 1) << L) - 1) / n; };
  for (int i = tid; i < n * LD; i += NT) Q[i] = 0.0;
  // scaled by a power of two to entries of at most one; couplings below TINY
  // are deflated, so the products and reciprocals of what is left stay normal
  double big = 0.0;
  const double tl = (S.flags & SE_TEAR_L) ? e[-1] : 0.0, tr = (S.flags & SE_TEAR_R) ? e[n - 1] : 0.0;
  auto diag = [&](int t) { return d[t] - (t == 0 ? tl : 0.0) - (t == n - 1 ? tr : 0.0); };
  for (int t = lane; t < n; t += 64) big = fmax(big, fmax(fabs(diag(t)), t < n - 1 ? fabs(e[t]) : 0.0));
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) big = fmax(big, __shfl_xor(big, o, 64));
  int ex = 0;
  if (big > 0.0 && isfinite(big)) (void)frexp(big, &ex);
  for (int t = tid; t < n - 1; t += NT) ee[t] = ldexp(e[t], -ex);
  __syncthreads();
  if (tid < n) {
    const int t = tid, lf = leaf_of(t), a = bnd(lf), sz = bnd(lf + 1) - a;
    if (t == a) {
      double p = ldexp(diag(t), -ex) - (t > 0 ? fabs(ee[t - 1]) : 0.0);
      if (sz == 1) {
        if (t < n - 1) p -= fabs(ee[t]);
        D[t] = p;
        Q[t * LD + t] = 1.0;
      } else {
        const double g = ee[t];
        const double q = ldexp(diag(t + 1), -ex) - (t + 1 < n - 1 ? fabs(ee[t + 1]) : 0.0);
        double c = 1.0, s = 0.0, tt = 0.0;
        if (g != 0.0) {
          const double zeta = (q - p) / (2.0 * g);
          if (fabs(zeta) > 1e150) tt = 0.5 / zeta;
          else tt = (zeta >= 0.0 ? 1.0 : -1.0) / (fabs(zeta) + sqrt(1.0 + zeta * zeta));
          c = 1.0 / sqrt(1.0 + tt * tt);
          s = c * tt;
        }
        D[t] = p - tt * g;
        D[t + 1] = q + tt * g;
        Q[t * LD + t] = c;
        Q[(t + 1) * LD + t] = -s;
        Q[t * LD + t + 1] = s;
        Q[(t + 1) * LD + t + 1] = c;
      }
    }
  }
  if (L == 0 && tid == 0) {  // n = 1
    Qg[0] = 1.0;
    lam[0] = diag(0);
  }
  __syncthreads();
  // four lanes per column (root)
  const int t = tid >> 2, sub = tid & 3;
  const bool act = t < n;
  for (int lev = 1; lev <= L; ++lev) {
    int a = 0, mid = 0, en = 0;
    double rho = 0.0;
    if (act) {
      const int b = leaf_of(t) >> lev;
      a = bnd(b << lev);
      mid = bnd((b << lev) + (1 << (lev - 1)));
      en = bnd((b + 1) << lev);
      const double beta = ee[mid - 1];
      rho = 2.0 * fabs(beta);
      if (sub == 0) {
        const double row = t < mid ? Q[(mid - 1) * LD + t] : copysign(1.0, beta) * Q[mid * LD + t];
        z[t] = row * 0.70710678118654752440;
        ba[t] = a;
        be[t] = en;
        perm[t] = t;
      }
    }
    __syncthreads();
    double tol = 0.0;
    if (act) {  // rank of this column in its block, and the deflation tolerance
      const double mine = D[t];
      int cnt = 0;
      double dm = 0.0, zm = 0.0;
#pragma unroll 2
      for (int u = a + sub; u < en; u += 4) {
        const double x = D[u];
        cnt += (x < mine || (x == mine && u < t)) ? 1 : 0;
        dm = fmax(dm, fabs(x));
        zm = fmax(zm, fabs(z[u]));
      }
#pragma unroll
      for (int o = 1; o < 4; o <<= 1) {
        cnt += __shfl_xor(cnt, o, 64);
        dm = fmax(dm, __shfl_xor(dm, o, 64));
        zm = fmax(zm, __shfl_xor(zm, o, 64));
      }
      tol = fmax(8.0 * EPS * fmax(dm, rho * zm), TINY);
      if (sub == 0) {
        perm[a + cnt] = t;
        tau[a + cnt] = mine;
        zh[a + cnt] = z[t];
        if (t == a) inv[a] = tol;
      }
    }
    __syncthreads();
    // deflation in pole order: one thread per merge, or (merges of more than
    // about 16 columns) one wavefront that passes the columns through its lanes
    if ((n >> (L - lev)) <= 16) {
      if (act && t == a && sub == 0) {
        Deflate df{D, src, nD, dK, zK, ra, rb, rc, rs, a, en, rho, tol};
        for (int i = a; i < en; ++i) df.column(perm[i], tau[i], zh[i]);
        df.finish(kc, nrot);
      }
    } else {
      for (int b = wave; b < (1 << (L - lev)); b += NT / 64) {
        const int A0 = bnd(b << lev), A1 = bnd((b + 1) << lev), m = A1 - A0;
        const double r = 2.0 * fabs(ee[bnd((b << lev) + (1 << (lev - 1))) - 1]);
        Deflate df{D, src, nD, dK, zK, ra, rb, rc, rs, A0, A1, r, inv[A0]};
        for (int h = 0; h < m; h += 64) {
          const int i = A0 + min(h + lane, m - 1);
          const int c = perm[i];
          const double dv = tau[i], zv = zh[i];
          for (int q = 0; q < min(64, m - h); ++q)
            df.column_wave(__builtin_amdgcn_readlane(c, q), read_lane(dv, q), read_lane(zv, q));
        }
        df.finish(kc, nrot);
      }
    }
    __syncthreads();
    const int k = act ? kc[a] : 0;
    const bool root = act && t - a < k;
    if (root && sub == 0) rz[t] = rho * zK[t] * zK[t];
    if (tid < n) {  // deflation rotations, row by row
      const int A0 = ba[tid], nr = nrot[A0];
      double* row = Q + tid * LD;
      for (int i = A0; i < A0 + nr; ++i) {
        const double x = row[ra[i]], y = row[rb[i]], c = rc[i], s = rs[i];
        row[ra[i]] = c * x + s * y;
        row[rb[i]] = c * y - s * x;
      }
    }
    __syncthreads();
    const double* dd = dK + a;
    if (root) {
      int o;
      double x;
      secular_root4(dd, rz + a, k, t - a, sub, o, x);
      if (sub == 0) {
        org[t] = o;
        tau[t] = x;
        nD[t] = dd[o] + x;
      }
    }
    __syncthreads();
    if (root) {  // Gu-Eisenstat: the computed roots are exact for z-hat
      const int j = t - a;
      const double dj = dd[j];
      double pr = 1.0;
#pragma unroll 2
      for (int i = sub; i < k - 1; i += 4) {
        const double den = (i < j) ? (dd[i] - dj) : (dd[i + 1] - dj);
        pr *= ((dd[org[a + i]] - dj) + tau[a + i]) * rcp2(den);
      }
      pr = prod4(pr) * (((dd[org[a + k - 1]] - dj) + tau[a + k - 1]) / rho);
      if (sub == 0) zh[t] = copysign(sqrt(fmax(pr, 0.0)), zK[t]);
    }
    __syncthreads();
    if (root) {  // norm of the root's eigenvector
      const double dO = dd[org[t]], x = tau[t];
      double s2 = 0.0;
#pragma unroll 2
      for (int j = sub; j < k; j += 4) {
        const double u = zh[a + j] * rcp2((dd[j] - dO) - x);
        s2 += u * u;
      }
      s2 = sum4(s2);
      if (sub == 0) inv[t] = 1.0 / sqrt(s2);
    }
    __syncthreads();
    // Q <- Q U: 16 columns per wavefront, over the row tiles their merges cover
    const int cl = wave * 16 + (lane & 15);
    d4 acc[NRT];
    int lo = 0, hi = 0;
    if (wave * 16 < n) {
      lo = ba[wave * 16];
      hi = be[min(n - 1, wave * 16 + 15)];
    }
    const int sb = lo / 16, ntile = hi > lo ? (hi - 1) / 16 - sb + 1 : 0;
    auto multiply = [&](auto width) {
      constexpr int W = decltype(width)::value;
      const bool cv = cl < n;
      const int ca = cv ? ba[cl] : 0, ck = cv ? kc[ca] : 0;
      const bool cr = cv && cl - ca < ck;
      const double cO = cr ? dK[ca + org[cl]] : 0.0, ctau = cr ? tau[cl] : 0.0, cinv = cr ? inv[cl] : 0.0;
      const double* row[W];
#pragma unroll
      for (int s = 0; s < W; ++s) {
        acc[s] = d4{0.0, 0.0, 0.0, 0.0};
        row[s] = Q + min((sb + s) * 16 + (lane & 15), n - 1) * LD;
      }
      // row q of U in this lane's column, and the column of Q it multiplies
      auto entry = [&](int q0, double& u, int& sc) {
        const int q = q0 + (lane >> 4), qq = min(q, n - 1);
        sc = src[qq];
        const double ur = zh[qq] * rcp2((dK[qq] - cO) - ctau) * cinv;  // a root's column
        const double ud = (q == cl) ? 1.0 : 0.0;                        // a deflated one
        u = cr ? ur : ud;
        u = (cv && q < n && ba[qq] == ca && (!cr || q - ca < ck)) ? u : 0.0;
      };
      double u;
      int sc;
      entry(lo & ~3, u, sc);
      for (int q0 = lo & ~3; q0 < hi; q0 += 4) {
        double f[W];
#pragma unroll
        for (int s = 0; s < W; ++s) f[s] = row[s][sc];
        const double uu = u;
        entry(q0 + 4, u, sc);  // the next step's, while this one's products run
#pragma unroll
        for (int s = 0; s < W; ++s) acc[s] = __builtin_amdgcn_mfma_f64_16x16x4f64(f[s], uu, acc[s], 0, 0, 0);
      }
    };
    if (ntile > 0) {
      if (ntile <= 2) multiply(std::integral_constant<int, 2>{});
      else if (NRT > 2 && ntile <= 4) multiply(std::integral_constant<int, NRT < 4 ? NRT : 4>{});
      else multiply(std::integral_constant<int, NRT>{});
    }
    if (lev < L) __syncthreads();
#pragma unroll
    for (int s = 0; s < NRT; ++s) {
      if (s < ntile && cl < n) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int r = (sb + s) * 16 + (lane >> 4) + 4 * q;
          if (r < n) {
            if (lev < L) Q[r * LD + cl] = acc[s][q];
            else Qg[(long)r * S.ldq + cl] = acc[s][q];
          }
        }
      }
    }
    if (act && sub == 0) {
      if (lev < L) D[t] = nD[t];
      else lam[t] = ldexp(nD[t], ex);
    }
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Back-transformation: Vt[i][r] = conj(E[r][i]), E = H_0 H_1 ... H_{n-2} Q with
// the reflectors in the rows of A (zeros left of and on the diagonal).  One
// wavefront per NC columns of Q, RPL rows per lane: a reflector costs one
// pass over registers, a sum over the wavefront and a second pass, with no
// barrier.  Bound by that chain, so the next three reflectors are on their way
// from the L2 meanwhile.  370 rows: 105 us (0.28 us a reflector).
// ---------------------------------------------------------------------------
template <bool CX, int RPL, int NC>
__global__ __launch_bounds__(64) void back_small_kernel(SmallEig one, const SmallEig* __restrict__ list,
                                                        const void* __restrict__ Abase,
                                                        const void* __restrict__ taubase,
                                                        const double* __restrict__ Qbase, void* __restrict__ Vbase) {
  typedef El<CX> E;
  typedef typename E::T T;
  const SmallEig S = pick(one, list, blockIdx.y);
  const int n = S.n, lane = threadIdx.x, col0 = blockIdx.x * NC;
  if (col0 >= n) return;
  const T* A = reinterpret_cast<const T*>(Abase) + S.a;
  const T* tauv = reinterpret_cast<const T*>(taubase) + S.de;
  const double* Q = Qbase + S.q;
  T q[NC][RPL];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      const int r = lane + 64 * i;
      const double x = (r < n && col0 + c < n) ? Q[(long)r * S.ldq + col0 + c] : 0.0;
      if constexpr (CX) q[c][i] = make_double2(x, 0.0);
      else q[c][i] = x;
    }
  // reflectors j with 64 s <= j + 1 < 64 (s + 1): entries of chunks s .. RPL - 1
  // (of 64, clamped at n), the next three reflectors on their way
  auto segment = [&](auto sg) {
    constexpr int I0 = decltype(sg)::value, PF = 4;
    if (64 * I0 - 1 > n - 2) return;
    const int jlo = max(64 * I0 - 1, 0), jhi = min(64 * I0 + 62, n - 2);
    T v[PF][RPL], tau[PF];
    auto load = [&](int j, int k) {
      const T* row = A + (long)max(j, 0) * S.lda;
      tau[k] = tauv[max(j, 0)];
#pragma unroll
      for (int i = I0; i < RPL; ++i) v[k][i] = row[min(lane + 64 * i, n - 1)];
    };
#pragma unroll
    for (int k = 0; k < PF - 1; ++k) load(jhi - k, k);
    for (int j0 = jhi; j0 >= jlo; j0 -= PF) {
#pragma unroll
      for (int k = 0; k < PF; ++k) {
        const int j = j0 - k;
        load(j - (PF - 1), (k + PF - 1) % PF);
        if (j < jlo) continue;
        T dot[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) dot[c] = E::zero();
#pragma unroll
        for (int i = I0; i < RPL; ++i) {
          v[k][i] = E::sel(lane + 64 * i < n, v[k][i], E::zero());
#pragma unroll
          for (int c = 0; c < NC; ++c) dot[c] = E::add(dot[c], E::cmul(v[k][i], q[c][i]));
        }
#pragma unroll
        for (int c = 0; c < NC; ++c)
          dot[c] = E::mul(tau[k], E::each(dot[c], [](double u) { return wave_sum64(u); }));
#pragma unroll
        for (int i = I0; i < RPL; ++i)
#pragma unroll
          for (int c = 0; c < NC; ++c) q[c][i] = E::sub(q[c][i], E::mul(v[k][i], dot[c]));
      }
    }
  };
  if constexpr (RPL > 11) segment(std::integral_constant<int, 11>{});
  if constexpr (RPL > 10) segment(std::integral_constant<int, 10>{});
  if constexpr (RPL > 9) segment(std::integral_constant<int, 9>{});
  if constexpr (RPL > 8) segment(std::integral_constant<int, 8>{});
  if constexpr (RPL > 7) segment(std::integral_constant<int, 7>{});
  if constexpr (RPL > 6) segment(std::integral_constant<int, 6>{});
  if constexpr (RPL > 5) segment(std::integral_constant<int, 5>{});
  if constexpr (RPL > 4) segment(std::integral_constant<int, 4>{});
  if constexpr (RPL > 3) segment(std::integral_constant<int, 3>{});
  if constexpr (RPL > 2) segment(std::integral_constant<int, 2>{});
  if constexpr (RPL > 1) segment(std::integral_constant<int, 1>{});
  segment(std::integral_constant<int, 0>{});
#pragma unroll
  for (int c = 0; c < NC; ++c) {
    if (col0 + c >= n) break;
    T* V = reinterpret_cast<T*>(Vbase) + S.v + (long)(col0 + c) * S.ldv;
#pragma unroll
    for (int i = 0; i < RPL; ++i) {
      const int r = lane + 64 * i;
      if (r < n) {
        if constexpr (CX) V[r] = make_double2(q[c][i].x, -q[c][i].y);
        else V[r] = q[c][i];
      }
    }
  }
}

template <bool CX, int GR, int GC, int NR, int NC>
void launch_trd(tn_ctx* c, int nb, const SmallEig& one, const SmallEig* list, void* A, double* d, double* e,
                void* tau) {
  constexpr int NM = GR * NR;
  constexpr size_t es = CX ? 16 : 8;
  const size_t shm = ((size_t)GR * (NM + 2) + 4 * NM) * es + 2 * (size_t)NM * sizeof(double);
  raise_lds_limit((const void*)trd_reg_kernel<CX, GR, GC, NR, NC>, shm);
  hipLaunchKernelGGL((trd_reg_kernel<CX, GR, GC, NR, NC>), dim3((unsigned)nb), dim3(GR * GC), shm, c->stream, one,
                     list, A, d, e, tau);
}

template <int NM>
void launch_dc(tn_ctx* c, int nb, const SmallEig& one, const SmallEig* list, const double* d, const double* e,
               double* Q, double* lam) {
  constexpr size_t shm = dc_small_lds<NM>();
  raise_lds_limit((const void*)dc_small_kernel<NM>, shm);
  hipLaunchKernelGGL(dc_small_kernel<NM>, dim3((unsigned)nb), dim3(4 * NM), shm, c->stream, one, list, d, e, Q, lam);
}

}  // namespace

void trd_small(tn_ctx* c, bool cplx, int nmax, int nb, const SmallEig& one, const SmallEig* list, void* A, double* d,
               double* e, void* tau) {
  TN_REQUIRE(nmax >= 1 && nmax <= (cplx ? TRD_SMALL_MAX_Z : TRD_SMALL_MAX), TN_E_INVALID, "trd_small: size");
  if (!cplx) {
    if (nmax <= 32) launch_trd<false, 8, 8, 4, 4>(c, nb, one, list, A, d, e, tau);
    else if (nmax <= 64) launch_trd<false, 16, 16, 4, 4>(c, nb, one, list, A, d, e, tau);
    else if (nmax <= 128) launch_trd<false, 16, 16, 8, 8>(c, nb, one, list, A, d, e, tau);
    else launch_trd<false, 16, 32, 12, 6>(c, nb, one, list, A, d, e, tau);
  } else {
    if (nmax <= 32) launch_trd<true, 8, 8, 4, 4>(c, nb, one, list, A, d, e, tau);
    else if (nmax <= 64) launch_trd<true, 16, 16, 4, 4>(c, nb, one, list, A, d, e, tau);
    else launch_trd<true, 16, 32, 8, 4>(c, nb, one, list, A, d, e, tau);
  }
  TN_HIP(hipGetLastError());
}

void dc_small(tn_ctx* c, int nmax, int nb, const SmallEig& one, const SmallEig* list, const double* d, const double* e,
              double* Q, double* lam) {
  TN_REQUIRE(nmax >= 1 && nmax <= DC_SMALL_MAX, TN_E_INVALID, "dc_small: size");
  if (nmax <= 32) launch_dc<32>(c, nb, one, list, d, e, Q, lam);
  else if (nmax <= 64) launch_dc<64>(c, nb, one, list, d, e, Q, lam);
  else launch_dc<128>(c, nb, one, list, d, e, Q, lam);
  TN_HIP(hipGetLastError());
}

void back_small(tn_ctx* c, bool cplx, int nmax, int nb, const SmallEig& one, const SmallEig* list, const void* A,
                const void* tau, const double* Q, void* V) {
  TN_REQUIRE(nmax >= 1 && nmax <= (cplx ? BACK_SMALL_MAX_Z : BACK_SMALL_MAX), TN_E_INVALID, "back_small: size");
  TN_REQUIRE(nb <= 65535, TN_E_INVALID, "back_small: too many blocks");
#define TN_BACK(CX, R, NC)                                                                                         \
  hipLaunchKernelGGL((back_small_kernel<CX, R, NC>), dim3((unsigned)((nmax + NC - 1) / NC), (unsigned)nb), dim3(64), \
                     0, c->stream, one, list, A, tau, Q, V)
  if (!cplx) {
    if (nmax <= 64) TN_BACK(false, 1, 1);
    else if (nmax <= 128) TN_BACK(false, 2, 1);
    else if (nmax <= 256) TN_BACK(false, 4, 1);
    else if (nmax <= 512) TN_BACK(false, 8, 2);
    else TN_BACK(false, 12, 2);
  } else {
    if (nmax <= 64) TN_BACK(true, 1, 1);
    else if (nmax <= 128) TN_BACK(true, 2, 1);
    else if (nmax <= 256) TN_BACK(true, 4, 1);
    else TN_BACK(true, 6, 2);
  }
#undef TN_BACK
  TN_HIP(hipGetLastError());
}

}  // namespace tn
