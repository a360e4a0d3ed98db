// H psi of a small bond in one launch:
//   T1[a, a', S, b]  = sum_al L[(a a'), al] psi[al, S, b]
//   T2[a', S', c, b] = sum_{a, S} Op[(c S'), (a S)] T1[a, a', S, b]
//   out[a', S', b']  = sum_{c, b} T2[a', S', c, b] R[(c b), b']
// Every step keeps a', so a workgroup takes GA of its values through all three
// with T1 and T2 in LDS (FP64 v_mfma_f64_16x16x4f64 throughout; complex values
// as separate planes, four real products).  Operands come from global memory
// straight into MFMA registers, a group of K steps ahead.  Three launches cost
// their issue and the latency of three first loads whatever the sizes: chi = 16,
// w = 5, d = 2 took kernels of 3.2, 5.0 and 3.2 us and the gaps between them;
// this one takes 6.6 us.  1024 threads a workgroup gained nothing (7.8 us there,
// 23 instead of 24 us at chi = 64).
#include "tn_internal.h"

#include <algorithm>
#include <type_traits>

namespace tn {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
constexpr int MV_THREADS = 512, MV_WAVES = MV_THREADS / 64;

struct MvArgs {
  const double* L;
  const double* v;
  const double* R;
  const double* op;
  double* out;
  int w0, w2, DD, cl, cr, GA;
  int ld1, ld2;    // row strides of T1 (GA w0 rows) and T2 (GA DD rows) in LDS
  int n1;          // doubles of one plane of T1, or of the partial tiles that replace it
  int ks;          // parts of the last product's K
  // 1 / divisor of the index arithmetic (a 32-bit division costs 40 instructions)
  float iGA, icr, iDD, int1, int2, itl2, itiles, int3;
};
// n / d for 0 <= n < 2^20 and inv = 1.0f / d: (n + 1/2) / d is at least 1 / (2 d)
// away from a whole number, and rounding moves it by less than 2^-22 n / d
__device__ __forceinline__ int mv_div(int n, float inv) { return (int)(((float)n + 0.5f) * inv); }

// operands in global memory: per-lane byte offsets, clamped to the last entry
typedef __amdgpu_buffer_rsrc_t Rsrc;
__device__ __forceinline__ Rsrc mv_rsrc(const void* p, long bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
template <typename T>
__device__ __forceinline__ T mv_ld(Rsrc r, unsigned off) {
  if constexpr (sizeof(T) == 16)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0));
}

constexpr int MV_U = 8;  // K steps (of four) per group of loads

__device__ __forceinline__ void mv_mul(d4 (&acc)[1], double a, double b) {
  acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc[0], 0, 0, 0);
}
__device__ __forceinline__ void mv_mul(d4 (&acc)[2], double2 a, double2 b) {
  acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, acc[1], 0, 0, 0);
  acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, acc[0], 0, 0, 0);
  acc[1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, acc[1], 0, 0, 0);
}

// Tiles u = wave, wave + MV_WAVES, ... of a product.  unit(u): the tile's state
// (s0, s1: its steps of four K, the last one ending at kend); la(t, s), lb(t,
// s): this lane's entries of A (row lane % 16) and B (column lane % 16) of step
// s (some valid entry past the end); done(t, acc).  The next group of loads, of
// the next tile at the end of one, is on its way while a group is multiplied.
// PRE: the first group of A (1) or B (2) has been loaded before (ga, gb).
__device__ __forceinline__ double mv_keep(bool in, double x) { return in ? x : 0.0; }
__device__ __forceinline__ double2 mv_keep(bool in, double2 x) { return make_double2(in ? x.x : 0.0, in ? x.y : 0.0); }
template <int C, int PRE, class T, class UN, class LA, class LB, class DN>
__device__ __forceinline__ void mv_stage(int wave, int units, const UN& unit, const LA& la, const LB& lb,
                                         const DN& done, T (&ga)[MV_U], T (&gb)[MV_U]) {
  const int kg = (threadIdx.x & 63) >> 4;
  int u = wave;
  if (u >= units) return;  // the whole wavefront leaves
  auto t = unit(u);
  int s = t.s0;
#pragma unroll
  for (int q = 0; q < MV_U; ++q) {
    if constexpr (PRE != 1) ga[q] = la(t, s + q);
    if constexpr (PRE != 2) gb[q] = lb(t, s + q);
  }
  d4 acc[C];
#pragma unroll
  for (int q = 0; q < C; ++q) acc[q] = d4{0, 0, 0, 0};
  while (true) {
    T na[MV_U], nb[MV_U];
    auto tn = t;
    int un = u, sn = s + MV_U;
    if (sn >= t.s1) {
      un = u + MV_WAVES;
      if (un < units) {
        tn = unit(un);
        sn = tn.s0;
      }
    }
    if (un < units) {
#pragma unroll
      for (int q = 0; q < MV_U; ++q) {
        na[q] = la(tn, sn + q);
        nb[q] = lb(tn, sn + q);
      }
    }
#pragma unroll
    for (int q = 0; q < MV_U; ++q) {
      if (s + q >= t.s1) break;
      if (4 * (s + q) + 4 > t.kend) {
        const bool in = 4 * (s + q) + kg < t.kend;
        ga[q] = mv_keep(in, ga[q]);
        gb[q] = mv_keep(in, gb[q]);
      }
      mv_mul(acc, ga[q], gb[q]);
    }
    if (un != u) {
      done(t, acc);
      if (un >= units) return;
#pragma unroll
      for (int q = 0; q < C; ++q) acc[q] = d4{0, 0, 0, 0};
    }
#pragma unroll
    for (int q = 0; q < MV_U; ++q) {
      ga[q] = na[q];
      gb[q] = nb[q];
    }
    t = tn;
    u = un;
    s = sn;
  }
}

template <bool CX>
__global__ __launch_bounds__(MV_THREADS) void mv_small_kernel(MvArgs g) {
  constexpr int C = CX ? 2 : 1;
  typedef typename std::conditional<CX, double2, double>::type T;
  extern __shared__ __attribute__((aligned(16))) unsigned char mv_smem[];
  const int M1 = g.w0 * g.GA, M2 = g.w2 * g.DD, K2 = g.w0 * g.DD, M3 = g.GA * g.DD, K3 = g.w2 * g.cr,
            NB = g.DD * g.cr, N2 = g.GA * g.cr;
  const int n2 = M3 * g.ld2;
  double* T1 = reinterpret_cast<double*>(mv_smem);  // C planes of n1
  double* T2 = T1 + C * g.n1;                       // C planes of n2
  int* koff = reinterpret_cast<int*>(T2 + C * n2);  // K2: T1 offset of (a, S)
  int* roff = koff + K2;                            // M2: T2 offset of (c, S')
  const int tid = threadIdx.x, lane = tid & 63, ln = lane & 15, kg = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int a0 = blockIdx.x * g.GA;
  constexpr unsigned ES = sizeof(T);
  const Rsrc L = mv_rsrc(g.L, (long)g.w0 * g.cl * g.cl * ES), v = mv_rsrc(g.v, (long)g.cl * NB * ES),
             R = mv_rsrc(g.R, (long)K3 * g.cr * ES), op = mv_rsrc(g.op, (long)M2 * K2 * 8);
  T* out = reinterpret_cast<T*>(g.out) + (long)a0 * g.DD * g.cr;
  // tiles of the three products, and their operands
  struct Unit {
    int s0, s1, m0, c0, kend;  // steps, first row and column, end of K
    unsigned oa, ob;           // this lane's offsets into A and B at step 0
    unsigned ea, eb;           // the last valid ones
    int x, u;
  };
  const int nt1 = (NB + 15) / 16, un1 = (M1 + 15) / 16 * nt1, st1 = (g.cl + 3) / 4;
  auto unit1 = [&](int u) {
    Unit t;
    t.s0 = 0; t.s1 = st1; t.kend = g.cl; t.u = u; t.x = 0;
    const int mi = mv_div(u, g.int1);
    t.m0 = mi * 16; t.c0 = (u - mi * nt1) * 16;
    const int m = min(t.m0 + ln, M1 - 1), a = mv_div(m, g.iGA);
    const unsigned row = (unsigned)(a * g.cl + min(a0 + m - a * g.GA, g.cl - 1)) * g.cl, col = min(t.c0 + ln, NB - 1);
    t.oa = (row + kg) * ES; t.ea = (row + g.cl - 1) * ES;
    t.ob = (col + kg * NB) * ES; t.eb = (col + (g.cl - 1) * NB) * ES;
    return t;
  };
  auto la1 = [&](const Unit& t, int s) { return mv_ld<T>(L, min(t.oa + 4u * s * ES, t.ea)); };
  auto lb1 = [&](const Unit& t, int s) { return mv_ld<T>(v, min(t.ob + 4u * s * NB * ES, t.eb)); };
  const int nt2 = (N2 + 15) / 16, tl2 = (M2 + 15) / 16 * nt2, un2 = C * tl2, st2 = (K2 + 3) / 4;
  auto unit2 = [&](int u) {  // the operator is real: planes apart
    Unit t;
    t.s0 = 0; t.s1 = st2; t.kend = K2; t.u = u;
    const int q = mv_div(u, g.itl2), x = u - q * tl2, mi = mv_div(x, g.int2);
    t.m0 = mi * 16; t.c0 = (x - mi * nt2) * 16;
    const unsigned row = min(t.m0 + ln, M2 - 1) * K2;
    t.oa = (row + kg) * 8; t.ea = (row + K2 - 1) * 8;
    const int n = min(t.c0 + ln, N2 - 1), ga = mv_div(n, g.icr), b = n - ga * g.cr;
    t.ob = q * g.n1 + ga * g.ld1 + b; t.eb = 0;
    t.x = q * n2 + ga * g.DD * g.ld2 + b;
    return t;
  };
  auto la2 = [&](const Unit& t, int s) { return mv_ld<double>(op, min(t.oa + 32u * s, t.ea)); };
  auto lb2 = [&](const Unit& t, int s) { return T1[t.ob + koff[min(4 * s + kg, K2 - 1)]]; };
  // K of the last product in ks parts where there are fewer tiles than wavefronts
  const int nt3 = (g.cr + 15) / 16, tiles = (M3 + 15) / 16 * nt3, un3 = tiles * g.ks, st3 = (K3 + 3) / 4;
  auto unit3 = [&](int u) {
    Unit t;
    const int part = mv_div(u, g.itiles), x = u - part * tiles, mi = mv_div(x, g.int3);
    t.u = u; t.x = x;
    t.m0 = mi * 16; t.c0 = (x - mi * nt3) * 16;
    t.s0 = part * st3 / g.ks; t.s1 = (part + 1) * st3 / g.ks; t.kend = min(K3, 4 * t.s1);
    const unsigned row = min(t.m0 + ln, M3 - 1) * g.ld2, col = min(t.c0 + ln, g.cr - 1);
    t.oa = row + kg; t.ea = row + K3 - 1;
    t.ob = (col + kg * g.cr) * ES; t.eb = (col + (K3 - 1) * g.cr) * ES;
    return t;
  };
  auto la3 = [&](const Unit& t, int s) {
    const unsigned i = min(t.oa + 4u * s, t.ea);
    if constexpr (CX) return make_double2(T2[i], T2[n2 + i]);
    else return T2[i];
  };
  auto lb3 = [&](const Unit& t, int s) { return mv_ld<T>(R, min(t.ob + 4u * s * g.cr * ES, t.eb)); };
  const int rows = min(M3, (g.cl - a0) * g.DD);
  auto put = [&](int row, int col, const double (&x)[C]) {
    if (row < rows && col < g.cr) {
      if constexpr (CX) out[row * g.cr + col] = make_double2(x[0], x[1]);
      else out[row * g.cr + col] = x[0];
    }
  };
  // the first loads of all three products are on their way from the start
  T ga1[MV_U], gb1[MV_U], ga3[MV_U], gb3[MV_U];
  double ga2[MV_U], gb2[MV_U];
  {
    const Unit t2 = unit2(min(wave, un2 - 1)), t3 = unit3(min(wave, un3 - 1));
#pragma unroll
    for (int q = 0; q < MV_U; ++q) ga2[q] = la2(t2, q);
#pragma unroll
    for (int q = 0; q < MV_U; ++q) gb3[q] = lb3(t3, t3.s0 + q);
  }
  for (int i = tid; i < K2; i += MV_THREADS) {
    const int a = mv_div(i, g.iDD);
    koff[i] = a * g.GA * g.ld1 + (i - a * g.DD) * g.cr;
  }
  for (int i = tid; i < M2; i += MV_THREADS) {
    const int c = mv_div(i, g.iDD);
    roff[i] = (i - c * g.DD) * g.ld2 + c * g.cr;
  }
  // T1: rows (a, ga), columns (S, b)
  mv_stage<C, 0>(wave, un1, unit1, la1, lb1, [&](const Unit& t, const d4 (&acc)[C]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = t.m0 + kg + 4 * r, col = t.c0 + ln;
      if (row < M1 && col < NB) {
#pragma unroll
        for (int q = 0; q < C; ++q) T1[q * g.n1 + row * g.ld1 + col] = acc[q][r];
      }
    }
  }, ga1, gb1);
  __syncthreads();
  // T2: rows (c, S'), columns (ga, b)
  mv_stage<1, 1>(wave, un2, unit2, la2, lb2, [&](const Unit& t, const d4 (&acc)[1]) {
    auto put2 = [&](const d4& x) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = t.m0 + kg + 4 * r;
        if (row < M2 && t.c0 + ln < N2) T2[t.x + roff[row]] = x[r];
      }
    };
    put2(acc[0]);
    // NaN if a result is not finite
    const double nf = fma(acc[0][0], 0.0, acc[0][1] * 0.0) + fma(acc[0][2], 0.0, acc[0][3] * 0.0);
    if (__any(nf != 0.0)) {  // only the operator's entries may meet an Inf or NaN, not its zeros: again, entry by entry
      d4 x{0, 0, 0, 0};
      for (int k = 0; k < K2; ++k) {
        const double v = T1[t.ob + koff[k]];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const double o = mv_ld<double>(op, (unsigned)(min(t.m0 + kg + 4 * r, M2 - 1) * K2 + k) * 8u);
          if (o != 0.0) x[r] = fma(o, v, x[r]);
        }
      }
      put2(x);
    }
  }, ga2, gb2);
  __syncthreads();
  // out: rows (ga, S'), columns b'
  mv_stage<C, 2>(wave, un3, unit3, la3, lb3, [&](const Unit& t, const d4 (&acc)[C]) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      double x[C];
#pragma unroll
      for (int q = 0; q < C; ++q) x[q] = acc[q][r];
      if (g.ks == 1) {
        put(t.m0 + kg + 4 * r, t.c0 + ln, x);
      } else {
#pragma unroll
        for (int q = 0; q < C; ++q) T1[((t.u * C + q) * 4 + r) * 64 + lane] = x[q];  // T1 is dead
      }
    }
  }, ga3, gb3);
  if (g.ks == 1) return;  // uniform
  __syncthreads();
  for (int i = tid; i < tiles * 256; i += MV_THREADS) {
    const int t = i >> 8, r = (i >> 6) & 3, l = i & 63;
    double x[C];
#pragma unroll
    for (int q = 0; q < C; ++q) x[q] = 0.0;
    for (int p = 0; p < g.ks; ++p)
#pragma unroll
      for (int q = 0; q < C; ++q) x[q] += T1[(((p * tiles + t) * C + q) * 4 + r) * 64 + l];
    const int mi = mv_div(t, g.int3);
    put(mi * 16 + (l >> 4) + 4 * r, (t - mi * nt3) * 16 + (l & 15), x);
  }
}

}  // namespace

bool mv_small(tn_ctx* c, bool cplx, const SparseOp& op, const void* L, const void* v, const void* R, void* out, int w0,
              int w2, int DD, long chil, long chir, bool timed) {
  if (!op.mat || chil > 512 || chir > 512) return false;
  const int C = cplx ? 2 : 1, cl = (int)chil, cr = (int)chir;
  // every workgroup reads all of v while others already write out; the three
  // launches have read v before the last one writes
  const size_t bytes = (size_t)cl * DD * cr * C * sizeof(double);
  const uintptr_t v0 = (uintptr_t)v, o0 = (uintptr_t)out;
  if (v0 < o0 + bytes && o0 < v0 + bytes) return false;
  MvArgs a;
  a.L = (const double*)L;
  a.v = (const double*)v;
  a.R = (const double*)R;
  a.op = op.d64();
  a.out = (double*)out;
  a.w0 = w0; a.w2 = w2; a.DD = DD; a.cl = cl; a.cr = cr;
  // as many values of a' as a tile's 16 rows hold in both products
  a.GA = std::max(1, std::min({16 / w0, 16 / DD, cl}));
  a.ld1 = DD * cr | 1;
  a.ld2 = w2 * cr | 1;
  auto t16 = [](long x) { return (x + 15) / 16; };
  auto t4 = [](long x) { return (x + 3) / 4; };
  const long tiles3 = t16(a.GA * DD) * t16(cr);
  // MFMAs of a workgroup
  const long m1 = t16(w0 * a.GA) * t16(DD * cr) * t4(cl), m2 = t16(w2 * DD) * t16(a.GA * cr) * t4(w0 * DD),
             m3 = tiles3 * t4((long)w2 * cr);
  // Three launches spread over the chip and win from some size on, later where
  // their operator step has a large operator to stage.  Time of a call, one and
  // three launches, us: w = 5, d = 2 (20 rows and columns) real chi = 16 16.7 and
  // 23.1, 32 20.5 and 24.1, 48 28.9 and 26.0; complex 32 25.3 and 30.0, 48 37.7
  // and 34.9; w = 20 (80) real 32 32.9 and 40.7, 48 54.5 and 41.9; complex 32 46.2
  // and 65.0, 48 86.0 and 82.6; w = 6, d = 4 (96) real 32 32.3 and 40.4, 48 51.0
  // and 42.1; w = 1 (4) real 48 21.8 and 22.2, 64 24.1 and 22.2.
  const long oo = (long)op.rows * op.cols;
  if ((m1 + m3) * C * C + m2 * C > (cplx ? 700 + oo / 4 : 250 + oo / 12)) return false;
  a.ks = (int)std::max<long>(1, std::min<long>(MV_WAVES / tiles3, t4((long)w2 * cr)));
  a.n1 = w0 * a.GA * a.ld1;
  if (a.ks > 1) a.n1 = std::max<int>(a.n1, (int)(tiles3 * a.ks * 256));
  a.iGA = 1.0f / a.GA; a.icr = 1.0f / cr; a.iDD = 1.0f / DD;
  a.int1 = 1.0f / t16(DD * cr); a.int2 = 1.0f / t16(a.GA * cr); a.itl2 = 1.0f / (t16(w2 * DD) * t16(a.GA * cr));
  a.itiles = 1.0f / tiles3; a.int3 = 1.0f / t16(cr);
  const size_t shm = ((size_t)C * (a.n1 + (size_t)a.GA * DD * a.ld2)) * sizeof(double) +
                     (size_t)(w0 + w2) * DD * sizeof(int);
  if (shm > 160 * 1024) return false;
  const dim3 grid((unsigned)((cl + a.GA - 1) / a.GA));
  auto launch = [&]() {
    const auto kern = cplx ? mv_small_kernel<true> : mv_small_kernel<false>;
    raise_lds_limit((const void*)kern, shm);
    hipLaunchKernelGGL(kern, grid, dim3(MV_THREADS), shm, c->stream, a);
    TN_HIP(hipGetLastError());
  };
  if (timed) {
    PhaseTimer pg(c, PH_MV_GEMM);
    launch();
  } else {
    launch();
  }
  return true;
}

}  // namespace tn
