// GEMM entry point, split-K, and generic MFMA kernels for gfx950 (CDNA4),
// row-major, batched, optional transposes:
//   F64    : v_mfma_f64_16x16x4_f64, FP64 accumulate
//   F32    : v_mfma_f32_32x32x2_f32, FP32 accumulate
//   Z64    : complex FP64 (interleaved), four real f64 MFMAs per complex product.
// The generic kernels take any stride; everything whose tiles span less than
// 2^31 bytes runs in gemm_fast.hip.
#include "tn_internal.h"

namespace tn {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));

struct GArgs {
  long M, N, K;
  const void* A; long lda; long sA; int tA; int cA;
  const void* B; long ldb; long sB; int tB; int cB;
  void* C; long ldc; long sC;
  double alpha, beta;
};

// XCD-aware tile order: consecutive workgroup ids are dealt round-robin to
// the 8 XCDs, so remap the linear id so that each XCD gets a contiguous run
// of output tiles (shared A/B panels stay in that XCD's L2).
__device__ __forceinline__ void tile_coords(int ntm, int ntn, int& tm, int& tn) {
  const int nt = ntm * ntn;
  int id = blockIdx.x;
  if (nt >= 64 && (nt % 8) == 0) {
    const int per = nt / 8;
    id = (id % 8) * per + (id / 8);
  }
  // group rows of tiles (GROUP_M = 8) for L2 reuse of B panels
  const int GM = 8;
  const int group = id / (GM * ntn);
  const int first_m = group * GM;
  const int gsz = min(ntm - first_m, GM);
  const int in_group = id % (GM * ntn);
  tm = first_m + (in_group % gsz);
  tn = in_group / gsz;
}

// ------------------------------------------------------------------------
// FP64 / FP32 kernel: LDS tiles As[BK][BM+PAD], Bs[BK][BN+PAD]
// ------------------------------------------------------------------------
template <typename T, int BM, int BN, int BK>
struct RealTile {
  static constexpr int NT = 256;
  static constexpr int PAD = (sizeof(T) == 8) ? 2 : 4;
  static constexpr int AE = BM * BK / NT;  // A elements per thread
  static constexpr int BE = BK * BN / NT;
};

template <typename T>
__device__ __forceinline__ T ldg(const T* p) { return *p; }

template <typename T, int BM, int BN, int BK>
__device__ __forceinline__ void load_tiles(const GArgs& a, const T* __restrict__ A,
                                           const T* __restrict__ B, long m0, long n0, long k0,
                                           T (&ra)[RealTile<T, BM, BN, BK>::AE],
                                           T (&rb)[RealTile<T, BM, BN, BK>::BE]) {
  using TT = RealTile<T, BM, BN, BK>;
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < TT::AE; ++i) {
    const int idx = tid + i * TT::NT;
    int mm, kk;
    if (!a.tA) { kk = idx % BK; mm = idx / BK; } else { mm = idx % BM; kk = idx / BM; }
    const long m = m0 + mm, k = k0 + kk;
    T v = T(0);
    if (m < a.M && k < a.K) v = a.tA ? A[k * a.lda + m] : A[m * a.lda + k];
    ra[i] = v;
  }
#pragma unroll
  for (int i = 0; i < TT::BE; ++i) {
    const int idx = tid + i * TT::NT;
    int nn, kk;
    if (!a.tB) { nn = idx % BN; kk = idx / BN; } else { kk = idx % BK; nn = idx / BK; }
    const long n = n0 + nn, k = k0 + kk;
    T v = T(0);
    if (n < a.N && k < a.K) v = a.tB ? B[n * a.ldb + k] : B[k * a.ldb + n];
    rb[i] = v;
  }
}

template <typename T, int BM, int BN, int BK>
__device__ __forceinline__ void store_tiles(const GArgs& a, T* As, T* Bs,
                                            const T (&ra)[RealTile<T, BM, BN, BK>::AE],
                                            const T (&rb)[RealTile<T, BM, BN, BK>::BE]) {
  using TT = RealTile<T, BM, BN, BK>;
  constexpr int LA = BM + TT::PAD, LB = BN + TT::PAD;
  const int tid = threadIdx.x;
#pragma unroll
  for (int i = 0; i < TT::AE; ++i) {
    const int idx = tid + i * TT::NT;
    int mm, kk;
    if (!a.tA) { kk = idx % BK; mm = idx / BK; } else { mm = idx % BM; kk = idx / BM; }
    As[kk * LA + mm] = ra[i];
  }
#pragma unroll
  for (int i = 0; i < TT::BE; ++i) {
    const int idx = tid + i * TT::NT;
    int nn, kk;
    if (!a.tB) { nn = idx % BN; kk = idx / BN; } else { kk = idx % BK; nn = idx / BK; }
    Bs[kk * LB + nn] = rb[i];
  }
}

// FP64: wave tile (BM/2) x (BN/2) made of 16x16 MFMA blocks
template <int BM, int BN, int BK>
__global__ __launch_bounds__(256) void gemm_f64_kernel(GArgs a) {
  using T = double;
  using TT = RealTile<T, BM, BN, BK>;
  constexpr int LA = BM + TT::PAD, LB = BN + TT::PAD;
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int FM = WTM / 16, FN = WTN / 16;
  __shared__ T As[BK * LA];
  __shared__ T Bs[BK * LB];

  const int ntm = (int)((a.M + BM - 1) / BM), ntn = (int)((a.N + BN - 1) / BN);
  int tm, tn;
  tile_coords(ntm, ntn, tm, tn);
  const long m0 = (long)tm * BM, n0 = (long)tn * BN;
  const long bz = blockIdx.z;
  const T* A = reinterpret_cast<const T*>(a.A) + bz * a.sA;
  const T* B = reinterpret_cast<const T*>(a.B) + bz * a.sB;
  T* C = reinterpret_cast<T*>(a.C) + bz * a.sC;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  d4 acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = d4{0, 0, 0, 0};

  T ra[TT::AE], rb[TT::BE];
  load_tiles<T, BM, BN, BK>(a, A, B, m0, n0, 0, ra, rb);
  for (long k0 = 0; k0 < a.K; k0 += BK) {
    __syncthreads();
    store_tiles<T, BM, BN, BK>(a, As, Bs, ra, rb);
    __syncthreads();
    if (k0 + BK < a.K) load_tiles<T, BM, BN, BK>(a, A, B, m0, n0, k0 + BK, ra, rb);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const int kr = kk + (lane >> 4);
      double fa[FM], fb[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[i] = As[kr * LA + wm * WTM + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[j] = Bs[kr * LB + wn * WTN + j * 16 + (lane & 15)];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  }
  // epilogue: register r of lane holds row lane/16 + 4r, column lane%16 of
  // each 16x16 block (v_mfma_f64_16x16x4f64 output layout)
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long m = m0 + wm * WTM + i * 16 + (lane >> 4) + 4 * r;
        const long n = n0 + wn * WTN + j * 16 + (lane & 15);
        if (m < a.M && n < a.N) {
          double v = a.alpha * acc[i][j][r];
          if (a.beta != 0.0) v += a.beta * C[m * a.ldc + n];
          C[m * a.ldc + n] = v;
        }
      }
}

// FP32: wave tile (BM/2) x (BN/2) made of 32x32 MFMA blocks
template <int BM, int BN, int BK>
__global__ __launch_bounds__(256) void gemm_f32_kernel(GArgs a) {
  using T = float;
  using TT = RealTile<T, BM, BN, BK>;
  constexpr int LA = BM + TT::PAD, LB = BN + TT::PAD;
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int FM = WTM / 32, FN = WTN / 32;
  __shared__ T As[BK * LA];
  __shared__ T Bs[BK * LB];

  const int ntm = (int)((a.M + BM - 1) / BM), ntn = (int)((a.N + BN - 1) / BN);
  int tm, tn;
  tile_coords(ntm, ntn, tm, tn);
  const long m0 = (long)tm * BM, n0 = (long)tn * BN;
  const long bz = blockIdx.z;
  const T* A = reinterpret_cast<const T*>(a.A) + bz * a.sA;
  const T* B = reinterpret_cast<const T*>(a.B) + bz * a.sB;
  T* C = reinterpret_cast<T*>(a.C) + bz * a.sC;

  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  f16v acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = f16v{};

  T ra[TT::AE], rb[TT::BE];
  load_tiles<T, BM, BN, BK>(a, A, B, m0, n0, 0, ra, rb);
  for (long k0 = 0; k0 < a.K; k0 += BK) {
    __syncthreads();
    store_tiles<T, BM, BN, BK>(a, As, Bs, ra, rb);
    __syncthreads();
    if (k0 + BK < a.K) load_tiles<T, BM, BN, BK>(a, A, B, m0, n0, k0 + BK, ra, rb);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 2) {
      const int kr = kk + (lane >> 5);
      float fa[FM], fb[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) fa[i] = As[kr * LA + wm * WTM + i * 32 + (lane & 31)];
#pragma unroll
      for (int j = 0; j < FN; ++j) fb[j] = Bs[kr * LB + wn * WTN + j * 32 + (lane & 31)];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
    }
  }
  // epilogue: register r of lane -> row 8*(r/4) + 4*(lane/32) + r%4, column lane%32
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long m = m0 + wm * WTM + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const long n = n0 + wn * WTN + j * 32 + (lane & 31);
        if (m < a.M && n < a.N) {
          float v = (float)a.alpha * acc[i][j][r];
          if (a.beta != 0.0) v += (float)a.beta * C[m * a.ldc + n];
          C[m * a.ldc + n] = v;
        }
      }
}

// ------------------------------------------------------------------------
// Complex FP64 (interleaved re/im).  LDS holds re and im planes; each complex
// multiply-accumulate is four f64 MFMAs into re/im accumulators.
// ------------------------------------------------------------------------
template <int BM, int BN, int BK>
__global__ __launch_bounds__(256) void gemm_z64_kernel(GArgs a) {
  constexpr int NT = 256;
  constexpr int LA = BM + 2, LB = BN + 2;
  constexpr int AE = BM * BK / NT, BE = BK * BN / NT;
  constexpr int WTM = BM / 2, WTN = BN / 2;
  constexpr int FM = WTM / 16, FN = WTN / 16;
  __shared__ double Ar[BK * LA], Ai[BK * LA];
  __shared__ double Br[BK * LB], Bi[BK * LB];

  const int ntm = (int)((a.M + BM - 1) / BM), ntn = (int)((a.N + BN - 1) / BN);
  int tm, tn;
  tile_coords(ntm, ntn, tm, tn);
  const long m0 = (long)tm * BM, n0 = (long)tn * BN;
  const long bz = blockIdx.z;
  const double2* A = reinterpret_cast<const double2*>(a.A) + bz * a.sA;
  const double2* B = reinterpret_cast<const double2*>(a.B) + bz * a.sB;
  double2* C = reinterpret_cast<double2*>(a.C) + bz * a.sC;
  const double sa = a.cA ? -1.0 : 1.0, sb = a.cB ? -1.0 : 1.0;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;

  d4 accr[FM][FN], acci[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) { accr[i][j] = d4{0, 0, 0, 0}; acci[i][j] = d4{0, 0, 0, 0}; }

  double2 ra[AE], rb[BE];
  auto gload = [&](long k0) {
#pragma unroll
    for (int i = 0; i < AE; ++i) {
      const int idx = tid + i * NT;
      int mm, kk;
      if (!a.tA) { kk = idx % BK; mm = idx / BK; } else { mm = idx % BM; kk = idx / BM; }
      const long m = m0 + mm, k = k0 + kk;
      double2 v = make_double2(0.0, 0.0);
      if (m < a.M && k < a.K) v = a.tA ? A[k * a.lda + m] : A[m * a.lda + k];
      ra[i] = v;
    }
#pragma unroll
    for (int i = 0; i < BE; ++i) {
      const int idx = tid + i * NT;
      int nn, kk;
      if (!a.tB) { nn = idx % BN; kk = idx / BN; } else { kk = idx % BK; nn = idx / BK; }
      const long n = n0 + nn, k = k0 + kk;
      double2 v = make_double2(0.0, 0.0);
      if (n < a.N && k < a.K) v = a.tB ? B[n * a.ldb + k] : B[k * a.ldb + n];
      rb[i] = v;
    }
  };
  auto sstore = [&]() {
#pragma unroll
    for (int i = 0; i < AE; ++i) {
      const int idx = tid + i * NT;
      int mm, kk;
      if (!a.tA) { kk = idx % BK; mm = idx / BK; } else { mm = idx % BM; kk = idx / BM; }
      Ar[kk * LA + mm] = ra[i].x;
      Ai[kk * LA + mm] = sa * ra[i].y;
    }
#pragma unroll
    for (int i = 0; i < BE; ++i) {
      const int idx = tid + i * NT;
      int nn, kk;
      if (!a.tB) { nn = idx % BN; kk = idx / BN; } else { kk = idx % BK; nn = idx / BK; }
      Br[kk * LB + nn] = rb[i].x;
      Bi[kk * LB + nn] = sb * rb[i].y;
    }
  };

  gload(0);
  for (long k0 = 0; k0 < a.K; k0 += BK) {
    __syncthreads();
    sstore();
    __syncthreads();
    if (k0 + BK < a.K) gload(k0 + BK);
#pragma unroll
    for (int kk = 0; kk < BK; kk += 4) {
      const int kr = kk + (lane >> 4);
      double far_[FM], fai[FM], fbr[FN], fbi[FN], fbin[FN];
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        far_[i] = Ar[kr * LA + wm * WTM + i * 16 + (lane & 15)];
        fai[i] = Ai[kr * LA + wm * WTM + i * 16 + (lane & 15)];
      }
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        fbr[j] = Br[kr * LB + wn * WTN + j * 16 + (lane & 15)];
        fbi[j] = Bi[kr * LB + wn * WTN + j * 16 + (lane & 15)];
        fbin[j] = -fbi[j];
      }
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          accr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(far_[i], fbr[j], accr[i][j], 0, 0, 0);
          accr[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fai[i], fbin[j], accr[i][j], 0, 0, 0);
          acci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(far_[i], fbi[j], acci[i][j], 0, 0, 0);
          acci[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fai[i], fbr[j], acci[i][j], 0, 0, 0);
        }
    }
  }
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const long m = m0 + wm * WTM + i * 16 + (lane >> 4) + 4 * r;
        const long n = n0 + wn * WTN + j * 16 + (lane & 15);
        if (m < a.M && n < a.N) {
          double vr = a.alpha * accr[i][j][r];
          double vi = a.alpha * acci[i][j][r];
          if (a.beta != 0.0) {
            vr += a.beta * C[m * a.ldc + n].x;
            vi += a.beta * C[m * a.ldc + n].y;
          }
          C[m * a.ldc + n] = make_double2(vr, vi);
        }
      }
}

template <int BM, int BN>
dim3 grid_for(const GemmDesc& g) {
  const long ntm = (g.M + BM - 1) / BM, ntn = (g.N + BN - 1) / BN;
  return dim3((unsigned)(ntm * ntn), 1, (unsigned)g.batch);
}

GArgs to_args(const GemmDesc& g) {
  GArgs a;
  a.M = g.M; a.N = g.N; a.K = g.K;
  a.A = g.A; a.lda = g.lda; a.sA = g.sA; a.tA = g.tA; a.cA = g.cA;
  a.B = g.B; a.ldb = g.ldb; a.sB = g.sB; a.tB = g.tB; a.cB = g.cB;
  a.C = g.C; a.ldc = g.ldc; a.sC = g.sC;
  a.alpha = g.alpha; a.beta = g.beta;
  return a;
}


}  // namespace

namespace {
// C = alpha * sum_p part[p] + beta * C   (part: P slices of M x N, ld N)
template <typename T>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const T* __restrict__ part, int P, long M, long N,
                                                            double alpha, double beta, T* __restrict__ C, long ldc) {
  const long tot = M * N;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < tot; i += (long)gridDim.x * 256) {
    double acc = 0.0;
    for (int q = 0; q < P; ++q) acc += (double)part[(long)q * tot + i];
    const long r = i / N, col = i - r * N;
    T* dst = C + r * ldc + col;
    const double prev = (beta != 0.0) ? beta * (double)*dst : 0.0;
    *dst = (T)(alpha * acc + prev);
  }
}
}  // namespace

static void gemm_impl(tn_ctx* c, Prec p, const GemmDesc& g);

// Few output tiles with a long K (K-reductions over whole tensors, Gram
// matrices of tall matrices) leave most of the chip idle: split K into
// chunks computed as one batched GEMM into FP64/FP32 partials, then reduce.
// Chunk length along K of the split (0: no split).  The reduction is one more
// launch (about 4 us); a 32 x 32 tile runs K at about 7 ns a row, so from
// half a chip of idle CUs and chunks of 256 rows on the split pays.
static long split_chunk(Prec p, const GemmDesc& g) {
  if (!(p == Prec::F64 || p == Prec::F32) || g.batch != 1) return 0;
  const long t128 = ((g.M + 127) / 128) * ((g.N + 127) / 128);
  const long b = p == Prec::F64 ? 32 : 64, tiles = ((g.M + b - 1) / b) * ((g.N + b - 1) / b);
  long P0;
  if (t128 < 64 && g.K >= 4096) P0 = std::min<long>(g.K / 512, 256 / t128);
  else if (tiles <= 128 && g.K >= 512) P0 = std::min<long>(g.K / 256, 256 / tiles);
  else return 0;
  if (P0 < 2) return 0;
  return ((g.K + P0 - 1) / P0 + 15) / 16 * 16;
}

static bool gemm_split_k(tn_ctx* c, Prec p, const GemmDesc& g) {
  const long Kc = split_chunk(p, g);
  if (Kc == 0) return false;
  const long P = (g.K + Kc - 1) / Kc;
  const long full = g.K / Kc;  // chunks of exactly Kc
  const size_t es = (p == Prec::F64) ? 8 : 4;
  const size_t need = (size_t)P * g.M * g.N * es;
  char* part;
  if (g.split_ws) {
    if (need > g.split_cap) return false;
    part = (char*)g.split_ws;
  } else {
    part = (char*)c->workspace(WS_GEMM_SPLIT, need);
  }
  GemmDesc q = g;
  q.alpha = 1.0;
  q.beta = 0.0;
  q.K = Kc;
  q.C = part;
  q.ldc = g.N;
  q.sC = g.M * g.N;
  q.sA = g.tA ? Kc * g.lda : Kc;
  q.sB = g.tB ? Kc : Kc * g.ldb;
  q.batch = (int)full;
  gemm_impl(c, p, q);
  if (full < P) {  // the shorter last chunk
    GemmDesc r = q;
    r.batch = 1;
    r.K = g.K - full * Kc;
    r.A = (const char*)g.A + (size_t)(full * q.sA) * es;
    r.B = (const char*)g.B + (size_t)(full * q.sB) * es;
    r.C = part + (size_t)(full * q.sC) * es;
    gemm_impl(c, p, r);
  }
  const long tot = g.M * g.N;
  const unsigned grid = (unsigned)std::max<long>(1, std::min<long>(2048, (tot + 255) / 256));
  if (p == Prec::F64)
    hipLaunchKernelGGL(splitk_reduce_kernel<double>, dim3(grid), dim3(256), 0, c->stream, (const double*)part, (int)P,
                       g.M, g.N, g.alpha, g.beta, (double*)g.C, g.ldc);
  else
    hipLaunchKernelGGL(splitk_reduce_kernel<float>, dim3(grid), dim3(256), 0, c->stream, (const float*)part, (int)P,
                       g.M, g.N, g.alpha, g.beta, (float*)g.C, g.ldc);
  TN_HIP(hipGetLastError());
  return true;
}

void gemm(tn_ctx* c, Prec p, const GemmDesc& g) {
  TN_REQUIRE(g.M >= 0 && g.N >= 0 && g.K >= 0 && g.batch >= 1, TN_E_INVALID, "gemm: bad sizes");
  if (g.M == 0 || g.N == 0) return;
  TN_REQUIRE(g.A && g.B && g.C, TN_E_INVALID, "gemm: null operand");
  TN_REQUIRE(g.batch <= 65535, TN_E_INVALID, "gemm: batch too large");
  if (gemm_split_k(c, p, g)) return;
  gemm_impl(c, p, g);
}

static void gemm_impl(tn_ctx* c, Prec p, const GemmDesc& g) {
  if (gemm_fast_ok(p, g)) {
    gemm_fast(c, p, g);
    return;
  }
  // row strides past 32-bit tile offsets
  const GArgs a = to_args(g);
  const dim3 gr = grid_for<64, 64>(g);
  switch (p) {
    case Prec::F64:
      hipLaunchKernelGGL((gemm_f64_kernel<64, 64, 16>), gr, dim3(256), 0, c->stream, a);
      break;
    case Prec::F32:
      hipLaunchKernelGGL((gemm_f32_kernel<64, 64, 16>), gr, dim3(256), 0, c->stream, a);
      break;
    case Prec::Z64:
      hipLaunchKernelGGL((gemm_z64_kernel<64, 64, 8>), gr, dim3(256), 0, c->stream, a);
      break;
    case Prec::BF16X3:
      throw Error(TN_E_INVALID, "gemm: BF16x3 operands come pre-split (gemm_bf16x3_nt)");
  }
  TN_HIP(hipGetLastError());
}

}  // namespace tn
