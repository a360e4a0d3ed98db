// GEMM entry point and split-K (row-major, batched, optional transposes):
//   F64    : v_mfma_f64_16x16x4_f64, FP64 accumulate
//   F32    : v_mfma_f32_32x32x2_f32, FP32 accumulate
//   Z64    : complex FP64 (interleaved), four real f64 MFMAs per complex product.
// The kernels are in gemm_fast.hip.
#include "tn_internal.h"

namespace tn {
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

// Few output tiles with a long K (K-reductions over whole tensors, Gram
// matrices of tall matrices) leave most of the chip idle: split K into chunks,
// the last one shorter, computed as one batched GEMM into FP64/FP32 partials,
// then reduce.  Chunk length along K (0: no split).  The reduction is one more
// launch (about 4 us); a 32 x 32 FP64 tile runs K at about 7 ns a row, so from
// half a chip of idle CUs and chunks of 256 rows on the split pays; the 64 x 64
// FP32 tile is slower per row: chunks of 128.  H psi with chi_l = 4, d = 2, in
// us, chunks of 64 / 128 / 256: FP32 w = 3, chi_r = 128 32.1 / 32.8 / 36.2; FP64
// 25.9 / 26.0 / 27.0.
static long split_chunk(Prec p, const GemmDesc& g) {
  if (!(p == Prec::F64 || p == Prec::F32) || g.batch != 1) return 0;
  const long t128 = ((g.M + 127) / 128) * ((g.N + 127) / 128);
  const long b = p == Prec::F64 ? 32 : 64, tiles = ((g.M + b - 1) / b) * ((g.N + b - 1) / b);
  const long chunk = p == Prec::F64 ? 256 : 128;
  long P0;
  if (t128 < 64 && g.K >= 4096) P0 = std::min<long>(g.K / 512, 256 / t128);
  else if (tiles <= 128 && g.K >= 2 * chunk) P0 = std::min<long>(g.K / chunk, 256 / tiles);
  else return 0;
  if (P0 < 2) return 0;
  return ((g.K + P0 - 1) / P0 + 15) / 16 * 16;
}

static bool gemm_split_k(tn_ctx* c, Prec p, const GemmDesc& g) {
  const long Kc = split_chunk(p, g);
  if (Kc == 0) return false;
  const long P = (g.K + Kc - 1) / Kc;
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
  q.kstep = Kc;
  q.C = part;
  q.ldc = g.N;
  q.sC = g.M * g.N;
  q.sA = g.tA ? Kc * g.lda : Kc;
  q.sB = g.tB ? Kc : Kc * g.ldb;
  // the shorter last chunk goes with the others, unless their workgroups fill
  // the chip and it would cost all of them another round: 32 x 181 outputs, K =
  // 543 in two, H psi 29.7 us together, 37.6 apart; 1020 x 253, K = 5060 in nine,
  // product 70 us together, 61 apart
  const long last = g.K - (P - 1) * Kc;
  const double others = gemm_tile_work(p, g.M, g.N, P - 1);
  const bool together = last == Kc || gemm_tile_work(p, g.M, g.N, P) * Kc <=
                                          others * Kc + gemm_tile_work(p, g.M, g.N, 1) * last;
  q.batch = (int)(together ? P : P - 1);
  gemm_tiles(c, p, q);
  if (!together) {
    GemmDesc r = q;
    r.batch = 1;
    r.K = last;
    r.kstep = 0;
    r.A = (const char*)g.A + (size_t)((P - 1) * q.sA) * es;
    r.B = (const char*)g.B + (size_t)((P - 1) * q.sB) * es;
    r.C = part + (size_t)((P - 1) * q.sC) * es;
    gemm_tiles(c, p, r);
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
  gemm_tiles(c, p, g);
}

}  // namespace tn
