// Truncated factorisation for replacebond!: symmetric eigen-decomposition of
// the two-site density matrix on the device, in FP64.
//
// For phi (m x n) the Gram matrix G = phi phi^T (m x m, "left") or
// G = phi^T phi (n x n, "right") is formed with one FP64 MFMA GEMM and
// diagonalised by Householder tridiagonalisation and divide and conquer
// (eig_dc.hip).  The eigenvalues are the weights P = s^2 with absolute
// accuracy ~eps * sum(P) (the accuracy of a density-matrix eigensolver), and
// the eigenvectors are orthonormal to rounding, so the orthonormal MPS factor
// is taken from them directly and the other factor is the exact product
// V^T phi (or phi V): no division by small singular values anywhere.
#include "tn_internal.h"

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <numeric>

namespace tn {
namespace {

constexpr int PR = 64;  // density matrices are padded to a multiple of this

}  // namespace

// eigen-decomposition of the padded Hermitian matrix G (ld ppad)
static void eig_padded(tn_ctx* c, void* G, long p, long ppad, void* Vt, bool cplx, GramEig& out) {
  out.p = p;
  out.ppad = ppad;
  out.cplx = cplx;
  out.Vt = Vt;
  if (!cplx) sym_eig_dc(c, (double*)G, p, ppad, (double*)Vt, ppad, out.w);
  else sym_eig_dc_z(c, (double*)G, p, ppad, (double*)Vt, ppad, out.w);
}

void gram_eig(tn_ctx* c, const void* M, long m, long n, bool left, bool cplx, GramEig& out, const void* X, long kx,
              double xs, long ldx) {
  TN_REQUIRE(m > 0 && n > 0, TN_E_INVALID, "svd: empty matrix");
  const long p = left ? m : n;
  const long ppad = ((p + PR - 1) / PR) * PR;
  const size_t es = cplx ? 16 : 8;
  void* G = c->workspace(WS_SVD_X, (size_t)ppad * ppad * es);
  void* Vt = c->workspace(WS_SVD_Q, (size_t)ppad * ppad * es);
  fill_f64(c, (double*)G, 0.0, ppad * ppad * (cplx ? 2 : 1));
  GemmDesc g;
  g.M = p; g.N = p; g.C = G; g.ldc = ppad;
  if (left) {  // G = M M^T  (M M^H)
    g.K = n; g.A = M; g.lda = n; g.B = M; g.ldb = n; g.tB = 1; g.cB = cplx;
  } else {     // G = M^T M  (M^H M)
    g.K = m; g.A = M; g.lda = n; g.tA = 1; g.cA = cplx; g.B = M; g.ldb = n;
  }
  gemm(c, cplx ? Prec::Z64 : Prec::F64, g);
  if (X && kx > 0 && xs != 0.0) {  // density-matrix perturbation
    GemmDesc h;
    h.M = p; h.N = p; h.K = kx; h.C = G; h.ldc = ppad;
    h.alpha = xs; h.beta = 1.0;
    const long ld = ldx > 0 ? ldx : kx;
    if (left) { h.A = X; h.lda = ld; h.B = X; h.ldb = ld; h.tB = 1; h.cB = cplx; }
    else      { h.A = X; h.lda = p; h.tA = 1; h.cA = cplx; h.B = X; h.ldb = p; }
    gemm(c, cplx ? Prec::Z64 : Prec::F64, h);
  }
  out.left = left;
  eig_padded(c, G, p, ppad, Vt, cplx, out);
}

void herm_eig(tn_ctx* c, const void* H, long p, long ldh, bool cplx, GramEig& out) {
  TN_REQUIRE(p > 0, TN_E_INVALID, "eigen: empty matrix");
  const long ppad = ((p + PR - 1) / PR) * PR;
  const size_t es = cplx ? 16 : 8;
  void* G = c->workspace(WS_SVD_X, (size_t)ppad * ppad * es);
  void* Vt = c->workspace(WS_SVD_Q, (size_t)ppad * ppad * es);
  fill_f64(c, (double*)G, 0.0, ppad * ppad * (cplx ? 2 : 1));
  TN_HIP(hipMemcpy2DAsync(G, (size_t)ppad * es, H, (size_t)ldh * es, (size_t)p * es, (size_t)p,
                          hipMemcpyDeviceToDevice, c->stream));
  out.left = true;
  eig_padded(c, G, p, ppad, Vt, cplx, out);
}

TruncRule truncate_weights(const std::vector<double>& Pin, long maxdim, long mindim, double cutoff) {
  // NDTensors truncate!! with the relative cutoff (ITensors' default)
  std::vector<double> P = Pin;
  const long origm = (long)P.size();
  TruncRule tr{0, 0.0, 0.0};
  if (origm == 0) return tr;
  for (long k = origm - 1; k >= 0; --k) {
    if (P[k] >= 0.0) break;
    P[k] = 0.0;
  }
  if (origm == 1) { tr.n = 1; tr.docut = std::fabs(P[0]) / 2; return tr; }
  long n = origm;
  double truncerr = 0.0;
  maxdim = std::min(maxdim, origm);
  mindim = std::max<long>(1, std::min(mindim, maxdim));
  while (n > maxdim) { truncerr += P[n - 1]; --n; }
  double scale = 0.0;
  for (double v : P) scale += v;
  if (scale == 0.0) scale = 1.0;
  while (n > mindim && truncerr + P[n - 1] <= cutoff * scale) { truncerr += P[n - 1]; --n; }
  truncerr /= scale;
  n = std::max<long>(n, 1);
  double docut = 0.0;
  if (n < origm) {
    docut = (P[n - 1] + P[n]) / 2;
    if (std::fabs(P[n - 1] - P[n]) < 1e-3 * P[n - 1]) docut += 1e-3 * P[n - 1];
  }
  tr.n = n;
  tr.truncerr = truncerr;
  tr.docut = docut;
  return tr;
}

}  // namespace tn
