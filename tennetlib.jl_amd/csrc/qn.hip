// Quantum-number (U(1), U(1)xU(1)) blocks of the truncating factorisation
// (replacebond! of a QN-conserving two-site tensor): qn_scatter_kernel makes
// the kept eigenvectors of every sector the columns of the orthonormal factor
// (rows of its transpose), each written to the rows of M that belong to its
// sector; everything else stays zero.
#include "tn_internal.h"

namespace tn {
namespace {

// kept column j: eigenvector col[4j+2] of the sector whose rows of M are
// rows[col[4j+1] .. +col[4j+3]), stored at V + col[4j] (rows of length p);
// out (rows x k, ld k) gets out[rows[roff + r]][j], or with trans the k x rows
// transpose out[j][rows[roff + r]]
__global__ __launch_bounds__(256) void qn_scatter_kernel(const double* __restrict__ V, const int* __restrict__ col,
                                                         const int* __restrict__ rows, int k, long ldo, int trans,
                                                         double* __restrict__ out) {
  const int j = blockIdx.x;
  const long vo = col[4 * j + 0];
  const int roff = col[4 * j + 1], idx = col[4 * j + 2], p = col[4 * j + 3];
  for (int r = threadIdx.x; r < p; r += 256) {
    const double x = V[vo + (long)idx * p + r];
    const long row = rows[roff + r];
    if (trans) out[(long)j * ldo + row] = x;
    else out[row * ldo + j] = x;
  }
}

}  // namespace

void qn_scatter(tn_ctx* c, const double* V, const int* col_dev, const int* rows_dev, int k, long ldo, bool trans,
                double* out) {
  if (k <= 0) return;
  hipLaunchKernelGGL(qn_scatter_kernel, dim3((unsigned)k), dim3(256), 0, c->stream, V, col_dev, rows_dev, k, ldo,
                     trans ? 1 : 0, out);
  TN_HIP(hipGetLastError());
}

}  // namespace tn
