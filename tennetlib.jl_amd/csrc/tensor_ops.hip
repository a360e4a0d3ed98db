// Memory-bound kernels of the hot path: the small MPO contraction ("W step")
// between the two big GEMMs of a matvec / environment update, precision
// conversions, the FP64 Krylov vector operations (fixed-order two-stage
// reductions, no atomics, so results are reproducible run to run) and the
// gather / transpose kernels used by the truncated SVD.
#include "tn_internal.h"

#include <type_traits>

#include <cmath>

namespace tn {
namespace {

constexpr int RED_BLOCKS = 1024;  // first-stage reduction blocks (4 per CU)
constexpr int RED_THREADS = 256;
constexpr int MAX_DOT = 32;       // basis vectors per multi-dot pass

// ---------------------------------------------------------------------------
// W step: out[g', A, S', B] = sum_nz val * in[g, A, S, B]
// block = 64 B-columns x 4 row groups; the (g S) x 64 input slab of one A is
// staged in LDS, each wavefront walks a quarter of the CSR output rows (rows
// are wave-uniform, so the CSR entries come through the scalar cache).
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned short f2bf_rne(float x) {
  unsigned int u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

// SPLIT: T is float and the result is stored as bf16 hi/lo pairs
template <typename T, bool SPLIT>
__global__ __launch_bounds__(256) void wstep_kernel(int G, int Gp, int D, int Dp, long nA, long nB,
                                                    const T* __restrict__ in, long in_sg, long in_sA,
                                                    long in_sS, T* __restrict__ out, long out_sg,
                                                    long out_sA, long out_sS,
                                                    const int* __restrict__ rowptr,
                                                    const int* __restrict__ colidx,
                                                    const double* __restrict__ vals,
                                                    unsigned short* __restrict__ ohi,
                                                    unsigned short* __restrict__ olo) {
  extern __shared__ unsigned char smem_raw[];
  T* slab = reinterpret_cast<T*>(smem_raw);  // [K][64]
  const int K = G * D;
  const int tb = threadIdx.x & 63;
  const int ty = threadIdx.x >> 6;
  const long A = blockIdx.y;
  const long B = (long)blockIdx.x * 64 + tb;
  const bool valid = B < nB;
  for (int i = ty; i < K; i += 4) {
    const int g = i / D, S = i % D;
    T v = T(0);
    if (valid) v = in[g * in_sg + A * in_sA + S * in_sS + B];
    slab[i * 64 + tb] = v;
  }
  __syncthreads();
  if (!valid) return;
  const int rows = Gp * Dp;
  for (int o = ty; o < rows; o += 4) {
    const int b = rowptr[o], e = rowptr[o + 1];
    T acc = T(0);
    for (int z = b; z < e; ++z) acc += (T)vals[z] * slab[colidx[z] * 64 + tb];
    const int gp = o / Dp, Sp = o % Dp;
    const long off = gp * out_sg + A * out_sA + Sp * out_sS + B;
    if constexpr (SPLIT) {
      const unsigned short h = f2bf_rne((float)acc);
      ohi[off] = h;
      olo[off] = f2bf_rne((float)acc - __uint_as_float(((unsigned int)h) << 16));
    } else {
      out[off] = acc;
    }
  }
}

// The same W step with VEC consecutive B per thread (16-byte loads and
// stores: 64 VEC columns per workgroup, so every row segment it touches is
// 1 KiB contiguous instead of 256 B); shapes and strides multiples of VEC.
// Dynamic LDS: K x 64 VEC elements.
template <typename T, int VEC>
__global__ __launch_bounds__(256) void wstep_vec_kernel(int G, int Gp, int D, int Dp, long nB,
                                                        const T* __restrict__ in, long in_sg, long in_sA,
                                                        long in_sS, T* __restrict__ out, long out_sg,
                                                        long out_sA, long out_sS,
                                                        const int* __restrict__ rowptr,
                                                        const int* __restrict__ colidx,
                                                        const double* __restrict__ vals) {
  typedef T vec_t __attribute__((ext_vector_type(VEC)));
  extern __shared__ unsigned char smem_raw[];
  vec_t* slab = reinterpret_cast<vec_t*>(smem_raw);  // [K][64] vectors
  const int K = G * D;
  const int tb = threadIdx.x & 63;
  const int ty = threadIdx.x >> 6;
  const long A = blockIdx.y;
  const long B = ((long)blockIdx.x * 64 + tb) * VEC;
  const bool valid = B < nB;
  for (int i = ty; i < K; i += 4) {
    const int g = i / D, S = i % D;
    vec_t v = (vec_t)(T(0));
    if (valid) v = *reinterpret_cast<const vec_t*>(in + g * in_sg + A * in_sA + S * in_sS + B);
    slab[i * 64 + tb] = v;
  }
  __syncthreads();
  if (!valid) return;
  const int rows = Gp * Dp;
  for (int o = ty; o < rows; o += 4) {
    const int b = rowptr[o], e = rowptr[o + 1];
    vec_t acc = (vec_t)(T(0));
    for (int z = b; z < e; ++z) acc += (T)vals[z] * slab[colidx[z] * 64 + tb];
    const int gp = o / Dp, Sp = o % Dp;
    *reinterpret_cast<vec_t*>(out + gp * out_sg + A * out_sA + Sp * out_sS + B) = acc;
  }
}

// The W step as an MFMA product: out[(g', S'), cols] = Op[(g', S'), (g, S)] *
// in[(g, S), cols] for one A index and a strip of columns.  Bound by HBM (the
// input read once, the output written once): the operator sits in LDS, and
// each wavefront streams strips on its own, without barriers: input rows go
// straight from global memory into MFMA operands (two columns per lane, five
// K steps on their way while five are multiplied) and the results straight
// out.  All output rows of a strip are accumulated at once (NMB blocks of 32
// rows, v_mfma_f32_32x32x2f32, or 16, v_mfma_f64_16x16x4f64).  A sparse
// operator costs its full M x K here and still stays under the HBM time; strips
// with a result that is not finite are done again entry by entry, so that its
// zeros do not spread an Inf or NaN (the check costs nothing measurable).
// K runs from the operator's last column to its first.  In place of a
// workgroup per 128 columns that staged operator and input in LDS, with the
// w = 20 pair operator: FP32 to bf16 pairs at chi = 2048 2.46 -> 0.85 ms
// (1.4 -> 4.0 TB/s), FP32 at chi = 4096 8.0 -> 2.65 ms, FP64 at chi = 255 39 ->
// 33 us (22 where pairs of columns are aligned).  In place of CSR rows from
// LDS: w = 5 at chi = 16 6.4 -> 4.7 us.
// SPLIT (T = float): the result goes out as bf16 hi/lo pairs (ohi, olo).
// VEC: nB and all strides are even and the bases two-element aligned.
typedef float f16v __attribute__((ext_vector_type(16)));
typedef double d4 __attribute__((ext_vector_type(4)));
constexpr int WM_PF = 5;  // K steps per group of loads

template <typename T>
struct WmArgs {
  int D, Dp, M, K, Kp;
  long nA, nB;
  unsigned nbt, strips;  // strips per A index, in all
  const T* in; long in_sg, in_sA, in_sS;
  T* out; long out_sg, out_sA, out_sS;
  const T* opd;
  unsigned short* ohi;
  unsigned short* olo;
};

template <typename T, bool SPLIT, bool VEC, int NMB>
__global__ __launch_bounds__(256, 2) void wstep_mfma_kernel(WmArgs<T> w) {
  constexpr bool F64 = sizeof(T) == 8;
  constexpr int MB = F64 ? 16 : 32, KS = F64 ? 4 : 2, NR = F64 ? 4 : 16, MP = NMB * MB;
  typedef T vec2 __attribute__((ext_vector_type(2)));
  typedef typename std::conditional<F64, d4, f16v>::type Acc;
  extern __shared__ __attribute__((aligned(16))) unsigned char wm_smem[];
  const int lda = w.Kp + 1;
  long* ioff = reinterpret_cast<long*>(wm_smem);  // Kp: input row offsets
  long* ooff = ioff + w.Kp;                       // MP: output row offsets
  T* Aop = reinterpret_cast<T*>(ooff + MP);       // MP x lda
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int ln = lane & (MB - 1), kg = lane / MB;
  const int nks = w.Kp / KS;
  const unsigned step = gridDim.x * 4;
  // offset of K index i's input row (the padding meets zero operator columns), a strip's
  // first column and one K step of its input at row offset off: this lane's two
  // columns, those past the end clamped (and not stored)
  auto row_offset = [&](int i) -> long {
    const int r = min(w.Kp - 1 - i, w.K - 1);
    return (r / w.D) * w.in_sg + (r % w.D) * w.in_sS;
  };
  auto first_col = [&](unsigned s) -> long { return (long)(s % w.nbt) * (2 * MB); };
  auto load = [&](unsigned s, long off) -> vec2 {
    const T* p = w.in + (s / w.nbt) * w.in_sA + off;
    const long c0 = first_col(s) + (VEC ? 2 * ln : ln);
    if constexpr (VEC) return *reinterpret_cast<const vec2*>(p + min(c0, w.nB - 2));
    else return vec2{p[min(c0, w.nB - 1)], p[min(c0 + MB, w.nB - 1)]};
  };
  // the first strip's first rows are on their way while the operator is staged
  unsigned s = blockIdx.x * 4 + wave;
  vec2 cur[WM_PF], nxt[WM_PF];
#pragma unroll
  for (int p = 0; p < WM_PF; ++p) cur[p] = load(min(s, w.strips - 1), row_offset(p * KS + kg));
  for (int m = wave; m < MP; m += 4)
    for (int k = lane; k < w.Kp; k += 64) Aop[m * lda + (w.Kp - 1 - k)] = (m < w.M && k < w.K) ? w.opd[m * w.K + k] : T(0);
  for (int i = tid; i < w.Kp; i += 256) ioff[i] = row_offset(i);
  for (int i = tid; i < MP; i += 256) ooff[i] = (i / w.Dp) * w.out_sg + (i % w.Dp) * w.out_sS;
  __syncthreads();
  const T* arow = Aop + ln * lda + kg;
  for (; s < w.strips; s += step) {
    const unsigned Ai = s / w.nbt;
    const long c0 = first_col(s) + (VEC ? 2 * ln : ln), c1 = VEC ? c0 + 1 : c0 + MB;
    Acc acc[NMB][2];
#pragma unroll
    for (int i = 0; i < NMB; ++i) acc[i][0] = acc[i][1] = Acc{};
    for (int k0 = 0; k0 < nks; k0 += WM_PF) {
      // the next group of rows, or the next strip's first
      const bool last = k0 + WM_PF >= nks;
      const unsigned sn = last ? min(s + step, w.strips - 1) : s;
      const int kn = last ? 0 : k0 + WM_PF;
#pragma unroll
      for (int p = 0; p < WM_PF; ++p) nxt[p] = load(sn, ioff[(kn + p) * KS + kg]);
#pragma unroll
      for (int p = 0; p < WM_PF; ++p) {
#pragma unroll
        for (int i = 0; i < NMB; ++i) {
          const T av = arow[i * MB * lda + (k0 + p) * KS];
          if constexpr (F64) {
            acc[i][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, cur[p][0], acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, cur[p][1], acc[i][1], 0, 0, 0);
          } else {
            acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, cur[p][0], acc[i][0], 0, 0, 0);
            acc[i][1] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, cur[p][1], acc[i][1], 0, 0, 0);
          }
        }
      }
#pragma unroll
      for (int p = 0; p < WM_PF; ++p) cur[p] = nxt[p];
    }
    const long obase = Ai * w.out_sA;
    auto put = [&](int row, T x0, T x1) {
      if (row >= w.M) return;
      const long off = ooff[row] + obase;
      if constexpr (SPLIT) {
        const unsigned short h0 = f2bf_rne(x0), h1 = f2bf_rne(x1);
        const unsigned short l0 = f2bf_rne(x0 - __uint_as_float(((unsigned int)h0) << 16));
        const unsigned short l1 = f2bf_rne(x1 - __uint_as_float(((unsigned int)h1) << 16));
        if constexpr (VEC) {
          if (c0 < w.nB) {
            *reinterpret_cast<unsigned int*>(w.ohi + off + c0) = (unsigned int)h0 | ((unsigned int)h1 << 16);
            *reinterpret_cast<unsigned int*>(w.olo + off + c0) = (unsigned int)l0 | ((unsigned int)l1 << 16);
          }
        } else {
          if (c0 < w.nB) { w.ohi[off + c0] = h0; w.olo[off + c0] = l0; }
          if (c1 < w.nB) { w.ohi[off + c1] = h1; w.olo[off + c1] = l1; }
        }
      } else if constexpr (VEC) {
        if (c0 < w.nB) *reinterpret_cast<vec2*>(w.out + off + c0) = vec2{x0, x1};
      } else {
        if (c0 < w.nB) w.out[off + c0] = x0;
        if (c1 < w.nB) w.out[off + c1] = x1;
      }
    };
    T nf0 = T(0), nf1 = T(0);  // NaN if any result is not finite
#pragma unroll
    for (int i = 0; i < NMB; ++i)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        nf0 = fma(acc[i][0][r], T(0), nf0);
        nf1 = fma(acc[i][1][r], T(0), nf1);
      }
    if (__any(nf0 + nf1 != T(0))) {
      // only the operator's entries may meet an Inf or NaN, not its zeros: the strip again, entry by entry
      for (int m = kg; m < w.M; m += 64 / MB) {
        T x0 = T(0), x1 = T(0);
        for (int i = w.Kp - w.K; i < w.Kp; ++i) {
          const T o = Aop[m * lda + i];
          if (o != T(0)) {
            const vec2 v = load(s, ioff[i]);
            x0 = fma(o, v[0], x0);
            x1 = fma(o, v[1], x1);
          }
        }
        put(m, x0, x1);
      }
      continue;
    }
    // register r of a lane: f64 row lane / 16 + 4 r; f32 row 8 (r / 4) + 4 (lane / 32) + r % 4
#pragma unroll
    for (int i = 0; i < NMB; ++i)
#pragma unroll
      for (int r = 0; r < NR; ++r)
        put(i * MB + (F64 ? kg + 4 * r : 8 * (r >> 2) + 4 * kg + (r & 3)), acc[i][0][r], acc[i][1][r]);
  }
}

// ---------------------------------------------------------------------------
// complex <-> real FP32 layouts of the complex mixed-precision product: a
// complex product C = A B runs as one real GEMM [Cr | Ci] = [Ar | Ai] *
// [[Br, Bi], [-Bi, Br]] (four real products' flops, FP32 MFMA)
// ---------------------------------------------------------------------------
// dst (rows x 2 cols): [re | im] of the interleaved complex src (rows x cols)
__global__ void cplx_split_rows_kernel(const double* __restrict__ src, long rows, long cols,
                                       float* __restrict__ dst) {
  const long n = rows * cols;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long r = i / cols, c = i % cols;
    dst[r * 2 * cols + c] = (float)src[2 * i];
    dst[r * 2 * cols + cols + c] = (float)src[2 * i + 1];
  }
}
// dst (2 rows x 2 cols) = [[re, im], [-im, re]] of the interleaved complex src
__global__ void cplx_block_kernel(const double* __restrict__ src, long rows, long cols, float* __restrict__ dst) {
  const long n = rows * cols;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long r = i / cols, c = i % cols;
    const float re = (float)src[2 * i], im = (float)src[2 * i + 1];
    dst[r * 2 * cols + c] = re;
    dst[r * 2 * cols + cols + c] = im;
    dst[(rows + r) * 2 * cols + c] = -im;
    dst[(rows + r) * 2 * cols + cols + c] = re;
  }
}
// interleaved complex dst (rows x cols) from src (rows x 2 cols) = [re | im]
__global__ void cplx_join_rows_kernel(const float* __restrict__ src, long rows, long cols,
                                      double* __restrict__ dst) {
  const long n = rows * cols;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long r = i / cols, c = i % cols;
    dst[2 * i] = (double)src[r * 2 * cols + c];
    dst[2 * i + 1] = (double)src[r * 2 * cols + cols + c];
  }
}

// ---------------------------------------------------------------------------
// conversions / fills
// ---------------------------------------------------------------------------
__global__ void cvt_d2f_kernel(const double* __restrict__ x, float* __restrict__ y, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = (float)x[i];
}
// rows x cols block with row strides lds (source) and ldd (destination);
// destination columns cols .. ldd - 1 are set to zero
__global__ void cvt_d2f_2d_kernel(const double* __restrict__ x, long rows, long cols, long lds,
                                  float* __restrict__ y, long ldd) {
  const long n = rows * ldd;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long r = i / ldd, c = i % ldd;
    y[i] = c < cols ? (float)x[r * lds + c] : 0.0f;
  }
}
// rows x cols FP64 block copied to row stride ldd, columns cols .. ldd - 1 zero
__global__ void pad_rows_f64_kernel(const double* __restrict__ x, long rows, long cols, long lds,
                                    double* __restrict__ y, long ldd) {
  const long n = rows * ldd;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x) {
    const long r = i / ldd, c = i % ldd;
    y[i] = c < cols ? x[r * lds + c] : 0.0;
  }
}
__global__ void zero_cols_f64_kernel(double* __restrict__ y, long rows, long c0, long c1, long ld) {
  const long w = c1 - c0, n = rows * w;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[(i / w) * ld + c0 + i % w] = 0.0;
}
// columns c0 .. c1 - 1 of a rows x ld FP32 matrix set to zero
__global__ void zero_cols_f32_kernel(float* __restrict__ y, long rows, long c0, long c1, long ld) {
  const long w = c1 - c0, n = rows * w;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[(i / w) * ld + c0 + i % w] = 0.0f;
}
__global__ void zero_cols_u16_kernel(unsigned short* __restrict__ y, long rows, long c0, long c1, long ld) {
  const long w = c1 - c0, n = rows * w;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[(i / w) * ld + c0 + i % w] = 0;
}
__global__ void cvt_f2d_kernel(const float* __restrict__ x, double* __restrict__ y, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = (double)x[i];
}
__global__ void fill_kernel(double* __restrict__ x, double v, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    x[i] = v;
}
__global__ void scaled_copy_kernel(double* __restrict__ y, const double* __restrict__ x, double a, long n) {
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += (long)gridDim.x * blockDim.x)
    y[i] = a * x[i];
}
// ---------------------------------------------------------------------------
// Krylov: multi-dot (first stage + fixed-order second stage)
// part[v * nblk + blk] = partial sum of <basis_v, x> over the block's slice.
// Complex: data are interleaved (re, im); <u, x> = sum conj(u) x -> two parts.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) { return wave_sum64(v); }

template <bool CPLX>
__global__ __launch_bounds__(RED_THREADS) void multidot_stage1(const double* __restrict__ basis, long ld,
                                                               int count, const double* __restrict__ x,
                                                               long n, double* __restrict__ part,
                                                               double* __restrict__ hout) {
  __shared__ double red[RED_THREADS / 64][2 * MAX_DOT];
  const int nblk = gridDim.x;
  double acc[2 * MAX_DOT];
#pragma unroll
  for (int v = 0; v < 2 * MAX_DOT; ++v) acc[v] = 0.0;
  const long stride = (long)gridDim.x * blockDim.x;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += stride) {
    if (!CPLX) {
      const double xi = x[i];
#pragma unroll
      for (int v = 0; v < MAX_DOT; ++v)
        if (v < count) acc[v] = fma(basis[v * ld + i], xi, acc[v]);
    } else {
      const double xr = x[2 * i], xi = x[2 * i + 1];
#pragma unroll
      for (int v = 0; v < MAX_DOT; ++v)
        if (v < count) {
          const double ur = basis[v * ld + 2 * i], ui = basis[v * ld + 2 * i + 1];
          acc[2 * v] = fma(ur, xr, fma(ui, xi, acc[2 * v]));
          acc[2 * v + 1] = fma(ur, xi, fma(-ui, xr, acc[2 * v + 1]));
        }
    }
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int nacc = CPLX ? 2 * count : count;
#pragma unroll
  for (int v = 0; v < 2 * MAX_DOT; ++v) {
    if (v < nacc) {
      double s = wave_sum(acc[v]);
      if (lane == 0) red[wave][v] = s;
    }
  }
  __syncthreads();
  for (int v = threadIdx.x; v < nacc; v += blockDim.x) {
    double s = 0.0;
    for (int w = 0; w < RED_THREADS / 64; ++w) s += red[w][v];
    part[(long)v * nblk + blockIdx.x] = s;
    if (hout) hout[v] = s;  // one-workgroup launch: s is the final value
  }
}

__global__ __launch_bounds__(256) void multidot_stage2(const double* __restrict__ part, int nblk,
                                                       int nacc, double* __restrict__ out,
                                                       double* __restrict__ hout) {
  __shared__ double red[4];
  const int v = blockIdx.x;
  if (v >= nacc) return;
  double s = 0.0;
  for (int i = threadIdx.x; i < nblk; i += blockDim.x) s += part[(long)v * nblk + i];
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    const double r = red[0] + red[1] + red[2] + red[3];
    out[v] = r;
    if (hout) hout[v] = r;
  }
}

// ---------------------------------------------------------------------------
// Krylov steps: w <- w - V (V^H w) twice over K basis vectors, |w|^2, and the
// next basis vector w / |w|.  Short vectors: one workgroup with w in
// registers.  Others: a launch per pass over V -- dots; update and the second
// pass's dots, from one read of V; update and norm; scaling -- where every
// workgroup sums the previous launch's partial sums for itself, or a launch in
// between sums them (KP_SELF_SUM), in a fixed order.  Bound by launches and load
// latency up to about 10^6 elements (n = 1.4 10^5, 10 vectors: V is 11 MB, 3
// us), so all loads of a tile are issued before the first is used.  A solve of 7
// steps at n = 137k took 750 us with nine launches a step (dots and their sums,
// update, twice; norm and its sum; scaling) and the start's norm read by the
// host, with four 590 us, with six 550; two-site sweeps of 20 spins, mostly
// short vectors, 58 -> 49 ms.
// ---------------------------------------------------------------------------
constexpr int KS_THREADS = 1024;  // one-workgroup step
constexpr int KP_TILE = 512;      // elements per tile of the others, two a thread
constexpr int KP_BLOCKS = 1024;
constexpr long KS_MAX = 4L * KS_THREADS;

// n <= EP * blockDim elements.  hout (mapped host memory) receives the passes'
// coefficients at 0 and 128 (pairs when CX) and |w|^2 at 256.  K = 0: norm and
// scaling only, w stays as it is.
template <bool CX, int EP>
__global__ __launch_bounds__(KS_THREADS) void krylov_small_kernel(const double* __restrict__ basis, long ld, int K,
                                                                  double* __restrict__ w, int n,
                                                                  double* __restrict__ vnext,
                                                                  double* __restrict__ hout) {
  constexpr int C = CX ? 2 : 1;
  constexpr int KS_CH = EP == 1 ? 8 : 4;  // basis vectors whose loads are in flight at once
  __shared__ double part[KS_THREADS / 64][128];
  __shared__ double cf[128];  // zero past the last vector, as far as whole chunks reach
  __shared__ double red[KS_THREADS / 64];
  const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nw = nt >> 6;
  const int nacc = C * K;
  double x[EP][C];
  int idx[EP];
#pragma unroll
  for (int e = 0; e < EP; ++e) {
    const int j = tid + nt * e;
    idx[e] = C * min(j, n - 1);
#pragma unroll
    for (int q = 0; q < C; ++q) {
      const double t = w[idx[e] + q];
      x[e][q] = j < n ? t : 0.0;
    }
  }
  for (int pass = 0; pass < 2 && K > 0; ++pass) {
    for (int v0 = 0; v0 < K; v0 += KS_CH) {
      double b[KS_CH][EP][C], acc[KS_CH][C];
#pragma unroll
      for (int u = 0; u < KS_CH; ++u)
#pragma unroll
        for (int e = 0; e < EP; ++e)
#pragma unroll
          for (int q = 0; q < C; ++q) b[u][e][q] = basis[min(v0 + u, K - 1) * ld + idx[e] + q];
#pragma unroll
      for (int u = 0; u < KS_CH; ++u) {
#pragma unroll
        for (int q = 0; q < C; ++q) acc[u][q] = 0.0;
#pragma unroll
        for (int e = 0; e < EP; ++e) {
          acc[u][0] = fma(b[u][e][0], x[e][0], acc[u][0]);
          if constexpr (CX) {
            acc[u][0] = fma(b[u][e][1], x[e][1], acc[u][0]);
            acc[u][1] = fma(b[u][e][0], x[e][1], fma(-b[u][e][1], x[e][0], acc[u][1]));
          }
        }
#pragma unroll
        for (int q = 0; q < C; ++q) acc[u][q] = wave_sum64(acc[u][q]);
      }
      if (lane == 0) {
#pragma unroll
        for (int u = 0; u < KS_CH; ++u)
#pragma unroll
          for (int q = 0; q < C; ++q) part[wave][C * (v0 + u) + q] = acc[u][q];
      }
    }
    __syncthreads();
    for (int t = tid; t < 128; t += nt) {
      double s = 0.0;
      if (t < nacc) {
        for (int k = 0; k < nw; ++k) s += part[k][t];
        hout[128 * pass + t] = s;
      }
      cf[t] = s;
    }
    __syncthreads();
    double sub[EP][C];
#pragma unroll
    for (int e = 0; e < EP; ++e)
#pragma unroll
      for (int q = 0; q < C; ++q) sub[e][q] = 0.0;
    for (int v0 = 0; v0 < K; v0 += KS_CH) {
      double b[KS_CH][EP][C];
#pragma unroll
      for (int u = 0; u < KS_CH; ++u)
#pragma unroll
        for (int e = 0; e < EP; ++e)
#pragma unroll
          for (int q = 0; q < C; ++q) b[u][e][q] = basis[min(v0 + u, K - 1) * ld + idx[e] + q];
#pragma unroll
      for (int u = 0; u < KS_CH; ++u)
#pragma unroll
        for (int e = 0; e < EP; ++e) {
          const double cr = cf[C * (v0 + u)];
          if constexpr (CX) {
            const double ci = cf[C * (v0 + u) + 1];
            sub[e][0] = fma(cr, b[u][e][0], fma(-ci, b[u][e][1], sub[e][0]));
            sub[e][1] = fma(cr, b[u][e][1], fma(ci, b[u][e][0], sub[e][1]));
          } else {
            sub[e][0] = fma(cr, b[u][e][0], sub[e][0]);
          }
        }
    }
#pragma unroll
    for (int e = 0; e < EP; ++e)
#pragma unroll
      for (int q = 0; q < C; ++q) x[e][q] = tid + nt * e < n ? x[e][q] - sub[e][q] : 0.0;
  }
  double s = 0.0;
#pragma unroll
  for (int e = 0; e < EP; ++e)
#pragma unroll
    for (int q = 0; q < C; ++q) s = fma(x[e][q], x[e][q], s);
  s = wave_sum64(s);
  if (lane == 0) red[wave] = s;
  __syncthreads();
  double r2 = 0.0;
  for (int k = 0; k < nw; ++k) r2 += red[k];
  if (tid == 0) hout[256] = r2;
  const double a = 1.0 / sqrt(fmax(0.0, r2));
#pragma unroll
  for (int e = 0; e < EP; ++e)
#pragma unroll
    for (int q = 0; q < C; ++q)
      if (tid + nt * e < n) {
        if (K > 0) w[idx[e] + q] = x[e][q];
        vnext[idx[e] + q] = a * x[e][q];
      }
}

// sums of the previous launch's partial results: 16 threads per value
__device__ __forceinline__ double sum_parts16(const double* __restrict__ pin, int np) {
  const int l = threadIdx.x & 15;
  double s = 0.0;
  for (int i = l; i < np; i += 16) s += pin[i];
#pragma unroll
  for (int o = 8; o > 0; o >>= 1) s += __shfl_xor(s, o, 16);
  return s;
}

// sums of np partial results each, one workgroup per value
__global__ __launch_bounds__(256) void krylov_sum_kernel(const double* __restrict__ pin, int np,
                                                         double* __restrict__ out) {
  __shared__ double red[4];
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += 256) s += pin[(long)blockIdx.x * np + i];
  s = wave_sum64(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}

// PHASE 0: dots of w with the basis vectors.  PHASE 1: their sums, w updated,
// dots of the new w.  PHASE 2: sums, update, |w|^2.  NV >= K, or 16 (then the
// dots of PHASE 1 read V once more).  Partial results of workgroup g at
// pout[value * gridDim.x + g], np of the previous launch per value at pin;
// hout: the coefficients of this phase.
template <bool CX, int PHASE, int NV>
__global__ __launch_bounds__(256) void krylov_pass_kernel(const double* __restrict__ basis, long ld, int K,
                                                          double* __restrict__ w, long n,
                                                          const double* __restrict__ pin, int np,
                                                          double* __restrict__ pout, double* __restrict__ hout) {
  constexpr int C = CX ? 2 : 1;
  __shared__ double cf[128];
  __shared__ double red[4][C * NV];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, nblk = gridDim.x;
  const int nacc = C * K;
  if constexpr (PHASE > 0) {
    if (tid < 128) cf[tid] = 0.0;
    __syncthreads();
    for (int v = tid >> 4; v < nacc; v += 16) {
      const double s = sum_parts16(pin + (long)v * np, np);
      if ((tid & 15) == 0) {
        cf[v] = s;
        if (blockIdx.x == 0) hout[v] = s;
      }
    }
    __syncthreads();
  }
  double acc[NV][C];
#pragma unroll
  for (int u = 0; u < NV; ++u)
#pragma unroll
    for (int q = 0; q < C; ++q) acc[u][q] = 0.0;
  double nrm = 0.0;
  auto load = [&](int v0, const long (&o)[2], double (&b)[NV][2][C]) {
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int q = 0; q < C; ++q) b[u][e][q] = basis[min(v0 + u, K - 1) * ld + o[e] + q];
  };
  auto dots = [&](const double (&b)[NV][2][C], const double (&x)[2][C]) {
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        acc[u][0] = fma(b[u][e][0], x[e][0], acc[u][0]);
        if constexpr (CX) {
          acc[u][0] = fma(b[u][e][1], x[e][1], acc[u][0]);
          acc[u][1] = fma(b[u][e][0], x[e][1], fma(-b[u][e][1], x[e][0], acc[u][1]));
        }
      }
  };
  auto offsets = [&](long i0, long (&o)[2]) {
    o[0] = C * min(i0 + tid, n - 1);
    o[1] = C * min(i0 + tid + 256, n - 1);
  };
  auto read = [&](long i0, const long (&o)[2], double (&x)[2][C]) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const double t = w[o[e] + q];
        x[e][q] = i0 + tid + 256 * e < n ? t : 0.0;
      }
  };
  auto flush = [&](int v0) {  // this workgroup's sums of the dots with vectors v0 ..
#pragma unroll
    for (int u = 0; u < NV; ++u)
#pragma unroll
      for (int q = 0; q < C; ++q) {
        const double s = wave_sum64(acc[u][q]);
        if (lane == 0) red[wave][C * u + q] = s;
        acc[u][q] = 0.0;
      }
    __syncthreads();
    for (int t = tid; t < C * NV; t += 256)
      if (C * v0 + t < nacc)
        pout[(long)(C * v0 + t) * nblk + blockIdx.x] = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
    __syncthreads();
  };
  const long step = (long)nblk * KP_TILE;
  const bool one = K <= NV;
  if (PHASE > 0 || one) {
    for (long i0 = (long)blockIdx.x * KP_TILE; i0 < n; i0 += step) {
      long o[2];
      double x[2][C], b[NV][2][C];
      offsets(i0, o);
      read(i0, o, x);
      if constexpr (PHASE == 0) {
        load(0, o, b);
      } else {
        double sub[2][C];
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int q = 0; q < C; ++q) sub[e][q] = 0.0;
        for (int v0 = 0; v0 < K; v0 += NV) {
          load(v0, o, b);
#pragma unroll
          for (int u = 0; u < NV; ++u)
#pragma unroll
            for (int e = 0; e < 2; ++e) {
              const double cr = cf[C * (v0 + u)];
              if constexpr (CX) {
                const double ci = cf[C * (v0 + u) + 1];
                sub[e][0] = fma(cr, b[u][e][0], fma(-ci, b[u][e][1], sub[e][0]));
                sub[e][1] = fma(cr, b[u][e][1], fma(ci, b[u][e][0], sub[e][1]));
              } else {
                sub[e][0] = fma(cr, b[u][e][0], sub[e][0]);
              }
            }
        }
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int q = 0; q < C; ++q)
            if (i0 + tid + 256 * e < n) {
              x[e][q] -= sub[e][q];
              w[o[e] + q] = x[e][q];
            }
      }
      if constexpr (PHASE == 2) {
#pragma unroll
        for (int e = 0; e < 2; ++e)
#pragma unroll
          for (int q = 0; q < C; ++q) nrm = fma(x[e][q], x[e][q], nrm);
      } else if (one) {
        dots(b, x);
      }
    }
  }
  if constexpr (PHASE < 2) {
    if (one) {
      flush(0);
    } else {
      for (int v0 = 0; v0 < K; v0 += NV) {
        for (long i0 = (long)blockIdx.x * KP_TILE; i0 < n; i0 += step) {
          long o[2];
          double x[2][C], b[NV][2][C];
          offsets(i0, o);
          read(i0, o, x);
          load(v0, o, b);
          dots(b, x);
        }
        flush(v0);
      }
    }
  } else {
    nrm = wave_sum64(nrm);
    if (lane == 0) red[wave][0] = nrm;
    __syncthreads();
    if (tid == 0) pout[blockIdx.x] = (red[0][0] + red[1][0]) + (red[2][0] + red[3][0]);
  }
}

// out = sum_v co[v] V_v (pairs when CX); norm: with the partial sums of |out|^2
struct KryCoef {
  double c[128];
};
template <bool CX>
__global__ __launch_bounds__(256) void krylov_combine_kernel(const double* __restrict__ basis, long ld, int K,
                                                             KryCoef co, double* __restrict__ out, long n,
                                                             double* __restrict__ pout) {
  constexpr int C = CX ? 2 : 1;
  __shared__ double red[4];
  double nrm = 0.0;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += gridDim.x * 256L) {
    double a[C];
#pragma unroll
    for (int q = 0; q < C; ++q) a[q] = 0.0;
    for (int v = 0; v < K; ++v) {
      const double* b = basis + v * ld + C * i;
      if constexpr (CX) {
        const double br = b[0], bi = b[1], cr = co.c[2 * v], ci = co.c[2 * v + 1];
        a[0] = fma(cr, br, fma(-ci, bi, a[0]));
        a[1] = fma(cr, bi, fma(ci, br, a[1]));
      } else {
        a[0] = fma(co.c[v], b[0], a[0]);
      }
    }
#pragma unroll
    for (int q = 0; q < C; ++q) {
      out[C * i + q] = a[q];
      nrm = fma(a[q], a[q], nrm);
    }
  }
  if (!pout) return;  // uniform over the grid
  nrm = wave_sum64(nrm);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = nrm;
  __syncthreads();
  if (threadIdx.x == 0) pout[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}
__global__ __launch_bounds__(256) void krylov_norm_kernel(const double* __restrict__ x, long nd,
                                                          double* __restrict__ pout) {
  __shared__ double red[4];
  double s = 0.0;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < nd; i += gridDim.x * 256L) s = fma(x[i], x[i], s);
  s = wave_sum64(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) pout[blockIdx.x] = (red[0] + red[1]) + (red[2] + red[3]);
}
// y = x / |x| from the partial sums of |x|^2 (y may be x)
__global__ __launch_bounds__(256) void krylov_scale_kernel(double* y, const double* x, long nd,
                                                           const double* __restrict__ pin, int np,
                                                           double* __restrict__ hout) {
  __shared__ double red[4];
  double s = 0.0;
  for (int i = threadIdx.x; i < np; i += 256) s += pin[i];
  s = wave_sum64(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  const double r2 = (red[0] + red[1]) + (red[2] + red[3]);
  if (hout && blockIdx.x == 0 && threadIdx.x == 0) *hout = r2;
  const double a = 1.0 / sqrt(fmax(0.0, r2));
  for (long i = blockIdx.x * 256L + threadIdx.x; i < nd; i += gridDim.x * 256L) y[i] = a * x[i];
}

// row sums of squares: one block per row
__global__ __launch_bounds__(256) void row_norms2_kernel(const double* __restrict__ X, long L, long ld,
                                                         double* __restrict__ out) {
  __shared__ double red[4];
  const long r = blockIdx.x;
  double s = 0.0;
  for (long j = threadIdx.x; j < L; j += blockDim.x) {
    const double v = X[r * ld + j];
    s = fma(v, v, s);
  }
  s = wave_sum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) out[r] = red[0] + red[1] + red[2] + red[3];
}

// out (C x R) = in^T, in is R x C; 32x32 LDS tiles
__global__ __launch_bounds__(256) void transpose_kernel(const double* __restrict__ in, long R, long C,
                                                        double* __restrict__ out) {
  __shared__ double t[32][33];
  const long r0 = (long)blockIdx.y * 32, c0 = (long)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  for (int k = ty; k < 32; k += 8) {
    const long r = r0 + k, cc = c0 + tx;
    t[k][tx] = (r < R && cc < C) ? in[r * C + cc] : 0.0;
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const long cc = c0 + k, r = r0 + tx;
    if (cc < C && r < R) out[cc * R + r] = t[tx][k];
  }
}

__global__ __launch_bounds__(256) void gather_rows_kernel(const double* __restrict__ src, long ld,
                                                          const int* __restrict__ perm,
                                                          const double* __restrict__ scale, long L,
                                                          double* __restrict__ out) {
  const long k = blockIdx.y;
  const long j = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (j < L) out[k * L + j] = src[(long)perm[k] * ld + j] * scale[k];
}

// out[j][k] = src[perm[k]][j] * scale[k]; 32x32 tiles through LDS
__global__ __launch_bounds__(256) void gather_rows_T_kernel(const double* __restrict__ src, long ld,
                                                            const int* __restrict__ perm,
                                                            const double* __restrict__ scale, long kcount,
                                                            long L, double* __restrict__ out) {
  __shared__ double t[32][33];
  const long k0 = (long)blockIdx.y * 32, j0 = (long)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int a = ty; a < 32; a += 8) {
    const long k = k0 + a, j = j0 + tx;
    t[a][tx] = (k < kcount && j < L) ? src[(long)perm[k] * ld + j] * scale[k] : 0.0;
  }
  __syncthreads();
  for (int a = ty; a < 32; a += 8) {
    const long j = j0 + a, k = k0 + tx;
    if (j < L && k < kcount) out[j * kcount + k] = t[tx][a];
  }
}

// complex: out[j][k] = conj?(src[perm[k]][j]) * scale[k]; 16x16 complex tiles
__global__ __launch_bounds__(256) void gather_rows_T_z_kernel(const double2* __restrict__ src, long ld,
                                                              const int* __restrict__ perm,
                                                              const double* __restrict__ scale, long kcount,
                                                              long L, double2* __restrict__ out, int conj) {
  __shared__ double2 t[16][17];
  const long k0 = (long)blockIdx.y * 16, j0 = (long)blockIdx.x * 16;
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;  // 16 x 16
  {
    const long k = k0 + ty, j = j0 + tx;
    double2 v = make_double2(0.0, 0.0);
    if (k < kcount && j < L) {
      v = src[(long)perm[k] * ld + j];
      if (conj) v.y = -v.y;
      v.x *= scale[k];
      v.y *= scale[k];
    }
    t[ty][tx] = v;
  }
  __syncthreads();
  const long j = j0 + ty, k = k0 + tx;
  if (j < L && k < kcount) out[j * kcount + k] = t[tx][ty];
}

inline int grid1d(long n, int threads = 256) {
  long g = (n + threads - 1) / threads;
  if (g > 4096) g = 4096;
  if (g < 1) g = 1;
  return (int)g;
}

}  // namespace

// ---------------------------------------------------------------------------
void build_sparse_op(SparseOp& op, int rows, int cols, const std::vector<double>& dense) {
  std::vector<int> rp(rows + 1, 0), ci;
  std::vector<double> v;
  for (int r = 0; r < rows; ++r) {
    for (int c = 0; c < cols; ++c) {
      const double x = dense[(size_t)r * cols + c];
      if (x != 0.0) { ci.push_back(c); v.push_back(x); }
    }
    rp[r + 1] = (int)ci.size();
  }
  op.rows = rows;
  op.cols = cols;
  op.nnz = (int)ci.size();
  op.mat = rows <= 128 && cols <= 128;
  op.dense = op.mat && op.nnz >= 8 * rows;
  // one allocation and one copy: values, FP64 matrix, FP32 matrix, row starts, columns
  const size_t n = v.size(), nm = op.mat ? (size_t)rows * cols : 0;
  op.o_d64 = n * sizeof(double);
  op.o_d32 = op.o_d64 + nm * sizeof(double);
  op.o_rp = op.o_d32 + nm * sizeof(float);
  op.o_ci = op.o_rp + rp.size() * sizeof(int);
  std::vector<unsigned char> h(op.o_ci + n * sizeof(int));
  std::copy_n(v.data(), n, reinterpret_cast<double*>(h.data()));
  std::copy_n(dense.data(), nm, reinterpret_cast<double*>(h.data() + op.o_d64));
  std::copy_n(dense.data(), nm, reinterpret_cast<float*>(h.data() + op.o_d32));
  std::copy_n(rp.data(), rp.size(), reinterpret_cast<int*>(h.data() + op.o_rp));
  std::copy_n(ci.data(), n, reinterpret_cast<int*>(h.data() + op.o_ci));
  op.buf.ensure(h.size());
  TN_HIP(hipMemcpy(op.buf.p, h.data(), h.size(), hipMemcpyHostToDevice));
}

namespace {
template <typename T, bool SPLIT, bool VEC, int NMB>
void launch_wm(tn_ctx* c, const WmArgs<T>& a) {
  constexpr int MP = NMB * (sizeof(T) == 8 ? 16 : 32);
  const size_t shm = ((size_t)a.Kp + MP) * sizeof(long) + (size_t)MP * (a.Kp + 1) * sizeof(T);
  raise_lds_limit((const void*)wstep_mfma_kernel<T, SPLIT, VEC, NMB>, shm);
  // wavefronts take strips until all are done: enough workgroups for three per CU
  const unsigned wg = std::min<unsigned>((a.strips + 3) / 4, 768);
  hipLaunchKernelGGL((wstep_mfma_kernel<T, SPLIT, VEC, NMB>), dim3(wg), dim3(256), shm, c->stream, a);
}
template <typename T, bool SPLIT, bool VEC>
void launch_wm_rows(tn_ctx* c, const WmArgs<T>& a) {
  const int nmb = (a.M + (sizeof(T) == 8 ? 15 : 31)) / (sizeof(T) == 8 ? 16 : 32);
  if constexpr (sizeof(T) == 8) {
    if (nmb <= 2) launch_wm<T, SPLIT, VEC, 2>(c, a);
    else if (nmb <= 4) launch_wm<T, SPLIT, VEC, 4>(c, a);
    else if (nmb <= 5) launch_wm<T, SPLIT, VEC, 5>(c, a);
    else if (nmb <= 6) launch_wm<T, SPLIT, VEC, 6>(c, a);
    else launch_wm<T, SPLIT, VEC, 8>(c, a);
  } else {
    if (nmb <= 1) launch_wm<T, SPLIT, VEC, 1>(c, a);
    else if (nmb <= 2) launch_wm<T, SPLIT, VEC, 2>(c, a);
    else if (nmb <= 3) launch_wm<T, SPLIT, VEC, 3>(c, a);
    else launch_wm<T, SPLIT, VEC, 4>(c, a);
  }
  TN_HIP(hipGetLastError());
}
template <typename T, bool SPLIT>
void wstep_mfma(tn_ctx* c, const WStepDesc& w, const T* opd, bool vec, unsigned short* hi, unsigned short* lo) {
  constexpr int CW = sizeof(T) == 8 ? 32 : 64, KG = (sizeof(T) == 8 ? 4 : 2) * WM_PF;
  WmArgs<T> a;
  a.D = w.D; a.Dp = w.Dp; a.M = w.Gp * w.Dp; a.K = w.G * w.D;
  a.Kp = (a.K + KG - 1) / KG * KG;
  a.nA = w.nA; a.nB = w.nB;
  const long nbt = (w.nB + CW - 1) / CW;
  TN_REQUIRE(nbt * w.nA < (1L << 31), TN_E_INVALID, "wstep: too many columns");
  a.nbt = (unsigned)nbt; a.strips = (unsigned)(nbt * w.nA);
  a.in = (const T*)w.in; a.in_sg = w.in_sg; a.in_sA = w.in_sA; a.in_sS = w.in_sS;
  a.out = (T*)w.out; a.out_sg = w.out_sg; a.out_sA = w.out_sA; a.out_sS = w.out_sS;
  a.opd = opd; a.ohi = hi; a.olo = lo;
  if (vec) launch_wm_rows<T, SPLIT, true>(c, a);
  else launch_wm_rows<T, SPLIT, false>(c, a);
}
}  // namespace

static void wstep_launch(tn_ctx* c, bool fp32, bool split, const WStepDesc& w, unsigned short* hi,
                         unsigned short* lo) {
  TN_REQUIRE(w.op && w.op->rows == w.Gp * w.Dp && w.op->cols == w.G * w.D, TN_E_SHAPE,
             "wstep: operator shape mismatch");
  if (w.nA == 0 || w.nB == 0) return;
  const int K = w.G * w.D;
  const int* rp = w.op->rowptr();
  const int* ci = w.op->colidx();
  const double* vv = w.op->vals();
  // the MFMA product, except for operators past its 128 rows or columns and
  // for inputs with undefined values where the operator is zero
  if (w.op->mat && !w.csr) {
    auto even = [](long x) { return x % 2 == 0; };
    const size_t es = fp32 ? sizeof(float) : sizeof(double), os = split ? 2 : es;
    const void* out0 = split ? (const void*)hi : w.out;
    const bool vec = even(w.nB) && even(w.in_sg) && even(w.in_sA) && even(w.in_sS) && even(w.out_sg) &&
                     even(w.out_sA) && even(w.out_sS) && (uintptr_t)w.in % (2 * es) == 0 &&
                     (uintptr_t)out0 % (2 * os) == 0 && (!split || (uintptr_t)lo % 4 == 0);
    if (split) wstep_mfma<float, true>(c, w, w.op->d32(), vec, hi, lo);
    else if (fp32) wstep_mfma<float, false>(c, w, w.op->d32(), vec, nullptr, nullptr);
    else wstep_mfma<double, false>(c, w, w.op->d64(), vec, nullptr, nullptr);
    return;
  }
  TN_REQUIRE(w.nA <= 65535L, TN_E_INVALID, "wstep: nA exceeds grid.y");
  if (!split) {
    // 16-byte vectors along B when every offset allows them and the slab fits
    const int vec = fp32 ? 4 : 2;
    const size_t es = fp32 ? sizeof(float) : sizeof(double);
    const size_t vshm = (size_t)K * 64 * vec * es;
    auto ok = [&](long x) { return x % vec == 0; };
    if (w.nB >= 64 * vec && ok(w.nB) && ok(w.in_sg) && ok(w.in_sA) && ok(w.in_sS) && ok(w.out_sg) &&
        ok(w.out_sA) && ok(w.out_sS) && (uintptr_t)w.in % 16 == 0 && (uintptr_t)w.out % 16 == 0 &&
        vshm <= 160 * 1024) {
      dim3 grid((unsigned)((w.nB / vec + 63) / 64), (unsigned)w.nA);
      if (fp32) {
        raise_lds_limit((const void*)wstep_vec_kernel<float, 4>, vshm);
        hipLaunchKernelGGL((wstep_vec_kernel<float, 4>), grid, dim3(256), vshm, c->stream, w.G, w.Gp, w.D, w.Dp,
                           w.nB, (const float*)w.in, w.in_sg, w.in_sA, w.in_sS, (float*)w.out, w.out_sg, w.out_sA,
                           w.out_sS, rp, ci, vv);
      } else {
        raise_lds_limit((const void*)wstep_vec_kernel<double, 2>, vshm);
        hipLaunchKernelGGL((wstep_vec_kernel<double, 2>), grid, dim3(256), vshm, c->stream, w.G, w.Gp, w.D, w.Dp,
                           w.nB, (const double*)w.in, w.in_sg, w.in_sA, w.in_sS, (double*)w.out, w.out_sg,
                           w.out_sA, w.out_sS, rp, ci, vv);
      }
      TN_HIP(hipGetLastError());
      return;
    }
  }
  const size_t shm = (size_t)K * 64 * (fp32 ? sizeof(float) : sizeof(double));
  TN_REQUIRE(shm <= 64 * 1024, TN_E_UNSUPPORTED, "wstep: MPO slab exceeds 64 KiB of LDS");
  dim3 grid((unsigned)((w.nB + 63) / 64), (unsigned)w.nA);
  if (split)
    hipLaunchKernelGGL((wstep_kernel<float, true>), grid, dim3(256), shm, c->stream, w.G, w.Gp, w.D, w.Dp, w.nA,
                       w.nB, (const float*)w.in, w.in_sg, w.in_sA, w.in_sS, (float*)nullptr, w.out_sg, w.out_sA,
                       w.out_sS, rp, ci, vv, hi, lo);
  else if (fp32)
    hipLaunchKernelGGL((wstep_kernel<float, false>), grid, dim3(256), shm, c->stream, w.G, w.Gp, w.D, w.Dp, w.nA,
                       w.nB, (const float*)w.in, w.in_sg, w.in_sA, w.in_sS, (float*)w.out, w.out_sg, w.out_sA,
                       w.out_sS, rp, ci, vv, (unsigned short*)nullptr, (unsigned short*)nullptr);
  else
    hipLaunchKernelGGL((wstep_kernel<double, false>), grid, dim3(256), shm, c->stream, w.G, w.Gp, w.D, w.Dp, w.nA,
                       w.nB, (const double*)w.in, w.in_sg, w.in_sA, w.in_sS, (double*)w.out, w.out_sg, w.out_sA,
                       w.out_sS, rp, ci, vv, (unsigned short*)nullptr, (unsigned short*)nullptr);
  TN_HIP(hipGetLastError());
}

void wstep(tn_ctx* c, bool fp32, const WStepDesc& w) { wstep_launch(c, fp32, false, w, nullptr, nullptr); }

void wstep_split(tn_ctx* c, const WStepDesc& w, unsigned short* hi, unsigned short* lo) {
  wstep_launch(c, true, true, w, hi, lo);
}

void cvt_f64_to_f32(tn_ctx* c, const double* x, float* y, long n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(cvt_d2f_kernel, dim3(grid1d(n)), dim3(256), 0, c->stream, x, y, n);
  TN_HIP(hipGetLastError());
}
void cvt_f64_to_f32_2d(tn_ctx* c, const double* x, long rows, long cols, long lds, float* y, long ldd) {
  if (rows * cols <= 0) return;
  if (lds == cols && ldd == cols) {
    cvt_f64_to_f32(c, x, y, rows * cols);
    return;
  }
  hipLaunchKernelGGL(cvt_d2f_2d_kernel, dim3(grid1d(rows * ldd)), dim3(256), 0, c->stream, x, rows, cols, lds, y,
                     ldd);
  TN_HIP(hipGetLastError());
}
void pad_rows_f64(tn_ctx* c, const double* x, long rows, long cols, long lds, double* y, long ldd) {
  if (rows * ldd <= 0) return;
  hipLaunchKernelGGL(pad_rows_f64_kernel, dim3(grid1d(rows * ldd)), dim3(256), 0, c->stream, x, rows, cols, lds, y,
                     ldd);
  TN_HIP(hipGetLastError());
}
void zero_cols_f64(tn_ctx* c, double* y, long rows, long c0, long c1, long ld) {
  if (rows <= 0 || c1 <= c0) return;
  hipLaunchKernelGGL(zero_cols_f64_kernel, dim3(grid1d(rows * (c1 - c0))), dim3(256), 0, c->stream, y, rows, c0, c1,
                     ld);
  TN_HIP(hipGetLastError());
}
void zero_cols_f32(tn_ctx* c, float* y, long rows, long c0, long c1, long ld) {
  if (rows <= 0 || c1 <= c0) return;
  hipLaunchKernelGGL(zero_cols_f32_kernel, dim3(grid1d(rows * (c1 - c0))), dim3(256), 0, c->stream, y, rows, c0, c1,
                     ld);
  TN_HIP(hipGetLastError());
}
void zero_cols_u16(tn_ctx* c, unsigned short* y, long rows, long c0, long c1, long ld) {
  if (rows <= 0 || c1 <= c0) return;
  hipLaunchKernelGGL(zero_cols_u16_kernel, dim3(grid1d(rows * (c1 - c0))), dim3(256), 0, c->stream, y, rows, c0, c1,
                     ld);
  TN_HIP(hipGetLastError());
}
void cvt_f32_to_f64(tn_ctx* c, const float* x, double* y, long n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(cvt_f2d_kernel, dim3(grid1d(n)), dim3(256), 0, c->stream, x, y, n);
  TN_HIP(hipGetLastError());
}
void cplx_split_rows_f32(tn_ctx* c, const double* src, long rows, long cols, float* dst) {
  if (rows * cols <= 0) return;
  hipLaunchKernelGGL(cplx_split_rows_kernel, dim3(grid1d(rows * cols)), dim3(256), 0, c->stream, src, rows, cols,
                     dst);
  TN_HIP(hipGetLastError());
}
void cplx_block_f32(tn_ctx* c, const double* src, long rows, long cols, float* dst) {
  if (rows * cols <= 0) return;
  hipLaunchKernelGGL(cplx_block_kernel, dim3(grid1d(rows * cols)), dim3(256), 0, c->stream, src, rows, cols, dst);
  TN_HIP(hipGetLastError());
}
void cplx_join_rows_f64(tn_ctx* c, const float* src, long rows, long cols, double* dst) {
  if (rows * cols <= 0) return;
  hipLaunchKernelGGL(cplx_join_rows_kernel, dim3(grid1d(rows * cols)), dim3(256), 0, c->stream, src, rows, cols,
                     dst);
  TN_HIP(hipGetLastError());
}
void fill_f64(tn_ctx* c, double* x, double v, long n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(fill_kernel, dim3(grid1d(n)), dim3(256), 0, c->stream, x, v, n);
  TN_HIP(hipGetLastError());
}
void copy_f64(tn_ctx* c, double* dst, const double* src, long n) {
  if (n <= 0) return;
  TN_HIP(hipMemcpyAsync(dst, src, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
}
void scale_f64(tn_ctx* c, double* x, double s, long n) { scaled_copy(c, x, x, s, n); }
void scaled_copy(tn_ctx* c, double* y, const double* x, double a, long n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(scaled_copy_kernel, dim3(grid1d(n)), dim3(256), 0, c->stream, y, x, a, n);
  TN_HIP(hipGetLastError());
}
void multi_dot(tn_ctx* c, const double* basis, long ld, int count, const double* x, long n, bool cplx,
               double* out_dev, double* out_host) {
  TN_REQUIRE(count >= 1, TN_E_INVALID, "multi_dot: count");
  // short vectors (small bonds): one workgroup sums everything and writes
  // the results itself (part[v * 1 + 0] is out[v]), so no second launch
  const bool one = n <= 16L * RED_THREADS;
  const int nblk = one ? 1 : (int)std::min<long>(RED_BLOCKS, std::max<long>(1, (n + RED_THREADS - 1) / RED_THREADS));
  double* part = one ? nullptr : (double*)c->workspace(WS_KRY_PART, (size_t)2 * MAX_DOT * nblk * sizeof(double));
  for (int v0 = 0; v0 < count; v0 += MAX_DOT) {
    const int cnt = std::min(MAX_DOT, count - v0);
    const int nacc = cplx ? 2 * cnt : cnt;
    double* o = out_dev + (cplx ? 2 * v0 : v0);
    double* ho = out_host ? out_host + (cplx ? 2 * v0 : v0) : nullptr;
    double* dst = one ? o : part;
    double* hdst = one ? ho : nullptr;
    if (cplx)
      hipLaunchKernelGGL(multidot_stage1<true>, dim3(nblk), dim3(RED_THREADS), 0, c->stream, basis + v0 * ld,
                         ld, cnt, x, n, dst, hdst);
    else
      hipLaunchKernelGGL(multidot_stage1<false>, dim3(nblk), dim3(RED_THREADS), 0, c->stream, basis + v0 * ld,
                         ld, cnt, x, n, dst, hdst);
    TN_HIP(hipGetLastError());
    if (one) continue;
    hipLaunchKernelGGL(multidot_stage2, dim3(nacc), dim3(256), 0, c->stream, part, nblk, nacc, o, ho);
    TN_HIP(hipGetLastError());
  }
}

namespace {
// y += scale * coef[0] * x (coef on the device; complex pair when cplx)
__global__ __launch_bounds__(256) void add_scaled_dev_kernel(double* __restrict__ y, const double* __restrict__ x,
                                                             const double* __restrict__ coef, double scale, long n,
                                                             int cplx) {
  const double cr = scale * coef[0], ci = cplx ? scale * coef[1] : 0.0;
  const long stride = (long)gridDim.x * blockDim.x;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < n; i += stride) {
    if (!cplx) {
      y[i] = fma(cr, x[i], y[i]);
    } else {
      const double xr = x[2 * i], xi = x[2 * i + 1];
      y[2 * i] += cr * xr - ci * xi;
      y[2 * i + 1] += cr * xi + ci * xr;
    }
  }
}

}  // namespace

void add_scaled_dev(tn_ctx* c, double* y, const double* x, const double* coef_dev, double scale, long n, bool cplx) {
  if (n <= 0) return;
  hipLaunchKernelGGL(add_scaled_dev_kernel, dim3(grid1d(n)), dim3(256), 0, c->stream, y, x, coef_dev, scale, n,
                     cplx ? 1 : 0);
  TN_HIP(hipGetLastError());
}

// |x|^2 partial sums per workgroup, and workgroups of a scaling
static int krylov_blocks(long n) { return (int)std::min<long>(KP_BLOCKS, std::max<long>(1, (n + KP_TILE - 1) / KP_TILE)); }

template <bool CX>
static bool krylov_small(tn_ctx* c, const double* basis, long ld, int K, double* w, long n, double* vnext,
                         double* hout) {
  if (n > KS_MAX) return false;
  // one element a thread, or four
  if (n <= KS_THREADS)
    hipLaunchKernelGGL((krylov_small_kernel<CX, 1>), dim3(1), dim3((unsigned)((n + 63) / 64 * 64)), 0, c->stream, basis,
                       ld, K, w, (int)n, vnext, hout);
  else
    hipLaunchKernelGGL((krylov_small_kernel<CX, 4>), dim3(1), dim3(KS_THREADS), 0, c->stream, basis, ld, K, w, (int)n,
                       vnext, hout);
  TN_HIP(hipGetLastError());
  return true;
}

// Partial results a value up to which the next launch's workgroups sum them
// each for itself; more take a launch of their own, since all workgroups
// together read values * np^2 of them.  Kernel times of a solve, us, summed by
// the passes and by launches of their own: real 14 400 elements and 10 vectors
// (np 29) 173 and 222, complex 40 000 and 30 (79) 1068 and 1189; real 137 000
// and 10 (268) 295 and 255, complex 160 000 and 30 (313) 2670 and 1810, complex
// 600 000 and 10 (1024) 1180 and 647, and 30 9810 and 4050.
constexpr int KP_SELF_SUM = 128;

template <bool CX, int NV>
static void krylov_passes(tn_ctx* c, const double* basis, long ld, int K, double* w, long n, int nb, double* p1,
                          double* p2, double* p3, double* sums, double* hout) {
  const dim3 g(nb), b(256);
  const bool self = nb <= KP_SELF_SUM;
  auto summed = [&](double* p) {
    if (self) return p;
    hipLaunchKernelGGL(krylov_sum_kernel, dim3(CX ? 2 * K : K), b, 0, c->stream, (const double*)p, nb, sums);
    return sums;
  };
  const int np = self ? nb : 1;
  hipLaunchKernelGGL((krylov_pass_kernel<CX, 0, NV>), g, b, 0, c->stream, basis, ld, K, w, n, nullptr, 0, p1, nullptr);
  const double* s1 = summed(p1);
  hipLaunchKernelGGL((krylov_pass_kernel<CX, 1, NV>), g, b, 0, c->stream, basis, ld, K, w, n, s1, np, p2, hout);
  const double* s2 = summed(p2);
  hipLaunchKernelGGL((krylov_pass_kernel<CX, 2, NV>), g, b, 0, c->stream, basis, ld, K, w, n, s2, np, p3, hout + 128);
  TN_HIP(hipGetLastError());
}

template <bool CX>
static void krylov_step_t(tn_ctx* c, const double* basis, long ld, int K, double* w, long n, double* vnext,
                          double* hout) {
  if (krylov_small<CX>(c, basis, ld, K, w, n, vnext, hout)) return;
  const int nb = krylov_blocks(n), nacc = CX ? 2 * K : K;
  const long nd = CX ? 2 * n : n;
  double* p1 = (double*)c->workspace(WS_KRY_PART, ((size_t)(2 * nacc + 1) * nb + nacc) * sizeof(double));
  double* p2 = p1 + (size_t)nacc * nb;
  double* p3 = p2 + (size_t)nacc * nb;
  double* sums = p3 + nb;
  if (K <= 4) krylov_passes<CX, 4>(c, basis, ld, K, w, n, nb, p1, p2, p3, sums, hout);
  else if (K <= 8) krylov_passes<CX, 8>(c, basis, ld, K, w, n, nb, p1, p2, p3, sums, hout);
  else krylov_passes<CX, 16>(c, basis, ld, K, w, n, nb, p1, p2, p3, sums, hout);
  hipLaunchKernelGGL(krylov_scale_kernel, dim3(grid1d(nd)), dim3(256), 0, c->stream, vnext, (const double*)w, nd,
                     (const double*)p3, nb, hout + 256);
  TN_HIP(hipGetLastError());
}

void krylov_step(tn_ctx* c, const double* basis, long ld, int K, double* w, long n, bool cplx, double* vnext,
                 double* hout) {
  TN_REQUIRE(K >= 1 && K <= KRY_MAX && n >= 1, TN_E_INVALID, "Krylov step: basis size");
  if (cplx) krylov_step_t<true>(c, basis, ld, K, w, n, vnext, hout);
  else krylov_step_t<false>(c, basis, ld, K, w, n, vnext, hout);
}

void krylov_normalize(tn_ctx* c, double* y, const double* x, long nd, double* hout) {
  // the one-workgroup step without basis vectors leaves x as it is
  if (krylov_small<false>(c, nullptr, 0, 0, const_cast<double*>(x), nd, y, hout - 256)) return;
  const int nb = krylov_blocks(nd);
  double* p = (double*)c->workspace(WS_KRY_PART, (size_t)nb * sizeof(double));
  hipLaunchKernelGGL(krylov_norm_kernel, dim3(nb), dim3(256), 0, c->stream, x, nd, p);
  hipLaunchKernelGGL(krylov_scale_kernel, dim3(grid1d(nd)), dim3(256), 0, c->stream, y, x, nd, (const double*)p, nb,
                     hout);
  TN_HIP(hipGetLastError());
}

void krylov_combine(tn_ctx* c, const double* basis, long ld, int K, const double* co, double* out, long n, bool cplx,
                    bool normalize) {
  TN_REQUIRE(K >= 1 && K <= KRY_MAX && n >= 1, TN_E_INVALID, "Krylov combination: basis size");
  KryCoef kc{};
  std::copy(co, co + (cplx ? 2 * K : K), kc.c);
  const int nb = krylov_blocks(n);
  const long nd = cplx ? 2 * n : n;
  double* p = normalize ? (double*)c->workspace(WS_KRY_PART, (size_t)nb * sizeof(double)) : nullptr;
  if (cplx) hipLaunchKernelGGL(krylov_combine_kernel<true>, dim3(nb), dim3(256), 0, c->stream, basis, ld, K, kc, out, n, p);
  else hipLaunchKernelGGL(krylov_combine_kernel<false>, dim3(nb), dim3(256), 0, c->stream, basis, ld, K, kc, out, n, p);
  if (normalize)
    hipLaunchKernelGGL(krylov_scale_kernel, dim3(grid1d(nd)), dim3(256), 0, c->stream, out, (const double*)out, nd,
                       (const double*)p, nb, (double*)nullptr);
  TN_HIP(hipGetLastError());
}

void row_norms2(tn_ctx* c, const double* X, long rows, long L, long ld, double* out) {
  if (rows <= 0) return;
  TN_REQUIRE(rows <= 2147483647L, TN_E_INVALID, "row_norms2: rows");
  hipLaunchKernelGGL(row_norms2_kernel, dim3((unsigned)rows), dim3(256), 0, c->stream, X, L, ld, out);
  TN_HIP(hipGetLastError());
}

void transpose_f64(tn_ctx* c, const double* in, long R, long C, double* out) {
  if (R <= 0 || C <= 0) return;
  dim3 grid((unsigned)((C + 31) / 32), (unsigned)((R + 31) / 32));
  TN_REQUIRE((R + 31) / 32 <= 65535, TN_E_INVALID, "transpose: too many rows");
  hipLaunchKernelGGL(transpose_kernel, grid, dim3(256), 0, c->stream, in, R, C, out);
  TN_HIP(hipGetLastError());
}

void gather_rows(tn_ctx* c, const double* src, long ld_src, const int* perm, const double* scale, long kcount,
                 long L, double* out) {
  if (kcount <= 0 || L <= 0) return;
  TN_REQUIRE(kcount <= 65535, TN_E_INVALID, "gather_rows: kcount");
  dim3 grid((unsigned)((L + 255) / 256), (unsigned)kcount);
  hipLaunchKernelGGL(gather_rows_kernel, grid, dim3(256), 0, c->stream, src, ld_src, perm, scale, L, out);
  TN_HIP(hipGetLastError());
}

void gather_rows_T_z(tn_ctx* c, const double* src, long ld_src, const int* perm, const double* scale,
                     long kcount, long L, double* out, bool conj) {
  if (kcount <= 0 || L <= 0) return;
  dim3 grid((unsigned)((L + 15) / 16), (unsigned)((kcount + 15) / 16));
  TN_REQUIRE((kcount + 15) / 16 <= 65535, TN_E_INVALID, "gather_rows_T_z: kcount");
  hipLaunchKernelGGL(gather_rows_T_z_kernel, grid, dim3(256), 0, c->stream, (const double2*)src, ld_src, perm,
                     scale, kcount, L, (double2*)out, (int)conj);
  TN_HIP(hipGetLastError());
}

void gather_rows_T(tn_ctx* c, const double* src, long ld_src, const int* perm, const double* scale,
                   long kcount, long L, double* out) {
  if (kcount <= 0 || L <= 0) return;
  dim3 grid((unsigned)((L + 31) / 32), (unsigned)((kcount + 31) / 32));
  TN_REQUIRE((kcount + 31) / 32 <= 65535, TN_E_INVALID, "gather_rows_T: kcount");
  hipLaunchKernelGGL(gather_rows_T_kernel, grid, dim3(256), 0, c->stream, src, ld_src, perm, scale, kcount, L,
                     out);
  TN_HIP(hipGetLastError());
}

}  // namespace tn
