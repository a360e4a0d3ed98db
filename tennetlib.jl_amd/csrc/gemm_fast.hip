// Double-buffered MFMA GEMMs.
//
//  * gemm_fast<T, TA, TB, tile>: FP64 (v_mfma_f64_16x16x4_f64), FP32
//    (v_mfma_f32_32x32x2_f32) or complex FP64 (four f64 MFMAs per product),
//    square tiles of 128, 64 or 32, 4 wavefronts (2 x 2) of a quarter tile.
//    Each operand is staged with 16-byte loads along its contiguous
//    dimension into an LDS tile that keeps the global orientation
//    (A: [m][k] if k is contiguous, [k][m] if m is; B: [k][n] or [n][k]),
//    so staging never transposes; the MFMA fragment reads adapt instead.
//    Two LDS stages: the next tile is fetched into registers while the
//    current one feeds the MFMAs, then written to the other stage; one
//    barrier per K tile.  The same loop runs over a list of K segments, for
//    the grouped and the block-sparse products.
//  * gemm_bf16x3_nt: C = A * B^T with A (M x K) and B (N x K) given as bf16
//    hi/lo pairs (k contiguous, pre-split by split_bf16_*).  Each 32x32x16
//    step issues lo*hi + hi*lo + hi*hi with FP32 accumulation.
// Operands whose rows are 16-byte aligned with whole vectors take vector
// loads, others element loads, both with 32-bit offsets into the tile; row
// strides past those take element loads from 64-bit addresses.
#include <map>
#include <mutex>

#include "tn_internal.h"

#include <algorithm>
#include <cstdlib>
#include <type_traits>

namespace tn {
namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef unsigned short us8 __attribute__((ext_vector_type(8)));

struct FArgs {
  long M, N, K;
  const void* A; long lda; long sA; long wA;  // wA, wB: readable row widths
  const void* B; long ldb; long sB; long wB;
  void* C; long ldc; long sC;
  double alpha, beta;
  int cA, cB;  // complex: conjugated operands
  long Kall;   // K in parts: batch z sums rows z K .. (z + 1) K of Kall
};

__device__ __forceinline__ void tile_coords2(int ntm, int ntn, int& tm, int& tn) {
  const int nt = ntm * ntn;
  int id = blockIdx.x;
  if (nt >= 64 && (nt % 8) == 0) {  // contiguous tile runs per XCD
    const int per = nt / 8;
    id = (id % 8) * per + (id / 8);
  }
  const int GM = 8;
  const int group = id / (GM * ntn);
  const int first_m = group * GM;
  const int gsz = min(ntm - first_m, GM);
  const int in_group = id % (GM * ntn);
  tm = first_m + (in_group % gsz);
  tn = in_group / gsz;
}

// ---------------------------------------------------------------------------
// Tile loads through buffer resources.  A resource covers the rows of one
// tile of a row-major operand, from its first row to the last valid element
// ((rows_valid - 1) * ld + cols elements); the hardware returns zeros for any
// offset at or beyond that extent, and vectors past the last column get an
// offset far beyond it.  Tile edges therefore need no branches, the loads of
// the next tile stay in flight while the MFMAs run, and no load touches
// memory outside the operand.  Every row's valid width (cols) is a multiple
// of the 16-byte vector, so a vector is either fully valid or fully outside.
// ---------------------------------------------------------------------------
typedef __amdgpu_buffer_rsrc_t Rsrc;
constexpr unsigned OOB = 0x80000000u;  // offset past every extent (< 2^31 bytes)

__device__ __forceinline__ Rsrc tile_rsrc(const void* base, long r0, long rows, long tile_rows, long ld, long cols,
                                          int esz) {
  const long rv = min(tile_rows, rows - r0);
  const long bytes = rv > 0 ? ((rv - 1) * ld + cols) * esz : 0;
  return __builtin_amdgcn_make_buffer_rsrc(
      const_cast<void*>(reinterpret_cast<const void*>(reinterpret_cast<const char*>(base) + r0 * ld * esz)),
      (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ uint4 ld16(Rsrc r, unsigned off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0));
}
// byte offset of the vector at (tile row rr, column c) or OOB past the columns
__device__ __forceinline__ unsigned voff(int rr, long c, long ld, long cols, int esz) {
  return c < cols ? (unsigned)((rr * ld + c) * esz) : OOB;
}
// the VN elements at (tile row rr, columns c .. c + VN - 1) as one 16-byte
// value: AL = 1, one vector load (the row start and c are vector-aligned and
// the row width is whole vectors); AL = 0, element loads, each bounded by the
// row width on its own, for operands whose rows are not 16-byte aligned
template <typename T, int AL>
__device__ __forceinline__ uint4 ldvec(Rsrc r, int rr, long c, long ld, long cols) {
  constexpr int ES = (int)sizeof(T);
  if constexpr (AL || ES == 16) {
    return ld16(r, voff(rr, c, ld, cols, ES));
  } else if constexpr (ES == 8) {
    uint4 v;
    const unsigned long long x0 = __builtin_bit_cast(
        unsigned long long, __builtin_amdgcn_raw_buffer_load_b64(r, voff(rr, c, ld, cols, ES), 0, 0));
    const unsigned long long x1 = __builtin_bit_cast(
        unsigned long long, __builtin_amdgcn_raw_buffer_load_b64(r, voff(rr, c + 1, ld, cols, ES), 0, 0));
    v.x = (unsigned)x0; v.y = (unsigned)(x0 >> 32);
    v.z = (unsigned)x1; v.w = (unsigned)(x1 >> 32);
    return v;
  } else {
    uint4 v;
    v.x = __builtin_amdgcn_raw_buffer_load_b32(r, voff(rr, c, ld, cols, ES), 0, 0);
    v.y = __builtin_amdgcn_raw_buffer_load_b32(r, voff(rr, c + 1, ld, cols, ES), 0, 0);
    v.z = __builtin_amdgcn_raw_buffer_load_b32(r, voff(rr, c + 2, ld, cols, ES), 0, 0);
    v.w = __builtin_amdgcn_raw_buffer_load_b32(r, voff(rr, c + 3, ld, cols, ES), 0, 0);
    return v;
  }
}

// the same VN elements through 64-bit addresses: rows [0, rows) of the tile,
// columns [0, cols), both at least one; loads without branches, from the last
// valid element past the ends
template <typename T>
__device__ __forceinline__ uint4 ldvec_far(const T* base, int rr, long rows, long c, long ld, long cols) {
  constexpr int VN = 16 / (int)sizeof(T);
  struct alignas(16) V { T e[VN]; } v;
  const T* p = base + min((long)rr, rows - 1) * ld;
#pragma unroll
  for (int q = 0; q < VN; ++q) v.e[q] = p[min(c + q, cols - 1)];
  uint4 u = __builtin_bit_cast(uint4, v);
  constexpr int D = (int)sizeof(T) / 4;  // words an element
#pragma unroll
  for (int q = 0; q < VN; ++q) {
    const bool in = rr < rows && c + q < cols;
    unsigned* w = &u.x + q * D;
#pragma unroll
    for (int i = 0; i < D; ++i) w[i] = in ? w[i] : 0u;
  }
  return u;
}

// how a kernel loads its operands: LOAD_ELEM and LOAD_VEC as in ldvec, LOAD_FAR
// as in ldvec_far.  Factorisation of 200 rows of 2.1 10^6 numbers with LOAD_FAR
// 15.5 ms, of 1.05 10^6 complex ones 93 ms (kernels of their own for such rows:
// 16.2 to 17.2 and 207 ms); with branches around each load 13.3 and 165 ms.
constexpr int LOAD_ELEM = 0, LOAD_VEC = 1, LOAD_FAR = 2;

// ---------------------------------------------------------------------------
// bf16 hi/lo split: hi = rne(x), lo = rne(x - hi); from FP64 or FP32 sources
// ---------------------------------------------------------------------------
__device__ __forceinline__ unsigned short f2bf(float x) {
  unsigned int u = __float_as_uint(x);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f_(unsigned short h) { return __uint_as_float(((unsigned int)h) << 16); }

template <typename T>
__device__ __forceinline__ void split1(T x, unsigned short& h, unsigned short& l) {
  h = f2bf((float)x);
  l = f2bf((float)(x - (T)bf2f_(h)));
}

// ---------------------------------------------------------------------------
// One output tile.  T: float, double or double2 (complex).
// Tile sizes: BM x BM outputs, K tiles of BK.  128 x 128 keeps the MFMAs busy
// with two workgroups per CU; launch bounds of two wavefronts per SIMD keep
// the 128 accumulator registers of the FP64 tile in place (without them the
// compiler moved them between the two register files in every K tile: 4096^3
// FP64 at 47 TF/s, with them 63).  64 and 32 put four and sixteen times the
// workgroups on products with fewer tiles than CUs; they are bound by the
// latency of a K tile, so theirs are longer.
// ---------------------------------------------------------------------------
template <typename T> struct Acc;
template <> struct Acc<double> { typedef d4 type; static constexpr int MB = 16, NR = 4; };
template <> struct Acc<float> { typedef f16v type; static constexpr int MB = 32, NR = 16; };
struct Z4 {
  d4 re, im;
};
template <> struct Acc<double2> { typedef Z4 type; static constexpr int MB = 16, NR = 4; };

template <typename T, int TA, int TB, int BM_, int BK_>
struct TileCfg {
  static constexpr int BM = BM_, BN = BM_, BK = BK_;
  static constexpr int VN = 16 / (int)sizeof(T);
  static constexpr int PAD = VN;  // keeps 16-byte alignment of every LDS row
  // A stage: [BM][BK+PAD] if TA == 0 else [BK][BM+PAD]
  static constexpr int A_ROWS = TA ? BK : BM, A_COLS = TA ? BM : BK, A_LD = A_COLS + PAD;
  static constexpr int B_ROWS = TB ? BN : BK, B_COLS = TB ? BK : BN, B_LD = B_COLS + PAD;
  static constexpr int A_VECS = A_ROWS * A_COLS / VN / 256;  // per thread
  static constexpr int B_VECS = B_ROWS * B_COLS / VN / 256;
  static constexpr int A_ELEMS = A_ROWS * A_LD, B_ELEMS = B_ROWS * B_LD;
  static constexpr int WT = BM / 2, F = WT / Acc<T>::MB;  // wave tile, MFMA blocks per side
  // K tiles on their way in registers: one where the MFMAs of a tile cover a
  // load, more where they do not (a 32 x 32 FP64 tile multiplies 32 rows of K
  // in 0.2 us): 370 x 185 x 925 FP64 20.2 us with one, 17.4 with four.  64 x 64
  // FP64 and complex tiles gained nothing (40.4 and 40.7 us, 35.3 and 36.6).
  static constexpr int PF = BM == 128 || (BM == 64 && sizeof(T) >= 8) ? 1 : (A_VECS + B_VECS) <= 4 ? 4 : 2;
  static constexpr size_t LDS = 2 * (size_t)(A_ELEMS + B_ELEMS) * sizeof(T);
  static_assert(A_VECS * VN * 256 == A_ROWS * A_COLS && B_VECS * VN * 256 == B_ROWS * B_COLS, "whole vectors");
};
// K tile of a tile size: 128 holds two 35 KB stages per operand pair, the
// small tiles trade LDS for fewer barriers
template <typename T> constexpr int tile_bk(int bm) {
  return sizeof(T) == 8 ? (bm == 128 ? 16 : 32) : sizeof(T) == 4 ? 32 : 16;
}

// acc += sum over the K segments of seg of A_s (rows m0..) * B_s (columns
// n0..).  Seg: done(), next() and the current A, B, K, wA, wB, weight w
// (SCALE: A_s is multiplied by w).  SPLIT: FP32 fragments as bf16 hi/lo parts.
template <class CF, typename T, int TA, int TB, int AL, bool SCALE, bool SPLIT, class Seg>
__device__ __forceinline__ void tile_product(Seg& seg, long M, long N, long m0, long n0, long lda, long ldb, int cA,
                                             int cB, T* smem, typename Acc<T>::type (&acc)[CF::F][CF::F]) {
  constexpr int BM = CF::BM, BN = CF::BN, BK = CF::BK, VN = CF::VN, F = CF::F, MB = Acc<T>::MB, ES = (int)sizeof(T);
  T* As = smem;  // 2 stages
  T* Bs = As + 2 * CF::A_ELEMS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave >> 1) * CF::WT, wn = (wave & 1) * CF::WT;
  constexpr int PF = CF::PF;
  uint4 ra[PF][CF::A_VECS], rb[PF][CF::B_VECS];
  long k0 = 0;
  double w[PF];
  // the next K tile of the current segment: rows m (TA = 0, k contiguous) or rows k (TA = 1, m contiguous)
  auto gload = [&](auto slot) {
    constexpr int Q = decltype(slot)::value;
    const T* A = reinterpret_cast<const T*>(seg.A);
    const T* B = reinterpret_cast<const T*>(seg.B);
    const long ra0 = TA ? k0 : m0, na = TA ? seg.K : M, rb0 = TB ? n0 : k0, nb = TB ? N : seg.K;  // first row, rows
    const Rsrc ar = tile_rsrc(A, ra0, na, TA ? BK : BM, lda, seg.wA, ES);
    const Rsrc br = tile_rsrc(B, rb0, nb, TB ? BN : BK, ldb, seg.wB, ES);
#pragma unroll
    for (int i = 0; i < CF::A_VECS; ++i) {
      const int idx = tid + i * 256;
      const int rr = idx / (CF::A_COLS / VN), cc = (idx % (CF::A_COLS / VN)) * VN;
      if constexpr (AL == LOAD_FAR)
        ra[Q][i] = ldvec_far<T>(A + ra0 * lda, rr, na - ra0, (TA ? m0 : k0) + cc, lda, seg.wA);
      else
        ra[Q][i] = ldvec<T, AL>(ar, rr, (TA ? m0 : k0) + cc, lda, seg.wA);
    }
#pragma unroll
    for (int i = 0; i < CF::B_VECS; ++i) {
      const int idx = tid + i * 256;
      const int rr = idx / (CF::B_COLS / VN), cc = (idx % (CF::B_COLS / VN)) * VN;
      if constexpr (AL == LOAD_FAR)
        rb[Q][i] = ldvec_far<T>(B + rb0 * ldb, rr, nb - rb0, (TB ? k0 : n0) + cc, ldb, seg.wB);
      else
        rb[Q][i] = ldvec<T, AL>(br, rr, (TB ? k0 : n0) + cc, ldb, seg.wB);
    }
    if constexpr (SCALE) w[Q] = seg.w;
    k0 += BK;
    if (k0 >= seg.K) {
      k0 = 0;
      seg.next();
    }
  };
  auto sstore = [&](auto slot, int st) {
    constexpr int Q = decltype(slot)::value;
    T* as = As + st * CF::A_ELEMS;
    T* bs = Bs + st * CF::B_ELEMS;
    if constexpr (SCALE) {
#pragma unroll
      for (int i = 0; i < CF::A_VECS; ++i) {
        double2 v = __builtin_bit_cast(double2, ra[Q][i]);
        v.x *= w[Q];
        v.y *= w[Q];
        ra[Q][i] = __builtin_bit_cast(uint4, v);
      }
    }
    if constexpr (ES == 16) {  // conjugated operands: the sign of the imaginary part
#pragma unroll
      for (int i = 0; i < CF::A_VECS; ++i) ra[Q][i].w ^= cA ? 0x80000000u : 0u;
#pragma unroll
      for (int i = 0; i < CF::B_VECS; ++i) rb[Q][i].w ^= cB ? 0x80000000u : 0u;
    }
#pragma unroll
    for (int i = 0; i < CF::A_VECS; ++i) {
      const int idx = tid + i * 256;
      const int rr = idx / (CF::A_COLS / VN), cc = (idx % (CF::A_COLS / VN)) * VN;
      *reinterpret_cast<uint4*>(&as[rr * CF::A_LD + cc]) = ra[Q][i];
    }
#pragma unroll
    for (int i = 0; i < CF::B_VECS; ++i) {
      const int idx = tid + i * 256;
      const int rr = idx / (CF::B_COLS / VN), cc = (idx % (CF::B_COLS / VN)) * VN;
      *reinterpret_cast<uint4*>(&bs[rr * CF::B_LD + cc]) = rb[Q][i];
    }
  };
  // element (m, k) of the A stage and (k, n) of the B stage
  auto Ael = [&](const T* as, int m, int k) -> T { return TA ? as[k * CF::A_LD + m] : as[m * CF::A_LD + k]; };
  auto Bel = [&](const T* bs, int k, int n) -> T { return TB ? bs[n * CF::B_LD + k] : bs[k * CF::B_LD + n]; };
  auto compute = [&](int st) {
    const T* as = As + st * CF::A_ELEMS;
    const T* bs = Bs + st * CF::B_ELEMS;
    if constexpr (SPLIT) {
      // lane: row / column lane % 32, the 8 k values 8 (lane / 32) .. + 7 of every 16
#pragma unroll
      for (int kk = 0; kk < BK; kk += 16) {
        const int kb = kk + 8 * (lane >> 5);
        bf8 ah[F], al[F], bh[F], bl[F];
#pragma unroll
        for (int i = 0; i < F; ++i) {
          us8 h, l;
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            unsigned short hq, lq;
            split1<float>(Ael(as, wm + i * MB + (lane & 31), kb + q), hq, lq);
            h[q] = hq;
            l[q] = lq;
          }
          ah[i] = __builtin_bit_cast(bf8, h);
          al[i] = __builtin_bit_cast(bf8, l);
        }
#pragma unroll
        for (int j = 0; j < F; ++j) {
          us8 h, l;
#pragma unroll
          for (int q = 0; q < 8; ++q) {
            unsigned short hq, lq;
            split1<float>(Bel(bs, kb + q, wn + j * MB + (lane & 31)), hq, lq);
            h[q] = hq;
            l[q] = lq;
          }
          bh[j] = __builtin_bit_cast(bf8, h);
          bl[j] = __builtin_bit_cast(bf8, l);
        }
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j) {
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
          }
      }
    } else if constexpr (ES == 4) {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 2) {
        const int kr = kk + (lane >> 5);
        float fa[F], fb[F];
#pragma unroll
        for (int i = 0; i < F; ++i) fa[i] = Ael(as, wm + i * MB + (lane & 31), kr);
#pragma unroll
        for (int j = 0; j < F; ++j) fb[j] = Bel(bs, kr, wn + j * MB + (lane & 31));
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
    } else if constexpr (ES == 8) {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        const int kr = kk + (lane >> 4);
        double fa[F], fb[F];
#pragma unroll
        for (int i = 0; i < F; ++i) fa[i] = Ael(as, wm + i * MB + (lane & 15), kr);
#pragma unroll
        for (int j = 0; j < F; ++j) fb[j] = Bel(bs, kr, wn + j * MB + (lane & 15));
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i], fb[j], acc[i][j], 0, 0, 0);
      }
    } else {
#pragma unroll
      for (int kk = 0; kk < BK; kk += 4) {
        const int kr = kk + (lane >> 4);
        double2 fa[F], fb[F];
#pragma unroll
        for (int i = 0; i < F; ++i) fa[i] = Ael(as, wm + i * MB + (lane & 15), kr);
#pragma unroll
        for (int j = 0; j < F; ++j) fb[j] = Bel(bs, kr, wn + j * MB + (lane & 15));
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < F; ++j) {
            acc[i][j].re = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i].x, fb[j].x, acc[i][j].re, 0, 0, 0);
            acc[i][j].im = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i].x, fb[j].y, acc[i][j].im, 0, 0, 0);
            acc[i][j].re = __builtin_amdgcn_mfma_f64_16x16x4f64(-fa[i].y, fb[j].y, acc[i][j].re, 0, 0, 0);
            acc[i][j].im = __builtin_amdgcn_mfma_f64_16x16x4f64(fa[i].y, fb[j].x, acc[i][j].im, 0, 0, 0);
          }
      }
    }
  };
  if (seg.done()) return;
  using S0 = std::integral_constant<int, 0>;
  if constexpr (PF == 1) {
    gload(S0{});
    sstore(S0{}, 0);
    __syncthreads();
    for (int st = 0;; st ^= 1) {
      const bool more = !seg.done();
      if (more) gload(S0{});
      __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the MFMAs
      compute(st);
      __builtin_amdgcn_sched_barrier(0);
      if (!more) break;
      sstore(S0{}, st ^ 1);
      __syncthreads();
    }
  } else {
    // PF tiles ahead in registers: slot q holds tiles q, q + PF, ...
    using S1 = std::integral_constant<int, 1>;
    using S2 = std::integral_constant<int, PF == 4 ? 2 : 0>;
    using S3 = std::integral_constant<int, PF == 4 ? 3 : 1>;
    int ahead = 1;  // tiles loaded and not yet multiplied
    gload(S0{});
    auto fetch = [&](auto slot) {
      if (!seg.done()) {
        gload(slot);
        ++ahead;
      }
    };
    fetch(S1{});
    if constexpr (PF == 4) {
      fetch(S2{});
      fetch(S3{});
    }
    sstore(S0{}, 0);
    fetch(S0{});
    __syncthreads();
    // one tile: multiply it from stage st, then move the next one (slot) to the other stage
    auto step = [&](int st, auto slot) -> bool {
      compute(st);
      if (--ahead == 0) return false;
      sstore(slot, st ^ 1);
      fetch(slot);
      __syncthreads();
      return true;
    };
    while (true) {
      if (!step(0, S1{})) break;
      if (!step(1, S2{})) break;
      if constexpr (PF == 4) {
        if (!step(0, S3{})) break;
        if (!step(1, S0{})) break;
      }
    }
  }
}

// C tile = alpha acc + beta C.  Registers of an MFMA block: f64 (complex: re
// and im alike) register r of a lane is row lane / 16 + 4 r, column lane %
// 16; f32 row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32.
template <class CF, typename T>
__device__ __forceinline__ void tile_store(T* C, long ldc, long M, long N, long m0, long n0, double alpha, double beta,
                                           const typename Acc<T>::type (&acc)[CF::F][CF::F]) {
  constexpr int F = CF::F, MB = Acc<T>::MB, NR = Acc<T>::NR;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long mw = m0 + (wave >> 1) * CF::WT, nw = n0 + (wave & 1) * CF::WT;
#pragma unroll
  for (int i = 0; i < F; ++i)
#pragma unroll
    for (int j = 0; j < F; ++j)
#pragma unroll
      for (int r = 0; r < NR; ++r) {
        const long m = mw + i * MB + (MB == 32 ? 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3) : (lane >> 4) + 4 * r);
        const long n = nw + j * MB + (lane & (MB - 1));
        if (m < M && n < N) {
          T* p = C + m * ldc + n;
          if constexpr (std::is_same<T, double2>::value) {
            double2 v = make_double2(alpha * acc[i][j].re[r], alpha * acc[i][j].im[r]);
            if (beta != 0.0) {
              const double2 o = *p;
              v.x += beta * o.x;
              v.y += beta * o.y;
            }
            *p = v;
          } else {
            T v = (T)alpha * acc[i][j][r];
            if (beta != 0.0) v += (T)beta * *p;
            *p = v;
          }
        }
      }
}

template <class CF, typename T>
__device__ __forceinline__ void tile_zero(typename Acc<T>::type (&acc)[CF::F][CF::F]) {
#pragma unroll
  for (int i = 0; i < CF::F; ++i)
#pragma unroll
    for (int j = 0; j < CF::F; ++j) acc[i][j] = typename Acc<T>::type{};
}

struct OneSeg {  // a plain product: one segment
  const void* A;
  const void* B;
  long K, wA, wB;
  bool end;
  __device__ __forceinline__ bool done() const { return end; }
  __device__ __forceinline__ void next() { end = true; }
};

// PARTS: K in parts (a kernel of its own: the last part's length costs the
// others 0.1 to 0.2 us)
template <typename T, int TA, int TB, int AL, int BM, bool PARTS>
__global__ __launch_bounds__(256, 2) void gemm_fast_kernel(FArgs a) {
  using CF = TileCfg<T, TA, TB, BM, tile_bk<T>(BM)>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int ntm = (int)((a.M + BM - 1) / BM), ntn = (int)((a.N + BM - 1) / BM);
  int tm, tn;
  tile_coords2(ntm, ntn, tm, tn);
  const long m0 = (long)tm * BM, n0 = (long)tn * BM, bz = blockIdx.z;
  OneSeg seg{reinterpret_cast<const T*>(a.A) + bz * a.sA, reinterpret_cast<const T*>(a.B) + bz * a.sB, a.K, a.wA, a.wB,
             a.K <= 0};
  if constexpr (PARTS) {  // the last part may be shorter
    const long kb = bz * a.K;
    seg.K = min(a.K, a.Kall - kb);
    if (!TA) seg.wA = min(a.K, a.wA - kb);
    if (TB) seg.wB = min(a.K, a.wB - kb);
  }
  typename Acc<T>::type acc[CF::F][CF::F];
  tile_zero<CF, T>(acc);
  tile_product<CF, T, TA, TB, AL, false, false>(seg, a.M, a.N, m0, n0, a.lda, a.ldb, a.cA, a.cB,
                                                reinterpret_cast<T*>(smem), acc);
  tile_store<CF, T>(reinterpret_cast<T*>(a.C) + bz * a.sC, a.ldc, a.M, a.N, m0, n0, a.alpha, a.beta, acc);
}

// ---------------------------------------------------------------------------
// Grouped FP64 GEMM: output group g (grid y) and batch z (grid z) accumulate
// sum over the terms t of group g of w_t A_{ia_t} B_{ib_t}, every term an
// M x N x K product; the output tile is written once (no read of C).  The
// terms are the K segments of one tile loop, so the next term's first tile
// is on its way while a term ends.
// ---------------------------------------------------------------------------
struct TermSeg {
  const GroupedDesc& g;
  const double* A0;
  const double* B0;
  const void* A;
  const void* B;
  long K, wA, wB;
  double w;
  int t, t1;
  __device__ __forceinline__ void set() {
    if (t < t1) {
      A = A0 + (long)g.ia[t] * g.tsA;
      B = B0 + (long)g.ib[t] * g.tsB;
      w = g.w[t];
    }
  }
  __device__ __forceinline__ bool done() const { return t >= t1; }
  __device__ __forceinline__ void next() {
    ++t;
    set();
  }
};

template <int AL, int BM>
__global__ __launch_bounds__(256, 2) void gemm_grouped_kernel(GroupedDesc d) {
  using CF = TileCfg<double, 0, 0, BM, tile_bk<double>(BM)>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  int tm, tn;
  tile_coords2((int)((d.M + BM - 1) / BM), (int)((d.N + BM - 1) / BM), tm, tn);
  const long m0 = (long)tm * BM, n0 = (long)tn * BM, z = blockIdx.z;
  const int g = blockIdx.y;
  TermSeg seg{d, d.A + z * d.sA, d.B + z * d.sB, nullptr, nullptr, d.K, d.K, d.N, 0.0, d.off[g], d.off[g + 1]};
  if (d.K <= 0) seg.t = seg.t1;
  seg.set();
  d4 acc[CF::F][CF::F];
  tile_zero<CF, double>(acc);
  tile_product<CF, double, 0, 0, AL, true, false>(seg, d.M, d.N, m0, n0, d.lda, d.ldb, 0, 0,
                                                  reinterpret_cast<double*>(smem), acc);
  tile_store<CF, double>(d.C + (long)g * d.gsC + z * d.sC, d.ldc, d.M, d.N, m0, n0, 1.0, 0.0, acc);
}

// ---------------------------------------------------------------------------
// Block-sparse GEMM over uneven blocks (QN sectors): one launch covers a list
// of output tiles; tile t belongs to task tiles[t].x, whose output block
// C + c_off (M x N, ld ldc) is the sum over the task's K segments of
// A_s (M x K_s, ld lda) * B_s (K_s x N, ld ldb), A_s = A + a_off, B_s = B +
// b_off.  A task without segments writes zeros.  The tile list is laid out
// XCD-major: workgroup id i runs list entry (i % 8) * per + i / 8, so the
// contiguous run of tiles one XCD runs shares its tasks' A and B panels in
// that XCD's L2; padding entries (task < 0) exit at once.  Blocks start at
// any element, so the operands take element loads.
// SPLIT (FP32 operands only): each FP32 fragment is split into bf16 hi/lo
// parts in registers and the product accumulates lo*hi + hi*lo + hi*hi with
// the bf16 MFMA 32x32x16.
// ---------------------------------------------------------------------------
struct BlockSeg {
  const BsSeg* segs;
  const char* A0;
  const char* B0;
  int es, tB;
  long N;
  const void* A;
  const void* B;
  long K, wA, wB;
  int s, s1;
  __device__ __forceinline__ void set() {
    while (s < s1) {
      const BsSeg g = segs[s];
      A = A0 + g.a_off * es;
      B = B0 + g.b_off * es;
      K = wA = g.K;
      wB = tB ? g.K : N;
      if (K > 0) return;
      ++s;
    }
  }
  __device__ __forceinline__ bool done() const { return s >= s1; }
  __device__ __forceinline__ void next() {
    ++s;
    set();
  }
};

template <typename T, int TB, bool SPLIT, int AL>
__global__ __launch_bounds__(256, 2) void gemm_bs_kernel(BsDesc d) {
  using CF = TileCfg<T, 0, TB, BS_TILE, SPLIT ? 16 : tile_bk<T>(BS_TILE)>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int4 tl = d.tiles[(long)(blockIdx.x % 8) * (d.ntiles / 8) + blockIdx.x / 8];
  if (tl.x < 0) return;
  const BsTask tk = d.tasks[tl.x];
  BlockSeg seg{d.segs, reinterpret_cast<const char*>(d.A), reinterpret_cast<const char*>(d.B), (int)sizeof(T), TB,
               tk.N, nullptr, nullptr, 0, 0, 0, tk.seg0, tk.seg0 + tk.nseg};
  seg.set();
  typename Acc<T>::type acc[CF::F][CF::F];
  tile_zero<CF, T>(acc);
  tile_product<CF, T, 0, TB, AL, false, SPLIT>(seg, tk.M, tk.N, tl.y, tl.z, d.lda, d.ldb, 0, 0,
                                              reinterpret_cast<T*>(smem), acc);
  tile_store<CF, T>(reinterpret_cast<T*>(d.C) + tk.c_off, d.ldc, tk.M, tk.N, tl.y, tl.z, d.alpha, 0.0, acc);
}

// ---------------------------------------------------------------------------
// BF16x3, C (float) = A * B^T, A = (Ah + Al) M x K, B = (Bh + Bl) N x K
// ---------------------------------------------------------------------------
struct SArgs {
  long M, N, K;
  const unsigned short* Ah; const unsigned short* Al; long lda;
  const unsigned short* Bh; const unsigned short* Bl; long ldb;
  float* C; long ldc;
};

// 128 x 128 output tile, 4 wavefronts of 64 x 64 (2 x 2 blocks of 32 x 32);
// K tile SBK = 32 (two 80 KiB stages: two workgroups per CU) or 64 (one).
constexpr int SBM = 128, SBN = 128;
template <int SBK> struct SCfg {
  static constexpr int SLD = SBK + 8;                      // bf16 per LDS row (16 B pad)
  static constexpr int STAGE = (2 * SBM + 2 * SBN) * SLD;  // hi+lo of A and B, bf16 elements
  static constexpr int VPR = SBK / 8;                      // 16-byte vectors per row
  static constexpr int NV = SBM * VPR / 256;               // per thread, per operand part
};

template <int SBK>
__global__ __launch_bounds__(256) void gemm_bf16x3_nt_kernel(SArgs a) {
  using CF = SCfg<SBK>;
  constexpr int SLD = CF::SLD, VPR = CF::VPR, NV = CF::NV;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned short* S = reinterpret_cast<unsigned short*>(smem);
  const int ntm = (int)((a.M + SBM - 1) / SBM), ntn = (int)((a.N + SBN - 1) / SBN);
  int tm, tn;
  tile_coords2(ntm, ntn, tm, tn);
  const long m0 = (long)tm * SBM, n0 = (long)tn * SBN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  // rows are zero-padded to Kp (a multiple of 8): vectors below Kp are valid
  const long Kp = (a.K + 7) & ~7L;
  const Rsrc rah_r = tile_rsrc(a.Ah, m0, a.M, SBM, a.lda, Kp, 2);
  const Rsrc ral_r = tile_rsrc(a.Al, m0, a.M, SBM, a.lda, Kp, 2);
  const Rsrc rbh_r = tile_rsrc(a.Bh, n0, a.N, SBN, a.ldb, Kp, 2);
  const Rsrc rbl_r = tile_rsrc(a.Bl, n0, a.N, SBN, a.ldb, Kp, 2);
  uint4 rah[NV], ral[NV], rbh[NV], rbl[NV];
  auto gload = [&](long k0) {
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * 256;
      const int rr = idx / VPR, cc = (idx % VPR) * 8;
      const unsigned oa = voff(rr, k0 + cc, a.lda, Kp, 2), ob = voff(rr, k0 + cc, a.ldb, Kp, 2);
      rah[i] = ld16(rah_r, oa);
      ral[i] = ld16(ral_r, oa);
      rbh[i] = ld16(rbh_r, ob);
      rbl[i] = ld16(rbl_r, ob);
    }
  };
  auto sstore = [&](int st) {
    unsigned short* Ah = S + st * CF::STAGE;
    unsigned short* Al = Ah + SBM * SLD;
    unsigned short* Bh = Al + SBM * SLD;
    unsigned short* Bl = Bh + SBN * SLD;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const int idx = tid + i * 256;
      const int rr = idx / VPR, cc = (idx % VPR) * 8;
      *reinterpret_cast<uint4*>(&Ah[rr * SLD + cc]) = rah[i];
      *reinterpret_cast<uint4*>(&Al[rr * SLD + cc]) = ral[i];
      *reinterpret_cast<uint4*>(&Bh[rr * SLD + cc]) = rbh[i];
      *reinterpret_cast<uint4*>(&Bl[rr * SLD + cc]) = rbl[i];
    }
  };
  f16v acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f16v{};
  const long nk = (a.K + SBK - 1) / SBK;
  gload(0);
  sstore(0);
  __syncthreads();
  for (long t = 0; t < nk; ++t) {
    gload((t + 1) * SBK);  // past the last tile this loads zeros and touches no memory
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch ahead of the MFMAs
    const unsigned short* Ah = S + (t & 1) * CF::STAGE;
    const unsigned short* Al = Ah + SBM * SLD;
    const unsigned short* Bh = Al + SBM * SLD;
    const unsigned short* Bl = Bh + SBN * SLD;
#pragma unroll
    for (int kk = 0; kk < SBK; kk += 16) {
      const int kc = kk + 8 * (lane >> 5);
      bf8 ah[2], al[2], bh[2], bl[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = wm * 64 + i * 32 + (lane & 31);
        ah[i] = __builtin_bit_cast(bf8, *reinterpret_cast<const us8*>(&Ah[row * SLD + kc]));
        al[i] = __builtin_bit_cast(bf8, *reinterpret_cast<const us8*>(&Al[row * SLD + kc]));
      }
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const int col = wn * 64 + j * 32 + (lane & 31);
        bh[j] = __builtin_bit_cast(bf8, *reinterpret_cast<const us8*>(&Bh[col * SLD + kc]));
        bl[j] = __builtin_bit_cast(bf8, *reinterpret_cast<const us8*>(&Bl[col * SLD + kc]));
      }
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    sstore((t + 1) & 1);
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const long m = m0 + wm * 64 + i * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        const long n = n0 + wn * 64 + j * 32 + (lane & 31);
        if (m < a.M && n < a.N) a.C[m * a.ldc + n] = acc[i][j][r];
      }
}

// dst[r][c] (ld_dst) = split(src[r][c]); columns cols..ld_dst-1 zeroed
template <typename T>
__global__ __launch_bounds__(256) void split_rows_kernel(const T* __restrict__ src, long rows, long cols,
                                                         long lds, unsigned short* __restrict__ hi,
                                                         unsigned short* __restrict__ lo, long ldd) {
  const long total = rows * ldd;
  for (long i = blockIdx.x * (long)blockDim.x + threadIdx.x; i < total; i += (long)gridDim.x * blockDim.x) {
    const long r = i / ldd, c = i % ldd;
    unsigned short h = 0, l = 0;
    if (c < cols) split1<T>(src[r * lds + c], h, l);
    hi[i] = h;
    lo[i] = l;
  }
}

// dst[c][r] (ld_dst) = split(src[r][c]) for r < rows, c < cols; 32x32 tiles
template <typename T>
__global__ __launch_bounds__(256) void split_transpose_kernel(const T* __restrict__ src, long rows, long cols,
                                                              long lds, unsigned short* __restrict__ hi,
                                                              unsigned short* __restrict__ lo, long ldd) {
  __shared__ T t[32][33];
  const long r0 = (long)blockIdx.y * 32, c0 = (long)blockIdx.x * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const long r = r0 + k, c = c0 + tx;
    t[k][tx] = (r < rows && c < cols) ? src[r * lds + c] : T(0);
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const long c = c0 + k, r = r0 + tx;  // output row c, column r
    if (c < cols && r < ldd) {
      unsigned short h = 0, l = 0;
      if (r < rows) split1<T>(t[tx][k], h, l);
      hi[c * ldd + r] = h;
      lo[c * ldd + r] = l;
    }
  }
}

}  // namespace

// ---------------------------------------------------------------------------
std::recursive_mutex& api_mutex() {
  static std::recursive_mutex m;
  return m;
}

// Every launch of a kernel with dynamic LDS goes through this first.  The
// first call for a kernel sets its dynamic-LDS limit once, to everything the
// 160 KB LDS leaves beside its static LDS, and it is never changed again, so
// no attribute change can meet a launch of the same kernel on another thread.
void raise_lds_limit(const void* fn, size_t bytes) {
  constexpr size_t LDS_BYTES = 160 * 1024;
  static std::mutex mu;
  static std::map<const void*, size_t> done;  // kernel -> dynamic-LDS limit
  std::lock_guard<std::mutex> lock(mu);
  auto it = done.find(fn);
  if (it == done.end()) {
    hipFuncAttributes attr;
    TN_HIP(hipFuncGetAttributes(&attr, fn));
    const size_t lim = LDS_BYTES - std::min(LDS_BYTES, (size_t)attr.sharedSizeBytes);
    TN_HIP(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lim));
    it = done.emplace(fn, lim).first;
  }
  TN_REQUIRE(bytes <= it->second, TN_E_UNSUPPORTED,
             "kernel needs " + std::to_string(bytes) + " bytes of dynamic LDS, more than the " +
                 std::to_string(it->second) + " available");
}
static void allow_lds(const void* fn, size_t bytes) { raise_lds_limit(fn, bytes); }

// readable row widths of A and B: the valid width, rounded up to whole
// vectors for an operand the caller marks zero-padded
static int vec_elems(Prec p) { return p == Prec::F64 ? 2 : p == Prec::Z64 ? 1 : 4; }
static size_t elem_bytes(Prec p) { return p == Prec::F64 ? 8 : p == Prec::Z64 ? 16 : 4; }
static long width_a(Prec p, const GemmDesc& g) {
  const int vn = vec_elems(p);
  if (g.tA) return g.M;
  return g.zpA ? (g.K + vn - 1) / vn * vn : g.K;
}
static long width_b(Prec p, const GemmDesc& g) {
  const int vn = vec_elems(p);
  if (g.tB) return g.K;
  return g.zpB ? (g.N + vn - 1) / vn * vn : g.N;
}
// operands whose rows are 16-byte aligned with a valid width of whole
// vectors take the vector loads; any other operand takes element loads
static bool fast_aligned(Prec p, const GemmDesc& g) {
  const int vn = vec_elems(p);
  auto al = [&](const void* ptr, long ld, long s, long cols) {
    return ((uintptr_t)ptr % 16 == 0) && (ld % vn == 0) && (s % vn == 0) && (cols % vn == 0) && cols <= ld;
  };
  return al(g.A, g.lda, g.sA, width_a(p, g)) && al(g.B, g.ldb, g.sB, width_b(p, g));
}

// Operands whose tiles have 32-bit offsets: the rows that a tile holds span less
// than 2^31 bytes, and the offsets that the kernel forms for all rows of the
// tile stay below 2^32, so that those past the operand's end are past its
// extent and do not wrap into it.
static bool extent_ok(long ld, long rows, long tile_rows, size_t es) {
  const size_t row = (size_t)ld * es;
  return row * (size_t)(std::min(rows, tile_rows) + 1) < ((size_t)1 << 31) &&
         row * (size_t)(tile_rows + 1) < ((size_t)1 << 32);
}

// Tile of an M x N product over a batch: the one with the least work on the
// busiest CU, tiles / 256 rounds of b^2 outputs each, weighted by how well a
// tile size keeps the MFMAs fed (measured on full grids: FP64 128 63 TF/s,
// 64 55, 32 30).  Complex products and FP32 have no 128 / 32 tile respectively.
// Complex products take the FP64 weights; 64 and 32 tiles run at about the same
// rate there.  H psi (w = 5), us, by the rule and on 32 tiles throughout: chi =
// 200 112 and 114, 256 168 and 152, 400 552 and 484, 512 800 and 855.
static int pick_tile(Prec p, long M, long N, long batch, double* work = nullptr) {
  int best = 0;
  double cost = 0.0;
  for (int b : {128, 64, 32}) {
    if ((p == Prec::Z64 && b == 128) || (p == Prec::F32 && b == 32)) continue;
    const double eff = b == 128 ? 1.0 : b == 64 ? 0.87 : 0.5;
    const long tiles = ((M + b - 1) / b) * ((N + b - 1) / b) * batch;
    const double t = (double)((tiles + 255) / 256) * b * b / eff;
    if (best == 0 || t < cost) {
      best = b;
      cost = t;
    }
  }
  if (work) *work = cost;
  return best;
}
double gemm_tile_work(Prec p, long M, long N, long batch) {
  double work;
  pick_tile(p, M, N, batch, &work);
  return work;
}

namespace {
template <typename T, int TA, int TB, int AL, int BM>
void launch_tile(tn_ctx* c, const FArgs& a, int batch) {
  constexpr size_t shm = TileCfg<T, TA, TB, BM, tile_bk<T>(BM)>::LDS;
  const long tiles = ((a.M + BM - 1) / BM) * ((a.N + BM - 1) / BM);
  TN_REQUIRE(tiles < (1L << 31), TN_E_INVALID, "gemm: too many tiles");
  auto launch = [&](auto kern) {
    allow_lds((const void*)kern, shm);
    hipLaunchKernelGGL(kern, dim3((unsigned)tiles, 1, (unsigned)batch), dim3(256), shm, c->stream, a);
  };
  if constexpr (sizeof(T) != 16)
    if (a.Kall > a.K) return launch(gemm_fast_kernel<T, TA, TB, AL, BM, true>);
  launch(gemm_fast_kernel<T, TA, TB, AL, BM, false>);
}
template <typename T, int TA, int TB, int AL>
void launch_bm(tn_ctx* c, const FArgs& a, int batch, int bm) {
  if constexpr (sizeof(T) != 16 && AL != LOAD_FAR)
    if (bm == 128) return launch_tile<T, TA, TB, AL, 128>(c, a, batch);
  if constexpr (sizeof(T) != 4)
    if (bm == 32) return launch_tile<T, TA, TB, AL, 32>(c, a, batch);
  launch_tile<T, TA, TB, AL, 64>(c, a, batch);
}
template <typename T, int AL>
void launch_ops(tn_ctx* c, const FArgs& a, const GemmDesc& g, int bm) {
  if (!g.tA && !g.tB) launch_bm<T, 0, 0, AL>(c, a, g.batch, bm);
  else if (g.tA && !g.tB) launch_bm<T, 1, 0, AL>(c, a, g.batch, bm);
  else if (!g.tA && g.tB) launch_bm<T, 0, 1, AL>(c, a, g.batch, bm);
  else launch_bm<T, 1, 1, AL>(c, a, g.batch, bm);
}
}  // namespace

void gemm_tiles(tn_ctx* c, Prec p, const GemmDesc& g) {
  TN_REQUIRE(p != Prec::BF16X3, TN_E_INVALID, "gemm: BF16x3 operands come pre-split (gemm_bf16x3_nt)");
  const size_t es = elem_bytes(p);
  const bool far = !extent_ok(g.lda, g.tA ? g.K : g.M, 128, es) || !extent_ok(g.ldb, g.tB ? g.N : g.K, 128, es) ||
                   (p == Prec::Z64 && ((uintptr_t)g.A % 16 != 0 || (uintptr_t)g.B % 16 != 0));
  const bool aligned = !far && fast_aligned(p, g);
  FArgs a;
  a.M = g.M; a.N = g.N; a.K = g.K;
  a.A = g.A; a.lda = g.lda; a.sA = g.sA; a.cA = g.cA;
  a.B = g.B; a.ldb = g.ldb; a.sB = g.sB; a.cB = g.cB;
  // the vector kernel reads the padded widths; the element kernels the valid ones
  a.wA = aligned ? width_a(p, g) : (g.tA ? g.M : g.K);
  a.wB = aligned ? width_b(p, g) : (g.tB ? g.K : g.N);
  a.C = g.C; a.ldc = g.ldc; a.sC = g.sC;
  a.alpha = g.alpha; a.beta = g.beta;
  a.Kall = g.K;
  if (g.kstep) a.K = g.kstep;
  const int bm = pick_tile(p, g.M, g.N, g.batch);
  if (p == Prec::Z64) {
    if (far) launch_ops<double2, LOAD_FAR>(c, a, g, bm);
    else launch_ops<double2, LOAD_VEC>(c, a, g, bm);
  } else if (p == Prec::F64) {
    if (far) launch_ops<double, LOAD_FAR>(c, a, g, bm);
    else if (aligned) launch_ops<double, LOAD_VEC>(c, a, g, bm);
    else launch_ops<double, LOAD_ELEM>(c, a, g, bm);
  } else {
    if (far) launch_ops<float, LOAD_FAR>(c, a, g, bm);
    else if (aligned) launch_ops<float, LOAD_VEC>(c, a, g, bm);
    else launch_ops<float, LOAD_ELEM>(c, a, g, bm);
  }
  TN_HIP(hipGetLastError());
}

void gemm_grouped_f64(tn_ctx* c, const GroupedDesc& d) {
  if (d.M <= 0 || d.N <= 0 || d.ngroups <= 0 || d.batch <= 0) return;
  TN_REQUIRE(d.ngroups <= 65535 && d.batch <= 65535, TN_E_INVALID, "grouped gemm: grid too large");
  const bool far = !extent_ok(d.lda, d.M, 64, 8) || !extent_ok(d.ldb, d.K, 64, 8);
  const int bm = far ? 64 : std::min(64, pick_tile(Prec::F64, d.M, d.N, (long)d.ngroups * d.batch));
  const long tiles = ((d.M + bm - 1) / bm) * ((d.N + bm - 1) / bm);
  TN_REQUIRE(tiles < (1L << 31), TN_E_INVALID, "grouped gemm: too many tiles");
  const bool al = (uintptr_t)d.A % 16 == 0 && (uintptr_t)d.B % 16 == 0 &&
                  ((d.lda | d.sA | d.tsA | d.K | d.ldb | d.sB | d.tsB | d.N) & 1) == 0;
  const dim3 gr((unsigned)tiles, (unsigned)d.ngroups, (unsigned)d.batch);
  auto launch = [&](auto kern, size_t shm) {
    allow_lds((const void*)kern, shm);
    hipLaunchKernelGGL(kern, gr, dim3(256), shm, c->stream, d);
  };
  constexpr size_t s64 = TileCfg<double, 0, 0, 64, tile_bk<double>(64)>::LDS;
  constexpr size_t s32 = TileCfg<double, 0, 0, 32, tile_bk<double>(32)>::LDS;
  if (far) launch(gemm_grouped_kernel<LOAD_FAR, 64>, s64);
  else if (bm == 64 && al) launch(gemm_grouped_kernel<LOAD_VEC, 64>, s64);
  else if (bm == 64) launch(gemm_grouped_kernel<LOAD_ELEM, 64>, s64);
  else if (al) launch(gemm_grouped_kernel<LOAD_VEC, 32>, s32);
  else launch(gemm_grouped_kernel<LOAD_ELEM, 32>, s32);
  TN_HIP(hipGetLastError());
}

void gemm_blocksparse(tn_ctx* c, Prec p, const BsDesc& d) {
  if (d.ntiles <= 0) return;
  TN_REQUIRE(p == Prec::F64 || p == Prec::F32 || p == Prec::BF16X3, TN_E_INVALID,
             "block-sparse gemm: FP64, FP32 or BF16x3 (FP32 operands) only");
  TN_REQUIRE(d.ntiles % 8 == 0 && d.ntiles < (1L << 31), TN_E_INVALID, "block-sparse gemm: bad tile list");
  const size_t es = p == Prec::F64 ? 8 : 4;
  const bool far = !extent_ok(d.lda, BS_TILE, BS_TILE, es) || !extent_ok(d.ldb, BS_TILE, BS_TILE, es);
  auto launch = [&](auto kern, size_t shm) {
    allow_lds((const void*)kern, shm);
    hipLaunchKernelGGL(kern, dim3((unsigned)d.ntiles), dim3(256), shm, c->stream, d);
  };
#define TN_BS(T, TB, SPLIT)                                                                                   \
  do {                                                                                                        \
    constexpr size_t shm = TileCfg<T, 0, TB, BS_TILE, SPLIT ? 16 : tile_bk<T>(BS_TILE)>::LDS;                 \
    if (far) launch(gemm_bs_kernel<T, TB, SPLIT, LOAD_FAR>, shm);                                             \
    else launch(gemm_bs_kernel<T, TB, SPLIT, LOAD_ELEM>, shm);                                                \
  } while (0)
  if (p == Prec::F64) {
    if (d.tB) TN_BS(double, 1, false);
    else TN_BS(double, 0, false);
  } else if (p == Prec::F32) {
    if (d.tB) TN_BS(float, 1, false);
    else TN_BS(float, 0, false);
  } else {
    if (d.tB) TN_BS(float, 1, true);
    else TN_BS(float, 0, true);
  }
#undef TN_BS
  TN_HIP(hipGetLastError());
}

void gemm_bf16x3_nt(tn_ctx* c, long M, long N, long K, const unsigned short* Ah, const unsigned short* Al,
                    long lda, const unsigned short* Bh, const unsigned short* Bl, long ldb, float* C, long ldc) {
  if (M == 0 || N == 0) return;
  TN_REQUIRE(lda % 8 == 0 && ldb % 8 == 0 && lda >= ((K + 7) / 8) * 8 && ldb >= ((K + 7) / 8) * 8,
             TN_E_INVALID, "gemm_bf16x3_nt: rows must be padded to 8 bf16");
  TN_REQUIRE((size_t)std::max(lda, ldb) * 2 * 130 < ((size_t)1 << 31), TN_E_INVALID,
             "gemm_bf16x3_nt: row stride too large for 32-bit tile offsets");
  SArgs a{M, N, K, Ah, Al, lda, Bh, Bl, ldb, C, ldc};
  const long ntm = (M + SBM - 1) / SBM, ntn = (N + SBN - 1) / SBN;
  const size_t shm = 2 * (size_t)SCfg<32>::STAGE * sizeof(unsigned short);
  allow_lds((const void*)gemm_bf16x3_nt_kernel<32>, shm);
  hipLaunchKernelGGL(gemm_bf16x3_nt_kernel<32>, dim3((unsigned)(ntm * ntn)), dim3(256), shm, c->stream, a);
  TN_HIP(hipGetLastError());
}

void split_bf16(tn_ctx* c, const void* src, bool src_f64, long rows, long cols, long lds, bool transpose,
                unsigned short* hi, unsigned short* lo, long ldd) {
  if (rows == 0 || cols == 0) return;
  if (!transpose) {
    const long total = rows * ldd;
    const int g = (int)std::min<long>(8192, (total + 255) / 256);
    if (src_f64)
      hipLaunchKernelGGL(split_rows_kernel<double>, dim3(g), dim3(256), 0, c->stream, (const double*)src, rows,
                         cols, lds, hi, lo, ldd);
    else
      hipLaunchKernelGGL(split_rows_kernel<float>, dim3(g), dim3(256), 0, c->stream, (const float*)src, rows,
                         cols, lds, hi, lo, ldd);
  } else {
    // output is cols x ldd with ldd >= rows
    const long orows = std::max(rows, ldd);
    dim3 grid((unsigned)((cols + 31) / 32), (unsigned)((orows + 31) / 32));
    TN_REQUIRE((orows + 31) / 32 <= 65535, TN_E_INVALID, "split_bf16: too many rows");
    if (src_f64)
      hipLaunchKernelGGL(split_transpose_kernel<double>, grid, dim3(256), 0, c->stream, (const double*)src, rows,
                         cols, lds, hi, lo, ldd);
    else
      hipLaunchKernelGGL(split_transpose_kernel<float>, grid, dim3(256), 0, c->stream, (const float*)src, rows,
                         cols, lds, hi, lo, ldd);
  }
  TN_HIP(hipGetLastError());
}

}  // namespace tn
