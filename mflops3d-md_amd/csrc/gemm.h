// MFMA tensor-mode products for the diagonalisation solver (gfx950).
//
// Every eigenvector transform of solve_3d (dgx/dgy/dgz,
// class_solver_3d.f90:307-378) is a column-major GEMM C = A B:
//   x-transform:  C(n1, n2 n3) = W(n1,n1) . F(n1, n2 n3)          (W left)
//   y-transform:  C_k(n1, n2)  = F_k(n1,n2) . Wt(n2,n2), k = 1..n3 (W right, batched)
//   z-transform:  C(n1 n2, n3) = F(n1 n2, n3) . Wt(n3,n3)         (W right)
// In all three A is M-contiguous.  B is K-contiguous where it is the field
// (x) and N-contiguous where it is the matrix (y and z: W itself, whose
// columns are Wt's rows).
//
// One wave forms one (16 MI) x (16 NI) tile of C on its own: the MFMA
// operands come straight from global memory into registers, D k-steps ahead,
// with no LDS and no barrier.  A 16 x 16 x 4 FP64 MFMA occupies its SIMD for
// 64 cycles, so a 64 x 64 tile spends 1024 cycles on a k-step's 8 loads of
// 512 bytes; the waves of a block take the tiles that share the field's
// values, which then come from L1, and the matrix streams from L2.  What bounds
// it is the matrix rate on large problems and, on small ones, the latency of
// one pass of loads: there the tiles shrink until every SIMD has a wave
// (gemm_tile_of), and with 16 k-steps ahead a 62-point axis is one pass.
//
// MFMA operand order is swapped (D = B^T-fragment x A-fragment) so that the
// 16 lanes holding one D row are 16 consecutive m: stores of the
// column-major C are 128-byte contiguous segments.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "gemm_tile.h"

namespace mf {

typedef double d4_t __attribute__((ext_vector_type(4)));
typedef float f4_t __attribute__((ext_vector_type(4)));

template <typename T>
struct Mfma;
// Operand layout (both types): lane l supplies A[l%16][l/16] and B[l/16][l%16].
// Output layout differs: result r of lane l is D[row(l,r)][l%16] with
// row = l/16 + 4r for the f64 instruction and 4(l/16) + r for the f32 one
// (measured on gfx950).
template <>
struct Mfma<double> {
  typedef d4_t acc_t;
  static __device__ __forceinline__ acc_t op(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return (lane >> 4) + 4 * r; }
};
template <>
struct Mfma<float> {
  typedef f4_t acc_t;
  static __device__ __forceinline__ acc_t op(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int lane, int r) { return 4 * (lane >> 4) + r; }
};

// R = 1 / (lx + ly + lz + sigma), 0 where max(|sigma|, |l|) < 1e-11 (the
// eigen-divide's null-mode guard, class_solver_3d.f90:202-225)
__device__ __forceinline__ double inv_eig(double lx, double ly, double lz, double sigma) {
  const double big = fmax(fmax(fabs(sigma), fmax(fabs(lx), fabs(ly))), fabs(lz));
  return big < 1e-11 ? 0.0 : 1.0 / (((lx + ly) + lz) + sigma);
}

enum EpiMode {
  EPI_STORE = 0, EPI_DIVIDE = 1, EPI_SCATTER = 2, EPI_SCATTER_ADD = 3, EPI_FIELDS = 4, EPI_TAU = 5
};

struct EpiArgs {
  // EPI_DIVIDE: m = i1 + n1*i2, n = i3 -> value / (lx[i1]+ly[i2]+lz[i3]+sigma),
  // 0 where max(|sigma|,|lx|,|ly|,|lz|) < 1e-11 (class_solver_3d.f90:202-225)
  const double *lx, *ly, *lz;
  double sigma;
  int n1, n2;
  // EPI_SCATTER(_ADD): m = i, n = j + n2*k -> u[(i+1) + nx((j+1) + ny(k+1))]
  double *u;
  int nx, ny;
  // EPI_FIELDS: batch b -> out[b] instead of C + sC b.  EPI_TAU: batch b is the
  // filtered product of fields p and q, point t = m + ldc n:
  // tau[6 t + col[b]] = (value - p[b][t] q[b][t]) inv
  double *out[3];
  const double *p[3], *q[3];
  float *tau;
  int col[3];
  double inv;
};

// The products of one tile of C = A B, rows from m0 and columns from n0, by one
// wave: lane l ends with C(m0 + 16 mi + l%16, n0 + 16 ni + row(l, r)) in
// acc[mi][ni][r].  A: M-contiguous; B: K-contiguous (KB) or N-contiguous.
template <typename T, int MI, int NI, int D, bool KB>
__device__ __forceinline__ void gemm_tile(const T *__restrict__ A, long lda,
                                          const T *__restrict__ B, long ldb, int M, int N, int K,
                                          int m0, int n0, typename Mfma<T>::acc_t (&acc)[MI][NI]) {
  typedef typename Mfma<T>::acc_t acc_t;
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int a = 0; a < MI; ++a)
#pragma unroll
    for (int b = 0; b < NI; ++b) acc[a][b] = (acc_t){0, 0, 0, 0};

  // Operand pointers at k = 4 s + g of step s.  Rows and columns past the
  // edge repeat the last one (their results are not stored); in the last step
  // lanes past K repeat k = K - 1 and their operands are set to zero.
  const int KS = (K + 3) / 4;
  const int over = max(0, 4 * (KS - 1) + g - (K - 1));
  const long sb = KB ? 1 : ldb;
  const long a4 = 4 * lda, b4 = 4 * sb, aL = (4 - over) * lda, bL = (4 - over) * sb;
  const T *pa[MI], *pb[NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
    pa[i] = A + min(m0 + 16 * i + c, M - 1) + lda * (KS == 1 ? g - over : g);
#pragma unroll
  for (int i = 0; i < NI; ++i)
    pb[i] = B + (long)min(n0 + 16 * i + c, N - 1) * (KB ? ldb : 1) + sb * (KS == 1 ? g - over : g);
  T af[D][MI], bf[D][NI];
  // fetch step s into slot d and move the pointers to step s + 1
  auto fetch = [&](int d, int s) {
#pragma unroll
    for (int i = 0; i < MI; ++i) af[d][i] = *pa[i];
#pragma unroll
    for (int i = 0; i < NI; ++i) bf[d][i] = *pb[i];
    const bool last = s + 2 == KS, end = s + 2 > KS;
    const long da = end ? 0 : (last ? aL : a4), db = end ? 0 : (last ? bL : b4);
#pragma unroll
    for (int i = 0; i < MI; ++i) pa[i] += da;
#pragma unroll
    for (int i = 0; i < NI; ++i) pb[i] += db;
  };
  auto mma = [&](int d) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        acc[mi][ni] = Mfma<T>::op(bf[d][ni], af[d][mi], acc[mi][ni]);
  };
  auto mma_end = [&](int d, int s) {  // a step that may be the last
    if (s + 1 == KS && over > 0) {
#pragma unroll
      for (int i = 0; i < MI; ++i) af[d][i] = (T)0;
#pragma unroll
      for (int i = 0; i < NI; ++i) bf[d][i] = (T)0;
    }
    mma(d);
  };
  // every fetch is unconditional (past the last step it repeats it), so that the
  // compiler waits for exactly the loads each step needs
#pragma unroll
  for (int d = 0; d < D; ++d) fetch(d, d);
  int s = 0;
  for (; s + 2 * D <= KS; s += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      mma(d);
      fetch(d, s + d + D);
    }
  }
  if (s + D < KS) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      mma(d);
      fetch(d, s + d + D);
    }
    s += D;
  }
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (s + d < KS) mma_end(d, s + d);
}

// The same for a K-contiguous B, 16 k at a time (K >= 16): in step r of four,
// lane (c, g) takes k = 16 q + 4 g + r, so that it loads the four steps' values
// of B as one vector (at any alignment of T).  One value a step touches 16 cache
// lines for 256 bytes where T is 32 bits wide, and that bound the FP32 x
// transform: 124 us at 254^3 on 64 x 64 tiles, 61 at 192 x 256 x 192 on 64 x 48.
// With vectors, four quads ahead, 32 x 32 tiles do best: 96 and 44 us (staged
// through LDS 101 and 46); 3.5 us for 4.7 at 64^3 on 16 x 16.
template <typename T, int MI, int NI, int Q>
__device__ __forceinline__ void gemm_tile_quads(const T *__restrict__ A, long lda,
                                                const T *__restrict__ B, long ldb, int M, int N,
                                                int K, int m0, int n0,
                                                typename Mfma<T>::acc_t (&acc)[MI][NI]) {
  typedef typename Mfma<T>::acc_t acc_t;
  typedef T vec_t __attribute__((ext_vector_type(4), aligned(sizeof(T))));
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
#pragma unroll
  for (int a = 0; a < MI; ++a)
#pragma unroll
    for (int b = 0; b < NI; ++b) acc[a][b] = (acc_t){0, 0, 0, 0};

  // The last 16 k are K - 16 .. K - 1; the first `over` of them, which the quad
  // before holds, are set to zero.
  const int KQ = (K + 15) / 16, over = 16 * KQ - K;
  const T *pa[MI], *pb[NI];
#pragma unroll
  for (int i = 0; i < MI; ++i) pa[i] = A + min(m0 + 16 * i + c, M - 1) + lda * (4 * g);
#pragma unroll
  for (int i = 0; i < NI; ++i) pb[i] = B + (long)min(n0 + 16 * i + c, N - 1) * ldb + 4 * g;
  T af[Q][4][MI];
  vec_t bf[Q][NI];
  // k from quad q to the next
  auto step = [&](int q) { return q + 2 > KQ ? 0 : (q + 2 == KQ ? 16 - over : 16); };
  auto fetch_a = [&](int d, int r, int q) {
#pragma unroll
    for (int i = 0; i < MI; ++i) af[d][r][i] = *pa[i];
    const long da = r < 3 ? lda : (step(q) - 3) * lda;
#pragma unroll
    for (int i = 0; i < MI; ++i) pa[i] += da;
  };
  auto fetch_b = [&](int d, int q) {
#pragma unroll
    for (int i = 0; i < NI; ++i) bf[d][i] = *(const vec_t *)pb[i];
    const int db = step(q);
#pragma unroll
    for (int i = 0; i < NI; ++i) pb[i] += db;
  };
  auto mma = [&](int d, int r) {
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int ni = 0; ni < NI; ++ni)
        acc[mi][ni] = Mfma<T>::op(bf[d][ni][r], af[d][r][mi], acc[mi][ni]);
  };
#pragma unroll
  for (int d = 0; d < Q; ++d) {
    fetch_b(d, d);
#pragma unroll
    for (int r = 0; r < 4; ++r) fetch_a(d, r, d);
  }
  int q = 0;
  for (; q + Q < KQ; q += Q) {
#pragma unroll
    for (int d = 0; d < Q; ++d) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        mma(d, r);
        fetch_a(d, r, q + d + Q);
      }
      fetch_b(d, q + d + Q);
    }
  }
#pragma unroll
  for (int d = 0; d < Q; ++d)
    if (q + d < KQ) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (q + d + 1 == KQ && 4 * g + r < over) {
#pragma unroll
          for (int i = 0; i < MI; ++i) af[d][r][i] = (T)0;
#pragma unroll
          for (int i = 0; i < NI; ++i) bf[d][i][r] = (T)0;
        }
        mma(d, r);
      }
    }
}

// A: M-contiguous; B: K-contiguous (KB) or N-contiguous.  tm x tn x batch
// tiles, one per wave: the M tiles of a column group in turn when the field is
// B, the N tiles of a row group when it is A.  QUADS: the products by gemm_tile_quads, D / 4 quads ahead.
template <typename T, typename TC, int MI, int NI, int D, bool KB, bool QUADS, int EPI>
__global__ void __launch_bounds__(256, 2)
    gemm_mode_kernel(const T *__restrict__ A, long lda, long sA, const T *__restrict__ B, long ldb,
                     TC *__restrict__ C, long ldc, long sC, int M, int N, int K, int tm, int tn,
                     long waves, EpiArgs ep) {
  typedef typename Mfma<T>::acc_t acc_t;
  const int lane = threadIdx.x & 63, c = lane & 15;
  const int wv = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wv >= waves) return;
  int im, in, ib;
  if (KB) { im = wv % tm; in = (wv / tm) % tn; }
  else { in = wv % tn; im = (wv / tn) % tm; }
  ib = wv / (tm * tn);
  const int m0 = im * 16 * MI, n0 = in * 16 * NI;
  A += (long)ib * sA;
  if (EPI == EPI_STORE || EPI == EPI_DIVIDE) C += (long)ib * sC;
  if (EPI == EPI_FIELDS) C = (TC *)ep.out[ib];

  acc_t acc[MI][NI];
  if constexpr (QUADS)
    gemm_tile_quads<T, MI, NI, D / 4>(A, lda, B, ldb, M, N, K, m0, n0, acc);
  else
    gemm_tile<T, MI, NI, D, KB>(A, lda, B, ldb, M, N, K, m0, n0, acc);
  // epilogue: lane holds C(m0+16mi+lane%16, n0+16ni+row(lane,r)).
  // Index splits (m -> i1,i2; n -> j,k) take one 32-bit division per lane and
  // then advance with wrap-around.
  int i1 = 0, i2 = 0;
  if (EPI == EPI_DIVIDE) {
    const int mb = m0 + c;
    i1 = mb % ep.n1;
    i2 = mb / ep.n1;
  }
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = m0 + mi * 16 + c;
    if (mi > 0 && EPI == EPI_DIVIDE) {
      i1 += 16;
      while (i1 >= ep.n1) { i1 -= ep.n1; ++i2; }
    }
    if (m >= M) continue;
    double lxy = 0.0, big_xy = 0.0;
    if (EPI == EPI_DIVIDE) {
      lxy = ep.lx[i1] + ep.ly[i2];
      big_xy = fmax(fabs(ep.lx[i1]), fabs(ep.ly[i2]));
    }
    long ubase = 0;
    int jb = 0, kb = 0;
    if (EPI == EPI_SCATTER || EPI == EPI_SCATTER_ADD) {
      ubase = m + 1;
      const int nb = n0;
      jb = nb % ep.n2;
      kb = nb / ep.n2;
    }
#pragma unroll
    for (int ni = 0; ni < NI; ++ni)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int dn = ni * 16 + Mfma<T>::row(lane, r);
        const int n = n0 + dn;
        if (n >= N) continue;
        const double v = (double)acc[mi][ni][r];
        if (EPI == EPI_STORE || EPI == EPI_FIELDS) {
          C[m + ldc * n] = (TC)v;
        } else if (EPI == EPI_TAU) {
          const long t = m + ldc * n;
          ep.tau[6 * t + ep.col[ib]] = (float)((v - ep.p[ib][t] * ep.q[ib][t]) * ep.inv);
        } else if (EPI == EPI_DIVIDE) {
          const double lzn = ep.lz[n];
          const double big = fmax(fmax(fabs(ep.sigma), big_xy), fabs(lzn));
          const double den = lxy + lzn + ep.sigma;
          if (sizeof(TC) == 8)
            C[m + ldc * n] = (TC)((big < 1e-11) ? 0.0 : v / den);
          else  // FP32 inner solve: FP32 reciprocal
            C[m + ldc * n] = (TC)((big < 1e-11) ? 0.0f : (float)v * __builtin_amdgcn_rcpf((float)den));
        } else {
          int j = jb + dn, k = kb;
          while (j >= ep.n2) { j -= ep.n2; ++k; }
          double *p = ep.u + ubase + (long)ep.nx * ((j + 1) + (long)ep.ny * (k + 1));
          if (EPI == EPI_SCATTER)
            *p = v;
          else
            *p += v;
        }
      }
  }
}

// C = A B (per batch) with the epilogue EPI, enqueued on st.
template <typename T, typename TC, bool KB, int EPI>
void gemm_launch(const T *A, long lda, long sA, const T *B, long ldb, TC *C, long ldc, long sC,
                 int M, int N, int K, int batch, const EpiArgs &ep, int ncu, hipStream_t st) {
  // FP32: x by quads; y and z with more k-steps ahead, since a step's MFMAs take
  // half the time (a z transform at 254^3 on 64 x 64 tiles 106 -> 90 us, at
  // 192 x 256 x 192 on 64 x 48 ones 50 -> 45)
  constexpr bool F32 = sizeof(T) == 4, X32 = KB && F32;
  const bool quads = X32 && K >= 16;
  const GemmTile t = X32 ? gemm_tile_x32(M, N, K, batch, ncu) : gemm_tile_of(M, N, K, batch, ncu);
  const int tm = (M + 16 * t.mi - 1) / (16 * t.mi), tn = (N + 16 * t.ni - 1) / (16 * t.ni);
  const long waves = (long)tm * tn * batch;
  const dim3 grid((unsigned)((waves + 3) / 4));
  auto go = [&](auto mi, auto ni, auto d, auto qd) {
    hipLaunchKernelGGL((gemm_mode_kernel<T, TC, decltype(mi)::value, decltype(ni)::value,
                                         decltype(d)::value, KB, decltype(qd)::value, EPI>),
                       grid, dim3(256), 0, st, A, lda, sA, B, ldb, C, ldc, sC, M, N, K, tm, tn,
                       waves, ep);
  };
  typedef std::integral_constant<int, 1> I1;
  typedef std::integral_constant<int, 2> I2;
  typedef std::integral_constant<int, 3> I3;
  typedef std::integral_constant<int, 4> I4;
  typedef std::integral_constant<int, F32 ? 6 : 4> D6;
  typedef std::integral_constant<int, F32 ? 8 : 4> D8;
  typedef std::integral_constant<int, 8> I8;
  typedef std::integral_constant<int, 16> I16;
  typedef std::false_type no;
  if constexpr (X32) {
    if (!quads) go(I1(), I1(), I16(), no());
    else if (t.mi == 2) go(I2(), I2(), I16(), std::true_type());
    else go(I1(), I1(), I16(), std::true_type());
  } else {
    switch (10 * t.mi + t.ni) {
      case 44: go(I4(), I4(), D8(), no()); break;
      case 43: go(I4(), I3(), D6(), no()); break;
      case 34: go(I3(), I4(), D6(), no()); break;
      case 33: go(I3(), I3(), D8(), no()); break;
      case 42: go(I4(), I2(), D8(), no()); break;
      case 24: go(I2(), I4(), D6(), no()); break;
      case 22: go(I2(), I2(), I8(), no()); break;
      default: go(I1(), I1(), I16(), no()); break;
    }
  }
}

}  // namespace mf
