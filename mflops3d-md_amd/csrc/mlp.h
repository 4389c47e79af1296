// The learned closure's network, 10 -> 64 -> 64 -> 6 (tanh), on the FP32
// matrix cores: inference and the gradient of a training pass.
//
// Every product is v_mfma_f32_16x16x4f32 on FP32 operands (the bf16 weights
// widened, which is exact) with FP32 accumulation, units along the rows and
// 16 samples along the columns.  Such a product leaves lane l with units
// 4 (l/16) + r (r = 0..3) of sample l%16, and the next one wants, in lane l,
// one unit of sample l%16 per k-step: taking k-step r over the units
// {4 g + r} makes register r the operand as it stands, so the whole forward
// and backward chain of 16 samples stays in one wave's registers, without
// LDS.  The first layer's bias rides in its padded k (input 10 is 1).
//
// What bounds it: 5 120 multiply-adds per sample forward (92 MFMAs of 32
// cycles per 16 samples with the padding), 15 000 with the gradient (268), on
// 154 TFLOP/s of measured FP32 matrix rate, beside 128 tanhf per sample on
// the vector units; the input and output rows are 64 B per sample.  Measured
// at 1 045 568 samples: loss and gradient 0.44 ms (9.96 ms with one sample per
// lane on vector FMAs, 64-sample partials in memory and a serial sum of them).
#pragma once
#include <hip/hip_runtime.h>

namespace mf {
namespace les {

constexpr int I0 = 10, H = 64, O = 6;
constexpr int NW1 = H * I0, NW2 = H * H, NW3 = O * H;
constexpr int OB1 = NW1, OW2 = OB1 + H, OB2 = OW2 + NW2, OW3 = OB2 + H, OB3 = OW3 + NW3;
constexpr int NPARAM = OB3 + O;  // 5254

constexpr int MLP_WAVES = 4;               // wavefronts per block, 16 samples each per pass
constexpr int MLP_TILE = 16 * MLP_WAVES;   // samples per block and pass

typedef float mlp_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(unsigned short b) { return __uint_as_float((unsigned)b << 16); }

// four bf16 at an 8-byte aligned address, widened
__device__ __forceinline__ mlp_f4 mlp_widen4(const unsigned short *q) {
  const uint2 v = *(const uint2 *)q;
  return (mlp_f4){__uint_as_float(v.x << 16), __uint_as_float(v.x & 0xffff0000u),
                  __uint_as_float(v.y << 16), __uint_as_float(v.y & 0xffff0000u)};
}

__device__ __forceinline__ mlp_f4 mlp_mma(float a, float b, mlp_f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// The first layer's operand: W1 and, as input 10, b1; a[ib][st] is row
// 16 ib + l%16, input g + 4 st
__device__ __forceinline__ void mlp_load_w1(float (&a)[4][3], const unsigned short *wb,
                                            const float *p, int c, int g) {
#pragma unroll
  for (int ib = 0; ib < 4; ++ib)
#pragma unroll
    for (int st = 0; st < 3; ++st) {
      const int i = 16 * ib + c, k = g + 4 * st;
      a[ib][st] = k < I0 ? bf2f(wb[i * I0 + k]) : (k == I0 ? p[OB1 + i] : 0.0f);
    }
}

// Inputs g + 4 st of sample s (1 for input 10; 0 beyond the inputs and the samples)
__device__ __forceinline__ void mlp_load_x(float (&x)[3], const float *X, long s, long n, int g) {
#pragma unroll
  for (int st = 0; st < 3; ++st) {
    const int k = g + 4 * st;
    x[st] = k < I0 ? (s < n ? X[s * I0 + k] : 0.0f) : (k == I0 ? 1.0f : 0.0f);
  }
}

// Inference.  Each wave keeps the three weight operands in registers (92) and
// walks 16-sample tiles with the grid's stride, one tile's inputs ahead.
__global__ void __launch_bounds__(64 * MLP_WAVES, 2)
    mlp_forward_kernel(const float *__restrict__ X, float *__restrict__ Y, long n,
                       const unsigned short *__restrict__ wb, const float *__restrict__ p) {
  const int l = threadIdx.x & 63, c = l & 15, g = l >> 4;
  const long wave = (long)blockIdx.x * MLP_WAVES + (threadIdx.x >> 6);
  const long nwaves = (long)gridDim.x * MLP_WAVES, tiles = (n + 15) / 16;
  if (wave >= tiles) return;
  float w1[4][3], x[3];
  mlp_f4 w2[4][4], w3[4], b2[4], b3;
  mlp_load_x(x, X, wave * 16 + c, n, g);
  mlp_load_w1(w1, wb, p, c, g);
#pragma unroll
  for (int ib = 0; ib < 4; ++ib)
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
      w2[ib][kb] = mlp_widen4(wb + NW1 + (16 * ib + c) * H + 16 * kb + 4 * g);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb) {
    w3[kb] = mlp_widen4(wb + NW1 + NW2 + min(c, O - 1) * H + 16 * kb + 4 * g);
#pragma unroll
    for (int r = 0; r < 4; ++r) b2[kb][r] = p[OB2 + 16 * kb + 4 * g + r];
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) b3[r] = 4 * g + r < O ? p[OB3 + 4 * g + r] : 0.0f;
  for (long t = wave; t < tiles; t += nwaves) {
    float xn[3];
    mlp_load_x(xn, X, (t + nwaves) * 16 + c, n, g);
    mlp_f4 h[4], z[4], y[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) h[ib] = (mlp_f4){0, 0, 0, 0};
#pragma unroll
    for (int st = 0; st < 3; ++st)
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) h[ib] = mlp_mma(w1[ib][st], x[st], h[ib]);
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      z[ib] = b2[ib];
      y[ib] = ib == 0 ? b3 : (mlp_f4){0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) h[ib][r] = tanhf(h[ib][r]);
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) z[ib] = mlp_mma(w2[ib][kb][r], h[kb][r], z[ib]);
#pragma unroll
    for (int kb = 0; kb < 4; ++kb)
#pragma unroll
      for (int r = 0; r < 4; ++r) y[kb] = mlp_mma(w3[kb][r], tanhf(z[kb][r]), y[kb]);
    const long s = t * 16 + c;
    if (s < n && g < 2) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (4 * g + r < O) Y[s * O + 4 * g + r] = (y[0][r] + y[1][r]) + (y[2][r] + y[3][r]);
    }
#pragma unroll
    for (int st = 0; st < 3; ++st) x[st] = xn[st];
  }
}

// Gradient of sum_s sum_c (Y - T)^2 / n: part[blk (NPARAM + 1) + q], FP64
// (q = NPARAM: the block's loss term).
//
// A block walks 64-sample tiles with the grid's stride.  Per tile each wave
// runs its 16 samples forward and backward in registers; the weight gradients
// contract over samples, which needs the transposed operands: the wave puts
// h1, h2, dh2, dh1 into LDS as [unit][sample] (row pitch 68: both the 4-byte
// writes along a row and the 16-byte reads down 16 rows are conflict-free),
// and wave w then forms rows 16 w .. 16 w + 15 of dW2 and dW1 and columns
// 16 w .. of dW3 over the tile's 64 samples.  So a block holds one copy of the
// gradient (24 FP32 accumulators per lane), and each tile's FP32 sums are
// added into FP64 ones, as many samples per FP32 sum as the tile has.  Three
// LDS buffers (dh1 reuses h2's) let two blocks share a CU: one's tanhf and
// barriers run beside the other's MFMAs.  W2 lies in LDS once, widened: as two
// bf16 copies (one transposed) every operand had to be widened in each tile,
// which took 0.03 of 0.47 ms.
constexpr int MLP_PITCH = MLP_TILE + 4;
constexpr int MLP_WP = H + 8;  // bf16 pitch of the weight matrices in LDS

__global__ void __launch_bounds__(64 * MLP_WAVES, 2)
    mlp_grad_kernel(const float *__restrict__ X, const float *__restrict__ T, long n,
                    const unsigned short *__restrict__ wb, const float *__restrict__ p,
                    double *__restrict__ part) {
  // read four values at a time (mlp_f4, mlp_widen4): aligned bases and pitches
  __shared__ alignas(16) float S[3][H][MLP_PITCH];     // h2 then dh1 | dh2 | h1
  __shared__ alignas(16) float SX[I0 + 1][MLP_PITCH];  // inputs and a row of ones
  __shared__ alignas(16) float SD[O][MLP_PITCH];       // dY
  __shared__ alignas(16) float W2[H][MLP_PITCH];       // widened; rows forward, columns backward
  __shared__ alignas(16) unsigned short W3[O][MLP_WP], W3t[H][8];
  __shared__ alignas(16) float B2[H];
  static_assert(MLP_PITCH * sizeof(float) % sizeof(mlp_f4) == 0 &&
                MLP_WP * sizeof(unsigned short) % sizeof(uint2) == 0, "rows stay aligned");
  const int tid = threadIdx.x, l = tid & 63, c = l & 15, g = l >> 4;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int t = tid; t < NW2; t += 64 * MLP_WAVES) W2[t / H][t % H] = bf2f(wb[NW1 + t]);
  for (int t = tid; t < NW3; t += 64 * MLP_WAVES) W3[t / H][t % H] = wb[NW1 + NW2 + t];
  for (int t = tid; t < 8 * H; t += 64 * MLP_WAVES)
    W3t[t / 8][t % 8] = t % 8 < O ? wb[NW1 + NW2 + (t % 8) * H + t / 8] : (unsigned short)0;
  if (tid < H) B2[tid] = p[OB2 + tid];
  float w1[4][3];
  mlp_load_w1(w1, wb, p, c, g);
  mlp_f4 b3;
#pragma unroll
  for (int r = 0; r < 4; ++r) b3[r] = 4 * g + r < O ? p[OB3 + 4 * g + r] : 0.0f;
  const float inv_n = 1.0f / (float)n;
  const long tiles = (n + MLP_TILE - 1) / MLP_TILE;
  const int sl = 16 * w + c;  // this lane's sample within the tile
  const int oc = min(c, O - 1), kc = min(c, I0);
  double g2[4][4] = {}, g1[4] = {}, g3[4] = {}, gb2 = 0.0, gb3 = 0.0, loss = 0.0;
  float x[3], tv[4];
  auto load_t = [&](long s) {
#pragma unroll
    for (int r = 0; r < 4; ++r)
      tv[r] = (4 * g + r < O && s < n) ? T[s * O + 4 * g + r] : 0.0f;
  };
  mlp_load_x(x, X, (long)blockIdx.x * MLP_TILE + sl, n, g);
  load_t((long)blockIdx.x * MLP_TILE + sl);
  __syncthreads();
  for (long t = blockIdx.x; t < tiles; t += gridDim.x) {
    const long s = t * MLP_TILE + sl;
    mlp_f4 h1[4], h2[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) h1[ib] = (mlp_f4){0, 0, 0, 0};
#pragma unroll
    for (int st = 0; st < 3; ++st)
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) h1[ib] = mlp_mma(w1[ib][st], x[st], h1[ib]);
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      h2[ib] = *(const mlp_f4 *)&B2[16 * ib + 4 * g];
#pragma unroll
      for (int r = 0; r < 4; ++r) h1[ib][r] = tanhf(h1[ib][r]);
    }
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      mlp_f4 a[4];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib) a[ib] = *(const mlp_f4 *)&W2[16 * ib + c][16 * kb + 4 * g];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) h2[ib] = mlp_mma(a[ib][r], h1[kb][r], h2[ib]);
    }
    mlp_f4 y[4];
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const mlp_f4 a = mlp_widen4(&W3[oc][16 * kb + 4 * g]);
      y[kb] = kb == 0 ? b3 : (mlp_f4){0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        h2[kb][r] = tanhf(h2[kb][r]);
        y[kb] = mlp_mma(a[r], h2[kb][r], y[kb]);
      }
    }
    mlp_f4 dy;
    float ls = 0.0f;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const float yr = (y[0][r] + y[1][r]) + (y[2][r] + y[3][r]);
      const float d = (4 * g + r < O && s < n) ? yr - tv[r] : 0.0f;
      ls = fmaf(d, d, ls);
      dy[r] = 2.0f * d * inv_n;
    }
    loss += (double)ls;
    // dh2 = (W3^T dY) (1 - h2^2); outputs 8.. of the padded k carry zero weights
    mlp_f4 d2[4], d1[4];
#pragma unroll
    for (int ib = 0; ib < 4; ++ib) {
      mlp_f4 a = mlp_widen4(&W3t[16 * ib + c][4 * (g & 1)]);
      d2[ib] = d1[ib] = (mlp_f4){0, 0, 0, 0};
#pragma unroll
      for (int r = 0; r < 4; ++r) d2[ib] = mlp_mma(g < 2 ? a[r] : 0.0f, dy[r], d2[ib]);
    }
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) d2[ib][r] *= 1.0f - h2[ib][r] * h2[ib][r];
    // the previous tile's last reads of the buffers are behind this barrier
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int u = 16 * ib + 4 * g + r;
        S[0][u][sl] = h2[ib][r];
        S[1][u][sl] = d2[ib][r];
        S[2][u][sl] = h1[ib][r];
      }
#pragma unroll
    for (int st = 0; st < 3; ++st)
      if (g + 4 * st <= I0) SX[g + 4 * st][sl] = x[st];
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (4 * g + r < O) SD[4 * g + r][sl] = dy[r];
    // the next tile's inputs and targets, a whole tile ahead of their use
    mlp_load_x(x, X, s + (long)gridDim.x * MLP_TILE, n, g);
    load_t(s + (long)gridDim.x * MLP_TILE);
    // dh1 = (W2^T dh2) (1 - h1^2), over the barrier's wait
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      mlp_f4 a[4];
#pragma unroll
      for (int ib = 0; ib < 4; ++ib)
#pragma unroll
        for (int r = 0; r < 4; ++r) a[ib][r] = W2[16 * kb + 4 * g + r][16 * ib + c];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int ib = 0; ib < 4; ++ib) d1[ib] = mlp_mma(a[ib][r], d2[kb][r], d1[ib]);
    }
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) d1[ib][r] *= 1.0f - h1[ib][r] * h1[ib][r];
    __syncthreads();
    // dW3 (columns 16 w ..), dW2 (rows 16 w ..) over the tile's samples
    {
      mlp_f4 a3 = {0, 0, 0, 0}, a2[4];
      float s3 = 0.0f, s2 = 0.0f;
#pragma unroll
      for (int q = 0; q < 4; ++q) a2[q] = (mlp_f4){0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < MLP_TILE / 16; ++m) {
        const int o = 16 * m + 4 * g;
        const mlp_f4 fd = *(const mlp_f4 *)&SD[oc][o], fh = *(const mlp_f4 *)&S[0][16 * w + c][o];
        const mlp_f4 fa = *(const mlp_f4 *)&S[1][16 * w + c][o];
        mlp_f4 fb[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) fb[q] = *(const mlp_f4 *)&S[2][16 * q + c][o];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          a3 = mlp_mma(fd[r], fh[r], a3);
#pragma unroll
          for (int q = 0; q < 4; ++q) a2[q] = mlp_mma(fa[r], fb[q][r], a2[q]);
          s3 += fd[r];
          s2 += fa[r];
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        g3[r] += (double)a3[r];
#pragma unroll
        for (int q = 0; q < 4; ++q) g2[q][r] += (double)a2[q][r];
      }
      gb3 += (double)s3;
      gb2 += (double)s2;
    }
    __syncthreads();
#pragma unroll
    for (int ib = 0; ib < 4; ++ib)
#pragma unroll
      for (int r = 0; r < 4; ++r) S[0][16 * ib + 4 * g + r][sl] = d1[ib][r];
    __syncthreads();
    // dW1 and, as its column 10, db1 (rows 16 w ..)
    {
      mlp_f4 a1 = {0, 0, 0, 0};
#pragma unroll
      for (int m = 0; m < MLP_TILE / 16; ++m) {
        const int o = 16 * m + 4 * g;
        const mlp_f4 fa = *(const mlp_f4 *)&S[0][16 * w + c][o], fx = *(const mlp_f4 *)&SX[kc][o];
#pragma unroll
        for (int r = 0; r < 4; ++r) a1 = mlp_mma(fa[r], fx[r], a1);
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) g1[r] += (double)a1[r];
    }
  }
  double *out = part + (long)blockIdx.x * (NPARAM + 1);
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int i = 16 * w + 4 * g + r;
#pragma unroll
    for (int q = 0; q < 4; ++q) out[OW2 + i * H + 16 * q + c] = g2[q][r];
    if (4 * g + r < O) out[OW3 + (4 * g + r) * H + 16 * w + c] = g3[r];
    if (c < I0) out[i * I0 + c] = g1[r];
    else if (c == I0) out[OB1 + i] = g1[r];
  }
  for (int o = 16; o < 64; o <<= 1) {
    gb2 += __shfl_xor(gb2, o, 64);
    gb3 += __shfl_xor(gb3, o, 64);
  }
  if (g == 0) out[OB2 + 16 * w + c] = gb2;
  if (w == 0 && g == 0 && c < O) out[OB3 + c] = gb3;
  for (int o = 1; o < 64; o <<= 1) loss += __shfl_xor(loss, o, 64);
  __shared__ double ls[MLP_WAVES];
  if (l == 0) ls[w] = loss;
  __syncthreads();
  if (tid == 0) {
    double a = 0.0;
    for (int q = 0; q < MLP_WAVES; ++q) a += ls[q];
    out[NPARAM] = a / (double)n;
  }
}

// grad[q] = sum_b part[b (NPARAM + 1) + q] in a fixed order: 64 parameters per
// block, wave v the partials v, v + 16, ..., then the 16 waves' sums in order
constexpr int MLP_RED = 16;
__global__ void __launch_bounds__(64 * MLP_RED)
    mlp_reduce_kernel(const double *__restrict__ part, int nb, float *__restrict__ grad) {
  __shared__ double sh[MLP_RED][64];
  const int l = threadIdx.x & 63, v = threadIdx.x >> 6;
  const int q = blockIdx.x * 64 + l;
  double a = 0.0;
  if (q <= NPARAM) {
#pragma unroll 8
    for (int b = v; b < nb; b += MLP_RED) a += part[(long)b * (NPARAM + 1) + q];
  }
  sh[v][l] = a;
  __syncthreads();
  if (v == 0 && q <= NPARAM) {
    for (int k = 1; k < MLP_RED; ++k) a += sh[k][l];
    grad[q] = (float)a;
  }
}

}  // namespace les
}  // namespace mf
