// The influence operator y = M x applied without its matrix
// (md_influence_matrix_set, class_field.f90:1396-1510, as the solve needs it).
//
// With the blocks' one-axis factors (infl_spec.h), the response of a subdomain
// to values x on its interface faces and its boundary derivatives are
//   Xhat_f = W_b x_f W_c^T                     (face axes b < c of each face f)
//   U(a,b,c) = R(a,b,c) sum_f ahat_f(its axis) Xhat_f(the other two)
//   Ghat_t = sum over t's axis of what_t U,    y_t = V_b Ghat_t V_c^T
// plus dcoef x_f on the faces of t's own axis.  That is O(n^3) work and
// O(n^2) memory per subdomain, where the dense block is O(n^4) doubles to
// read per product: at 2 x 2 x 2 subdomains of 48-96 points 8.6 GB and 1.72 ms
// (5 TB/s) against six launches; a solve (9 iterations) 20.4 -> 2.8 ms, 2.0 with
// one wait per iteration.  The four transforms of all faces of all subdomains run
// as grouped launches of one-wave 16 x 16 tiles
// (gemm_tile), bounded by their latency at these sizes, as is the spectral
// sum, which forms R anew for each of the three axes it sums along rather than
// storing U.
#pragma once
#include <hip/hip_runtime.h>

#include "gemm.h"

namespace mf {

// One face's product of a grouped launch: C = A B, M x N x K.  Stages 0 and 2
// multiply from the left (B K-contiguous), 1 and 3 from the right (B
// N-contiguous).  a, b, c: offsets into the launch's base where the pointer is
// null.  x0, x1 (stage 3): offsets of the faces of this axis in the launch's x,
// -1 for none, with their weights.
struct ApplyProblem {
  const double *A, *B;
  long a, b, c;
  long lda, ldb, ldc;
  int M, N, K, tn;
  long x0, x1;
  double c0, c1;
};

// tile: tile of the launch -> (problem, tile within it)
template <bool KB, bool DIAG>
__global__ void __launch_bounds__(256)
    apply_gemm_kernel(const ApplyProblem *__restrict__ probs, const int2 *__restrict__ tile,
                      int tiles, const double *__restrict__ abase, const double *__restrict__ bbase,
                      double *__restrict__ cbase, const double *__restrict__ x) {
  const int wv = (int)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (wv >= tiles) return;
  const int2 t = tile[wv];
  const ApplyProblem &p = probs[t.x];
  const int m0 = 16 * (t.y / p.tn), n0 = 16 * (t.y % p.tn);
  const double *A = p.A ? p.A : abase + p.a, *B = p.B ? p.B : bbase + p.b;
  Mfma<double>::acc_t acc[1][1];
  gemm_tile<double, 1, 1, 16, KB>(A, p.lda, B, p.ldb, p.M, p.N, p.K, m0, n0, acc);
  const int lane = threadIdx.x & 63, m = m0 + (lane & 15);
  if (m >= p.M) return;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int n = n0 + Mfma<double>::row(lane, r);
    if (n >= p.N) continue;
    const long o = m + p.ldc * n;
    double v = acc[0][0][r];
    if (DIAG) {
      if (p.x0 >= 0) v = fma(p.c0, x[p.x0 + o], v);
      if (p.x1 >= 0) v = fma(p.c1, x[p.x1 + o], v);
    }
    cbase[p.c + o] = v;
  }
}

// The spectral sum along axis a of one subdomain for its no (1 or 2)
// interface faces on a.  Faces f: their axis, ahat and Xhat (offset; face
// axes ascending, lower one contiguous).
struct ApplyRole {
  int n[3];
  int a, nf, no;
  int fax[6];
  const double *ahat[6];
  long xoff[6];
  const double *what[2];
  long goff[2];
  const double *lam[3];
};

constexpr int APPLY_SPLIT = 4;  // waves per 64 face points, each a part of the summed axis

// NF: the most faces of any subdomain (a role with fewer adds zero times a
// finite value for the rest, so that the line's loads need no branch and four
// points' loads are in flight together: 33 us a product with one point at a
// time, at the sizes above)
template <int NF>
__global__ void __launch_bounds__(64 * APPLY_SPLIT)
    apply_sum_kernel(const ApplyRole *__restrict__ roles, const double *__restrict__ xhat,
                     double *__restrict__ ghat, double sigma) {
  __shared__ double red[2][APPLY_SPLIT][64];
  const ApplyRole &r = roles[blockIdx.y];
  const int a = r.a, b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
  const int na = r.n[a], nb = r.n[b], nc = r.n[c];
  const int lane = threadIdx.x, w = threadIdx.y;
  if ((long)blockIdx.x * 64 >= (long)nb * nc) return;
  const int pt = min((int)blockIdx.x * 64 + lane, nb * nc - 1);
  const int ib = pt % nb, ic = pt / nb;
  // per face, its term along the line: k q[st al], Xhat times ahat(al) on the
  // line's own axis, ahat of the line times Xhat along it otherwise
  double k[NF];
  const double *q[NF];
  int st[NF];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    k[f] = 0.0;
    q[f] = r.ahat[0];
    st[f] = 0;
    if (f < r.nf) {
      const double *xh = xhat + r.xoff[f];
      const int ax = r.fax[f];
      if (ax == a) {  // Xhat(b, c)
        k[f] = xh[pt];
        q[f] = r.ahat[f];
        st[f] = 1;
      } else if (ax == b) {  // Xhat over a and c
        k[f] = r.ahat[f][ib];
        q[f] = a < c ? xh + (long)na * ic : xh + ic;
        st[f] = a < c ? 1 : nc;
      } else {  // Xhat over a and b
        k[f] = r.ahat[f][ic];
        q[f] = a < b ? xh + (long)na * ib : xh + ib;
        st[f] = a < b ? 1 : nb;
      }
    }
  }
  const double *la = r.lam[a], *w0 = r.what[0], *w1 = r.what[1];
  const double lb = r.lam[b][ib], lc = r.lam[c][ic];
  const int per = (na + APPLY_SPLIT - 1) / APPLY_SPLIT, a0 = w * per, a1 = min(na, a0 + per);
  double s0 = 0.0, s1 = 0.0;
#pragma unroll 4
  for (int al = a0; al < a1; ++al) {
    double v = 0.0;
#pragma unroll
    for (int f = 0; f < NF; ++f) v = fma(k[f], q[f][(long)st[f] * al], v);
    v *= a == 0 ? inv_eig(la[al], lb, lc, sigma)
                : (a == 1 ? inv_eig(lb, la[al], lc, sigma) : inv_eig(lb, lc, la[al], sigma));
    s0 = fma(w0[al], v, s0);
    s1 = fma(w1[al], v, s1);
  }
  red[0][w][lane] = s0;
  red[1][w][lane] = s1;
  __syncthreads();
  if (w < r.no && (int)blockIdx.x * 64 + lane < nb * nc) {
    double s = red[w][0][lane];
    for (int t = 1; t < APPLY_SPLIT; ++t) s += red[w][t][lane];
    ghat[r.goff[w] + pt] = s;
  }
}

}  // namespace mf
