// Compact finite-difference derivatives on gfx950.
//
// Lines of up to 528 points take the segmented solve (der_seg.h), 3-D fields
// and batches of contiguous lines alike.  Longer ones (and contiguous lines
// that lie more than 2^25 points apart) take the kernels of this file:
// one lane owns one grid line and runs the reference's per-line algorithm:
// the explicit stencil right-hand side (class_derivatives.f90:262-295) fused
// with the forward recurrence of the packed quasi-pentadiagonal LU solve
// (pentares, class_derivatives.f90:425-466), then the backward recurrence.
// All lanes of a wavefront walk their lines in lockstep, so the coefficient
// loads are wave-uniform (scalar loads) and, for y- and z-lines whose
// neighbouring lanes are neighbouring i, every field access is a coalesced
// 512-byte wavefront access.  Field values are prefetched CH positions ahead
// into registers so that a wave keeps CH loads in flight per lane; the
// forward-sweep intermediate goes through the output array and comes back
// from L2/MALL in the backward sweep.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <type_traits>
#include <vector>

#include "conv.h"
#include "der_seg3d.h"
#include "internal.h"
#include "stage.h"
#include "mflops/mf.h"

namespace mf {

struct LineTab {      // device view of one packed scheme (dl LU + dr)
  const double *dr;   // (n,7) row-major: dr[7*i + m]
  const double *p, *f, *d, *e, *c;  // (n) each
  const double *rc;   // 1/c
  double alpha, beta;
  int n;
};

// y[i*ys] <- scheme applied to x[i*xs], i = 0..n-1 (n = T.n >= 8).
// The interior rows run in chunks of CH with the next chunk's inputs loaded
// ahead; every load and store is unconditional (addresses clamped into the
// line) and every branch is wave-uniform, so the compiler can wait for
// exactly the loads it needs.  A surplus lane of a block passes a scratch
// line as y (ys = 1): it walks the recurrences and stores only there.
// The coefficient rows come from CP-typed pointers: the block's copy of the
// scheme in LDS (coef_lds), whose wave-uniform reads are broadcasts that the
// compiler can issue ahead of the recurrence.
struct Coef {
  const double *dr, *p, *f, *d, *e, *rc;
  double alpha, beta;
  int n;
};

// Copy the packed scheme (dr 7n | p | f | d | e | c | 1/c) into LDS.
__device__ __forceinline__ Coef coef_lds(const LineTab &T, double *lds) {
  const int n = T.n;
  for (int q = threadIdx.x; q < 13 * n; q += blockDim.x) lds[q] = T.dr[q];
  __syncthreads();
  Coef c;
  c.dr = lds;
  c.p = lds + 7 * n;
  c.f = c.p + n;
  c.d = c.f + n;
  c.e = c.d + n;
  c.rc = c.e + 2 * n;
  c.alpha = T.alpha;
  c.beta = T.beta;
  c.n = n;
  return c;
}

template <int CH>
__device__ __forceinline__ void solve_line(const double *__restrict__ x, long xs,
                                           double *__restrict__ y, long ys, const Coef &T) {
  const int n = T.n;
  typedef const double *cptr;
  const cptr dr = T.dr, Tp = T.p, Tf = T.f, Td = T.d, Te = T.e, Trc = T.rc;
  auto X = [&](int q) { return x[(long)q * xs]; };
  // ---- rows 0 and 1: 7-point one-sided stencils on f[0..6]
  double w[7];
#pragma unroll
  for (int m = 0; m < 7; ++m) w[m] = X(m);
  double r0 = 0.0, r1 = 0.0;
#pragma unroll
  for (int m = 0; m < 7; ++m) {
    r0 = fma(dr[m], w[m], r0);
    r1 = fma(dr[7 + m], w[m], r1);
  }
  double ym2 = r0;
  double ym1 = r1 - Tf[1] * ym2;
  double ym3 = 0.0;
  y[0] = ym2;
  y[ys] = ym1;
  // window a[0..4] = f[i-2..i+2] for the interior rows 2..n-3
  double a0 = w[0], a1 = w[1], a2 = w[2], a3 = w[3], a4 = w[4];
  auto row = [&](int i, double fnext) {
    a0 = a1; a1 = a2; a2 = a3; a3 = a4; a4 = fnext;
    const cptr c = dr + 7 * i;
    const double rr = c[0] * a0 + c[1] * a1 + c[2] * a2 + c[3] * a3 + c[4] * a4;
    const double yi = rr - Tp[i] * ym2 - Tf[i] * ym1;
    y[(long)i * ys] = yi;
    ym3 = ym2; ym2 = ym1; ym1 = yi;
  };
  // row 2: its window f[0..4] is complete already
  {
    const cptr c = dr + 7 * 2;
    const double rr = c[0] * a0 + c[1] * a1 + c[2] * a2 + c[3] * a3 + c[4] * a4;
    const double yi = rr - Tp[2] * ym2 - Tf[2] * ym1;
    y[2 * ys] = yi;
    ym3 = ym2; ym2 = ym1; ym1 = yi;
  }
  const int last = n - 3;  // last interior row
  int i0 = 3;
  double buf[CH];
#pragma unroll
  for (int r = 0; r < CH; ++r) buf[r] = X(min(i0 + 2 + r, n - 1));  // f[i+2], rows i0..
  for (; i0 + CH - 1 <= last; i0 += CH) {
    double nbuf[CH];
#pragma unroll
    for (int r = 0; r < CH; ++r) nbuf[r] = X(min(i0 + CH + 2 + r, n - 1));
#pragma unroll
    for (int r = 0; r < CH; ++r) row(i0 + r, buf[r]);
#pragma unroll
    for (int r = 0; r < CH; ++r) buf[r] = nbuf[r];
  }
  // remaining interior rows (fewer than CH): buf holds their inputs
#pragma unroll
  for (int r = 0; r < CH - 1; ++r)
    if (i0 + r <= last) row(i0 + r, buf[r]);
  // ---- rows n-2 and n-1: 7-point stencils on f[n-7..n-1]
  double v[7];
#pragma unroll
  for (int m = 0; m < 7; ++m) v[m] = X(n - 7 + m);
  {
    cptr c = dr + 7 * (n - 2);
    double rr = 0.0;
#pragma unroll
    for (int m = 0; m < 7; ++m) rr = fma(c[m], v[m], rr);
    double yi = rr - Tp[n - 2] * ym2 - Tf[n - 2] * ym1;
    y[(long)(n - 2) * ys] = yi;
    ym3 = ym2; ym2 = ym1; ym1 = yi;
    c = dr + 7 * (n - 1);
    rr = 0.0;
#pragma unroll
    for (int m = 0; m < 7; ++m) rr = fma(c[m], v[m], rr);
    yi = rr - Tp[n - 1] * ym2 - Tf[n - 1] * ym1 - T.beta * ym3;
    // ---- backward sweep
    double xp1 = yi * Trc[n - 1];                                    // x[n-1]
    y[(long)(n - 1) * ys] = xp1;
    double xc = (ym1 - Td[n - 2] * xp1) * Trc[n - 2];               // x[n-2]
    y[(long)(n - 2) * ys] = xc;
    double xp2 = xp1;
    xp1 = xc;
    double x1 = 0.0, x2 = 0.0, x3 = 0.0;  // x[1], x[2], x[3] for row 0
    auto brow = [&](int i, double yv) {
      const double xi = (yv - Te[i] * xp2 - Td[i] * xp1) * Trc[i];
      y[(long)i * ys] = xi;
      xp2 = xp1;
      xp1 = xi;
    };
    // rows n-3 .. 1 in chunks, prefetching y downward
    int j0 = n - 3;
    double yb[CH];
#pragma unroll
    for (int r = 0; r < CH; ++r) yb[r] = y[(long)max(j0 - r, 1) * ys];
    for (; j0 - CH + 1 >= 4; j0 -= CH) {  // full chunks that stay above row 3
      double nyb[CH];
#pragma unroll
      for (int r = 0; r < CH; ++r) nyb[r] = y[(long)max(j0 - CH - r, 1) * ys];
#pragma unroll
      for (int r = 0; r < CH; ++r) brow(j0 - r, yb[r]);
#pragma unroll
      for (int r = 0; r < CH; ++r) yb[r] = nyb[r];
    }
    // remaining rows j0 .. 1 (fewer than CH + 3), keeping x[3], x[2], x[1]
#pragma unroll
    for (int r = 0; r < CH + 2; ++r) {
      const int i = j0 - r;
      if (i >= 1) {
        const double yv = r < CH ? yb[r] : y[(long)i * ys];
        brow(i, yv);
        if (i == 3) x3 = xp1;
        if (i == 2) x2 = xp1;
        if (i == 1) x1 = xp1;
      }
    }
    const double y0 = y[0];
    y[0] = (y0 - Te[0] * x2 - Td[0] * x1 - T.alpha * x3) * Trc[0];
  }
}

constexpr int kCH = 16;
constexpr int kMaxLine = 630;  // 13 coefficient doubles per point in 64 KiB of LDS

// 3-D driver (class_field.f90:629-978).  mode 0 = plain (every line full
// scheme), 1 = solver (interior lines full, one-boundary-plane lines on the
// sub-line scheme with zero ends, two-boundary-plane lines zero).  Blocks
// [0, b_full) take full-scheme lines, [b_full, b_full + b_sub) the sub-line
// ones and the last block the zero lines, so every line solve runs in
// wave-uniform control flow (the coefficients then come through the scalar
// cache); surplus lanes of a block walk its last line and store into the
// handle's scratch line.
template <int AXIS>
__global__ void __launch_bounds__(256) der3d_kernel(FieldSet fs, int nx, int ny, int nz,
                                                    LineTab full, LineTab sub, int mode,
                                                    int b_full, int b_sub,
                                                    double *__restrict__ scratch) {
  const double *__restrict__ x = fs.x[blockIdx.y];
  double *__restrict__ out = fs.out[blockIdx.y];
  int na, nb;
  long s;
  if (AXIS == 0) { na = ny; nb = nz; s = 1; }
  else if (AXIS == 1) { na = nx; nb = nz; s = nx; }
  else { na = nx; nb = ny; s = (long)nx * ny; }
  auto base_of = [&](int a, int b) -> long {
    if (AXIS == 0) return (long)nx * (a + (long)ny * b);
    if (AXIS == 1) return a + (long)nx * ny * b;
    return a + (long)nx * b;
  };
  extern __shared__ double coef[];
  const int n = full.n;
  const int blk = blockIdx.x;
  const long tid = threadIdx.x;
  if (!mode) {
    const Coef C = coef_lds(full, coef);
    const long cnt = (long)na * nb;
    long t = (long)blk * 256 + tid;
    const bool act = t < cnt;
    t = act ? t : cnt - 1;
    const long base = base_of((int)(t % na), (int)(t / na));
    solve_line<kCH>(x + base, s, act ? out + base : scratch, act ? s : 1, C);
  } else if (blk < b_full) {
    const Coef C = coef_lds(full, coef);
    const long cnt = (long)(na - 2) * (nb - 2);
    long t = (long)blk * 256 + tid;
    const bool act = t < cnt;
    t = act ? t : cnt - 1;
    const long base = base_of(1 + (int)(t % (na - 2)), 1 + (int)(t / (na - 2)));
    solve_line<kCH>(x + base, s, act ? out + base : scratch, act ? s : 1, C);
  } else if (blk < b_full + b_sub) {
    const Coef C = coef_lds(sub, coef);
    const long cnt = 2L * (na - 2) + 2L * (nb - 2);
    long t = (long)(blk - b_full) * 256 + tid;
    const bool act = t < cnt;
    t = act ? t : cnt - 1;
    int a, b;
    if (t < 2L * (na - 2)) {
      a = 1 + (int)(t % (na - 2));
      b = (t / (na - 2)) ? nb - 1 : 0;
    } else {
      t -= 2L * (na - 2);
      b = 1 + (int)(t % (nb - 2));
      a = (t / (nb - 2)) ? na - 1 : 0;
    }
    const long base = base_of(a, b);
    if (act) {
      out[base] = 0.0;
      out[base + (long)(n - 1) * s] = 0.0;
    }
    solve_line<kCH>(x + base + s, s, act ? out + base + s : scratch, act ? s : 1, C);
  } else {
    for (long t = tid; t < 4L * n; t += 256) {
      const int line = (int)(t / n), i = (int)(t % n);
      const long base = base_of((line & 1) ? na - 1 : 0, (line & 2) ? nb - 1 : 0);
      out[base + (long)i * s] = 0.0;
    }
  }
}

// One axis of the convective term of all components (SegConv): 32 lines of one
// component per block, blocks of the three components of the same lines next to
// each other (the advecting component they share then comes from the L2).
// Bounds: HBM, 6 fields on the first axis and 9 on the others (stored products
// and derivatives take 78 in all, with their kernels and the sum's), and
// registers: a pair's values, results and addresses need more than the 128
// that launch bounds for 16 waves leave, so that a lane keeps 161 to 185 of them
// (240 to 243 pentadiagonal) in scratch memory, 268 bytes a lane on the first
// axis.  192 x 256 x 192: 246 + 193 + 204 us (1.8, 3.5 and
// 3.3 TB/s), where products, 18 derivatives and the sum with the right-hand
// sides took 1330, and right-hand sides on their own now take 207; a time
// step 4.09 -> 3.53 ms.  At 24^3 to 64^3, three launches in turn for five with
// the middle three beside each other: 0.42 -> 0.38 and 0.44 -> 0.41 ms a step.
// Taken back: the right-hand sides formed here on the last axis (1.06 ms for
// that launch; the many pointers cost the registers of the solve).
template <int AXIS, bool TRI>
__global__ void __launch_bounds__(64 * SEG_KMAX) conv3d_kernel(ConvArgs a, SegGrid G) {
  extern __shared__ double lds[];
  int c, blk;
  seg_place(G, true, blk, c);
  const SegConv<AXIS != 0> job{a.q[c], a.u, a.acc[c], a.out[c]};
  seg_block<AXIS, TRI, false>(job, G, blk, lds);
}

// batched contiguous lines (der/dder/der_s/dder_s), one lane per line, where they
// are longer than the segmented solve takes; surplus lanes walk the last line into the scratch line (as der3d_kernel)
__global__ void __launch_bounds__(256) der_lines_kernel(const double *__restrict__ x,
                                                        double *__restrict__ out, int nlines,
                                                        long ld, LineTab T, int offset,
                                                        double *__restrict__ scratch) {
  extern __shared__ double coef[];
  const Coef C = coef_lds(T, coef);
  long l = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const bool act = l < nlines;
  l = act ? l : nlines - 1;
  solve_line<kCH>(x + l * ld + offset, 1, act ? out + l * ld + offset : scratch, 1, C);
}

}  // namespace mf

// ---------------------------------------------------------------------------
// Handle and C ABI
// ---------------------------------------------------------------------------
struct mf_der {
  int n = 0, so = 6, solver = 0;
  mutable mf::HostStage stage;  // device staging of the host-array entry points
  double *dbuf = nullptr;      // device tables, then one scratch line of n
  double *scratch = nullptr;   // surplus lanes' output line
  mf::LineTab tab[2][2];       // [order-1][sub]
  mf::SegTab seg[2][2];        // the segmented solve's tables (lines it takes)
  bool tri[2] = {false, false};  // [order-1]: tridiagonal factors, full and sub scheme
  std::vector<double> host[2][2][2];  // [order-1][sub][0: dl_lu(n,5), 1: dr(n,7)]
};

bool mf::der_host_tables(const mf_der *dc, int order, int sub, const double **dl_lu,
                         const double **dr, int *n) {
  if (!dc || order < 1 || order > 2 || (sub && !dc->solver)) return false;
  const auto &t = dc->host[order - 1][sub ? 1 : 0];
  *dl_lu = t[0].data();
  *dr = t[1].data();
  *n = sub ? dc->n - 2 : dc->n;
  return true;
}

namespace {
// pack one scheme: dr row-major (7n) | p | f | d | e | c | 1/c, then the
// segmented solve's table (seg_tables) on lines it takes
constexpr int kLinePack = 13;
void pack_scheme(int n, const std::vector<double> &dl, const std::vector<double> &dr, bool tri,
                 std::vector<double> &dst) {
  const int K = mf::seg_count(n, tri);
  const bool seg = K <= mf::SEG_KMAX;
  dst.assign((size_t)kLinePack * n + (seg ? mf::seg_table_doubles(K) : 0), 0.0);
  for (int i = 0; i < n; ++i)
    for (int m = 0; m < 7; ++m) dst[(size_t)7 * i + m] = dr[i + (size_t)n * m];
  double *p = &dst[(size_t)7 * n];
  for (int i = 0; i < n; ++i) {
    p[i] = dl[i];
    p[n + i] = dl[n + i];
    p[2 * n + i] = dl[3 * (size_t)n + i];
    p[3 * n + i] = dl[4 * (size_t)n + i];
    p[4 * n + i] = dl[2 * (size_t)n + i];
    p[5 * n + i] = 1.0 / dl[2 * (size_t)n + i];
  }
  // alpha = dl(1,1) and beta = dl(n,5) of the factored matrix
  if (seg)
    mf::seg_tables(n, dr.data(), p, p + n, p + 2 * n, p + 3 * n, p + 5 * n, dl[0],
                   dl[4 * (size_t)n + n - 1], tri, p + 6 * n);
}

// whether the factored matrix has two diagonals per sweep only: p and e zero
// (and with them alpha = dl(1,1) and beta = dl(n,5))
bool factors_tri(int n, const std::vector<double> &dl) {
  for (int i = 0; i < n; ++i)
    if (dl[i] != 0.0 || dl[4 * (size_t)n + i] != 0.0) return false;
  return true;
}
#define HIPCHK(call)                                                             \
  do {                                                                           \
    hipError_t e_ = (call);                                                      \
    if (e_ != hipSuccess)                                                        \
      return mf::fail(MF_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)
}  // namespace

extern "C" int mf_der_coeffs_1d(const double *grid, int n, int der, int so, double *dl_lu,
                                double *dr) {
  if (!grid || !dl_lu || !dr || n < 8 || (der != 1 && der != 2) ||
      (so != 2 && so != 4 && so != 6 && so != 8))
    return mf::fail(MF_ERR_ARG, "mf_der_coeffs_1d: invalid argument");
  if (!mf::der_coeffs_global(grid, n, der, so, dl_lu, dr))
    return mf::fail(MF_ERR_SETUP, "mf_der_coeffs_1d: singular Taylor system");
  mf::pentalu(n, dl_lu);
  return MF_OK;
}

extern "C" int mf_der_create(const double *grid, int n, int solver_mode, int so, mf_der **out) {
  if (!grid || !out) return mf::fail(MF_ERR_ARG, "mf_der_create: null pointer");
  const int nmin = solver_mode ? 10 : 8;
  if (n < nmin) return mf::fail(MF_ERR_ARG, "mf_der_create: line too short for the 7-point closures");
  if (n > mf::kMaxLine)
    return mf::fail(MF_ERR_ARG, "mf_der_create: lines longer than " + std::to_string(mf::kMaxLine) +
                                    " points exceed the per-block coefficient copy (64 KiB LDS)");
  if (so != 2 && so != 4 && so != 6 && so != 8)
    return mf::fail(MF_ERR_ARG, "mf_der_create: so must be 2, 4, 6 or 8");
  mf_der *h = new mf_der();
  h->n = n;
  h->so = so;
  h->solver = solver_mode ? 1 : 0;
  std::vector<double> packed[2][2];
  for (int o = 0; o < 2; ++o)
    for (int sub = 0; sub < 1 + h->solver; ++sub) {
      const int m = sub ? n - 2 : n;
      auto &dl = h->host[o][sub][0];
      auto &dr = h->host[o][sub][1];
      dl.assign((size_t)5 * m, 0.0);
      dr.assign((size_t)7 * m, 0.0);
      if (!mf::der_coeffs_global(grid + sub, m, o + 1, so, dl.data(), dr.data())) {
        delete h;
        return mf::fail(MF_ERR_SETUP, "mf_der_create: singular Taylor system");
      }
      mf::pentalu(m, dl.data());
    }
  for (int o = 0; o < 2; ++o) {
    h->tri[o] = true;
    for (int sub = 0; sub < 1 + h->solver; ++sub)
      h->tri[o] = h->tri[o] && factors_tri(sub ? n - 2 : n, h->host[o][sub][0]);
    for (int sub = 0; sub < 1 + h->solver; ++sub)
      pack_scheme(sub ? n - 2 : n, h->host[o][sub][0], h->host[o][sub][1], h->tri[o],
                  packed[o][sub]);
  }
  size_t total = 0;
  for (int o = 0; o < 2; ++o)
    for (int sub = 0; sub < 2; ++sub) total += packed[o][sub].size();
  hipError_t e = hipMalloc(&h->dbuf, (total + n) * sizeof(double));
  if (e == hipSuccess) h->scratch = h->dbuf + total;
  if (e != hipSuccess) {
    delete h;
    return mf::fail(MF_ERR_DEVICE, std::string("mf_der_create: hipMalloc: ") + hipGetErrorString(e));
  }
  size_t off = 0;
  for (int o = 0; o < 2; ++o)
    for (int sub = 0; sub < 2; ++sub) {
      auto &pk = packed[o][sub];
      mf::LineTab &T = h->tab[o][sub];
      std::memset(&T, 0, sizeof(T));
      h->seg[o][sub] = mf::SegTab{nullptr, 0, 0, 0};
      if (pk.empty()) continue;
      const int m = sub ? n - 2 : n;
      e = hipMemcpy(h->dbuf + off, pk.data(), pk.size() * sizeof(double), hipMemcpyHostToDevice);
      if (e != hipSuccess) {
        (void)hipFree(h->dbuf);
        delete h;
        return mf::fail(MF_ERR_DEVICE, std::string("mf_der_create: hipMemcpy: ") + hipGetErrorString(e));
      }
      double *b = h->dbuf + off;
      T.dr = b;
      T.p = b + 7 * (size_t)m;
      T.f = T.p + m;
      T.d = T.f + m;
      T.e = T.d + m;
      T.c = T.e + m;
      T.rc = T.c + m;
      T.alpha = h->host[o][sub][0][0];                       // dl(1,1)
      T.beta = h->host[o][sub][0][4 * (size_t)m + m - 1];    // dl(m,5) after pentalu
      T.n = m;
      if (pk.size() > (size_t)kLinePack * m) {
        const int K = mf::seg_count(m, h->tri[o]);
        h->seg[o][sub] = mf::SegTab{b + (size_t)kLinePack * m, m, K, mf::seg_len(m, K)};
      }
      off += pk.size();
    }
  *out = h;
  return MF_OK;
}

extern "C" int mf_der_destroy(mf_der *dc) {
  if (!dc) return MF_OK;
  if (dc->dbuf) (void)hipFree(dc->dbuf);
  delete dc;
  return MF_OK;
}

extern "C" int mf_der_lines(const mf_der *dc, int order, int sub, const double *x, double *out,
                            int nlines, long long ld, void *stream) {
  if (!dc || !x || !out || (order != 1 && order != 2) || nlines < 0 || ld < dc->n)
    return mf::fail(MF_ERR_ARG, "mf_der_lines: invalid argument");
  if (sub && !dc->solver)
    return mf::fail(MF_ERR_ARG, "mf_der_lines: sub-line scheme needs a solver-mode handle");
  if (nlines == 0) return MF_OK;
  const mf::LineTab &T = dc->tab[order - 1][sub ? 1 : 0];
  const mf::SegTab &S = dc->seg[order - 1][sub ? 1 : 0];
  if (S.pack && mf::seg_fits(ld)) {
    const dim3 grid((nlines + 63) / 64), block(64 * S.K);
    const size_t lds = mf::seg_lds_doubles(S.K, true) * sizeof(double);
    const int o = sub ? 1 : 0;
    auto go = S.len > mf::SEG_LEN ? mf::der_lines_seg_launch<true> : mf::der_lines_seg_launch<false>;
    go(dc->tri[order - 1], grid, block, lds, (hipStream_t)stream, x + o, out + o, nlines, (long)ld, S);
    HIPCHK(hipGetLastError());
    return MF_OK;
  }
  const int blocks = (nlines + 255) / 256;
  hipLaunchKernelGGL(mf::der_lines_kernel, dim3(blocks), dim3(256), 13 * T.n * sizeof(double),
                     (hipStream_t)stream, x, out, nlines, (long)ld, T, sub ? 1 : 0, dc->scratch);
  HIPCHK(hipGetLastError());
  return MF_OK;
}

namespace {
// Blocks of `lines` lines along an axis: the grid's geometry and block count
mf::SegGrid seg_grid(const mf_der *dc, int axis, int order, int lines, int nx, int ny, int nz,
                     int *blocks) {
  const int na = axis == 0 ? ny : nx, nb = axis == 2 ? ny : nz;
  mf::SegGrid G;
  std::memset(&G, 0, sizeof(G));
  G.nx = nx; G.ny = ny; G.nz = nz;
  G.full = dc->seg[order - 1][0];
  G.sub = dc->seg[order - 1][1];
  G.mode = dc->solver;
  G.groups = axis != 0 && mf::seg_aligned(nx, lines) ? (nx + lines - 1) / lines : 0;
  auto count = [&](long m) { return (int)((m + lines - 1) / lines); };
  if (!G.mode) {
    *blocks = G.b_full = G.groups ? G.groups * nb : count((long)na * nb);
  } else {
    G.b_full = G.groups ? G.groups * (nb - 2) : count((long)(na - 2) * (nb - 2));
    G.nb4.x = G.nb4.y = count(na - 2);
    G.nb4.z = G.nb4.w = count(nb - 2);
    *blocks = G.b_full + G.nb4.x + G.nb4.y + G.nb4.z + G.nb4.w + 1;
  }
  return G;
}
}  // namespace

namespace mf {
bool conv3d_takes(const ::mf_der *const dc[3], int nx, int ny, int nz) {
  for (int a = 0; a < 3; ++a)
    if (!dc[a]->seg[0][0].pack || dc[a]->seg[0][0].len > SEG_LEN) return false;
  return seg_fits((long)nx * ny) && nx > 2 && ny > 2 && nz > 2;
}

int conv3d(const ::mf_der *dc, int axis, const ConvArgs &a, int nx, int ny, int nz, void *stream) {
  const int n = axis == 0 ? nx : (axis == 1 ? ny : nz);
  if (dc->n != n || !dc->solver) return fail(MF_ERR_ARG, "conv3d: not the handle of this axis");
  int blocks;
  const SegGrid G = seg_grid(dc, axis, 1, 32, nx, ny, nz, &blocks);
  const size_t lds = seg_lds_doubles(G.full.K, axis == 0) * sizeof(double);
  auto go = [&](auto ax, auto tri) {
    hipLaunchKernelGGL((conv3d_kernel<decltype(ax)::value, decltype(tri)::value>), dim3(blocks, 3),
                       dim3(64 * G.full.K), lds, (hipStream_t)stream, a, G);
  };
  auto pick = [&](auto ax) {
    if (dc->tri[0]) go(ax, std::true_type());
    else go(ax, std::false_type());
  };
  if (axis == 0) pick(std::integral_constant<int, 0>());
  else if (axis == 1) pick(std::integral_constant<int, 1>());
  else pick(std::integral_constant<int, 2>());
  HIPCHK(hipGetLastError());
  return MF_OK;
}
}  // namespace mf

extern "C" int mf_der3d_batch(const mf_der *dc, int axis, int order, int nfields,
                              const double *const *x, double *const *out, int nx, int ny, int nz,
                              void *stream) {
  if (!dc || !x || !out || axis < 0 || axis > 2 || (order != 1 && order != 2) || nx < 1 ||
      ny < 1 || nz < 1 || nfields < 1 || nfields > mf::kMaxBatch)
    return mf::fail(MF_ERR_ARG, "mf_der3d: invalid argument");
  const int dims[3] = {nx, ny, nz};
  if (dims[axis] != dc->n)
    return mf::fail(MF_ERR_ARG, "mf_der3d: field size along the axis differs from the handle's grid");
  mf::FieldSet fs;
  std::memset(&fs, 0, sizeof(fs));
  for (int f = 0; f < nfields; ++f) {
    if (!x[f] || !out[f]) return mf::fail(MF_ERR_ARG, "mf_der3d: null field pointer");
    for (int g = 0; g < nfields; ++g)
      if (x[g] == out[f]) return mf::fail(MF_ERR_ARG, "mf_der3d: an output aliases an input");
    fs.x[f] = x[f];
    fs.out[f] = out[f];
  }
  const int na = axis == 0 ? ny : nx, nb = axis == 2 ? ny : nz;
  const mf::LineTab &F = dc->tab[order - 1][0];
  const mf::LineTab &S = dc->tab[order - 1][1];
  const int mode = dc->solver;
  int blocks, b_full = 0, b_sub = 0;
  if (!mode) {
    blocks = (int)(((long)na * nb + 255) / 256);
  } else {
    if (na < 3 || nb < 3) return mf::fail(MF_ERR_ARG, "mf_der3d: solver mode needs 3+ points across the lines");
    b_full = (int)(((long)(na - 2) * (nb - 2) + 255) / 256);
    b_sub = (int)((2L * (na - 2) + 2L * (nb - 2) + 255) / 256);
    blocks = b_full + b_sub + 1;
  }
  hipStream_t st = (hipStream_t)stream;
  if (dc->seg[order - 1][0].pack && (axis != 0 || mf::seg_fits((long)nx * ny))) {
    // segmented solves: 64 lines per block, one wavefront per segment
    int sblocks;
    const mf::SegGrid G = seg_grid(dc, axis, order, 64, nx, ny, nz, &sblocks);
    const size_t lds = mf::seg_lds_doubles(G.full.K, axis == 0) * sizeof(double);
    const dim3 grid(sblocks, nfields), block(64 * G.full.K);
    auto go = G.full.len > mf::SEG_LEN ? mf::der3d_seg_launch<true> : mf::der3d_seg_launch<false>;
    go(axis, dc->tri[order - 1], grid, block, lds, st, fs, G);
    HIPCHK(hipGetLastError());
    return MF_OK;
  }
  const size_t lds = 13 * (size_t)F.n * sizeof(double);  // the larger (full) scheme
  const dim3 grid(blocks, nfields);
  if (axis == 0)
    hipLaunchKernelGGL(mf::der3d_kernel<0>, grid, dim3(256), lds, st, fs, nx, ny, nz, F, S, mode, b_full, b_sub, dc->scratch);
  else if (axis == 1)
    hipLaunchKernelGGL(mf::der3d_kernel<1>, grid, dim3(256), lds, st, fs, nx, ny, nz, F, S, mode, b_full, b_sub, dc->scratch);
  else
    hipLaunchKernelGGL(mf::der3d_kernel<2>, grid, dim3(256), lds, st, fs, nx, ny, nz, F, S, mode, b_full, b_sub, dc->scratch);
  HIPCHK(hipGetLastError());
  return MF_OK;
}

extern "C" int mf_der3d(const mf_der *dc, int axis, int order, const double *x, double *out,
                        int nx, int ny, int nz, void *stream) {
  if (x && x == out) return mf::fail(MF_ERR_ARG, "mf_der3d: in-place derivative is not supported");
  return mf_der3d_batch(dc, axis, order, 1, &x, &out, nx, ny, nz, stream);
}

extern "C" int mf_der3d_host(const mf_der *dc, int axis, int order, const double *x, double *out,
                             int nx, int ny, int nz) {
  if (!dc || !x || !out || nx < 1 || ny < 1 || nz < 1)
    return mf::fail(MF_ERR_ARG, "mf_der3d_host: invalid argument");
  const size_t bytes = (size_t)nx * ny * nz * sizeof(double);
  std::lock_guard<std::mutex> lock(dc->stage.mu);
  hipError_t e = dc->stage.reserve(2 * bytes);
  if (e != hipSuccess)
    return mf::fail(MF_ERR_DEVICE, std::string("mf_der3d_host: staging: ") + hipGetErrorString(e));
  double *dx = (double *)dc->stage.dev, *dy = dx + (size_t)nx * ny * nz;
  int rc = MF_OK;
  e = hipMemcpy(dx, x, bytes, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    rc = mf_der3d(dc, axis, order, dx, dy, nx, ny, nz, nullptr);
    if (rc == MF_OK) e = hipMemcpy(out, dy, bytes, hipMemcpyDeviceToHost);
  }
  if (rc != MF_OK) return rc;
  if (e != hipSuccess)
    return mf::fail(MF_ERR_DEVICE, std::string("mf_der3d_host: ") + hipGetErrorString(e));
  return MF_OK;
}

extern "C" int mf_der_lines_host(const mf_der *dc, int order, int sub, const double *x, double *out,
                                 int nlines, long long ld) {
  if (!dc || !x || !out || nlines < 0 || ld < dc->n)
    return mf::fail(MF_ERR_ARG, "mf_der_lines_host: invalid argument");
  if (nlines == 0) return MF_OK;
  const size_t bytes = (size_t)nlines * (size_t)ld * sizeof(double);
  std::lock_guard<std::mutex> lock(dc->stage.mu);
  hipError_t e = dc->stage.reserve(2 * bytes);
  if (e != hipSuccess)
    return mf::fail(MF_ERR_DEVICE, std::string("mf_der_lines_host: staging: ") + hipGetErrorString(e));
  double *dx = (double *)dc->stage.dev, *dy = dx + (size_t)nlines * ld;
  e = hipMemcpy(dx, x, bytes, hipMemcpyHostToDevice);
  // the sub-line scheme leaves the end points of out untouched
  if (e == hipSuccess && sub) e = hipMemcpy(dy, out, bytes, hipMemcpyHostToDevice);
  int rc = MF_OK;
  if (e == hipSuccess) {
    rc = mf_der_lines(dc, order, sub, dx, dy, nlines, ld, nullptr);
    if (rc == MF_OK) e = hipMemcpy(out, dy, bytes, hipMemcpyDeviceToHost);
  }
  if (rc != MF_OK) return rc;
  if (e != hipSuccess)
    return mf::fail(MF_ERR_DEVICE, std::string("mf_der_lines_host: ") + hipGetErrorString(e));
  return MF_OK;
}
