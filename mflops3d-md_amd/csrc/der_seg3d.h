// The segmented line solves (der_seg.h) over 3-D fields and batches of lines:
// kernels and their launches.  The instances for lines beyond 16 segments of 32
// rows (LONG) are a code object of their own (der_long.hip): together with the
// others, which fill 2 MB, they moved those to other pages, and second
// derivatives along x, y and z of 201 x 256 x 187 took 190 us instead of 184 with
// the same instructions.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "der_seg.h"

namespace mf {

// Up to kMaxBatch fields of one shape go in one launch, field = blockIdx.y.
constexpr int kMaxBatch = 8;
struct FieldSet {
  const double *x[kMaxBatch];
  double *out[kMaxBatch];
};

// 3-D driver on segmented line solves (seg_solve): blocks of 64 lines, one
// wavefront per segment.  Plain mode (mode 0): every line on the full scheme,
// blocks [0, b_full).  Solver mode: blocks [0, b_full) take the interior lines
// (full scheme), the next nb4.x .. nb4.w blocks the four families of
// one-boundary-plane lines (sub-line scheme on points 1..n-2), and the last
// block writes the zeros (two-boundary-plane lines, sub-line end points).
struct SegGrid {
  int nx, ny, nz;
  SegTab full, sub;
  int mode, b_full;
  int4 nb4;
  int groups;
};

// Block and field of this block: the boundary-plane blocks come first (at y
// and z half of them read one point per cache line and take longest), then
// the full-scheme blocks, a contiguous run of them on each of the 8 XCDs that
// consecutive block ids go to in turn: groups of lines start at any byte, so
// neighbours share cache lines at both ends, which then come from the XCD's
// own L2.  inner: fields next to each other rather than one after the other.
__device__ __forceinline__ void seg_place(const SegGrid &G, bool inner, int &blk, int &fld) {
  const int nf = gridDim.y, nsub = gridDim.x - G.b_full;
  int bid = blockIdx.x + gridDim.x * blockIdx.y;
  if (bid < nsub * nf) {
    fld = bid % nf;
    blk = G.b_full + bid / nf;
    return;
  }
  bid -= nsub * nf;
  const int nb = G.b_full * nf, off = nsub * nf % 8;
  // XCD of this block and its place among the XCD's full-scheme blocks
  const int xc = (bid + off) % 8, first = (xc - off + 8) % 8, l = (bid - first) / 8;
  int start = 0;
  for (int q = 0; q < xc; ++q) start += (nb - (q - off + 8) % 8 + 7) / 8;
  const int t = start + l;
  blk = inner ? t / nf : t % G.b_full;
  fld = inner ? t % nf : t / G.b_full;
}

template <int AXIS, bool TRI, bool LONG, class Job>
__device__ __forceinline__ void seg_block(const Job &job, const SegGrid &G, int blk, double *lds) {
  const int nx = G.nx, ny = G.ny, nz = G.nz;
  const int4 nb4 = G.nb4;
  int na, nb;
  long s, sa, sb;
  if (AXIS == 0) { na = ny; nb = nz; s = 1; sa = nx; sb = (long)nx * ny; }
  else if (AXIS == 1) { na = nx; nb = nz; s = nx; sa = 1; sb = (long)nx * ny; }
  else { na = nx; nb = ny; s = (long)nx * ny; sa = 1; sb = nx; }
  const int n = G.full.n;
  SegLines L;
  L.sa = sa; L.sb = sb; L.s = s;
  // one call site of seg_solve: pick the scheme, the line family and the
  // field offset of this block, then solve
  SegTab T = G.full;
  long off = 0;
  bool solve = true;
  L.groups = 0;
  if (blk < G.b_full) {
    L.groups = G.groups;
    if (G.mode) { L.a0 = 1; L.na = na - 2; L.b0 = 1; L.nb = nb - 2; }
    else { L.a0 = 0; L.na = na; L.b0 = 0; L.nb = nb; }
  } else {
    blk -= G.b_full;
    if (blk < nb4.x + nb4.y) {
      const int f = blk >= nb4.x;
      blk -= f ? nb4.x : 0;
      L.a0 = 1; L.na = na - 2; L.b0 = f ? nb - 1 : 0; L.nb = 1;
    } else if (blk < nb4.x + nb4.y + nb4.z + nb4.w) {
      blk -= nb4.x + nb4.y;
      const int f = blk >= nb4.z;
      blk -= f ? nb4.z : 0;
      L.a0 = f ? na - 1 : 0; L.na = 1; L.b0 = 1; L.nb = nb - 2;
    } else {
      solve = false;
    }
    T = G.sub;
    off = s;  // the sub-line scheme acts on points 1..n-2
  }
  if (solve) {
    L.nlines = L.na * L.nb;
    seg_solve<TRI, AXIS == 0, LONG>(job, off, T, L, blk, lds);
    return;
  }
  // zeros: the four two-boundary-plane lines and both ends of the sub lines
  const int nt = blockDim.x;
  for (long t = threadIdx.x; t < 4L * n; t += nt) {
    const int line = (int)(t / n), i = (int)(t % n);
    job.edge(((line & 1) ? na - 1 : 0) * sa + (long)((line & 2) ? nb - 1 : 0) * sb + (long)i * s);
  }
  const long ns = 2L * (na - 2) + 2L * (nb - 2);
  for (long t = threadIdx.x; t < ns; t += nt) {
    int a, b;
    if (t < 2L * (na - 2)) { a = 1 + (int)(t % (na - 2)); b = (t / (na - 2)) ? nb - 1 : 0; }
    else { const long r = t - 2L * (na - 2); b = 1 + (int)(r % (nb - 2)); a = (r / (nb - 2)) ? na - 1 : 0; }
    const long base = a * sa + b * sb;
    job.edge(base);
    job.edge(base + (long)(n - 1) * s);
  }
}

template <int AXIS, bool TRI, bool LONG>
__global__ void __launch_bounds__(64 * SEG_KMAX) der3d_seg_kernel(FieldSet fs, SegGrid G) {
  extern __shared__ double lds[];
  int blk, fld;
  seg_place(G, false, blk, fld);
  const SegDer job{fs.x[fld], fs.out[fld]};
  seg_block<AXIS, TRI, LONG>(job, G, blk, lds);
}

// batched lines on segmented line solves: line l at x + l*ld, contiguous
// points (der/dder/der_s/dder_s)
template <bool TRI, bool LONG>
__global__ void __launch_bounds__(64 * SEG_KMAX)
    der_lines_seg_kernel(const double *__restrict__ x, double *__restrict__ out, int nlines,
                         long ld, SegTab T) {
  extern __shared__ double lds[];
  SegLines L;
  L.sa = ld; L.sb = 0; L.s = 1;
  L.a0 = 0; L.na = nlines; L.b0 = 0; L.nb = 1;
  L.nlines = nlines;
  L.groups = 0;
  seg_solve<TRI, true, LONG>(SegDer{x, out}, 0, T, L, blockIdx.x, lds);
}

template <bool LONG>
void der3d_seg_launch(int axis, bool tri, dim3 grid, dim3 block, size_t lds, hipStream_t st,
                      const FieldSet &fs, const SegGrid &G) {
  auto go = [&](auto ax, auto t) {
    hipLaunchKernelGGL((der3d_seg_kernel<decltype(ax)::value, decltype(t)::value, LONG>), grid, block,
                       lds, st, fs, G);
  };
  auto pick = [&](auto ax) {
    if (tri) go(ax, std::true_type());
    else go(ax, std::false_type());
  };
  if (axis == 0) pick(std::integral_constant<int, 0>());
  else if (axis == 1) pick(std::integral_constant<int, 1>());
  else pick(std::integral_constant<int, 2>());
}

template <bool LONG>
void der_lines_seg_launch(bool tri, dim3 grid, dim3 block, size_t lds, hipStream_t st,
                          const double *x, double *out, int nlines, long ld, const SegTab &T) {
  if (tri)
    hipLaunchKernelGGL((der_lines_seg_kernel<true, LONG>), grid, block, lds, st, x, out, nlines, ld, T);
  else
    hipLaunchKernelGGL((der_lines_seg_kernel<false, LONG>), grid, block, lds, st, x, out, nlines, ld, T);
}

extern template void der3d_seg_launch<true>(int, bool, dim3, dim3, size_t, hipStream_t,
                                            const FieldSet &, const SegGrid &);
extern template void der_lines_seg_launch<true>(bool, dim3, dim3, size_t, hipStream_t, const double *,
                                                double *, int, long, const SegTab &);

}  // namespace mf
