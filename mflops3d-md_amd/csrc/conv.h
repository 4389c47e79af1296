// The convective term formed by the derivative kernels themselves (der.hip),
// for the Navier-Stokes step (ns.hip).
#pragma once

struct mf_der;

namespace mf {

// One axis' share of the skew-symmetric convective term of the three
// components, with solver-mode derivatives:
//   out[c] = acc[c] + (u d(q[c]) + d(q[c] u)) / 2,   0 on the edges,
// u the component along the axis; acc is not read on axis 0.  The outputs
// alias no input.
struct ConvArgs {
  const double *q[3], *u, *acc[3];
  double *out[3];
};
// whether conv3d takes these axes' handles and sizes
bool conv3d_takes(const ::mf_der *const dc[3], int nx, int ny, int nz);
int conv3d(const ::mf_der *dc, int axis, const ConvArgs &a, int nx, int ny, int nz, void *stream);

}  // namespace mf
