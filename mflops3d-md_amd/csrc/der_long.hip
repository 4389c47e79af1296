// Derivatives along lines of 513 to 528 points (der_seg3d.h): segments of up to 33
// rows.
#include "der_seg3d.h"

namespace mf {
template void der3d_seg_launch<true>(int, bool, dim3, dim3, size_t, hipStream_t, const FieldSet &,
                                     const SegGrid &);
template void der_lines_seg_launch<true>(bool, dim3, dim3, size_t, hipStream_t, const double *,
                                         double *, int, long, const SegTab &);
}  // namespace mf
