// Which tile a product of gemm.h takes (host code only).
#pragma once
#include <algorithm>
#include <cmath>

namespace mf {

struct GemmTile {
  int mi, ni;
};

// Tile of a product, in MFMA blocks: the one whose waves take the least time
// on the busiest SIMD, a k-step of a wave costing its MFMAs (64 cycles each)
// or its loads (512 B each, a CU's L1 delivering 64 B a cycle to 4 SIMDs),
// whichever is more, and each wave the latency of its first loads.  At 254
// points 64 x 64 tiles (4 waves per SIMD); 48 wide where that pads less (130
// columns in three); a 62^3 field 16 x 16 tiles, since 64-wide ones would leave
// fifteen SIMDs of sixteen empty.  Measured against block tiles staged through
// LDS (one barrier pair per 16-deep step, two blocks per CU), bit for bit the
// same results: a 256^3 FP64 solve 1.397 -> 1.051 ms, a 64^3 one 121 -> 37 us,
// training targets 256^3 -> 64^3 1.90 -> 1.33 ms.  The FP32 y and z transforms
// follow the same rule: their MFMAs and loads take half the time each, which
// picks the same tiles from 66^3 on.
inline GemmTile gemm_tile_of(int M, int N, int K, int batch, int ncu) {
  static const GemmTile all[] = {{4, 4}, {4, 3}, {3, 4}, {3, 3}, {4, 2}, {2, 4}, {2, 2}, {1, 1}};
  GemmTile best = all[0];
  double least = 0.0;
  for (const GemmTile &t : all) {
    const double w = (double)((M + 16 * t.mi - 1) / (16 * t.mi)) *
                     ((N + 16 * t.ni - 1) / (16 * t.ni)) * batch;
    const double per = std::ceil(w / (4.0 * ncu));
    const double step = std::max(64.0 * t.mi * t.ni, 32.0 * (t.mi + t.ni));
    const double cost = per * ((K + 3) / 4) * step + 2000.0 * std::ceil(per / 2.0);
    if (least == 0.0 || cost < least) {
      least = cost;
      best = t;
    }
  }
  return best;
}

// The FP32 x transform's (gemm_tile_quads): 32 x 32, or 16 x 16 where those
// would leave SIMDs without a wave (64^3: 3.5 us for 5.0; 128^3 with 2048 waves of
// 32 x 32: 10.8 for 12.2) and where K holds no quad.
inline GemmTile gemm_tile_x32(int M, int N, int K, int batch, int ncu) {
  const long w = (long)((M + 31) / 32) * ((N + 31) / 32) * batch;
  return K >= 16 && w >= 4L * ncu ? GemmTile{2, 2} : GemmTile{1, 1};
}

}  // namespace mf
