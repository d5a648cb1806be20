// Instantiation of the four f16/bf16 tile shapes for one (element type, B layout,
// K check) -- one translation unit per combination, so that they build in
// parallel: 256 x 256 and 256 x 224 tiles with 8 waves and one workgroup per CU
// (128 KiB of LDS); 128 x 128 tiles with 4 waves and two workgroups per CU, or one with a
// deeper ring;
// 64 x 256 tiles (M <= 64, short K) with 4 waves and two workgroups per CU.
#pragma once

#include "kernels.h"
#include "tile16_kernel.h"

namespace cmpext3 {

// 128 x 128 tiles that leave every CU at most one workgroup take a ring of four K steps
// (128 KiB of LDS) instead of two: alone on its CU a workgroup has no other to run while
// its loads are on their way, and with two slots each load has only a step (~0.2 us of
// matrix products) to arrive.  With four, three steps are in flight and what a CU can
// take in from L2 bounds it (~34 bytes per cycle; 8 waves instead of 4: no change).
// MI355X, two slots -> four: x[1024, 4096] W[4096, 4096]^T bf16 41.6 -> 30.3 us, fp16
// 2048^3 24.0 -> 19.3, 1024^3 12.6 -> 9.7, x[4096, 512] W[1024, 512]^T 9.8 -> 8.5.  Below
// 8 steps per workgroup there is nothing to keep in flight and filling the ring costs more
// (2048 x 2048 x 128 5.7 -> 6.1, x[200, 320] W[2048, 320]^T 6.0 -> 6.1).
inline bool deep_ring(const GemmParams& p, dim3 grid) {
  const int k = p.splits > 1 ? p.ksplit : p.K;
  return k >= 512 && (uint64_t)grid.x * grid.z <= 256;
}

template <typename T, bool KN, bool KCHECK>
hipError_t launch_tiles(KernelId id, const GemmParams& p, dim3 grid, hipStream_t s) {
  switch (id) {
    case kTile256x256:
      return launch_tile16_k<T, KN, 256, 256, 4, 2, 1, KCHECK>(p, grid, s);
    case kTile256x224:
      return launch_tile16_k<T, KN, 256, 224, 4, 2, 1, KCHECK>(p, grid, s);
    case kTile128x128:
      if (deep_ring(p, grid)) return launch_tile16_k<T, KN, 128, 128, 2, 2, 1, KCHECK, 4>(p, grid, s);
      return launch_tile16_k<T, KN, 128, 128, 2, 2, 2, KCHECK>(p, grid, s);
    case kTile64x256:
      return launch_tile16_k<T, KN, 64, 256, 1, 4, 2, KCHECK>(p, grid, s);
    default:
      return hipErrorInvalidValue;
  }
}

}  // namespace cmpext3

#define CMPEXT3_TILE_TU(NAME, T, KN, KCHECK)                                               \
  namespace cmpext3 {                                                                      \
  hipError_t NAME(KernelId id, const GemmParams& p, dim3 grid, hipStream_t s) {            \
    return launch_tiles<T, KN, KCHECK>(id, p, grid, s);                                    \
  }                                                                                        \
  }
