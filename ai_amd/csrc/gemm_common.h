// Device helpers shared by the product kernels (gemm.hip, gemm_h2.hip).
#pragma once

#include <hip/hip_runtime.h>

namespace fa {

// Tile index of this workgroup. Workgroup ids are dealt to the 8 XCDs
// round-robin; each XCD gets a contiguous run of tiles (row-major over n) so
// the tiles sharing A rows and B columns share that XCD's L2.
__device__ __forceinline__ int xcd_tile(int tiles_m, int tiles_n) {
  constexpr int kXcd = 8;
  const int total = tiles_m * tiles_n;
  int tile = blockIdx.x;
  const int per = total / kXcd;
  if (per > 0 && tile < per * kXcd) tile = (tile % kXcd) * per + tile / kXcd;
  return tile;
}

}  // namespace fa
