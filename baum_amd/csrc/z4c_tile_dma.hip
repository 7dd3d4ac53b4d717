// z4c_tile_dma.hip -- the Z4c tile kernel (z4c_tile.h) with LDS-DMA staging in dwords.
#include "z4c_tile.h"

namespace bamhip {

int tile_dma(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return launch_tiles<3, 1>(P, R, K, flag, st);
}

}  // namespace bamhip
