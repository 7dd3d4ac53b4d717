// z4c_tile_reg.hip -- the Z4c tile kernel (z4c_tile.h) with staging through registers.
#include "z4c_tile.h"

namespace bamhip {

int tile_reg(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return launch_tiles<0, 1>(P, R, K, flag, st);
}

}  // namespace bamhip
