// z4c_tile_bulk.hip -- variants of the Z4c tile kernel (z4c_tile.h).
#include "z4c_tile.h"

namespace bamhip {

int tile_bulk_dma(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return bulk_variant<LBulk, 3, 1, 2>(P, R, K, flag, st);
}
int tile_bulk_reg(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return bulk_variant<LBulk, 0, 1, 2>(P, R, K, flag, st);
}
int tile_bulk_dma_x4(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return bulk_variant<LBulk, 3, 4, 2>(P, R, K, flag, st);
}

}  // namespace bamhip
