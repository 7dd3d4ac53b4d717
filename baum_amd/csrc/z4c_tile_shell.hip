// z4c_tile_shell.hip -- variants of the Z4c tile kernel (z4c_tile.h).
#include "z4c_tile.h"

namespace bamhip {

int tile_shell_dma(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return shell_variant<3, 1, 1>(P, R, K, flag, st);
}
int tile_shell_reg(const Z4cPtrs &P, const RegionLists &R, const Z4cK &K, int *flag, hipStream_t st) {
  return shell_variant<0, 1, 1>(P, R, K, flag, st);
}

}  // namespace bamhip
