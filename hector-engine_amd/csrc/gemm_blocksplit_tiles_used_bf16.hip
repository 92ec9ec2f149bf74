// Tilings of the block-split product (gemm_blocksplit_tiles.h): bf16 results, groups of the weight that no row uses left out.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_used_bf16(HE_BS_DISPATCH_ARGS) {
  HE_BS_SIXTEEN_ROWS(BS_PLAIN, true, bf16_t)
  HE_BS_ORDERED(BS_PLAIN, true, bf16_t)
  HE_BS_NO_TILING;
}
