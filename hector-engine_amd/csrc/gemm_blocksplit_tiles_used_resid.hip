// Tilings of the block-split product (gemm_blocksplit_tiles.h): the residual epilogue, groups of the weight that no row uses left out.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_used_resid(HE_BS_DISPATCH_ARGS) {
  HE_BS_SIXTEEN_ROWS(BS_RESID, true, bf16_t)
  HE_BS_NO_TILING;
}
