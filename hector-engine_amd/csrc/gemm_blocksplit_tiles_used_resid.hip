// Tilings of the block-split product (gemm_blocksplit_tiles.h): the residual epilogue, groups of the weight that no row uses left out.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_used_resid(HE_BS_DISPATCH_ARGS) {
  HE_BS_SIXTEEN_ROWS(BS_RESID, true, bf16_t)
  he_set_error("he_gemm_blocksplit_bf16: no kernel for SP=%d MT=%d NA=%d S=%d", p.SP, p.MT, p.NA, p.S);
  return -1;
}
