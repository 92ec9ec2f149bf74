// Tilings of the few-rows product (gemm_blocksplit_tiles.h): the residual epilogue.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_resid(HE_BS_DISPATCH_ARGS) {
  HE_BS_SIXTEEN_ROWS(BS_RESID, false, bf16_t)
  HE_BS_THIRTY_TWO_ROWS(BS_RESID, bf16_t)
  HE_BS_NO_TILING;
}
