// Tilings of the few-rows product (gemm_blocksplit_tiles.h): gated SiLU x up epilogue, 32-bit output.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_gated_f32(HE_BS_DISPATCH_ARGS) {
  HE_BS_SIXTEEN_ROWS(BS_GATED, false, float)
  HE_BS_ORDERED(BS_GATED, false, float)
  HE_BS_THIRTY_TWO_ROWS(BS_GATED, float)
  HE_BS_NO_TILING;
}
