// Tilings of the few-rows product (gemm_blocksplit_tiles.h): plain and bias epilogues, bfloat16 output.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_bf16(HE_BS_DISPATCH_ARGS) {
  HE_BS_SIXTEEN_ROWS(BS_PLAIN, false, bf16_t)
  HE_BS_ORDERED(BS_PLAIN, false, bf16_t)
  HE_BS_THIRTY_TWO_ROWS(BS_PLAIN, bf16_t)
  HE_BS_NO_TILING;
}
