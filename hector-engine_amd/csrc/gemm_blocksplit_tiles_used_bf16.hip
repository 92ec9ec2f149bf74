// Tilings of the block-split product (gemm_blocksplit_tiles.h): bf16 results, groups of the weight that no row uses left out.
#include "gemm_blocksplit_tiles.h"

int he_blocksplit_tiles_used_bf16(HE_BS_DISPATCH_ARGS) {
#define HE_BS_USED(R_, U_) HE_BS_TILING_OF(1, R_, U_, false, true, bf16_t)
  HE_BS_USED(1, 1) HE_BS_USED(1, 2) HE_BS_USED(1, 4) HE_BS_USED(2, 1) HE_BS_USED(2, 2) HE_BS_USED(2, 4) HE_BS_USED(4, 1) HE_BS_USED(4, 2)
  he_set_error("he_gemm_blocksplit_bf16: no kernel for R=%d U=%d", p.R, p.U);
  return -1;
}
