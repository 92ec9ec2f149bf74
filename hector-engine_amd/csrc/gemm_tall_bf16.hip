// Products of many rows (gemm_tall_tiles.h): plain bf16 results.
#include "gemm_tall_tiles.h"

int gt_run_bf16(const GtCase& c, int tile, int mtiles, hipStream_t s) {
  return gt_run_tile<GT_BF16, false>(c, tile, mtiles, s);
}
