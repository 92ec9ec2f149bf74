// Products of many rows (gemm_tall_tiles.h): SiLU-gated results.
#include "gemm_tall_tiles.h"

int gt_run_gated(const GtCase& c, int tile, int mtiles, hipStream_t s) {
  return gt_run_tile<GT_GATED, false>(c, tile, mtiles, s);
}
