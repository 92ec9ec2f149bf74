// Products of many rows (gemm_tall_tiles.h): fp32 results, whole or of K slices.
#include "gemm_tall_tiles.h"

int gt_run_f32(const GtCase& c, int tile, int mtiles, hipStream_t s) {
  return gt_run_tile<GT_F32, false>(c, tile, mtiles, s);
}
