// Products of many rows (gemm_tall_tiles.h): results of the other gated activations.
#include "gemm_tall_tiles.h"

int gt_run_clamped(const GtCase& c, int tile, int mtiles, hipStream_t s) {
  return gt_run_tile<GT_GATED, true>(c, tile, mtiles, s);
}
