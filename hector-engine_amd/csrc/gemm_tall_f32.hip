// Products of many rows (gemm_tall_tiles.h): fp32 results, whole or of K slices.
#include "gemm_tall_tiles.h"

int gt_run_f32(const GtCase& c, int tile, int mtiles, hipStream_t s) {
#define GT_CASE(BM, BN, NX, NW) if (tile == ((BM) << 16 | (BN))) return gt_run<BM, BN, NX, NW, GT_F32, false>(c, mtiles, s);
  GT_TILES(GT_CASE)
  return -1;
}
