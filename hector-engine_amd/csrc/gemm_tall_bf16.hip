// Products of many rows (gemm_tall_tiles.h): plain bf16 results.
#include "gemm_tall_tiles.h"

int gt_run_bf16(const GtCase& c, int tile, int mtiles, hipStream_t s) {
#define GT_CASE(BM, BN, NX, NW) if (tile == ((BM) << 16 | (BN))) return gt_run<BM, BN, NX, NW, GT_BF16, false>(c, mtiles, s);
  GT_TILES(GT_CASE)
  return -1;
}
