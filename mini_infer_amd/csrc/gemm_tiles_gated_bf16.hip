// The gated products of gemm_tiles_bf16.hip (a file of their own: the two compile side by side).
#include "gemm_tiles.h"

void gemm_tiles_gated_launch(int shape, bool odd, const GemmTilesLaunch& l) {
#define X(...) gemm_tiles_launch<TileProduct<__VA_ARGS__>, PAIRED_GATED, false>,
  static void (*const launches[])(const GemmTilesLaunch&) = {GEMM_TILE_SHAPES(X)};
#undef X
  if (odd) gemm_tiles_launch<TileProduct<GEMM_TILE_ODD_SHAPE>, PAIRED_GATED, true>(l);
  else launches[shape](l);
}

// Tiles of 32 rows that sum K in eighths, which are added in order: the sums of gemm_skinny_bf16, whose waves take an eighth each.  That kernel reads W once and the
// rows of A once for every 32 features of W, from L2 and by each wave for itself, which at 17 to 32 rows bounds it; here A goes through LDS as W does.  gate|up
// 16384 x 3072 / 16384 x 2048 / 28672 x 5120 at 32 rows 23.8 -> 20.9, 19.6 -> 15.1, 73.7 -> 55.8 us (4.8, 4.4 and 5.3 TB/s); 24 requests decoding at 3B sizes 3,190 -> 3,113,
// 17 at 1B 1,110 -> 1,042, 24 at 8B 3,801 -> 3,737.
void gemm_tiles_eighths_launch(int features, const GemmTilesLaunch& l) {
  if (features == 64) gemm_tiles_launch<TileProduct<1, 2, 2, 2, 2, 6>, PAIRED_GATED, false, true>(l);
  else gemm_tiles_launch<TileProduct<1, 4, 2, 2, 2, 6>, PAIRED_GATED, false, true>(l);
}
