// The gated products of gemm_tiles_bf16.hip (a file of their own: the two compile side by side).
#include "gemm_tiles.h"

void gemm_tiles_gated_launch(int shape, bool odd, const GemmTilesLaunch& l) {
#define X(...) gemm_tiles_launch<TileProduct<__VA_ARGS__>, PAIRED_GATED, false>,
  static void (*const launches[])(const GemmTilesLaunch&) = {GEMM_TILE_SHAPES(X)};
#undef X
  if (odd) gemm_tiles_launch<TileProduct<GEMM_TILE_ODD_SHAPE>, PAIRED_GATED, true>(l);
  else launches[shape](l);
}
