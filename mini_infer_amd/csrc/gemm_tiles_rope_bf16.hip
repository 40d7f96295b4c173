// The rotary products of gemm_tiles_bf16.hip: [q | k | v] of some hundreds of rows, rotated and written where it belongs in the last step
// (gated_tile.h), in the tiles that the product alone is made in, so that the results are the same.
//
// What this saves is a launch that reads and writes the whole projection again.
#include "gemm_tiles.h"

extern "C" int mi_gemm_tiles_rope(const void* a, int64_t lda, const void* w, int64_t ldw, void* q, int64_t ldq, const float* cos_t, const float* sin_t,
                                  const int* slots, void* k_pages, void* v_pages, int m, int k, int q_heads, int kv_heads, int head_dim, int page_size,
                                  int num_pages, int v_transposed, int shape, hipStream_t stream) {
#define X(...) gemm_tiles_launch<TileProduct<__VA_ARGS__>, PAIRED_ROTARY, false>,
  static void (*const launches[])(const GemmTilesLaunch&) = {GEMM_TILE_SHAPES(X)};
#undef X
  const RotaryWrite how = {cos_t, sin_t, slots, (bf16_t*)q, (bf16_t*)k_pages, (bf16_t*)v_pages, ldq, q_heads, kv_heads, head_dim, page_size, v_transposed};
  MI_REQUIRE(rotary_write_fits(how, m, num_pages), "gemm_tiles_rope: m=%d, %d + 2 * %d heads of %d, pages of %d", m, q_heads, kv_heads, head_dim, page_size);
  MI_REQUIRE(k >= 64 && k % 64 == 0 && lda >= k && ldw >= k && lda % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0 &&
                 shape >= 0 && shape < (int)(sizeof(launches) / sizeof(launches[0])),
             "gemm_tiles_rope: takes K a multiple of 64 and rows on 16 bytes; got k=%d lda=%lld ldw=%lld shape %d", k, (long long)lda, (long long)ldw, shape);
  const int pairs = (q_heads + 2 * kv_heads) * (head_dim / 2);
  MI_REQUIRE((int64_t)ceil_div(m, 32) * ceil_div(pairs, 16) < (1 << 30), "gemm_tiles_rope: too many tiles");
  launches[shape]({a, w, nullptr, lda, ldw, 0, 0, 1.f, {}, how, true, m, pairs, k, k / 64, stream});
  MI_CHECK_LAUNCH("gemm_tiles_rope");
  return MI_OK;
}
