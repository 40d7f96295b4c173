// How the pairs of routed experts are cut into row tiles (expert_tiles.hip makes their products, routed_experts.hip lists them).
#pragma once

#include "common.h"

constexpr int CUT_FORMS = 4;  // the first forms of turns_product.h, 256 rows of W each
__host__ __device__ constexpr int cut_rows(int form) { return form == 0 ? 64 : form == 1 ? 128 : form == 2 ? 160 : 256; }

// Cut c < CUTS - 1: an expert's pairs into as few tiles as hold them where none is larger than form c + 1, as many pairs in each, of the smallest
// form that holds those.  The last cut: full tiles of the largest form, and one of the smallest that holds the rest.
constexpr int CUTS = CUT_FORMS;
struct Cover {  // an expert's: full tiles of the largest form in front, then tiles of a form with `each` pairs, the last one perhaps fewer
  int full, tiles, each, form;
};
__host__ __device__ inline Cover cover(int pairs, int cut) {
  Cover c = {0, 0, 0, 0};
  if (pairs <= 0) return c;
  if (cut == CUTS - 1) {
    c.full = (pairs - 1) / cut_rows(CUT_FORMS - 1);
    pairs -= c.full * cut_rows(CUT_FORMS - 1);
    c.tiles = 1;
  } else {
#pragma unroll
    for (int f = 1; f < CUT_FORMS; ++f)
      if (f == cut + 1) c.tiles = (pairs + cut_rows(f) - 1) / cut_rows(f);
  }
  c.each = (pairs + c.tiles - 1) / c.tiles;
#pragma unroll
  for (int f = 0; f + 1 < CUT_FORMS; ++f)
    if (c.each > cut_rows(f)) c.form = f + 1;
  return c;
}
__host__ __device__ inline int tiles_of(const Cover& c, int form) { return (c.form == form ? c.tiles : 0) + (form == CUT_FORMS - 1 ? c.full : 0); }

// A cut: row tiles of each form; experts with pairs; those whose weights are read again by a tile of another form, some time later.
struct CutSums {
  int tiles[CUT_FORMS], used, again;
};
__host__ __device__ inline void add(CutSums& sums, const Cover& c) {
#pragma unroll
  for (int f = 0; f < CUT_FORMS; ++f) sums.tiles[f] += tiles_of(c, f);
  sums.used += c.tiles > 0;
  sums.again += c.full > 0 && c.form < CUT_FORMS - 1;
}

// The row tiles that a cut can have at most.
__host__ __device__ inline int most_row_tiles(int pairs, int experts, int cut) {
  const int rows = cut == 0 ? cut_rows(1) : cut == 1 ? cut_rows(2) : cut_rows(3);
  return pairs / rows + (experts < pairs ? experts : pairs);
}

// The plan of a list: the sums of each cut, then its row tiles, the largest form first, expert by expert.
struct RowTile {
  int expert, row0, end, form;
};
struct CutsPlan {
  CutSums sums[CUTS];
};
static_assert(sizeof(CutsPlan) % 16 == 0 && sizeof(RowTile) == 16);
__host__ __device__ inline int64_t row_tiles_before(int cut, int pairs, int experts) {
  int64_t at = 0;
  for (int c = 0; c < cut; ++c) at += most_row_tiles(pairs, experts, c);
  return at;
}
__device__ __forceinline__ const RowTile* row_tiles_of(const CutsPlan* plan, int cut, int pairs, int experts) {
  return reinterpret_cast<const RowTile*>(plan + 1) + row_tiles_before(cut, pairs, experts);
}

// One wave makes one cut's part of the plan from the list's `first`.
__device__ __forceinline__ void plan_cut(const int* first, int pairs, int experts, int cut, CutsPlan* __restrict__ plan) {
  const int lane = threadIdx.x % MI_WAVE;
  CutSums sums = {};
  for (int e = lane; e < experts; e += MI_WAVE) add(sums, cover(first[e + 1] - first[e], cut));
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) {
    sums.used += __shfl_xor(sums.used, off, MI_WAVE);
    sums.again += __shfl_xor(sums.again, off, MI_WAVE);
#pragma unroll
    for (int f = 0; f < CUT_FORMS; ++f) sums.tiles[f] += __shfl_xor(sums.tiles[f], off, MI_WAVE);
  }
  RowTile* list = const_cast<RowTile*>(row_tiles_of(plan, cut, pairs, experts));
  int start[CUT_FORMS];  // of a form's row tiles that are still to come
  start[CUT_FORMS - 1] = 0;
#pragma unroll
  for (int f = CUT_FORMS - 2; f >= 0; --f) start[f] = start[f + 1] + sums.tiles[f + 1];
  for (int base = 0; base < experts; base += MI_WAVE) {
    const int e = base + lane, begin = e < experts ? first[e] : 0, end = e < experts ? first[e + 1] : 0;
    const Cover c = cover(end - begin, cut);
#pragma unroll
    for (int f = CUT_FORMS - 1; f >= 0; --f) {
      const int tiles = tiles_of(c, f);
      int upto = tiles;
#pragma unroll
      for (int off = 1; off < MI_WAVE; off <<= 1) {
        const int other = __shfl_up(upto, off, MI_WAVE);
        if (lane >= off) upto += other;
      }
      for (int i = 0; i < tiles; ++i) {
        const int rest = f == CUT_FORMS - 1 ? i - c.full : i;  // behind the full tiles
        const int row0 = begin + (rest < 0 ? i * cut_rows(CUT_FORMS - 1) : c.full * cut_rows(CUT_FORMS - 1) + rest * c.each);
        list[start[f] + upto - tiles + i] = {e, row0, min(row0 + (rest < 0 ? cut_rows(CUT_FORMS - 1) : c.each), end), f};
      }
      start[f] += __shfl(upto, MI_WAVE - 1, MI_WAVE);
    }
  }
  if (lane == 0) plan->sums[cut] = sums;
}
