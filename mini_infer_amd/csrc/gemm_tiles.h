// The kernel of gemm_tiles_bf16.hip, gemm_tiles_gated_bf16.hip and gemm_tiles_rope_bf16.hip, and the shapes that they compile it for.
#pragma once

#include "gated_tile.h"
#include "tile_product.h"

// Of the 20 shapes measured those that are the best anywhere by more than 1 %.
#define GEMM_TILE_SHAPES(X) \
  X(1, 2, 2, 2, 2, 6)  /* 32 x 64 */ \
  X(1, 4, 2, 2, 2, 6)  /* 32 x 128 */ \
  X(1, 2, 2, 3, 2, 5)  /* 48 x 64 */ \
  X(1, 2, 2, 4, 2, 5)  /* 64 x 64 */ \
  X(1, 4, 2, 4, 2, 6)  /* 64 x 128 */ \
  X(1, 2, 2, 5, 2, 4)  /* 80 x 64 */ \
  X(2, 2, 2, 3, 2, 6)  /* 96 x 64 */ \
  X(1, 4, 2, 6, 2, 5)  /* 96 x 128 */ \
  X(2, 2, 2, 4, 2, 6)  /* 128 x 64 */ \
  X(2, 2, 2, 4, 4, 5)  /* 128 x 128 */ \
  X(1, 4, 2, 9, 2, 4)  /* 144 x 128 */ \
  X(2, 4, 1, 5, 4, 3)  /* 160 x 256 */ \
  X(2, 2, 2, 6, 4, 3)  /* 192 x 128 */ \
  X(2, 4, 1, 8, 4, 2)  /* 256 x 256 */
#define GEMM_TILE_ODD_SHAPE 1, 2, 2, 4, 2, 5  // of a K of odd 32s

// pieces of 32 of K of range `range` of `ranges`, and the first of them; ranges are whole steps of 64
struct KRange {
  int first, halves;
};
__host__ __device__ __forceinline__ KRange k_range(int k, int steps_each, int range) {
  const int first = range * steps_each * 2;
  return {first, min(steps_each * 2, k / 32 - first)};
}

// Which rows of W stand beside one another in a tile: none, gate and up, or the two elements that are rotated together.
enum { PAIRED_NOT = 0, PAIRED_GATED = 1, PAIRED_ROTARY = 2 };

// (A type picked by comparing with one of those would put an unnamed enumeration into the kernel's symbol, which the compiler numbers otherwise for
// the host than for the device: the kernel is then not found.)
template <int PAIRED>
struct PairedHow {
  using type = GatedActivation;
};
template <>
struct PairedHow<2> {
  using type = RotaryWrite;
};

// Where rows of W are a multiple of 4 KB apart, blocks that walk K in step all ask the same memory channels; gated products and the output head then begin
// a step later from tile to tile, and go round.  Microseconds, from the beginning / so: gate|up 16384 x 2048 at 33 / 48 / 96 / 192 rows 16.5, 16.6, 19.3, 25.1 / 14.1, 14.1,
// 18.8, 24.5, 28672 x 4096 48.1, 48.8, 52.5, 64.9 / 43.4, 44.7, 48.9, 63.5; 128256 x 2048 at 17 / 32 / 64 / 128 102, 109, 125, 135 / 90, 96, 107, 107, x 4096
// 176, 182, 202, 219 / 173, 178, 196, 218, 64128 x 6144 145, 154, 169, 174 / 125, 131, 145, 146.  (Of 16384 x 3072, 28672 x 5120 and 128256 x 1024 the same or 3 % more; five
// or eight steps later for one: 128256 x 4096 189 and 176.  Ranges of K, which begin apart: the same.  Plain whole products and those with a rotation give the
// same bits as one another, which have their rows of W in other tiles: from the beginning.)
//
// Not with so few tiles that the channels are not what they wait for (1,024 features x 4096 at 66 rows 14.8 / 15.9, 512 x 8192 at 109 25.2 / 27.5), not with several
// tiles of rows to few of features, whose blocks read the same rows of W, and not in tiles 64 wide where rows of W are an odd multiple of 8 KB apart, whose
// halves of 32 features then meet again (4,096 features x 4096 at 33 / 48 rows 17.6 / 19.7 and 18.9 / 21.4, 8,192 at 33 / 96 1.15 times as long, 18,432 1.2; in tiles
// 128 wide 0.8 to 0.95).
static bool turned(int kind, int64_t ldw, int tile_width, int feature_tiles) {
  return kind >= 2 && ldw % 2048 == 0 && feature_tiles > 128 && !(tile_width == 64 && ldw % 8192 == 4096);
}

// (the second bound: two blocks a CU where LDS holds two)
template <class T, int PAIRED, bool ONCE, bool ODD, bool ROUND, bool EIGHTHS = false>
__global__ __launch_bounds__(T::THREADS, T::RING * 4 <= 163840 ? 2 : 1) void gemm_tiles_kernel(
    const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int64_t ldw, void* __restrict__ out, int64_t ldc,
    int kind, float scale, const typename PairedHow<PAIRED>::type how, bool vec, int m, int n, int k, int steps_each, int row_tiles, int feature_tiles,
    int total) {
  __shared__ __align__(16) bf16_t ring[T::RING];
  // Consecutive places go to one XCD (workgroups are dealt to the 8 of them in turn): the row tiles that read the same
  // rows of W run at the same time behind one L2.
  const int place = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  if (place >= total) return;
  const int row_tile = place % row_tiles, rest = place / row_tiles;
  const int feature_tile = rest % feature_tiles, range = rest / feature_tiles;
  const KRange part = k_range(k, steps_each, range);
  constexpr int FEATURES = PAIRED != PAIRED_NOT ? T::BN / 2 : T::BN;
  const int r0 = row_tile * T::BM, f0 = feature_tile * FEATURES;
  a += part.first * 32;
  w += part.first * 32;
  T tile;
  const auto a_row = [&](int r) { return a + (int64_t)min(r0 + r, m - 1) * lda; };
  const auto w_row = [&](int r) {
    if constexpr (PAIRED == PAIRED_ROTARY) return w + (int64_t)rotary_row_of(GatedTile<T::NT>::row_of(r, f0, n), n, how.head_dim) * ldw;
    else return w + (int64_t)(PAIRED == PAIRED_GATED ? GatedTile<T::NT>::row_of(r, f0, n) : min(f0 + r, n - 1)) * ldw;
  };
  if constexpr (EIGHTHS) tile.template run_eighths<ROUND>(ring, part.halves, a_row, w_row, feature_tile % 4);
  else tile.template run<ONCE, ODD, ROUND>(ring, part.halves, a_row, w_row, ROUND ? feature_tile % (part.halves / 2) : 0);
  if constexpr (PAIRED == PAIRED_ROTARY) {
    tile.leave(ring);
    write_rotated<GatedTile<T::NT>, T::BM, T::BN, T::MADE, T::THREADS>(ring, how, r0, m, f0, n);
    return;
  } else if constexpr (PAIRED == PAIRED_GATED) {
    tile.leave(ring);
#define MI_WRITE(ACT) write_activated<ACT, GatedTile<T::NT>, T::BM, T::BN, T::MADE, T::THREADS>(ring, how, (bf16_t*)out, ldc, vec, r0, m, f0, n)
    if (kind == 4) MI_WRITE(ACT_CLAMPED);
    else if (kind == 5) MI_WRITE(ACT_GELU);
    else MI_WRITE(ACT_SILU);
#undef MI_WRITE
    return;
  }
#pragma unroll
  for (int i = 0; i < T::MT; ++i) {
    const int row = r0 + tile.row(i);
    if (!tile.mine(i) || row >= m) continue;
#pragma unroll
    for (int j = 0; j < T::NT; ++j) {
      const int f = f0 + tile.feature(j);
      float v[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = kind == 2 ? to_f32(from_f32<bf16_t>(tile.acc[j][i][c])) * scale : tile.acc[j][i][c];
      const bool whole = vec && f + 4 <= n;
      if (kind != 0) {
        float* o = kind == 1 ? (float*)out + ((int64_t)range * m + row) * n + f : (float*)out + (int64_t)row * ldc + f;
        if (whole) {
          mi_store_cols<float, 4>(o, v);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (f + c < n) o[c] = v[c];
        }
      } else {
        bf16_t* o = (bf16_t*)out + (int64_t)row * ldc + f;
        if (whole) {
          mi_store_cols<bf16_t, 4>(o, v);
        } else {
#pragma unroll
          for (int c = 0; c < 4; ++c)
            if (f + c < n) o[c] = from_f32<bf16_t>(v[c]);
        }
      }
    }
  }
}

struct GemmTilesLaunch {
  const void *a, *w;
  void* out;
  int64_t lda, ldw, ldc;
  int kind;
  float scale;
  GatedActivation how;
  RotaryWrite rotary;
  bool vec;
  int m, n, k, steps_each;
  hipStream_t stream;
};

template <class T, int PAIRED, bool ODD, bool EIGHTHS = false>
static void gemm_tiles_launch(const GemmTilesLaunch& l) {
  const int row_tiles = ceil_div(l.m, T::BM), feature_tiles = ceil_div(l.n, PAIRED != PAIRED_NOT ? T::BN / 2 : T::BN);
  const int total = row_tiles * feature_tiles * ceil_div(ceil_div(l.k, 64), l.steps_each);
  auto kernel = gemm_tiles_kernel<T, PAIRED, true, ODD, false, EIGHTHS>;
  if constexpr (!EIGHTHS) {  // (of eighths: one row tile)
    if (row_tiles > 1) kernel = gemm_tiles_kernel<T, PAIRED, false, ODD, false>;
  }
  if constexpr (!ODD && PAIRED != PAIRED_ROTARY) {
    if (turned(l.kind, l.ldw, T::BN, feature_tiles)) {
      kernel = gemm_tiles_kernel<T, PAIRED, true, false, true, EIGHTHS>;
      if constexpr (!EIGHTHS) {
        if (row_tiles > 1) kernel = gemm_tiles_kernel<T, PAIRED, false, false, true>;
      }
    }
  }
  const auto& how = [&]() -> const auto& {
    if constexpr (PAIRED == PAIRED_ROTARY) return l.rotary;
    else return l.how;
  }();
  kernel<<<ceil_div(total, 8) * 8, T::THREADS, 0, l.stream>>>((const bf16_t*)l.a, l.lda, (const bf16_t*)l.w, l.ldw, l.out, l.ldc, l.kind,
                                                             l.scale, how, l.vec, l.m, l.n, l.k, l.steps_each, row_tiles, feature_tiles, total);
}

// gemm_tiles_gated_bf16.hip
void gemm_tiles_gated_launch(int shape, bool odd, const GemmTilesLaunch& l);
void gemm_tiles_eighths_launch(int features, const GemmTilesLaunch& l);
