// Products of some tens to some hundreds of rows: C = A * W^T, bfloat16, as tiles that stream both operands through LDS
// (tile_product.h, gemm_tiles.h), whole or left as float32 sums over ranges of K:
//   kind 0  C bfloat16
//   kind 1  part[s][M][N] float32: the sums over the s-th range of K, added up in order by whoever takes them
//   kind 2  C float32: the bfloat16 values times `scale` (an output head)
//   kind 3  silu(A * gate^T) * (A * up^T) bfloat16, W = [gate; up]; both products rounded to bfloat16 first
//   kind 4  the clamped activation of clamped_glu in its place, with biases or without; kind 5  gelu (tanh form) in the place of silu
//
// Which tile, and how many ranges, is chosen by the time that gemm_tiles_micros expects, a sum of what a launch costs anyhow, the
// bytes a CU brings in (see tile_product.h), its products, the bytes of W, later rounds of blocks, and the bytes written.  Its six
// numbers are a least-squares fit to 5,130 launches (12 matrices of 3072 x 2048 to 4096 x 14336 and 28672 x 4096, 24 to 768 rows,
// 20 tile shapes, every sensible number of ranges; relative error 8 %); the shape it picks is on average 1.4 % slower than the
// best one measured.  A rule by sizes alone would have to say the same in thresholds.
//
// Measured against what stood here before, microseconds, weights from memory (MI355X; a product in pieces without the reading of
// the pieces; gated with the activation): 3072 x 3072 at 24 / 64 / 128 / 271 rows 6.6 / 7.9 / 10.2 / 15.0 against the vendor
// library's 11.1 / 16.1 / 20.1 / 17.6, 3072 x 8192 11.6 / 13.3 / 18.0 / 25.9 against 16.8 / 23.6 / 42.4 / 31.9, 4096 x 14336 22 / 24
// / 30 / 47 against 33 / 41 / 76 / 77 (a product of one range of K and 128 features a block, which stood here for the last up to 128
// rows: 24 / 28 / 40); gate|up 16384 x 3072 19.8 / 24.3 / 35 / 41 against 23.9 (one launch, up to 32 rows) / 28.5 / 34 / 44 (two).
//
// This stands where the reference's engine calls the vendor BLAS (distributed/linear.py:167).
#include "gemm_tiles.h"

#include <math.h>

namespace {

struct Shape {
  int rows, features, ring_bytes, halves;  // halves: waves that share the K of a stage
  void (*launch)(const GemmTilesLaunch&);
};
template <class T, bool ODD = false>
constexpr Shape shape() {
  return {T::BM, T::BN, T::RING * 2, T::WK, gemm_tiles_launch<T, PAIRED_NOT, ODD>};
}
#define X(...) shape<TileProduct<__VA_ARGS__>>(),
const Shape SHAPES[] = {GEMM_TILE_SHAPES(X)};
#undef X
constexpr int SHAPE_COUNT = sizeof(SHAPES) / sizeof(SHAPES[0]);
constexpr int MOST_RANGES = 16;

// Microseconds that a launch is expected to take (rows: of W, gate and up together).
double gemm_tiles_micros(const Shape& s, int m, int rows, int k, int steps_each, int cus) {
  const int steps = ceil_div(k, 64), ranges = ceil_div(steps, steps_each);
  const int64_t blocks = (int64_t)ceil_div(m, s.rows) * ceil_div(rows, s.features) * ranges;
  const int xcds = max(1, cus / 32);  // (blocks are dealt to them in turn)
  const int64_t a_cu = ceil_div64(ceil_div64(blocks, xcds), max(1, cus / xcds));
  const int together = s.ring_bytes * 2 <= 163840 ? 2 : 1;
  const double brought = (double)a_cu * steps_each * (s.rows + s.features) * 128;
  const double products = (double)a_cu * steps_each * s.rows * s.features * 128;
  const double written = (double)m * rows * (ranges > 1 ? 4.0 * ranges : 2.0);
  return 3.63 + brought / 93.9e3 + products / 13.41e6 + (double)rows * k * 2 / 12.58e6 + 2.21 * (double)(ceil_div64(a_cu, together) - 1) +
         written / 4.84e6;
}

}  // namespace

// The best way to make a product: *shape and *ranges of K (1: whole), for a caller to whom sums over r > 1 ranges cost sum_base +
// sum_each * r microseconds more than the whole product.  most_ranges: 1 whole products only.  same_order: ranges by n and k alone, and
// every shape that is chosen sums a range in the same order, so that a row's sums do not depend on the other rows.
// Where rows of W are a multiple of 16 KB long, up to 128 rows are not cut into ranges of K that begin 4 KB apart: all blocks then ask the
// same memory channels at once, which the expected time does not know.  With the sum's launch, 8192 x 8192 at 17 / 64 rows in 4
// ranges 35.3 / 36.7 us, in 2 29.8 / 32.2 (the vendor library 31.0 / 33.0), 4096 x 16384 at 24 / 64 rows in 8 ranges 47.3 / 50.7, in 4, which
// begin 8 KB apart, 31.6 / 33.4 (the library 32.8 / 42.1).  More rows read little of W for what they multiply: 4096 x 8192 at 200 rows in 4 ranges 31.2, otherwise 36.6.
// cus: the device's compute units.  *micros: the expected microseconds, that extra included.
extern "C" int mi_gemm_tiles_plan(int m, int n, int k, int gated, int most_ranges, int same_order, float sum_base, float sum_each, int cus, int* shape,
                                  int* ranges, float* micros) {
  MI_REQUIRE(m >= 1 && n >= 1 && k >= 1 && cus >= 1, "gemm_tiles_plan: m=%d n=%d k=%d on %d compute units", m, n, k, cus);
  const int rows = gated ? 2 * n : n;
  const int steps = ceil_div(k, 64);
  double best = INFINITY;
  *shape = 0, *ranges = 1;
  int from = 1, to = max(1, min(min(most_ranges, MOST_RANGES), steps / 4));
  if (same_order) {  // a block a CU with tiles of 64 features
    to = max(1, min(min(MOST_RANGES, steps / 4), cus / ceil_div(n, 64)));
    from = to;
  }
  for (int i = 0; i < SHAPE_COUNT; ++i) {
    if (same_order && SHAPES[i].halves != 2) continue;
    for (int r = from; r <= to; ++r) {
      const int each = ceil_div(steps, r), got = ceil_div(steps, each);
      if (got != r && !same_order) continue;
      if (got > 1 && !same_order && m <= 128 && k % 8192 == 0 && each % 64 == 32) continue;  // (see above: the same memory channels)
      const double t = gemm_tiles_micros(SHAPES[i], m, rows, k, each, cus) + (got > 1 ? sum_base + sum_each * got : 0.0);
      if (t < best) best = t, *shape = i, *ranges = got;
    }
  }
  *micros = (float)best;
  return MI_OK;
}

// Rows and features of a shape (0: there is none of that number).
extern "C" int mi_gemm_tiles_rows(int shape) { return shape >= 0 && shape < SHAPE_COUNT ? SHAPES[shape].rows : 0; }
extern "C" int mi_gemm_tiles_features(int shape) { return shape >= 0 && shape < SHAPE_COUNT ? SHAPES[shape].features : 0; }

extern "C" int mi_gemm_tiles_take(int m, int n, int k, int64_t lda, int64_t ldw) {
  return m >= 1 && n >= 1 && k >= 32 && k % 32 == 0 && lda >= k && ldw >= k && lda % 8 == 0 && ldw % 8 == 0 &&
                 (int64_t)ceil_div(m, 32) * ceil_div(n, 32) * MOST_RANGES < (1 << 30)
             ? 1
             : 0;
}

// kind, out: as at the top; n: features written (kinds 3 to 5: W has 2 n rows; 8 ranges of these: shapes 0 and 1, whole, the sums of K's eighths added
// in order).  part of kind 1: [ranges][m][n], contiguous.
extern "C" int mi_gemm_tiles_bf16(int kind, const void* a, int64_t lda, const void* w, int64_t ldw, void* out, int64_t ldc, float scale,
                                  const float* bias, float limit, float slope, int m, int n, int k, int shape, int ranges, hipStream_t stream) {
  MI_REQUIRE(mi_gemm_tiles_take(m, n, k, lda, ldw) && ((uintptr_t)a | (uintptr_t)w) % 16 == 0,
             "gemm_tiles_bf16: takes K a multiple of 32 and rows on 16 bytes; got m=%d n=%d k=%d lda=%lld ldw=%lld", m, n, k, (long long)lda,
             (long long)ldw);
  const bool eighths = kind >= 3 && ranges == 8;
  MI_REQUIRE(!eighths || (m <= 32 && k % 512 == 0 && shape >= 0 && shape <= 1), "gemm_tiles_bf16: eighths of K of m=%d k=%d, shape %d", m, k, shape);
  MI_REQUIRE(kind >= 0 && kind <= 5 && (kind != 4 || limit > 0.f) && shape >= 0 && shape < SHAPE_COUNT && ranges >= 1 && ranges <= MOST_RANGES && (kind == 1 || ranges == 1 || eighths) &&
                 (kind == 1 || ldc >= n),
             "gemm_tiles_bf16: kind %d, shape %d, %d ranges", kind, shape, ranges);
  const int steps = ceil_div(k, 64), each = eighths ? steps : ceil_div(steps, ranges);
  MI_REQUIRE(eighths || ceil_div(steps, each) == ranges, "gemm_tiles_bf16: %d steps of K do not make %d ranges", steps, ranges);
  const int element = kind == 1 || kind == 2 ? 4 : 2, at_once = kind >= 3 ? 8 : 4;
  const bool vec = (uintptr_t)out % (at_once * element) == 0 && (kind == 1 ? n : ldc) % at_once == 0;
  const GemmTilesLaunch l = {a, w, out, lda, ldw, ldc, kind, scale, {bias, limit, slope}, {}, vec, m, n, k, each, stream};
  const bool odd = k % 64 != 0;  // (one shape for these: nothing real is made so)
  if (eighths) gemm_tiles_eighths_launch(SHAPES[shape].features, l);
  else if (kind >= 3) gemm_tiles_gated_launch(shape, odd, l);
  else if (odd) gemm_tiles_launch<TileProduct<GEMM_TILE_ODD_SHAPE>, PAIRED_NOT, true>(l);
  else SHAPES[shape].launch(l);
  MI_CHECK_LAUNCH("gemm_tiles_bf16");
  return MI_OK;
}

// out[i] = the sum over s of pieces[s][i], in order, as bfloat16; four values a thread.
namespace {
__global__ __launch_bounds__(256) void sum_pieces_kernel(const float* __restrict__ pieces, bf16_t* __restrict__ out, int count, int64_t size) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= size) return;
  float sum[4] = {0.f, 0.f, 0.f, 0.f};
  if (size % 4 == 0) {
#pragma unroll 8
    for (int s = 0; s < count; ++s) {
      float v[4];
      mi_load_cols<float, 4>(pieces + s * size + i, v);
#pragma unroll
      for (int c = 0; c < 4; ++c) sum[c] += v[c];
    }
    mi_store_cols<bf16_t, 4>(out + i, sum);
  } else {
    for (int c = 0; c < 4 && i + c < size; ++c) {
      for (int s = 0; s < count; ++s) sum[c] += pieces[s * size + i + c];
      out[i + c] = from_f32<bf16_t>(sum[c]);
    }
  }
}
}  // namespace

// pieces [count][size] float32 and out [size] bfloat16, both contiguous.
extern "C" int mi_sum_pieces(const float* pieces, void* out, int count, int64_t size, hipStream_t stream) {
  MI_REQUIRE(count >= 1 && size >= 1 && size < ((int64_t)1 << 40) && (uintptr_t)pieces % 16 == 0 && (uintptr_t)out % 8 == 0,
             "sum_pieces: %d pieces of %lld", count, (long long)size);
  sum_pieces_kernel<<<(unsigned)ceil_div64(size, 1024), 256, 0, stream>>>(pieces, (bf16_t*)out, count, size);
  MI_CHECK_LAUNCH("sum_pieces");
  return MI_OK;
}
