// Products of some tens of rows with small matrices: C = A * W^T, bfloat16 in and out, whole in one launch.
//
// What bounds them is the way through K: a tile of gemm_tiles_bf16 walks all of it in steps of 64 that wait for one another, 0.15 us each, on as
// few compute units as there are tiles (2048 x 2048 at 32 rows: 32 blocks, 9.9 us for 8 MB), and cut into ranges it needs a second launch.  Here a
// block's 8 waves share K: each takes an eighth of it, with everything that it needs of it asked for at once (32 rows and 16 features, K 2048:
// two rounds of loads), and the eight sums meet in LDS in order.  So a block holds few rows and features, what two blocks have in common comes from L2, and the
// launch is about one trip to memory long.  The larger the matrix and the more rows, the more that second reading costs against a tile's: the
// expected time below says where.
//
// Microseconds, weights from memory (vendor library / best of gemm_tiles_bf16, the launch that adds its ranges up included / this; the form taken is the first
// of FORMS with no more blocks than compute units):
//
//     rows               17                  32                  48                  64                  96                  128
//     1024 x 1024        5.7 / 6.3 / 3.7     8.0 / 6.4 / 3.7     8.0 / 6.0 / 3.7     8.3 / 6.0 / 3.7     8.0 / 6.1 / 4.7     8.0 / 6.1 / 4.7
//     2048 x 1024        6.7 / 6.2 / 4.0     10.3 / 6.5 / 4.0    10.3 / 6.3 / 5.0    10.6 / 6.5 / 5.0    10.3 / 6.4 / 5.6    10.1 / 6.5 / 5.6
//     2048 x 2048        11.0 / 6.7 / 5.7    11.4 / 7.2 / 6.1    11.3 / 8.5 / 7.3    11.8 / 9.0 / 7.7    11.4 / 10.0 / 8.5   11.3 / 10.0 / 8.4
//     3072 x 2048        11.7 / 8.2 / 5.8    11.6 / 8.4 / 7.7    11.9 / 9.6 / 8.5    12.1 / 10.3 / 8.9
//     8192 x 2048        14.2 / 11.2 / 10.2  14.6 / 11.9 / 11.4
//     2048 x 3072        12.0 / 7.5 / 7.0    10.4 / 8.0 / 8.0    10.3 / 9.1 / 9.7    15.6 / 9.8 / 10.2   10.9 / 11.3 / 11.4
//     8192 x 3072        19.9 / 15.2 / 13.0  19.7 / 15.0 / 15.1
//     4096 x 4096        14.2 / 11.6 / 10.3  14.2 / 11.9 / 12.9  14.1 / 12.8 / 14.2
//
// (Wider blocks, 4 x 1 to 4 x 4 tiles, and 16 waves were the better form nowhere by more than 0.2 us.)  A row's sums depend on K alone.
#include "common.h"

#include <math.h>

#include <type_traits>

namespace {

typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int WAVES = 8;
// of the expected time: a launch, bytes a block brings in a microsecond, bytes of W from memory
constexpr double ROWS_BASE = 2.51, ROWS_INTAKE = 50.5e3, ROWS_MEMORY = 12.2e6;

// RT x FT: a block's tiles of 16 rows and of 16 features; U: steps of 32 of K whose loads are asked for together.  ONCE: one block reads these features.
template <int RT, int FT, int U, bool ONCE>
__global__ __launch_bounds__(WAVES * MI_WAVE, 2) void gemm_rows_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int64_t ldw,
                                                                       bf16_t* __restrict__ out, int64_t ldc, bool vec, int m, int n, int k, int row_tiles,
                                                                       int total) {
  __shared__ __align__(16) f32x4_t meet[WAVES][FT * RT][MI_WAVE];
  // consecutive places go to one XCD: the blocks that read the same features run behind one L2
  const int place = (blockIdx.x % 8) * (gridDim.x / 8) + blockIdx.x / 8;
  if (place >= total) return;
  const int r0 = place % row_tiles * (RT * 16), f0 = place / row_tiles * (FT * 16);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), lane = threadIdx.x % MI_WAVE;
  const int col = lane % 16, quad = lane / 16;
  uint32_t lower[FT], upper[FT];  // offsets of this lane's 16 bytes in the lower and upper 8 features (past the end: the last one again)
#pragma unroll
  for (int t = 0; t < FT; ++t) {
    const int row = f0 + t * 16 + line_row_of_lane(lane);
    lower[t] = (uint32_t)min(row, n - 1) * (uint32_t)(ldw * 2) + line_chunk_of_lane(lane);
    upper[t] = (uint32_t)min(row + 8, n - 1) * (uint32_t)(ldw * 2) + line_chunk_of_lane(lane);
  }
  const bf16_t* x[RT];
#pragma unroll
  for (int i = 0; i < RT; ++i) x[i] = a + (int64_t)min(r0 + i * 16 + col, m - 1) * lda + quad * 8;
  f32x4_t acc[FT][RT];
#pragma unroll
  for (int t = 0; t < FT; ++t)
#pragma unroll
    for (int i = 0; i < RT; ++i) acc[t][i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  auto some = [&](int step, auto count) {  // that many steps from `step` on
    constexpr int N = decltype(count)::value;
    bf16x8_t wv[N][FT], xv[N][RT];
#pragma unroll
    for (int u = 0; u < N; u += 2)
#pragma unroll
      for (int t = 0; t < FT; ++t) load_line_pair<ONCE>(w, step + u, lower[t], upper[t], wv[u][t], wv[u + 1][t]);
#pragma unroll
    for (int u = 0; u < N; ++u)
#pragma unroll
      for (int i = 0; i < RT; ++i) xv[u][i] = *reinterpret_cast<const bf16x8_t*>(x[i] + (step + u) * 32);
    __builtin_amdgcn_sched_barrier(0);  // (or the compiler asks for half of them at a time)
#pragma unroll
    for (int u = 0; u < N; u += 2) {
#pragma unroll
      for (int t = 0; t < FT; ++t) lines_to_operands(wv[u][t], wv[u + 1][t]);
#pragma unroll
      for (int v = 0; v < 2; ++v)
#pragma unroll
        for (int t = 0; t < FT; ++t)
#pragma unroll
          for (int i = 0; i < RT; ++i) acc[t][i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wv[u + v][t], xv[u + v][i], acc[t][i], 0, 0, 0);
    }
  };
  const int pairs = k / 64, each = (pairs + WAVES - 1) / WAVES;
  int step = min(wave * each, pairs) * 2;
  const int last = min(wave * each + each, pairs) * 2;
  for (; step + U <= last; step += U) some(step, std::integral_constant<int, U>{});
  for (; step < last; step += 2) some(step, std::integral_constant<int, 2>{});
#pragma unroll
  for (int t = 0; t < FT; ++t)
#pragma unroll
    for (int i = 0; i < RT; ++i) meet[wave][t * RT + i][lane] = acc[t][i];
  __syncthreads();
  if (wave >= FT * RT) return;  // a wave adds up one tile
  f32x4_t sum = meet[0][wave][lane];
#pragma unroll
  for (int v = 1; v < WAVES; ++v) sum += meet[v][wave][lane];
  const int row = r0 + wave % RT * 16 + col, f = f0 + wave / RT * 16 + quad * 4;
  if (row >= m) return;
  bf16_t* o = out + (int64_t)row * ldc + f;
  if (vec && f + 4 <= n) {
    const float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    mi_store_cols<bf16_t, 4>(o, v);
  } else {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (f + c < n) o[c] = from_f32<bf16_t>(sum[c]);
  }
}

struct Launch {
  const void *a, *w;
  void* out;
  int64_t lda, ldw, ldc;
  bool vec;
  int m, n, k;
  hipStream_t stream;
};

template <int RT, int FT, int U>
void launch(const Launch& l) {
  static_assert(FT * RT <= WAVES, "a wave adds up a tile");
  const int row_tiles = ceil_div(l.m, RT * 16), total = row_tiles * ceil_div(l.n, FT * 16);
  const auto kernel = row_tiles == 1 ? gemm_rows_kernel<RT, FT, U, true> : gemm_rows_kernel<RT, FT, U, false>;
  kernel<<<ceil_div(total, 8) * 8, WAVES * MI_WAVE, 0, l.stream>>>((const bf16_t*)l.a, l.lda, (const bf16_t*)l.w, l.ldw, (bf16_t*)l.out, l.ldc, l.vec, l.m, l.n,
                                                                  l.k, row_tiles, total);
}

struct Form {
  int rows, features;
  void (*launch)(const Launch&);
};
const Form FORMS[] = {{16, 16, launch<1, 1, 8>}, {32, 16, launch<2, 1, 4>}, {32, 32, launch<2, 2, 4>}};
constexpr int FORM_COUNT = sizeof(FORMS) / sizeof(FORMS[0]);

}  // namespace

// The form in which a product is made, -1: it would have more blocks than compute units in each, and the microseconds expected: what a
// block brings in, and W from memory (a least-squares fit to 142 launches of 512 to 8,192 features, K 512 to 4,096, 17 to 256 rows; relative error 5 %).
extern "C" int mi_gemm_rows_plan(int m, int n, int k, int cus, int* form, float* micros) {
  MI_REQUIRE(m >= 1 && n >= 1 && k >= 1 && cus >= 1, "gemm_rows_plan: m=%d n=%d k=%d on %d compute units", m, n, k, cus);
  *form = -1, *micros = INFINITY;
  for (int i = 0; i < FORM_COUNT; ++i) {
    const Form& f = FORMS[i];
    if ((int64_t)ceil_div(m, f.rows) * ceil_div(n, f.features) > cus) continue;
    *form = i;
    *micros = (float)(ROWS_BASE + (double)(min(m, f.rows) + f.features) * k * 2 / ROWS_INTAKE + (double)n * k * 2 / ROWS_MEMORY);
    break;
  }
  return MI_OK;
}

// Whether the kernel takes these: rows of W in whole cache lines, all of W within 32-bit offsets.
extern "C" int mi_gemm_rows_take(const void* a, int64_t lda, const void* w, int64_t ldw, int m, int n, int k) {
  return m >= 1 && n >= 1 && k >= 64 && k % 64 == 0 && lda >= k && ldw >= k && lda % 8 == 0 && ldw % 64 == 0 && (uintptr_t)a % 16 == 0 &&
                 (uintptr_t)w % 128 == 0 && (int64_t)n * ldw * 2 < ((int64_t)1 << 32) && (int64_t)ceil_div(m, 16) * ceil_div(n, 16) < (1 << 30)
             ? 1
             : 0;
}

// Rows of a form (0: there is none of that number).
extern "C" int mi_gemm_rows_rows(int form) { return form >= 0 && form < FORM_COUNT ? FORMS[form].rows : 0; }

extern "C" int mi_gemm_rows_bf16(int form, const void* a, int64_t lda, const void* w, int64_t ldw, void* out, int64_t ldc, int m, int n, int k,
                                 hipStream_t stream) {
  MI_REQUIRE(form >= 0 && form < FORM_COUNT && ldc >= n && mi_gemm_rows_take(a, lda, w, ldw, m, n, k),
             "gemm_rows_bf16: form %d, m=%d n=%d k=%d lda=%lld ldw=%lld ldc=%lld; takes K a multiple of 64, rows of A on 16 bytes, of W on 128", form, m, n, k,
             (long long)lda, (long long)ldw, (long long)ldc);
  const bool vec = (uintptr_t)out % 8 == 0 && ldc % 4 == 0;
  FORMS[form].launch({a, w, out, lda, ldw, ldc, vec, m, n, k, stream});
  MI_CHECK_LAUNCH("gemm_rows_bf16");
  return MI_OK;
}
