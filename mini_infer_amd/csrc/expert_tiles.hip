// Routed experts for many rows (prompts): the two products of every chosen expert as one launch each over
// tiles of BM of the expert's (token, choice) pairs x BN of its output features on the matrix cores, with
// nothing the host has to know: the pairs are listed expert by expert on the device (`expert_sort`),
// and a block finds its tile in that list.
//
// The tiles are those of turns_product.h, 64, 128, 160 or 256 pairs x 256 weight rows, one block to a CU; all of them sum in the
// same order, so which one is taken does not show in the results.  What bounds such a launch is the matrix cores, and the
// last round of blocks, which may be nearly empty: 2,700 pairs over 16 experts are 22 to 50 row tiles, and a row tile more or less
// decides whether it takes one round or two.  The host does not know how many pairs an expert got, so every block works out
// from the list, before it looks for its tile, how long the launch takes in either size and takes the shortest: all
// blocks see the same list and take the same.  Measured (microseconds, the pairs as routers spread them, 58 to 333 an expert;
// before: tiles of 128 x 128 on two buffers, four waves in step, two blocks to a CU):
//     experts x gate|up, down            pairs    before        now
//     16 x 4096 x 3072, 3072 x 2048      1,942    133 +  40     102 +  42
//                                        3,238    161 +  70     126 +  52
//                                        4,122    173 +  70     123 +  56
//     16 x 7168 x 4096, 4096 x 3584      2,612    261 + 153     210 + 124
//                                        5,776    430 + 245     308 + 176
// and over 120 such pairs of launches 1.17 times as fast from 96 to 200 pairs an expert, 1.23 beyond, and below, where the weights' bytes
// bound both, 1.03 to 1.04 (a single launch at worst 0.93, both together 0.97).  A step of 1,501 tokens of 12 layers at the
// first sizes 6,708 -> 6,429 us.
//
// Tiles are numbered expert by expert, within an expert feature tile by feature tile with the row tiles of one
// feature tile side by side; each of the 8 XCDs takes one stretch of these numbers (workgroups are dealt
// to the XCDs in turn), so the row tiles that read the same weights run at the same time behind one
// L2, and an expert's rows stay in it.
//
// MODE as in routed_experts.hip: 0 plain, 1 silu(gate) * up (a block then makes BN / 2 features: gate and up rows
// side by side in its tile), 2 relu(weight * z)^2.
#include "turns_product.h"

namespace {

// The same on the device, from the list.  All threads of the block get the same answer.
__device__ __forceinline__ int pick_form(const int* __restrict__ first, int experts, bool smallest, int n, int k, int cus) {
  int row_tiles[TURNS_WIDE] = {}, used = 0;
  for (int e = threadIdx.x % MI_WAVE; e < experts; e += MI_WAVE) {
    const int pairs = first[e + 1] - first[e];
    used += pairs > 0;
#pragma unroll
    for (int f = 0; f < TURNS_WIDE; ++f) row_tiles[f] += (pairs + turns_form(f).rows - 1) / turns_form(f).rows;
  }
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) {
    used += __shfl_xor(used, off, MI_WAVE);
#pragma unroll
    for (int f = 0; f < TURNS_WIDE; ++f) row_tiles[f] += __shfl_xor(row_tiles[f], off, MI_WAVE);
  }
  if (!smallest) row_tiles[0] = 0;
  return __builtin_amdgcn_readfirstlane(turns_pick(row_tiles, used, n, k, cus));
}

// Which tile this block works on: expert, first pair of the row tile (an index into `listed`), feature tile.
// False: past the last tile.  All threads of the block get the same answer.
__device__ __forceinline__ bool find_tile(const int* __restrict__ first, int experts, int feature_tiles, int bm, int id,
                                          int& expert, int& row0, int& feature_tile) {
  const int lane = threadIdx.x % MI_WAVE;
  // row tiles in all
  int total = 0;
  for (int base = 0; base < experts; base += MI_WAVE) {
    const int e = base + lane;
    int tiles = e < experts ? (first[e + 1] - first[e] + bm - 1) / bm : 0;
#pragma unroll
    for (int off = MI_WAVE / 2; off > 0; off >>= 1) tiles += __shfl_xor(tiles, off, MI_WAVE);
    total += tiles;
  }
  total *= feature_tiles;
  const int per = (total + 7) / 8;
  const int place = (id % 8) * per + id / 8;
  if (id / 8 >= per || place >= total) return false;
  int before = 0;
  for (int base = 0; base < experts; base += MI_WAVE) {
    const int e = base + lane;
    const int tiles = e < experts ? (first[e + 1] - first[e] + bm - 1) / bm : 0;
    int upto = tiles;  // row tiles of the experts up to and including this lane's
#pragma unroll
    for (int off = 1; off < MI_WAVE; off <<= 1) {
      const int other = __shfl_up(upto, off, MI_WAVE);
      if (lane >= off) upto += other;
    }
    const uint64_t past = __ballot((before + upto) * feature_tiles > place);
    if (past != 0) {
      const int at = __builtin_ctzll(past);
      const int mine = __shfl(tiles, at, MI_WAVE), start = before + __shfl(upto, at, MI_WAVE) - mine;
      const int rest = place - start * feature_tiles;
      expert = base + at;
      row0 = first[expert] + (rest % mine) * bm;
      feature_tile = rest / mine;
      return true;
    }
    before += __shfl(upto, MI_WAVE - 1, MI_WAVE);
  }
  return false;
}

template <class T, int MODE>
__device__ __forceinline__ void make_tile(
    bf16_t* ring, const bf16_t* __restrict__ src, int64_t src_stride, int src_div, const bf16_t* __restrict__ weight,
    int64_t expert_stride, const int* __restrict__ listed, const int* __restrict__ first,
    const float* __restrict__ pair_weight, bf16_t* __restrict__ out, int64_t out_stride, int experts, int k_dim, int features) {
  constexpr bool GATED = MODE == 1;
  constexpr int FEATURES = GATED ? T::BN / 2 : T::BN;
  static_assert(T::BN == TURNS_FEATURES);
  const int feature_tiles = (features + FEATURES - 1) / FEATURES;
  int expert, row0, feature_tile;
  if (!find_tile(first, experts, feature_tiles, T::BM, blockIdx.x, expert, row0, feature_tile)) return;
  const int end = first[expert + 1], f0 = feature_tile * FEATURES;
  const bf16_t* w = weight + (int64_t)expert * expert_stride;
  T tile;
  tile.run(
      ring, k_dim / TURNS_K,
      [&](int r) {  // (past the expert's last pair: that one again, not written)
        return src + (int64_t)(listed[min(row0 + r, end - 1)] / src_div) * src_stride;
      },
      [&](int r) { return w + (int64_t)(GATED ? T::Pairs::row_of(r, f0, features) : min(f0 + r, features - 1)) * k_dim; });
  tile.leave(ring, [&](float sum, int r) {
    if (MODE != 2) return sum;
    const float z = fmaxf((pair_weight != nullptr ? pair_weight[listed[min(row0 + r, end - 1)]] : 1.f) * sum, 0.f);
    return z * z;
  });
  constexpr int CHUNKS = FEATURES / 8;
  const bool whole = (uintptr_t)out % 16 == 0 && out_stride % 8 == 0;
  for (int i = threadIdx.x; i < T::BM * CHUNKS; i += T::THREADS) {
    const int row = i / CHUNKS, f = i % CHUNKS * 8;
    if (row0 + row >= end || f0 + f >= features) continue;
    const bf16_t* at = ring + row * T::MADE + (GATED ? T::Pairs::at(f) : f);
    float v[8];
    mi_load_8(at, v);
    if constexpr (GATED) {  // the two products as the element type holds them, then silu(gate) * up
      float u[8];
      mi_load_8(at + T::Pairs::PAIR, u);
#pragma unroll
      for (int c = 0; c < 8; ++c) v[c] = silu_times<bf16_t>(v[c], u[c]);
    }
    mi_store_8(out + (int64_t)listed[row0 + row] * out_stride, f0 + f, features, whole, v);
  }
}

template <int MODE>
__global__ __launch_bounds__(512, 2) void expert_tiles_kernel(
    const bf16_t* __restrict__ src, int64_t src_stride, int src_div, const bf16_t* __restrict__ weight,
    int64_t expert_stride, const int* __restrict__ listed, const int* __restrict__ first,
    const float* __restrict__ pair_weight, bf16_t* __restrict__ out, int64_t out_stride, int experts, int k_dim,
    int features, bool smallest, int cus) {
  __shared__ __align__(16) bf16_t ring[TURNS_RING];
  const int form = pick_form(first, experts, smallest, MODE == 1 ? 2 * features : features, k_dim, cus);
#define MI_TILE(...) make_tile<__VA_ARGS__, MODE>(ring, src, src_stride, src_div, weight, expert_stride, listed, first, pair_weight, out, out_stride, experts, k_dim, features)
  if (form == 0) MI_TILE(TurnsOf<0>::type);
  else if (form == 1) MI_TILE(TurnsOf<1>::type);
  else if (form == 2) MI_TILE(TurnsOf<2>::type);
  else if (form == 3) MI_TILE(TurnsOf<3>::type);
#undef MI_TILE
}

// Pairs an expert has on average up to which tiles of 64 may be taken (they were the best of the four up to 71): a launch has a block for
// every tile that there can be of the smallest size, and the rest end when they have read the list.
constexpr int SMALLEST_UP_TO = 96;

template <int MODE>
void launch_tiles(const void* src, int64_t src_stride, int src_div, const void* weight, const int* listed, const int* first,
                  const float* pair_weight, void* out, int64_t out_stride, int pairs, int experts, int k_dim, int features, int cus,
                  hipStream_t stream) {
  const int feature_tiles = ceil_div(features, MODE == 1 ? TURNS_FEATURES / 2 : TURNS_FEATURES);
  const bool smallest = pairs <= (int64_t)SMALLEST_UP_TO * experts;
  const int most = feature_tiles * (pairs / turns_form(smallest ? 0 : 1).rows + min(experts, pairs));  // (an expert's last tile may be a short one)
  expert_tiles_kernel<MODE><<<ceil_div(most, 8) * 8, 512, 0, stream>>>(
      (const bf16_t*)src, src_stride, src_div, (const bf16_t*)weight, (int64_t)(MODE == 1 ? 2 : 1) * features * k_dim, listed,
      first, pair_weight, (bf16_t*)out, out_stride, experts, k_dim, features, smallest, cus);
}

}  // namespace

// Whether rows of k_dim bfloat16 elements are taken.
extern "C" int mi_expert_tiles_take(int k_dim) { return k_dim > 0 && k_dim % TURNS_K == 0; }

// Rows of the tile that a launch of n weight rows an expert takes where the experts got counts[0..experts) pairs (0: no pairs).
extern "C" int mi_expert_tiles_rows(const int* counts, int experts, int n, int k_dim, int cus) {
  int row_tiles[TURNS_WIDE] = {}, used = 0;
  int64_t pairs = 0;
  for (int e = 0; e < experts; ++e) {
    pairs += counts[e], used += counts[e] > 0;
    for (int f = 0; f < TURNS_WIDE; ++f) row_tiles[f] += ceil_div(counts[e], turns_form(f).rows);
  }
  if (pairs > (int64_t)SMALLEST_UP_TO * experts) row_tiles[0] = 0;
  const int form = turns_pick(row_tiles, used, n, k_dim, max(8, cus));
  return form < 0 ? 0 : turns_form(form).rows;
}

// Arguments as mi_expert_rows (bfloat16 only), with the number of listed pairs.
extern "C" int mi_expert_tiles(int mode, const void* src, int64_t src_stride, int src_div, const void* weight,
                               const int* listed, const int* first, const float* pair_weight, void* out,
                               int64_t out_stride, int pairs, int experts, int k_dim, int features, hipStream_t stream) {
  MI_REQUIRE(pairs >= 0 && experts > 0 && features > 0 && src_div > 0 && src_stride >= k_dim && out_stride >= features,
             "expert_tiles: bad sizes pairs=%d experts=%d k=%d features=%d", pairs, experts, k_dim, features);
  MI_REQUIRE(mi_expert_tiles_take(k_dim) && src_stride % 8 == 0 && ((uintptr_t)src | (uintptr_t)weight) % 16 == 0 && (uintptr_t)out % 8 == 0,
             "expert_tiles: rows of %d elements are not taken %d at a time", k_dim, TURNS_K);
  MI_REQUIRE(mode >= 0 && mode <= 2, "expert_tiles: mode %d", mode);
  MI_REQUIRE((int64_t)ceil_div(features, 128) * ((int64_t)pairs / 64 + experts) < (1 << 30), "expert_tiles: too many tiles");
  if (pairs == 0) return MI_OK;
  const int cus = max(8, mi_compute_units());
#define MI_TILES(MODE) \
  launch_tiles<MODE>(src, src_stride, src_div, weight, listed, first, pair_weight, out, out_stride, pairs, experts, k_dim, features, cus, stream)
  if (mode == 1) MI_TILES(1);
  else if (mode == 2) MI_TILES(2);
  else MI_TILES(0);
#undef MI_TILES
  MI_CHECK_LAUNCH("expert_tiles");
  return MI_OK;
}
