// Routed experts for many rows (prompts): the two products of every chosen expert as one launch each over
// tiles of BM of the expert's (token, choice) pairs x BN of its output features on the matrix cores, with
// nothing the host has to know: the pairs are listed expert by expert on the device (`expert_sort`),
// and a block finds its tile in that list.
//
// The tiles are those of turns_product.h, 64, 128, 160 or 256 pairs x 256 weight rows, one block to a CU; all of them sum in the
// same order, so which one is taken does not show in the results.  What bounds such a launch is the weights' bytes up to some 150 pairs an
// expert, the matrix cores beyond some 300, and anywhere the last round of blocks, which may be nearly empty: 2,700 pairs over 16 experts are 16 to 50
// row tiles of 16 blocks, and an expert with 257 pairs more decides whether 256 CUs take one round or two.  So each expert's pairs are cut by
// themselves (expert_cuts.h), whoever makes the list leaves the four ways to do so beside it, every block works out which of them its launch takes
// (the host does not know how many pairs an expert got), and the largest tiles run first, so that the small ones fill the gaps.
// Microseconds, gate and up + down, weights from memory, the pairs as routers spread them (two of 18 experts are not among the 16): all experts'
// tiles alike, cut expert by expert:
//     experts x gate|up, down          pairs     an expert        alike       by expert
//     16 x 4096 x 3072, 3072 x 2048      700      25 to 88       81 +  51      71 +  47
//                                      1,760      69 to 178      94 +  60      82 +  50
//                                      2,670     101 to 284     146 +  59     108 +  58
//                                      5,330     230 to 448     171 + 105     167 +  96
//                                     10,700     334 to 1001    254 + 159     268 + 147
//     16 x 7168 x 4096, 4096 x 3584    2,220      80 to 193     218 + 114     189 +  95
//                                      3,560     122 to 407     290 + 168     250 + 141
//     64 x 2048 x 2048, 2048 x 1024    5,800      35 to 173     165 +  84     133 +  61
// A step of 1,501 tokens of 12 layers at the first sizes 6,055 -> 5,800 us.  (Tiles of 128 x 128 on two buffers, four waves in step, two blocks to a
// CU, came before both: 1.17 to 1.23 times the time of tiles that are all alike from 96 pairs an expert on.)
//
// Each of the 8 XCDs takes an eighth of the tiles of every form (workgroups are dealt to the XCDs in turn), side by side in the list: an
// expert's row tile by row tile, a row tile's feature tiles one after the other, so that its pairs' rows stay behind one L2.  (Tiles
// dealt to the XCDs one by one, which brings every expert's rows into every L2: 16 x 4096 x 3072 with 5,330 pairs 157 -> 181.)
//
// MODE as in routed_experts.hip: 0 plain, 1 silu(gate) * up (a block then makes BN / 2 features: gate and up rows
// side by side in its tile), 2 relu(weight * z)^2.
#include "expert_cuts.h"
#include "turns_product.h"

namespace {

constexpr int TILE_FEATURES = 256;
static_assert(cut_rows(0) == turns_form(0).rows && cut_rows(1) == turns_form(1).rows && cut_rows(2) == turns_form(2).rows && cut_rows(3) == turns_form(3).rows);

// Microseconds of a launch over n weight rows of k elements an expert: what the compute units multiply, the largest tiles first, and what they
// bring in, of which neither hides the other quite.  Fitted to 48 spreads of pairs over experts of five sizes, weights from memory
// (profiles/expert_tiles_cuts_times.txt): the cut with the least of these is 0.3 % slower than the best one on average, 8 % at worst.
__host__ __device__ inline float launch_micros(const CutSums& sums, int n, int k, int cus) {
  const int feature_tiles = (n + TILE_FEATURES - 1) / TILE_FEATURES;
  constexpr float STEP[CUT_FORMS] = {0.84f, 1.04f, 1.15f, 1.30f};  // of 64 of K, with the pairs' rows from L2 and the weights from memory
  float micros[CUT_FORMS], work = 0.f, rows = 0.f;
  int all = 0;
#pragma unroll
  for (int f = 0; f < CUT_FORMS; ++f) {
    micros[f] = (float)(k / TURNS_K) * STEP[f] + 5.9f;
    work += micros[f] * (float)sums.tiles[f];
    rows += (float)cut_rows(f) * (float)sums.tiles[f];
    all += sums.tiles[f];
  }
  auto at = [&](int place) {  // of the tile at a place in the launch's order
    float of = 0.f;
    int past = 0;
#pragma unroll
    for (int f = CUT_FORMS - 1; f >= 0; --f) {
      past += sums.tiles[f] * feature_tiles;
      if (of == 0.f && place < past) of = micros[f];
    }
    return of;
  };
  float made = work * (float)feature_tiles / (float)cus;
  const float first = at(0), next = at(cus), two = next > 0.f ? at(cus - 1) + next : 0.f, three = 3.f * at(2 * cus);
  made = first > made ? first : made;
  made = two > made ? two : made;
  made = three > made ? three : made;
  const float matrix = (float)n * (float)k * 2.f;
  const float brought = 1.40e-7f * (float)sums.used * matrix + 0.78e-7f * rows * (float)feature_tiles * (float)k * 2.f +
                        0.69e-7f * (float)(all - sums.used) * matrix + 1.11e-7f * (float)sums.again * matrix;
  const float a = made * made, b = brought * brought;
  return sqrtf(sqrtf(a * a + b * b));
}

__global__ __launch_bounds__(CUTS * MI_WAVE) void expert_plan_kernel(const int* __restrict__ first, int pairs, int experts, CutsPlan* __restrict__ plan) {
  plan_cut(first, pairs, experts, __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), plan);
}

// Which tile block `id` works on.  False: past the last one.  All threads of the block get the same answer.
__device__ __forceinline__ bool find_tile(const CutsPlan* __restrict__ plan, int pairs, int experts, int n, int k, int cus, int id, RowTile& place,
                                          int& feature_tile) {
  const int lane = threadIdx.x % MI_WAVE, feature_tiles = (n + TILE_FEATURES - 1) / TILE_FEATURES;
  const CutSums sums = plan->sums[min(lane, CUTS - 1)];  // a lane a cut
  const float micros = launch_micros(sums, n, k, cus);
  int cut = 0;
  float least = 0.f;
#pragma unroll
  for (int c = CUTS - 1; c >= 0; --c) {
    const float its = __uint_as_float(__builtin_amdgcn_readlane(__float_as_uint(micros), c));
    if (c == CUTS - 1 || its < least) cut = c, least = its;
  }
  // each XCD has an eighth of the tiles of every form, the largest first, side by side in the list; what is left over of one form goes to
  // the XCDs behind those that got what was left over of the form before
  int slot = id / 8, row_tile = 0, given = 0, at = -1;
#pragma unroll
  for (int f = CUT_FORMS - 1; f >= 0; --f) {
    const int row_tiles = __builtin_amdgcn_readlane(sums.tiles[f], cut), tiles = row_tiles * feature_tiles, turn = (id - given) & 7;
    const int mine = tiles / 8 + (turn < tiles % 8);
    if (at < 0) {
      if (slot < mine) at = turn * (tiles / 8) + min(turn, tiles % 8) + slot;
      else slot -= mine, row_tile += row_tiles;
    }
    given += tiles;
  }
  if (at < 0) return false;
  row_tile += at / feature_tiles;
  feature_tile = at % feature_tiles;
  const RowTile* list = row_tiles_of(plan, cut, pairs, experts) + row_tile;
  place.expert = __builtin_amdgcn_readfirstlane(list->expert);
  place.row0 = __builtin_amdgcn_readfirstlane(list->row0);
  place.end = __builtin_amdgcn_readfirstlane(list->end);
  place.form = __builtin_amdgcn_readfirstlane(list->form);
  return true;
}

template <class T, int MODE, bool ONCE>
__device__ __forceinline__ void make_tile(
    bf16_t* ring, const bf16_t* __restrict__ src, int64_t src_stride, int src_div, const bf16_t* __restrict__ weight,
    int64_t expert_stride, const int* __restrict__ listed,
    const float* __restrict__ pair_weight, bf16_t* __restrict__ out, int64_t out_stride, int k_dim, int features, const RowTile& place, int feature_tile) {
  constexpr bool GATED = MODE == 1;
  constexpr int FEATURES = GATED ? T::BN / 2 : T::BN;
  static_assert(T::BN == TILE_FEATURES);
  const int expert = place.expert, row0 = place.row0, end = place.end, f0 = feature_tile * FEATURES;
  const bf16_t* w = weight + (int64_t)expert * expert_stride;
  T tile;
  tile.template run<ONCE>(
      ring, k_dim / TURNS_K,
      [&](int r) {  // (past the tile's last pair: that one again, not written)
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

// ONCE: weights are read past the caches, which pays where few experts have a second row tile.  The host knows only how many pairs an expert gets on
// average, and takes it up to 256; the cut, and with it who has one, is chosen later.  Microseconds through the caches / past them, gate and up:
//     one tile an expert     16 x 4096 x 3072  40 an expert 79.8 / 71.0    130  91.6 / 84.1    230 (all alike) 102 / 92     64 x 2048 x 2048  150  168 / 159
//     two for each           16 x 2048 x 2048  256 (all alike) 45.7 / 43.8
//     for some               16 x 4096 x 3072  256 146 / 142    230 133 / 134      16 x 2048 x 2048  230  48.6 / 52.4
//     beyond                 16 x 2048 x 2048  400 62.8 / 75.1    16 x 4096 x 3072  340 159 / 160     64 x 2048 x 2048  340  234 / 239
// (the second tile of an expert runs at the same time as the first and often finds its weights on the way all the same; over 108 launches of up to 256
// pairs an expert 0.93 to 1.24, one of 16 x 3072 x 2048 0.83, as a geometric mean 1.06; over 28 beyond 0.99).
template <int MODE, bool ONCE>
__global__ __launch_bounds__(512, 2) void expert_tiles_kernel(
    const bf16_t* __restrict__ src, int64_t src_stride, int src_div, const bf16_t* __restrict__ weight,
    int64_t expert_stride, const int* __restrict__ listed, const CutsPlan* __restrict__ plan,
    const float* __restrict__ pair_weight, bf16_t* __restrict__ out, int64_t out_stride, int pairs, int experts, int k_dim,
    int features, int cus) {
  __shared__ __align__(16) bf16_t ring[TURNS_RING];
  RowTile place;
  int feature_tile;
  if (!find_tile(plan, pairs, experts, MODE == 1 ? 2 * features : features, k_dim, cus, blockIdx.x, place, feature_tile)) return;
#define MI_TILE(...) \
  make_tile<__VA_ARGS__, MODE, ONCE>(ring, src, src_stride, src_div, weight, expert_stride, listed, pair_weight, out, out_stride, k_dim, features, place, feature_tile)
  if (place.form == 0) MI_TILE(TurnsOf<0>::type);
  else if (place.form == 1) MI_TILE(TurnsOf<1>::type);
  else if (place.form == 2) MI_TILE(TurnsOf<2>::type);
  else MI_TILE(TurnsOf<3>::type);
#undef MI_TILE
}

template <int MODE>
void launch_tiles(const void* src, int64_t src_stride, int src_div, const void* weight, const int* listed, const void* plan,
                  const float* pair_weight, void* out, int64_t out_stride, int pairs, int experts, int k_dim, int features, int cus,
                  hipStream_t stream) {
  const int feature_tiles = ceil_div(features, MODE == 1 ? TILE_FEATURES / 2 : TILE_FEATURES);
  const int most = feature_tiles * most_row_tiles(pairs, experts, 0);
  const auto kernel = pairs <= (int64_t)cut_rows(CUT_FORMS - 1) * experts ? expert_tiles_kernel<MODE, true> : expert_tiles_kernel<MODE, false>;
  kernel<<<ceil_div(most, 8) * 8, 512, 0, stream>>>((const bf16_t*)src, src_stride, src_div, (const bf16_t*)weight,
                                                    (int64_t)(MODE == 1 ? 2 : 1) * features * k_dim, listed, (const CutsPlan*)plan, pair_weight,
                                                    (bf16_t*)out, out_stride, pairs, experts, k_dim, features, cus);
}

}  // namespace

// Whether rows of k_dim bfloat16 elements are taken.
extern "C" int mi_expert_tiles_take(int k_dim) { return k_dim > 0 && k_dim % TURNS_K == 0; }

// How a launch of n weight rows an expert cuts experts with counts[0..experts) pairs: for each expert four numbers: full
// tiles of the largest form, tiles behind them, the pairs in each of these and the rows of their form.
extern "C" int mi_expert_tiles_cut(const int* counts, int experts, int n, int k_dim, int cus, int* cuts) {
  MI_REQUIRE(counts && cuts && experts > 0 && n > 0 && mi_expert_tiles_take(k_dim), "expert_tiles_cut: experts=%d n=%d k=%d", experts, n, k_dim);
  int best = -1;
  float least = 0.f;
  for (int c = CUTS - 1; c >= 0; --c) {
    CutSums sums = {};
    for (int e = 0; e < experts; ++e) add(sums, cover(counts[e], c));
    const float micros = launch_micros(sums, n, k_dim, max(8, cus));
    if (best < 0 || micros < least) best = c, least = micros;
  }
  for (int e = 0; e < experts; ++e) {
    const Cover c = cover(counts[e], best);
    cuts[4 * e] = c.full, cuts[4 * e + 1] = c.tiles, cuts[4 * e + 2] = c.each, cuts[4 * e + 3] = cut_rows(c.form);
  }
  return MI_OK;
}

// 32-bit words of the plan that mi_expert_plan leaves for mi_expert_tiles, on 16 bytes.
extern "C" int64_t mi_expert_plan_words(int pairs, int experts) {
  if (pairs < 0 || experts < 1) return 0;
  return (int64_t)(sizeof(CutsPlan) + row_tiles_before(CUTS, pairs, experts) * sizeof(RowTile)) / 4;
}

// (mi_expert_sort leaves the same where it is asked to)
extern "C" int mi_expert_plan(const int* first, int pairs, int experts, void* plan, hipStream_t stream) {
  MI_REQUIRE(pairs >= 0 && experts > 0 && first && plan && (uintptr_t)plan % 16 == 0, "expert_plan: pairs=%d experts=%d", pairs, experts);
  if (pairs == 0) return MI_OK;
  expert_plan_kernel<<<1, CUTS * MI_WAVE, 0, stream>>>(first, pairs, experts, (CutsPlan*)plan);
  MI_CHECK_LAUNCH("expert_plan");
  return MI_OK;
}

// Arguments as mi_expert_rows (bfloat16 only), with the number of pairs handed to the list, and the plan of mi_expert_plan for the list in place
// of `first`.
extern "C" int mi_expert_tiles(int mode, const void* src, int64_t src_stride, int src_div, const void* weight,
                               const int* listed, const void* plan, const float* pair_weight, void* out,
                               int64_t out_stride, int pairs, int experts, int k_dim, int features, hipStream_t stream) {
  MI_REQUIRE(pairs >= 0 && experts > 0 && features > 0 && src_div > 0 && src_stride >= k_dim && out_stride >= features,
             "expert_tiles: bad sizes pairs=%d experts=%d k=%d features=%d", pairs, experts, k_dim, features);
  MI_REQUIRE(mi_expert_tiles_take(k_dim) && src_stride % 8 == 0 && ((uintptr_t)src | (uintptr_t)weight) % 16 == 0 && (uintptr_t)out % 8 == 0,
             "expert_tiles: rows of %d elements are not taken %d at a time", k_dim, TURNS_K);
  MI_REQUIRE(mode >= 0 && mode <= 2 && (uintptr_t)plan % 16 == 0, "expert_tiles: mode %d", mode);
  MI_REQUIRE((int64_t)ceil_div(features, 128) * ((int64_t)pairs / 64 + experts) < (1 << 30), "expert_tiles: too many tiles");
  if (pairs == 0) return MI_OK;
  const int cus = max(8, mi_compute_units());
#define MI_TILES(MODE) \
  launch_tiles<MODE>(src, src_stride, src_div, weight, listed, plan, pair_weight, out, out_stride, pairs, experts, k_dim, features, cus, stream)
  if (mode == 1) MI_TILES(1);
  else if (mode == 2) MI_TILES(2);
  else MI_TILES(0);
#undef MI_TILES
  MI_CHECK_LAUNCH("expert_tiles");
  return MI_OK;
}
