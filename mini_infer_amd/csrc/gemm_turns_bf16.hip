// Products of many rows (prompts): C = A * W^T in bfloat16, or with W = [gate; up] act(A * gate^T, A * up^T), as ONE launch of tiles whose waves
// take turns (turns_product.h), the activation in the last step.
//
// What bounds such a launch is the matrix cores, or, where it runs long enough, the card's power, which lowers the clock for the vendor
// library's kernels and for these alike; and the last round of blocks.  The tile is the one whose rounds are expected to be the shortest, and where
// whole tiles would leave the last round partly empty, its tiles are cut into tiles of fewer rows: 2048 x 28672 x 4096 is three and
// a half rounds of 256 x 256, and the half is a round of 128 x 256 (gated 369 us in four rounds, 346 so); 1777 rows three rounds and 16
// tiles, cut into 64 rows (350, 327).  Results leave through LDS: in whole 16 bytes, and with little code (turns_product.h).
//
// Measured against the library, with the activation's launch where gated: `turns_pay` and `plain_turns_pay` (ops/kernels.py).  Steps without these tiles and
// with them, one machine in turn: 2,048 tokens at 8B sizes (Llama) 26,822 -> 25,461 us, of 12 layers with clamped feed-forwards 12,052 -> 11,266,
// 1,777 tokens of 12 layers at 3B widths with four streams 8,692 -> 8,252, 1,501 with routed experts 6,231 -> 5,900.
//
// This stands where the reference's engine calls the vendor BLAS (distributed/linear.py:167) and where its SiLU * up kernel stands
// (models/blocks/silu_mul_kernel.py:86-90).
#include "turns_product.h"

namespace {

// Which tiles a launch is made of: each of the 8 XCDs takes `places` tiles of form `form`, the first `whole` of them as they are, which fill
// its compute units in whole rounds, the rest, which would leave some of them idle, cut into `cut` tiles of fewer rows (form `rest`).
struct TurnsPlan {
  int form, rest, cut, whole, places;
};

constexpr int ACT_ROTARY = 4;  // not an activation: [q | k | v] rotated and written (gated_tile.h)
template <int ACT>
struct TurnsHow {
  using type = GatedActivation;
};
template <>
struct TurnsHow<4> {
  using type = RotaryWrite;
};

template <class T, int ACT>
__device__ __forceinline__ void make_tile(bf16_t* ring, const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int64_t ldw,
                                          bf16_t* __restrict__ out, int64_t ldo, const typename TurnsHow<ACT>::type& how, bool vec, int m, int n, int k, int r0,
                                          int feature_tile) {
  constexpr bool GATED = ACT != ACT_NONE;
  constexpr int FEATURES = GATED ? T::BN / 2 : T::BN;
  if (r0 >= m) return;
  const int f0 = feature_tile * FEATURES;
  T tile;
  tile.run(
      ring, k / TURNS_K, [&](int r) { return a + (int64_t)min(r0 + r, m - 1) * lda; },
      [&](int r) {
        if constexpr (ACT == ACT_ROTARY) return w + (int64_t)rotary_row_of(HalvedTile<T::BN>::row_of(r, f0, n), n, how.head_dim) * ldw;
        else return w + (int64_t)(GATED ? T::Pairs::row_of(r, f0, n) : min(f0 + r, n - 1)) * ldw;
      });
  tile.leave(ring, [](float sum, int) { return sum; });
  if constexpr (ACT == ACT_ROTARY) {
    write_rotated<HalvedTile<T::BN>, T::BM, T::BN, T::MADE, T::THREADS>(ring, how, r0, m, f0, n);
  } else if constexpr (GATED) {
    write_activated<ACT, typename T::Pairs, T::BM, T::BN, T::MADE, T::THREADS>(ring, how, out, ldo, vec, r0, m, f0, n);
  } else {
    constexpr int CHUNKS = FEATURES / 8;
    for (int i = threadIdx.x; i < T::BM * CHUNKS; i += T::THREADS) {
      const int row = i / CHUNKS, f = i % CHUNKS * 8;
      if (r0 + row >= m || f0 + f >= n) continue;
      float v[8];
      mi_load_8(ring + row * T::MADE + f, v);
      mi_store_8(out + (int64_t)(r0 + row) * ldo, f0 + f, n, vec, v);
    }
  }
}

template <int ACT>
__global__ __launch_bounds__(512, 2) void gemm_turns_kernel(const bf16_t* __restrict__ a, int64_t lda, const bf16_t* __restrict__ w, int64_t ldw,
                                                            bf16_t* __restrict__ out, int64_t ldo, const typename TurnsHow<ACT>::type how, bool vec, int m, int n, int k,
                                                            int row_tiles, int feature_tiles, const TurnsPlan plan) {
  __shared__ __align__(16) bf16_t ring[TURNS_RING];
  // (workgroups are dealt to the XCDs in turn)
  const int xcd = blockIdx.x % 8, at = blockIdx.x / 8;
  const bool cut = at >= plan.whole;
  const int behind = at - plan.whole;
  const int place = xcd * plan.places + (cut ? plan.whole + behind / plan.cut : at);
  if (place >= min((xcd + 1) * plan.places, row_tiles * feature_tiles)) return;
  // An XCD's stretch of places: up to BAND row tiles side by side, then the next feature tile, so that what runs at the same time behind one L2 shares
  // both operands.
  constexpr int BAND = 8;
  const int band = place / (BAND * feature_tiles), in_band = min(BAND, row_tiles - band * BAND), rest = place - band * BAND * feature_tiles;
  const int form = cut ? plan.rest : plan.form;
  const int r0 = (band * BAND + rest % in_band) * turns_form(plan.form).rows + (cut ? behind % plan.cut * turns_form(plan.rest).rows : 0);
#define X(I, ROWS, FEATURES, CAN_GATE, ...)                                                                                        \
  if constexpr (ACT == ACT_NONE || ACT == ACT_ROTARY || CAN_GATE) {                                                                             \
    if (form == I) make_tile<TurnsOf<I>::type, ACT>(ring, a, lda, w, ldw, out, ldo, how, vec, m, n, k, r0, rest / in_band);         \
  }
  TURNS_FORMS_OF(X)
#undef X
}

// The plan that is expected to be the shortest, and the microseconds it is expected to take beside what any launch does (n: rows of W).
TurnsPlan turns_plan(int m, int n, int k, bool gated, int only, int cus, double* micros) {
  const int each = max(1, cus / 8);
  TurnsPlan best = {};
  *micros = 0.0;
  for (int f = TURNS_FORMS - 1; f >= 0; --f) {
    const TurnsForm form = turns_form(f);
    if (only >= 0 ? f != only : gated && !form.gated) continue;
    const int feature_tiles = ceil_div(n, gated ? form.features / 2 : form.features);
    const int64_t total = (int64_t)ceil_div(m, form.rows) * feature_tiles;
    const int places = (int)ceil_div64(total, 8), whole = places / each * each;
    for (int rest = f; rest >= 0; --rest) {
      if (turns_form(rest).features != form.features || form.rows % turns_form(rest).rows != 0 || (only >= 0 && rest != f)) continue;
      const int cut = form.rows / turns_form(rest).rows;
      const double multiplied = turns_rounds_micros(f, whole, each, k) + turns_rounds_micros(rest, (places - whole) * cut, each, k);
      const double brought = turns_bytes_micros(f, total + (int64_t)(places - whole) * 8 * (cut - 1), gated ? 2 * n : n, k);
      const double t = multiplied > brought ? multiplied : brought;
      if (*micros == 0.0 || t < *micros) *micros = t, best = {f, rest, cut, whole, places};
    }
  }
  return best;
}

}  // namespace

// The plan of a product of n features, {rows and rows of W of its tiles, rows of those that the rest is cut into, whole, places}, and the
// microseconds that it is expected to take.
extern "C" int mi_gemm_turns_plan(int m, int n, int k, int gated, int cus, int* plan, float* micros) {
  MI_REQUIRE(m >= 1 && n >= 1 && k >= 1 && cus >= 1, "gemm_turns_plan: m=%d n=%d k=%d on %d compute units", m, n, k, cus);
  double t;
  const TurnsPlan p = turns_plan(m, n, k, gated != 0, -1, max(8, cus), &t);
  plan[0] = turns_form(p.form).rows, plan[1] = turns_form(p.form).features, plan[2] = turns_form(p.rest).rows, plan[3] = p.whole, plan[4] = p.places;
  *micros = (float)t;
  return MI_OK;
}

// Rows and rows of W of a form, and whether its tiles hold gate and up rows (0 rows: there is none of that number).
extern "C" int mi_gemm_turns_rows(int form) { return form >= 0 && form < TURNS_FORMS ? turns_form(form).rows : 0; }
extern "C" int mi_gemm_turns_features(int form) { return form >= 0 && form < TURNS_FORMS ? turns_form(form).features : 0; }
extern "C" int mi_gemm_turns_gated(int form) { return form >= 0 && form < TURNS_FORMS && turns_form(form).gated ? 1 : 0; }

// only: a form to make all tiles of, or -1.
extern "C" int mi_gemm_turns_bf16(int act, const void* a, int64_t lda, const void* w, int64_t ldw, const float* bias, float limit, float slope,
                                  void* out, int64_t ldo, int m, int n, int k, int only, hipStream_t stream) {
  MI_REQUIRE(m >= 1 && n >= 1 && k >= TURNS_K && k % TURNS_K == 0 && lda >= k && ldw >= k && lda % 8 == 0 && ldw % 8 == 0 && ldo >= n &&
                 ((uintptr_t)a | (uintptr_t)w) % 16 == 0,
             "gemm_turns_bf16: takes K a multiple of 64 and rows on 16 bytes; got m=%d n=%d k=%d lda=%lld ldw=%lld", m, n, k, (long long)lda, (long long)ldw);
  MI_REQUIRE(act >= 0 && act <= 3 && (act != ACT_CLAMPED || limit > 0.f), "gemm_turns_bf16: activation %d, limit %g", act, (double)limit);
  MI_REQUIRE((int64_t)ceil_div(m, 64) * ceil_div(n, 64) < (1 << 27), "gemm_turns_bf16: too many tiles");
  const bool vec = (uintptr_t)out % 16 == 0 && ldo % 8 == 0;
  const GatedActivation how = {bias, limit, slope};
  MI_REQUIRE(only >= -1 && only < TURNS_FORMS && (only < 0 || act == ACT_NONE || turns_form(only).gated), "gemm_turns_bf16: form %d", only);
  double micros;
  const TurnsPlan plan = turns_plan(m, n, k, act != ACT_NONE, only, max(8, mi_compute_units()), &micros);
  const TurnsForm form = turns_form(plan.form);
  const int row_tiles = ceil_div(m, form.rows), feature_tiles = ceil_div(n, act == ACT_NONE ? form.features : form.features / 2);
  const int blocks = 8 * (plan.whole + (plan.places - plan.whole) * plan.cut);
#define MI_LAUNCH(ACT) \
  gemm_turns_kernel<ACT><<<blocks, 512, 0, stream>>>((const bf16_t*)a, lda, (const bf16_t*)w, ldw, (bf16_t*)out, ldo, how, vec, m, n, k, row_tiles, feature_tiles, plan)
  if (act == ACT_NONE) MI_LAUNCH(ACT_NONE);
  else if (act == ACT_SILU) MI_LAUNCH(ACT_SILU);
  else if (act == ACT_CLAMPED) MI_LAUNCH(ACT_CLAMPED);
  else MI_LAUNCH(ACT_GELU);
#undef MI_LAUNCH
  MI_CHECK_LAUNCH("gemm_turns_bf16");
  return MI_OK;
}

// [q | k | v] rotated and written where it belongs in the last step; only: as above.
extern "C" int mi_gemm_turns_rope(const void* a, int64_t lda, const void* w, int64_t ldw, void* q, int64_t ldq, const float* cos_t, const float* sin_t,
                                  const int* slots, void* k_pages, void* v_pages, int m, int k, int q_heads, int kv_heads, int head_dim, int page_size,
                                  int num_pages, int v_transposed, int only, hipStream_t stream) {
  const RotaryWrite how = {cos_t, sin_t, slots, (bf16_t*)q, (bf16_t*)k_pages, (bf16_t*)v_pages, ldq, q_heads, kv_heads, head_dim, page_size, v_transposed};
  MI_REQUIRE(rotary_write_fits(how, m, num_pages), "gemm_turns_rope: m=%d, %d + 2 * %d heads of %d, pages of %d", m, q_heads, kv_heads, head_dim, page_size);
  MI_REQUIRE(k >= TURNS_K && k % TURNS_K == 0 && lda >= k && ldw >= k && lda % 8 == 0 && ldw % 8 == 0 && ((uintptr_t)a | (uintptr_t)w) % 16 == 0,
             "gemm_turns_rope: takes K a multiple of 64 and rows on 16 bytes; got k=%d lda=%lld ldw=%lld", k, (long long)lda, (long long)ldw);
  const int pairs = (q_heads + 2 * kv_heads) * (head_dim / 2);
  MI_REQUIRE((int64_t)ceil_div(m, 64) * ceil_div(pairs, 64) < (1 << 27), "gemm_turns_rope: too many tiles");
  MI_REQUIRE(only >= -1 && only < TURNS_FORMS, "gemm_turns_rope: form %d", only);
  double micros;
  const TurnsPlan plan = turns_plan(m, 2 * pairs, k, false, only, max(8, mi_compute_units()), &micros);
  const TurnsForm form = turns_form(plan.form);
  const int blocks = 8 * (plan.whole + (plan.places - plan.whole) * plan.cut);
  gemm_turns_kernel<ACT_ROTARY><<<blocks, 512, 0, stream>>>((const bf16_t*)a, lda, (const bf16_t*)w, ldw, nullptr, 0, how, true, m, pairs, k,
                                                            ceil_div(m, form.rows), ceil_div(pairs, form.features / 2), plan);
  MI_CHECK_LAUNCH("gemm_turns_rope");
  return MI_OK;
}
