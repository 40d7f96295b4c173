// Tiles of products of [gate; up] and of [q | k | v] (tile_product.h, turns_product.h): how the rows of gate and up, or of the two elements that are
// rotated together, lie in a tile, and what is made of its results.
#pragma once

#include "common.h"

#include <math.h>

// Of a wave's NT tiles of 16 rows of W the first half are gate rows, the second the up rows of the same features.
template <int NT>
struct GatedTile {
  static constexpr int PAIR = NT / 2 * 16;  // from a gate row of the tile to its up row
  // The row of [gate; up] of `features` features each that the tile's row r of W is, its features being those from f0 on.
  static __device__ __forceinline__ int row_of(int r, int f0, int features) {
    const int t = r % (2 * PAIR), f = min(f0 + r / (2 * PAIR) * PAIR + t % PAIR, features - 1);
    return t < PAIR ? f : f + features;
  }
  // Where the tile's feature f lies among its rows of W (its up row PAIR further on).
  static __device__ __forceinline__ int at(int f) { return f / PAIR * (2 * PAIR) + f % PAIR; }
};

// The same for results that meet in LDS only: gate rows (or first elements of pairs) are the first half of the tile's BN rows of W, whatever a wave's are.
template <int BN>
struct HalvedTile {
  static constexpr int PAIR = BN / 2;
  static_assert(PAIR % 8 == 0, "eight features of a thread lie side by side");
  static __device__ __forceinline__ int row_of(int r, int f0, int features) {
    const int f = min(f0 + r % PAIR, features - 1);
    return r < PAIR ? f : f + features;
  }
  static __device__ __forceinline__ int at(int f) { return f; }
};

enum { ACT_NONE = 0, ACT_SILU = 1, ACT_CLAMPED = 2, ACT_GELU = 3 };

struct GatedActivation {  // ACT_CLAMPED: float32 [2n] biases of gate and up (or null)
  const float* bias;
  float limit, slope;
};

// Eight bfloat16 values of LDS as floats, and eight floats as bfloat16 values of a row from column f on that has n of them (whole: 16 bytes at once).
__device__ __forceinline__ void mi_load_8(const bf16_t* p, float (&v)[8]) {
  const bf16x8_t got = *reinterpret_cast<const bf16x8_t*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = to_f32((bf16_t)got[i]);
}
__device__ __forceinline__ void mi_store_8(bf16_t* row, int f, int n, bool whole, const float (&v)[8]) {
  if (whole && f + 8 <= n) {
    bf16x8_t out;
#pragma unroll
    for (int i = 0; i < 8; ++i) out[i] = from_f32<bf16_t>(v[i]);
    *reinterpret_cast<bf16x8_t*>(row + f) = out;
  } else {
    for (int i = 0; i < 8 && f + i < n; ++i) row[f + i] = from_f32<bf16_t>(v[i]);
  }
}

// act(gate, up) of the BM x BN products that lie MADE elements a row apart in LDS, gate and up as Pairs says: rows r0 on (of m) and features f0 on (of n)
// of `out`.  The arithmetic of silu_mul, clamped_glu and gated_mul on the products as the element type holds them.
template <int ACT, class Pairs, int BM, int BN, int MADE, int THREADS>
__device__ __forceinline__ void write_activated(const bf16_t* made, const GatedActivation& how, bf16_t* out, int64_t ldo, bool whole, int r0, int m, int f0, int n) {
  constexpr int CHUNKS = BN / 16;
  static_assert(THREADS % CHUNKS == 0, "a thread's features are the same in every row");
  const int f = (int)threadIdx.x % CHUNKS * 8;
  float gate_bias[8] = {}, up_bias[8] = {};
  if (ACT == ACT_CLAMPED && how.bias != nullptr) {
#pragma unroll
    for (int c = 0; c < 8; ++c) gate_bias[c] = how.bias[min(f0 + f + c, n - 1)], up_bias[c] = how.bias[n + min(f0 + f + c, n - 1)];
  }
  if (f0 + f >= n) return;
  for (int row = threadIdx.x / CHUNKS; row < BM && r0 + row < m; row += THREADS / CHUNKS) {
    const bf16_t* at = made + row * MADE + Pairs::at(f);
    float v[8], u[8];
    mi_load_8(at, v);
    mi_load_8(at + Pairs::PAIR, u);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      if constexpr (ACT == ACT_CLAMPED) {
        const float gate = fminf(v[c] + gate_bias[c], how.limit);
        const float up = fminf(fmaxf(u[c] + up_bias[c], -how.limit), how.limit);
        v[c] = gate * mi_logistic(how.slope * gate) * (up + 1.f);
      } else if constexpr (ACT == ACT_GELU) {
        v[c] = 0.5f * v[c] * (1.f + tanhf(0.7978845608028654f * (v[c] + 0.044715f * v[c] * v[c] * v[c]))) * u[c];
      } else {
        v[c] = silu_times<bf16_t>(v[c], u[c]);
      }
    }
    mi_store_8(out + (int64_t)(r0 + row) * ldo, f0 + f, n, whole, v);
  }
}

// What becomes of a [q | k | v] product whose heads of `head_dim` are rotated in halves (element j with element j + head_dim / 2): rotated queries
// go to rows of q, rotated keys and values to their slots (values transposed within a page: [dim][slot]).
struct RotaryWrite {
  const float *cos, *sin;  // [m][head_dim / 2]
  const int* slots;        // of the rows; below 0: not written
  bf16_t *q, *k_pages, *v_pages;
  int64_t ldq;
  int q_heads, kv_heads, head_dim, page_size, v_transposed;
};

// The row of [q | k | v] that row_of's row of `pairs` pairs stands for: pair p is element p % half of head p / half, and the one half further on.
__device__ __forceinline__ int rotary_row_of(int row, int pairs, int head_dim) {
  const int half = head_dim / 2, p = row < pairs ? row : row - pairs;
  return p + p / half * half + (row < pairs ? 0 : half);
}

// Rotates and writes the BM x BN products that lie MADE elements a row apart in LDS: rows r0 on (of m), pairs f0 on (of n).  The arithmetic of
// rope_kv_write on the products as bfloat16.  A thread has 8 pairs of a row; of values that lie transposed 8 elements of the 8 rows
// that share 16 bytes of a page (two such windows side by side in a wave, the elements next: one row a thread, 2 bytes a store, would write
// a tile of values in four times the instructions).  What bounds it: the tile leaves LDS as it would without the rotation, beside the angles from
// L2 (asking for the next row's ahead of its turn measured the same).  The launch of rope_kv_write that it replaces read and wrote the projection once
// more: 6.3 us a layer at 271 rows x 5120, 11.8 at 2,048 x 6144, against products some 3 and 5 us longer; a step of 15 single tokens beside 256 at 3B
// sizes 4,281 -> 4,167 us (three times in turn, 1.026 to 1.030), a prompt of 2,048 tokens at 8B sizes 25,625 -> 25,370 (in tiles that keep both rows of a pair in one wave, of which
// there are none 192 wide, 25,825 -> 25,705).
template <class Pairs, int BM, int BN, int MADE, int THREADS>
__device__ __forceinline__ void write_rotated(const bf16_t* made, const RotaryWrite& how, int r0, int m, int f0, int n) {
  constexpr int CHUNKS = BN / 16;
  const int half = how.head_dim / 2, rows = min(BM, m - r0), ends = min(f0 + BN / 2, n);
  const int values_at = (how.q_heads + how.kv_heads) * half;  // pairs in front of the values
  const int direct = how.v_transposed ? min(ends, values_at) : ends;
  for (int i = threadIdx.x; f0 < direct && i < rows * CHUNKS; i += THREADS) {
    const int row = i / CHUNKS, f = i % CHUNKS * 8, p = f0 + f, t = r0 + row;
    if (p >= direct) continue;
    const int head = p / half, j = p % half;
    bf16_t* dst;
    if (head < how.q_heads) {
      dst = how.q + (int64_t)t * how.ldq + (int64_t)head * how.head_dim;
    } else {
      const int slot = how.slots[t];
      if (slot < 0) continue;
      const bool is_key = head < how.q_heads + how.kv_heads;
      const int h = head - how.q_heads - (is_key ? 0 : how.kv_heads);
      dst = (is_key ? how.k_pages : how.v_pages) + (((int64_t)(slot / how.page_size) * how.kv_heads + h) * how.page_size + slot % how.page_size) * how.head_dim;
    }
    const bf16_t* at = made + row * MADE + Pairs::at(f);
    float x0[8], x1[8], lo[8], hi[8];
    mi_load_8(at, x0);
    mi_load_8(at + Pairs::PAIR, x1);
    if (head < how.q_heads + how.kv_heads) {
      alignas(16) float c[8], s[8];
#pragma unroll
      for (int e = 0; e < 8; e += 4) {
        *reinterpret_cast<float4*>(c + e) = *reinterpret_cast<const float4*>(how.cos + (int64_t)t * half + j + e);
        *reinterpret_cast<float4*>(s + e) = *reinterpret_cast<const float4*>(how.sin + (int64_t)t * half + j + e);
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) mi_rotate(x0[e], x1[e], c[e], s[e], lo[e], hi[e]);
      mi_store_8(dst, j, how.head_dim, true, lo);
      mi_store_8(dst, j + half, how.head_dim, true, hi);
    } else {
      mi_store_8(dst, j, how.head_dim, true, x0);
      mi_store_8(dst, j + half, how.head_dim, true, x1);
    }
  }
  if (!how.v_transposed || ends <= max(values_at, f0)) return;
  // Windows of 8 rows begin where the first row's do in its page; a window whose rows do not follow one another there is written element by element.
  const int first = how.slots[r0], shift = first < 0 ? 0 : first % 8, windows = (rows + shift + 7) / 8;
  const bool eights = how.page_size % 8 == 0;
  for (int i = threadIdx.x; i < (windows + 1) / 2 * 2 * CHUNKS * 2; i += THREADS) {
    const int window = i / (4 * CHUNKS) * 2 + i % 2, part = i / 2 % (2 * CHUNKS), f = part / 2 * 8, p = f0 + f;
    const int begin = window * 8 - shift;
    if (window >= windows || p < values_at || p >= ends) continue;
    const int head = p / half, h = head - how.q_heads - how.kv_heads, d = p % half + part % 2 * half;
    const bf16_t* at = made + Pairs::at(f) + part % 2 * Pairs::PAIR;
    int slot[8];
    bf16x8_t got[8];
    bool together = eights;
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const int row = begin + r;
      const bool there = row >= 0 && row < rows;
      slot[r] = there ? how.slots[r0 + row] : -1;
      got[r] = *reinterpret_cast<const bf16x8_t*>(at + min(max(row, 0), rows - 1) * MADE);
      together = together && slot[r] >= 0 && slot[r] == slot[0] + r;
    }
    auto place = [&](int s) {
      return how.v_pages + (((int64_t)(s / how.page_size) * how.kv_heads + h) * how.head_dim + d) * how.page_size + s % how.page_size;
    };
    if (together && slot[0] % 8 == 0) {
      bf16_t* to = place(slot[0]);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        bf16x8_t out;
#pragma unroll
        for (int r = 0; r < 8; ++r) out[r] = got[r][e];
        *reinterpret_cast<bf16x8_t*>(to + (int64_t)e * how.page_size) = out;
      }
    } else {
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        if (slot[r] < 0) continue;
        bf16_t* to = place(slot[r]);
#pragma unroll
        for (int e = 0; e < 8; ++e) to[(int64_t)e * how.page_size] = (bf16_t)got[r][e];
      }
    }
  }
}

// What the entries of both kernels require of a rotary product's operands (m rows; the product's own are looked at there).
__host__ inline bool rotary_write_fits(const RotaryWrite& how, int m, int num_pages) {
  return m >= 1 && how.q_heads >= 1 && how.kv_heads >= 0 && how.head_dim >= 16 && how.head_dim % 16 == 0 && how.ldq >= (int64_t)how.q_heads * how.head_dim &&
         how.ldq % 8 == 0 && how.cos && how.sin && how.q && ((uintptr_t)how.cos | (uintptr_t)how.sin | (uintptr_t)how.q) % 16 == 0 &&
         (how.kv_heads == 0 || (how.slots && how.k_pages && how.v_pages && how.page_size > 0 && num_pages > 0 &&
                                ((uintptr_t)how.k_pages | (uintptr_t)how.v_pages) % 16 == 0));
}
