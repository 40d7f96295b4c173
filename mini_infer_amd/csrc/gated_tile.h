// Tiles of products of [gate; up] (tile_product.h, turns_product.h): how the rows of both lie in a tile, and what is made of its results.
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
