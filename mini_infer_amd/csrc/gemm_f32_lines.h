// The float32 product's order and its streaming loop, shared by gemm_f32.hip and the routed experts: 64-bit sums by the matrix instruction over SEGMENTS
// runs of K, each of whole slices of 32 values (gemm_f32.hip says how a run is summed).
#pragma once

#include "common.h"

typedef double f64x4_t __attribute__((ext_vector_type(4)));

#define SEGMENTS 8
#define SLICE 32       // values of K a step: one 128-byte line of a row

static __host__ __device__ inline int segment_slices(int k) { return (k + SEGMENTS * SLICE - 1) / (SEGMENTS * SLICE); }

__device__ __forceinline__ f64x4_t mma(float a, float w, f64x4_t acc) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64((double)a, (double)w, acc, 0, 0, 0);
}

// acc += the slices first .. last of RT tiles of 16 rows and FT tiles of 16 rows of W, a wave by itself.  a_row: lane's row (lane % 16 of each tile) from
// its first value on; lower, upper: byte offsets from w_block (the same for the wave) of the lane's 16 bytes in the lower and upper 8 rows of each
// tile of W (common.h): whole lines, non-temporal, brought into operand order by lane exchanges.  Two slices ahead.
template <int RT, int FT>
__device__ __forceinline__ void lines_product(const float* w_block, const uint32_t (&lower)[FT], const uint32_t (&upper)[FT], const float* const (&a_row)[RT],
                                              int first, int last, f64x4_t (&acc)[RT][FT]) {
  const int quad = threadIdx.x % MI_WAVE / 16;
  constexpr int AHEAD = 2;
  bf16x8_t lo[AHEAD][FT], hi[AHEAD][FT];  // 16-byte pieces; what they hold is float32
  float4 av[AHEAD][RT][2];
  auto fetch = [&](int slot, int slice) {
#pragma unroll
    for (int f = 0; f < FT; ++f) load_line_pair(w_block, 2 * (int64_t)slice, lower[f], upper[f], lo[slot][f], hi[slot][f]);
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      av[slot][i][0] = *reinterpret_cast<const float4*>(a_row[i] + slice * SLICE + 4 * quad);
      av[slot][i][1] = *reinterpret_cast<const float4*>(a_row[i] + slice * SLICE + 16 + 4 * quad);
    }
  };
#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
    if (first + s < last) fetch(s, first + s);
  for (int at = first; at < last; at += AHEAD) {
#pragma unroll
    for (int s = 0; s < AHEAD; ++s) {
      if (at + s < last) {
        float wv[FT][2][4], xv[RT][2][4];
#pragma unroll
        for (int f = 0; f < FT; ++f) {
          lines_to_operands(lo[s][f], hi[s][f]);
          __builtin_memcpy(wv[f][0], &lo[s][f], 16);
          __builtin_memcpy(wv[f][1], &hi[s][f], 16);
        }
        __builtin_memcpy(xv, av[s], sizeof(xv));
        if (at + s + AHEAD < last) fetch(s, at + s + AHEAD);
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int i = 0; i < RT; ++i)
#pragma unroll
              for (int f = 0; f < FT; ++f) acc[i][f] = mma(xv[i][half][e], wv[f][half][e], acc[i][f]);
      }
    }
  }
}
