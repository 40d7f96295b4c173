// Paged causal attention of the 32-bit path for steps with many tokens a request: the matrix cores' 64-bit instruction.
//
// The same attention as attn_generic (attention_generic.hip) makes of float32 inputs: scores, softmax and value sums are
// 64-bit, a result is rounded once, when it is written (weights, which that kernel rounds to float32, stay 64-bit here).
// Plain form only: causal, with or without a window; heads of 64 or 128, pages of whole 16s.
//
// A block owns 16 rows (a row is a token and a query head; the heads of a key/value head's group lie side by side, so that
// every key row read serves 16 of them), its 4 waves take every fourth tile of 16 keys and are merged at the end.  A row
// of attn_generic reads its keys for up to 4 heads, the query from LDS once a multiplication, and is bound by that: one
// layer of a prompt of 509 tokens, 32 heads of 64 over 8 key/value heads, took 147 us and takes 66 (the matrix
// instructions 30 of them; the rest is a tile's chain: loads, scores, maxima over 16 lanes, exponentials in 64-bit, the
// weights through LDS, with two waves a SIMD to cover one another).
#include "common.h"

#include <math.h>

typedef double f64x4_t __attribute__((ext_vector_type(4)));

namespace {

#define ROWS 16
#define KEYS 16
#define WAVES 4
#define P_ROW 18  // doubles: rows of weights on 16 bytes, 16-byte reads of 16 rows on different banks

__device__ __forceinline__ f64x4_t mma(double a, double b, f64x4_t acc) { return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0); }
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }

// grid: row tiles (the last, which see the most keys, first), key/value heads * blocks of up to 16 heads of the group.
// heads_each: query heads a tile holds; it holds 16 / heads_each tokens.  Operands of the instruction: lane = 16 * quad + c
// holds the first one's row c and the second one's column c, of the four values that the instructions s = 0..3 sum over
// number 4 * quad + s; results: register e is row 4 * e + quad, column c.
template <int HD>
__global__ __launch_bounds__(WAVES * MI_WAVE, HD == 64 ? 2 : 1) void attn_prompt_f32_kernel(
    const float* __restrict__ q, int64_t q_row_stride, const float* __restrict__ k_pages, const float* __restrict__ v_pages,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ token_request, const int* __restrict__ positions,
    float* __restrict__ out, int64_t out_row_stride, int num_tokens, int q_heads, int kv_heads, int page_size, double scale,
    int window, int heads_each) {
  constexpr int HALVES = HD / 64;
  __shared__ __align__(16) double weights[WAVES][ROWS * P_ROW];
  __shared__ __align__(16) double merge[WAVES - 1][HALVES * 4 * 4 + 4][MI_WAVE];
  __shared__ float maxima[WAVES][4][MI_WAVE];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), lane = threadIdx.x % MI_WAVE;
  const int c = lane % 16, quad = lane / 16;
  const int group = q_heads / kv_heads, head_blocks = (group + heads_each - 1) / heads_each;
  const int kvh = blockIdx.y / head_blocks, g0 = blockIdx.y % head_blocks * heads_each;
  const int nh = min(heads_each, group - g0), tokens_each = ROWS / heads_each;
  const int t0 = (gridDim.x - 1 - blockIdx.x) * tokens_each, nt = min(tokens_each, num_tokens - t0);
  const int head0 = kvh * group + g0;

  // the row whose queries this lane holds (of rows that are none the first one's)
  const int q_token = c / heads_each, q_head = c % heads_each;
  const bool q_real = q_token < nt && q_head < nh;
  const float* q_row = q + (int64_t)(t0 + (q_real ? q_token : 0)) * q_row_stride + (int64_t)(head0 + (q_real ? q_head : 0)) * HD;
  float4 query[HD / 16];
#pragma unroll
  for (int i = 0; i < HD / 16; ++i) query[i] = load4(q_row + 16 * i + 4 * quad);
  // the four rows whose scores and sums it holds
  int token[4], pos[4];
  bool real[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int row = 4 * e + quad;
    token[e] = row / heads_each;
    real[e] = token[e] < nt && row % heads_each < nh;
    pos[e] = positions[t0 + min(token[e], nt - 1)];
  }
  float m[4];
  double l[4];  // (of this lane's columns alone, until the end)
  f64x4_t acc[HALVES][4];
#pragma unroll
  for (int e = 0; e < 4; ++e) m[e] = -INFINITY, l[e] = 0.0;
#pragma unroll
  for (int h = 0; h < HALVES; ++h)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[h][j] = f64x4_t{0.0, 0.0, 0.0, 0.0};
  double* mine = weights[wave];

  // a tile's tokens are usually one request's; where it holds several, one after another
  for (int from = 0; from < nt;) {
    const int request = __builtin_amdgcn_readfirstlane(token_request[t0 + from]);
    int to = from + 1;
    while (to < nt && token_request[t0 + to] == request) ++to;
    const int* pages = block_table + (int64_t)request * max_blocks;
    const int first_pos = __builtin_amdgcn_readfirstlane(positions[t0 + from]), last_key = __builtin_amdgcn_readfirstlane(positions[t0 + to - 1]);
    const int lo = window > 0 ? max(0, first_pos - window + 1) : 0;
    for (int base = lo / KEYS * KEYS + wave * KEYS; base <= last_key; base += WAVES * KEYS) {
      const int64_t row0 = ((int64_t)pages[base / page_size] * kv_heads + kvh) * page_size + base % page_size;
      const int most = min(KEYS - 1, last_key - base);  // (keys past the last one: that one, with weight 0)
      const float* k_row = k_pages + (row0 + min(c, most)) * HD + 4 * quad;
      float4 key[HD / 16], value[4][HALVES];
#pragma unroll
      for (int i = 0; i < HD / 16; ++i) key[i] = load4(k_row + 16 * i);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int h = 0; h < HALVES; ++h) value[s][h] = load4(v_pages + (row0 + min(4 * quad + s, most)) * HD + 64 * h + 4 * c);
      f64x4_t score = {0.0, 0.0, 0.0, 0.0}, other = score;  // (two chains of instructions)
#pragma unroll
      for (int i = 0; i < HD / 16; ++i) {
        score = mma((double)query[i].x, (double)key[i].x, score);
        other = mma((double)query[i].y, (double)key[i].y, other);
        score = mma((double)query[i].z, (double)key[i].z, score);
        other = mma((double)query[i].w, (double)key[i].w, other);
      }
      bool sees[4], higher = false;
      float top[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int at = base + c;
        sees[e] = real[e] && token[e] >= from && token[e] < to && at <= pos[e] && (window <= 0 || at > pos[e] - window);
        score[e] = (score[e] + other[e]) * scale;
        top[e] = sees[e] ? (float)score[e] : -INFINITY;
#pragma unroll
        for (int off = 8; off > 0; off >>= 1) top[e] = fmaxf(top[e], __shfl_xor(top[e], off, MI_WAVE));
        top[e] = fmaxf(top[e], m[e]);
        higher = higher || top[e] > m[e];
      }
      if (__ballot(higher) != 0) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const double less = top[e] > m[e] ? exp((double)m[e] - (double)top[e]) : 1.0;  // (0 for the first keys)
          l[e] *= less;
#pragma unroll
          for (int h = 0; h < HALVES; ++h)
#pragma unroll
            for (int j = 0; j < 4; ++j) acc[h][j][e] *= less;
          m[e] = top[e];
        }
      }
      double p[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // (scores of -inf alone so far, of an infinite key say: weight 0, not the exponential of inf less inf)
        p[e] = sees[e] ? exp(score[e] - (m[e] == -INFINITY ? 0.0 : (double)m[e])) : 0.0;
        l[e] += p[e];
        mine[(4 * e + quad) * P_ROW + c] = p[e];
      }
      // (a wave's own LDS, whose accesses keep their order)
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const double2 p01 = *reinterpret_cast<const double2*>(&mine[c * P_ROW + 4 * quad]);
      const double2 p23 = *reinterpret_cast<const double2*>(&mine[c * P_ROW + 4 * quad + 2]);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      const double ps[4] = {p01.x, p01.y, p23.x, p23.y};
      // A value that is no number must not reach the rows that do not see its key (the instruction would make 0 * inf of
      // it): then key by key.
      float odd = 0.f;
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int h = 0; h < HALVES; ++h) odd += 0.f * value[s][h].x + 0.f * value[s][h].y + 0.f * value[s][h].z + 0.f * value[s][h].w;
      if (__ballot(!(odd == 0.f)) == 0) {
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int h = 0; h < HALVES; ++h) {
            acc[h][0] = mma(ps[s], (double)value[s][h].x, acc[h][0]);
            acc[h][1] = mma(ps[s], (double)value[s][h].y, acc[h][1]);
            acc[h][2] = mma(ps[s], (double)value[s][h].z, acc[h][2]);
            acc[h][3] = mma(ps[s], (double)value[s][h].w, acc[h][3]);
          }
      } else {
        for (int n = 0; n <= most; ++n) {
          float4 v[HALVES];
#pragma unroll
          for (int h = 0; h < HALVES; ++h) v[h] = load4(v_pages + (row0 + n) * HD + 64 * h + 4 * c);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const double weight = __shfl(p[e], 16 * quad + n, MI_WAVE);
            const bool seen = __shfl((int)sees[e], 16 * quad + n, MI_WAVE) != 0;
            if (seen) {
#pragma unroll
              for (int h = 0; h < HALVES; ++h) {
                acc[h][0][e] += weight * (double)v[h].x;
                acc[h][1][e] += weight * (double)v[h].y;
                acc[h][2][e] += weight * (double)v[h].z;
                acc[h][3][e] += weight * (double)v[h].w;
              }
            }
          }
        }
      }
    }
    from = to;
  }

  // the waves' sums, on the scale of the highest of their maxima; wave 0 takes over what the others have, in their order
#pragma unroll
  for (int e = 0; e < 4; ++e) maxima[wave][e][lane] = m[e];
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float top = maxima[0][e][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) top = fmaxf(top, maxima[w][e][lane]);
    const double less = m[e] == -INFINITY ? 0.0 : exp((double)m[e] - (double)top);  // (a wave without keys has nothing to add)
    l[e] *= less;
#pragma unroll
    for (int off = 8; off > 0; off >>= 1) l[e] += __shfl_xor(l[e], off, MI_WAVE);
#pragma unroll
    for (int h = 0; h < HALVES; ++h)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        acc[h][j][e] *= less;
        if (wave > 0) merge[wave - 1][(h * 4 + j) * 4 + e][lane] = acc[h][j][e];
      }
    if (wave > 0) merge[wave - 1][HALVES * 16 + e][lane] = l[e];
  }
  __syncthreads();
  if (wave > 0) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    double sum = l[e];
#pragma unroll
    for (int w = 0; w < WAVES - 1; ++w) sum += merge[w][HALVES * 16 + e][lane];
    const double inv = 1.0 / sum;
#pragma unroll
    for (int h = 0; h < HALVES; ++h) {
      float made[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        double total = acc[h][j][e];
#pragma unroll
        for (int w = 0; w < WAVES - 1; ++w) total += merge[w][(h * 4 + j) * 4 + e][lane];
        made[j] = (float)(total * inv);
      }
      if (real[e])
        *reinterpret_cast<float4*>(out + (int64_t)(t0 + token[e]) * out_row_stride + (int64_t)(head0 + (4 * e + quad) % heads_each) * HD +
                                   64 * h + 4 * c) = make_float4(made[0], made[1], made[2], made[3]);
    }
  }
}

// query heads a tile holds: a group's, up to 16
int heads_a_tile(int group) { return group < ROWS ? group : ROWS; }

}  // namespace

// Blocks that mi_attn_prompt_f32 starts for a step; 0: sizes it does not take.
extern "C" int64_t mi_attn_prompt_f32_blocks(int num_tokens, int q_heads, int kv_heads, int head_dim, int page_size) {
  if (num_tokens <= 0 || kv_heads <= 0 || q_heads <= 0 || q_heads % kv_heads != 0 || (head_dim != 64 && head_dim != 128) ||
      page_size <= 0 || page_size % KEYS != 0)
    return 0;
  const int each = heads_a_tile(q_heads / kv_heads);
  const int64_t y = (int64_t)kv_heads * ceil_div(q_heads / kv_heads, each);
  return y > 65535 ? 0 : ceil_div(num_tokens, ROWS / each) * y;
}

// q, k_pages, v_pages, out float32, their rows on 16 bytes; the rest as mi_attn_generic.
extern "C" int mi_attn_prompt_f32(const float* q, int64_t q_row_stride, const float* k_pages, const float* v_pages,
                                  const int* block_table, int max_blocks, const int* token_request, const int* positions, float* out,
                                  int64_t out_row_stride, int num_tokens, int q_heads, int kv_heads, int head_dim, int page_size,
                                  int num_pages, float scale, int window, hipStream_t stream) {
  MI_REQUIRE(num_tokens >= 0 && num_pages > 0 && max_blocks > 0 && window >= 0, "attn_prompt_f32: bad sizes tokens=%d pages=%d window=%d",
             num_tokens, num_pages, window);
  if (num_tokens == 0) return MI_OK;
  MI_REQUIRE(mi_attn_prompt_f32_blocks(num_tokens, q_heads, kv_heads, head_dim, page_size) > 0,
             "attn_prompt_f32: q_heads=%d kv_heads=%d head_dim=%d page_size=%d are not taken", q_heads, kv_heads, head_dim, page_size);
  MI_REQUIRE(q_row_stride >= (int64_t)q_heads * head_dim && out_row_stride >= (int64_t)q_heads * head_dim,
             "attn_prompt_f32: row strides shorter than q_heads*head_dim");
  MI_REQUIRE(q_row_stride % 4 == 0 && out_row_stride % 4 == 0 &&
                 ((uintptr_t)q | (uintptr_t)k_pages | (uintptr_t)v_pages | (uintptr_t)out) % 16 == 0,
             "attn_prompt_f32: rows must lie on 16 bytes");
  const int each = heads_a_tile(q_heads / kv_heads);
  dim3 grid(ceil_div(num_tokens, ROWS / each), kv_heads * ceil_div(q_heads / kv_heads, each));
#define MI_PROMPT(HD)                                                                                                        \
  attn_prompt_f32_kernel<HD><<<grid, WAVES * MI_WAVE, 0, stream>>>(q, q_row_stride, k_pages, v_pages, block_table, max_blocks, \
                                                                   token_request, positions, out, out_row_stride, num_tokens, \
                                                                   q_heads, kv_heads, page_size, (double)scale, window, each)
  if (head_dim == 64) MI_PROMPT(64);
  else MI_PROMPT(128);
#undef MI_PROMPT
  MI_CHECK_LAUNCH("attn_prompt_f32");
  return MI_OK;
}
