// What stands between the projections of a latent attention layer and its attention.
//
// Such a layer keeps ONE small row per token for all heads: a latent c (RMS-normed) from
// which every head's keys and values are linear maps, and a rotated part r that all heads
// share.  With the key map folded into the query (q' = W_uk^T q per head) a head's score is
// q' . c + q_rot . r: attention with a single key/value head whose key row is [c | r] and
// whose value row is c itself, the value map applied to the attention's output afterwards.
//
//   latent_prepare   per token: c = x_c / sqrt(mean(x_c^2) + eps) * weight and the rotated r go
//                    into the token's slot of the key pages as one row [c | r]; each head's
//                    rotated query part goes behind that head's folded part in the query rows
//                    the attention reads ([head][rank + rot]).
//   latent_expand_pages   for steps in which every request begins: keys and values written out per head.
//
// Rotation pairs entry 2i with 2i+1; cos and sin come as float32 tables [tokens, rot/2].
#include "common.h"

#include <math.h>

namespace {

template <typename T>
__global__ __launch_bounds__(256) void latent_prepare_kernel(
    const T* __restrict__ proj, int64_t proj_stride, int q_col, int q_head_width, int q_rot_at, int c_col,
    const float* __restrict__ cos_t, const float* __restrict__ sin_t, const float* __restrict__ norm_weight,
    const int* __restrict__ slot_mapping, T* __restrict__ k_pages, T* __restrict__ queries, int64_t queries_stride,
    T* __restrict__ latent_out, int heads, int rank, int rot, float eps, const T* __restrict__ down,
    int64_t down_stride) {
  __shared__ float scratch[4];
  __shared__ double scratch_wide[4];
  constexpr bool WIDE = sizeof(T) == 4;
  const int t = blockIdx.x;
  const int half = rot / 2;
  const T* row = proj + (int64_t)t * proj_stride;
  const float* c = cos_t + (int64_t)t * half;
  const float* s = sin_t + (int64_t)t * half;
  const int width = rank + rot;

  auto turn = [&](float x0, float x1, int i, float& y0, float& y1) {
    if constexpr (WIDE) {
      y0 = (float)((double)x0 * c[i] - (double)x1 * s[i]);
      y1 = (float)((double)x1 * c[i] + (double)x0 * s[i]);
    } else {
      y0 = x0 * c[i] - x1 * s[i];
      y1 = x1 * c[i] + x0 * s[i];
    }
  };

  T* q_out = queries + (int64_t)t * queries_stride;
  for (int e = threadIdx.x; queries != nullptr && e < heads * half; e += blockDim.x) {
    const int h = e / half, i = e % half;
    const T* x = row + q_col + h * q_head_width + q_rot_at;
    float y0, y1;
    turn(to_f32(x[2 * i]), to_f32(x[2 * i + 1]), i, y0, y1);
    T* dst = q_out + (int64_t)h * width + rank;
    dst[2 * i] = from_f32<T>(y0);
    dst[2 * i + 1] = from_f32<T>(y1);
  }

  const int slot = slot_mapping != nullptr ? slot_mapping[t] : -1;
  if (slot < 0 && latent_out == nullptr) return;  // (the whole block leaves together)
  // ([x_c | x_r] lie in `proj`'s rows, or in rows of their own where the queries come from a product of their own)
  const T* x = (down != nullptr ? down + (int64_t)t * down_stride : row) + c_col;
  float squares = 0.f;
  double squares_wide = 0.0;
  for (int d = threadIdx.x; d < rank; d += blockDim.x) {
    const float v = to_f32(x[d]);
    if constexpr (WIDE) squares_wide += (double)v * v;
    else squares += v * v;
  }
  T* dst = slot >= 0 ? k_pages + (int64_t)slot * width : nullptr;
  T* copy = latent_out ? latent_out + (int64_t)t * rank : nullptr;
  if constexpr (WIDE) {
    // (a fixed order: lanes by butterfly, waves one after another)
#pragma unroll
    for (int off = MI_WAVE / 2; off > 0; off >>= 1) squares_wide += __shfl_xor(squares_wide, off, MI_WAVE);
    if (threadIdx.x % MI_WAVE == 0) scratch_wide[threadIdx.x / MI_WAVE] = squares_wide;
    __syncthreads();
    double total = 0.0;
    for (int w = 0; w < (int)blockDim.x / MI_WAVE; ++w) total += scratch_wide[w];
    const double inv = 1.0 / sqrt(total / (double)rank + (double)eps);
    for (int d = threadIdx.x; d < rank; d += blockDim.x) {
      const float c_d = (float)((double)x[d] * inv * (double)norm_weight[d]);
      if (dst) dst[d] = c_d;
      if (copy) copy[d] = c_d;
    }
  } else {
    const float inv = rsqrtf(block_sum(squares, scratch) / (float)rank + eps);
    for (int d = threadIdx.x; d < rank; d += blockDim.x) {
      const T c_d = from_f32<T>(to_f32(x[d]) * inv * norm_weight[d]);
      if (dst) dst[d] = c_d;
      if (copy) copy[d] = c_d;
    }
  }
  for (int i = threadIdx.x; dst != nullptr && i < half; i += blockDim.x) {
    float y0, y1;
    turn(to_f32(x[rank + 2 * i]), to_f32(x[rank + 2 * i + 1]), i, y0, y1);
    dst[rank + 2 * i] = from_f32<T>(y0);
    dst[rank + 2 * i + 1] = from_f32<T>(y1);
  }
}

// Keys and values written out per head into pages of the step's own, for prompts that are in the step from their first
// token, and the queries' rotation:
//   q head: [plain part | rotated part], in place or into rows of their own      k head: [W_uk c | rotated shared part]
//   v head: [W_uv c | zeros up to v_width], transposed: a dim's slots side by side
// which the paged attention kernels take.  A block makes a page of some heads whole, zeros behind a request's last token
// included.  Bound by the bytes: each value is read and written once, 16 bytes a thread (EIGHTS: sizes and strides in
// whole 8s; without, an element a thread).  1,501 tokens of 24 heads of 128 + 64, 128 wide values (50 MB,
// 10.5 us at the rate of a large copy): 14.7 us, for 46.4 as one row [q | k | v] a token, a fill of the pages and a copy into them.
template <typename T>
struct BitsOf {
  using type = uint32_t;
};
template <>
struct BitsOf<bf16_t> {
  using type = uint16_t;
};

template <typename T, bool EIGHTS>
__global__ __launch_bounds__(256) void latent_expand_pages_kernel(
    const T* proj, int64_t proj_stride, const T* __restrict__ shared_key, int64_t shared_stride, const T* __restrict__ k_up,
    int64_t k_up_stride, const T* __restrict__ v_up, int64_t v_up_stride, const float* __restrict__ cos_t,
    const float* __restrict__ sin_t, T* queries, int64_t queries_stride, T* __restrict__ k_pages, T* __restrict__ v_pages,
    const int* __restrict__ page_first, const int* __restrict__ page_tokens, int heads, int dim, int rot, int vdim, int v_width,
    int page_size, int heads_each) {
  constexpr int V = EIGHTS ? 8 : 1;
  struct alignas(V * sizeof(T) < 16 ? V * sizeof(T) : 16) Piece {
    T v[V];
  };
  const int page = blockIdx.x, h0 = blockIdx.y * heads_each, nh = min(heads_each, heads - h0);
  const int t0 = page_first[page], n = page_tokens[page];
  const int D = dim + rot, half = rot / 2, pieces = D / V;
  const bool copies = queries != proj;
  for (int i = threadIdx.x; i < page_size * nh * pieces; i += blockDim.x) {
    const int d = i % pieces * V, h = h0 + i / pieces % nh, off = i / (pieces * nh);
    T* k_at = k_pages + (((int64_t)page * heads + h) * page_size + off) * D + d;
    Piece k;
    if (off >= n) {
#pragma unroll
      for (int j = 0; j < V; ++j) k.v[j] = from_f32<T>(0.f);
      *reinterpret_cast<Piece*>(k_at) = k;
      continue;
    }
    const int64_t t = t0 + off;
    const T* q_from = proj + t * proj_stride + (int64_t)h * D + d;
    T* q_to = queries + t * queries_stride + (int64_t)h * D + d;
    if (d < dim) {
      *reinterpret_cast<Piece*>(k_at) = *reinterpret_cast<const Piece*>(k_up + t * k_up_stride + (int64_t)h * dim + d);
      if (copies) *reinterpret_cast<Piece*>(q_to) = *reinterpret_cast<const Piece*>(q_from);
      continue;
    }
    // (which of the two products is fused is said, so that both forms, and steps of any size, round alike)
    const T* shared = shared_key + t * shared_stride + (d - dim);
    const float *c = cos_t + t * half + (d - dim) / 2, *s = sin_t + t * half + (d - dim) / 2;
    if constexpr (EIGHTS) {
      const Piece q = *reinterpret_cast<const Piece*>(q_from), r = *reinterpret_cast<const Piece*>(shared);
      float cj[4], sj[4];
      mi_load_cols<float, 4>(c, cj);
      mi_load_cols<float, 4>(s, sj);
      Piece turned;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float q0 = to_f32(q.v[2 * j]), q1 = to_f32(q.v[2 * j + 1]), k0 = to_f32(r.v[2 * j]), k1 = to_f32(r.v[2 * j + 1]);
        turned.v[2 * j] = from_f32<T>(fmaf(q0, cj[j], -(q1 * sj[j])));
        turned.v[2 * j + 1] = from_f32<T>(fmaf(q1, cj[j], q0 * sj[j]));
        k.v[2 * j] = from_f32<T>(fmaf(k0, cj[j], -(k1 * sj[j])));
        k.v[2 * j + 1] = from_f32<T>(fmaf(k1, cj[j], k0 * sj[j]));
      }
      *reinterpret_cast<Piece*>(q_to) = turned;
    } else {
      const int odd = (d - dim) & 1;
      const float q0 = to_f32(q_from[-odd]), q1 = to_f32(q_from[1 - odd]), k0 = to_f32(shared[-odd]), k1 = to_f32(shared[1 - odd]);
      q_to[0] = from_f32<T>(odd ? fmaf(q1, *c, q0 * *s) : fmaf(q0, *c, -(q1 * *s)));
      k.v[0] = from_f32<T>(odd ? fmaf(k1, *c, k0 * *s) : fmaf(k0, *c, -(k1 * *s)));
    }
    *reinterpret_cast<Piece*>(k_at) = k;
  }
  // (tokens past the last one and columns past the values: the last ones' bits, masked; a choice would be a branch a load)
  using Bits = typename BitsOf<T>::type;
  for (int i = threadIdx.x; i < nh * v_width; i += blockDim.x) {
    const int h = h0 + i / v_width, d = i % v_width;
    const Bits* from = reinterpret_cast<const Bits*>(v_up) + (int64_t)h * vdim + min(d, vdim - 1);
    Bits* to = reinterpret_cast<Bits*>(v_pages) + (((int64_t)page * heads + h) * v_width + d) * page_size;
    for (int o = 0; o < page_size; o += V) {
      struct alignas(V * sizeof(Bits) < 16 ? V * sizeof(Bits) : 16) Slots {
        Bits v[V];
      } x;
#pragma unroll
      for (int j = 0; j < V; ++j) x.v[j] = from[(int64_t)(t0 + min(o + j, n - 1)) * v_up_stride];
#pragma unroll
      for (int j = 0; j < V; ++j) x.v[j] &= (Bits)(o + j < n && d < vdim ? ~0u : 0u);
      *reinterpret_cast<Slots*>(to + o) = x;
    }
  }
}

}  // namespace

// proj: query heads [plain (dim) | to rotate (rot)] from column 0 on; shared_key: the shared part's rows, from its first
// column.  queries: rows of heads * (dim + rot), or proj itself (its heads are then rotated in place).  page_first,
// page_tokens: per page its first token and how many it holds, 1 .. page_size; every token lies in one page.
extern "C" int mi_latent_expand_pages(int dtype, const void* proj, int64_t proj_stride, const void* shared_key, int64_t shared_stride,
                                      const void* k_up, int64_t k_up_stride, const void* v_up, int64_t v_up_stride,
                                      const float* cos_t, const float* sin_t, void* queries, int64_t queries_stride, void* k_pages,
                                      void* v_pages, const int* page_first, const int* page_tokens, int num_pages, int heads, int dim,
                                      int rot, int vdim, int v_width, int page_size, hipStream_t stream) {
  MI_REQUIRE(num_pages >= 0 && heads > 0 && dim > 0 && rot >= 0 && rot % 2 == 0 && vdim > 0 && v_width >= vdim && page_size > 0,
             "latent_expand_pages: bad sizes pages=%d heads=%d dim=%d rot=%d vdim=%d v_width=%d page_size=%d", num_pages, heads, dim,
             rot, vdim, v_width, page_size);
  MI_REQUIRE(proj_stride >= (int64_t)heads * (dim + rot) && queries_stride >= (int64_t)heads * (dim + rot) && shared_stride >= rot &&
                 k_up_stride >= (int64_t)heads * dim && v_up_stride >= (int64_t)heads * vdim,
             "latent_expand_pages: row strides shorter than a row");
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "latent_expand_pages: unknown dtype %d", dtype);
  const bool eights = dim % 8 == 0 && rot % 8 == 0 && page_size % 8 == 0 &&
                      (proj_stride | shared_stride | k_up_stride | queries_stride) % 8 == 0 &&
                      ((uintptr_t)proj | (uintptr_t)shared_key | (uintptr_t)k_up | (uintptr_t)cos_t | (uintptr_t)sin_t |
                       (uintptr_t)queries | (uintptr_t)k_pages | (uintptr_t)v_pages) % 16 == 0;
  MI_REQUIRE(queries != proj || (eights && queries_stride == proj_stride), "latent_expand_pages: rows that cannot be rotated in place");
  if (num_pages == 0) return MI_OK;
  const int heads_each = eights ? 4 : 1;  // (4 heads of 100 + 20, an element a thread: a prompt of 300 tokens 24.4 us with 4, 9.1 with 1)
  MI_REQUIRE(ceil_div(heads, heads_each) <= 65535 && (int64_t)page_size * heads_each * (dim + rot) <= 2147483647,
             "latent_expand_pages: heads=%d or page_size=%d is too large", heads, page_size);
  dim3 grid(num_pages, ceil_div(heads, heads_each));
#define MI_EXPAND(T, EIGHTS)                                                                                                   \
  latent_expand_pages_kernel<T, EIGHTS><<<grid, 256, 0, stream>>>(                                                             \
      (const T*)proj, proj_stride, (const T*)shared_key, shared_stride, (const T*)k_up, k_up_stride, (const T*)v_up, v_up_stride, \
      cos_t, sin_t, (T*)queries, queries_stride, (T*)k_pages, (T*)v_pages, page_first, page_tokens, heads, dim, rot, vdim, v_width, \
      page_size, heads_each)
  if (dtype == MI_F32) {
    if (eights) MI_EXPAND(float, true);
    else MI_EXPAND(float, false);
  } else {
    if (eights) MI_EXPAND(bf16_t, true);
    else MI_EXPAND(bf16_t, false);
  }
#undef MI_EXPAND
  MI_CHECK_LAUNCH("latent_expand_pages");
  return MI_OK;
}

// proj: rows that hold the query projection (heads of q_head_width columns from q_col on, the
// part to rotate rot columns wide from q_rot_at inside a head) and, from c_col on, [x_c (rank) |
// x_r (rot)].  k_pages: [num_pages * page_size][rank + rot] (one key head); slot_mapping may be
// null (nothing is written: a call that reads another's pages).  queries: [tokens, heads * (rank
// + rot)] (row stride) or null; only the last rot columns of every head are written here.
// latent_out: [tokens, rank] or null, a copy of the normed latents.  down (may be null): rows of their own
// that hold [x_c | x_r] from c_col on, where the queries come from a product of their own.
extern "C" int mi_latent_prepare(int dtype, const void* proj, int64_t proj_stride, int q_col, int q_head_width,
                                 int q_rot_at, int c_col, const float* cos_t, const float* sin_t,
                                 const float* norm_weight, const int* slot_mapping, void* k_pages, void* queries,
                                 int64_t queries_stride, void* latent_out, int num_tokens, int heads, int rank, int rot,
                                 float eps, const void* down, int64_t down_stride, hipStream_t stream) {
  MI_REQUIRE(num_tokens >= 0 && heads > 0 && rank > 0 && rot >= 0 && rot % 2 == 0,
             "latent_prepare: bad sizes tokens=%d heads=%d rank=%d rot=%d", num_tokens, heads, rank, rot);
  MI_REQUIRE(q_rot_at >= 0 && q_rot_at + rot <= q_head_width, "latent_prepare: the rotated part lies outside a query head");
  MI_REQUIRE(q_col >= 0 && c_col >= 0 && proj_stride >= q_col + (int64_t)heads * q_head_width &&
                 (down != nullptr ? down_stride : proj_stride) >= c_col + (int64_t)rank + rot,
             "latent_prepare: columns outside a row of the projections");
  MI_REQUIRE(queries == nullptr || queries_stride >= (int64_t)heads * (rank + rot),
             "latent_prepare: query rows shorter than heads * (rank + rot)");
  MI_REQUIRE(slot_mapping == nullptr || k_pages != nullptr, "latent_prepare: pages are needed to write keys");
  MI_REQUIRE(eps > 0.f, "latent_prepare: eps must be positive, got %g", (double)eps);
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "latent_prepare: unknown dtype %d", dtype);
  if (num_tokens == 0) return MI_OK;
  if (dtype == MI_F32)
    latent_prepare_kernel<float><<<num_tokens, 256, 0, stream>>>(
        (const float*)proj, proj_stride, q_col, q_head_width, q_rot_at, c_col, cos_t, sin_t, norm_weight, slot_mapping,
        (float*)k_pages, (float*)queries, queries_stride, (float*)latent_out, heads, rank, rot, eps, (const float*)down, down_stride);
  else
    latent_prepare_kernel<bf16_t><<<num_tokens, 256, 0, stream>>>(
        (const bf16_t*)proj, proj_stride, q_col, q_head_width, q_rot_at, c_col, cos_t, sin_t, norm_weight, slot_mapping,
        (bf16_t*)k_pages, (bf16_t*)queries, queries_stride, (bf16_t*)latent_out, heads, rank, rot, eps, (const bf16_t*)down,
        down_stride);
  MI_CHECK_LAUNCH("latent_prepare");
  return MI_OK;
}
