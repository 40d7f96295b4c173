// Row kernels of a stack whose norms stand BEHIND the residual sum (post-norm), and of an
// embedding with a second table indexed by a hash of a token and the token before it.
//
//   embed_pair_hash   stream[t] = table[id_t] + pairs[row_t],
//                     row_t = (prev_t * mul_prev + id_t * mul_cur) mod buckets, and `buckets` (the
//                     table's last row) for a sequence's first token.  The token before a step's
//                     first one is read from the request's state row, and the step's last token
//                     is left there.
//   scale_add_norm    x[t] <- rms_norm(alpha * x[t] + scale[c] * y[t, c]) * factor[c]  in place on the
//                     float32 stream, with the new row's copy in the element type for the products
//                     that read it next; without y and for a list of rows: the norm alone (how
//                     such a stack ends).
//   norm_rows         out[t] = rms_norm(in[t, 0..width)) * weight: a norm inside a mixer, on the
//                     first columns of a wider row.
//
// Sums and statistics are float32 for bfloat16 rows and 64-bit for float32 rows (rounded once).
#include "common.h"

#include <math.h>

namespace {

template <typename T>
struct WideOf {
  using type = float;
};
template <>
struct WideOf<float> {
  using type = double;
};

__device__ __forceinline__ float lane_add(float v, int off) { return v + __shfl_xor(v, off, MI_WAVE); }
__device__ __forceinline__ double lane_add(double v, int off) { return v + __shfl_xor(v, off, MI_WAVE); }

// sum over a block in a fixed order: lanes by butterfly, waves one after another
template <typename A>
__device__ __forceinline__ A block_add(A v, A* scratch) {
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) v = lane_add(v, off);
  const int wave = threadIdx.x / MI_WAVE, lane = threadIdx.x % MI_WAVE;
  const int n_waves = (blockDim.x + MI_WAVE - 1) / MI_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  A total = 0;
  for (int w = 0; w < n_waves; ++w) total += scratch[w];
  return total;
}

// The same, the waves' sums (16 at most) read at once and added in order.
template <typename A>
__device__ __forceinline__ A block_add_at_once(A v, A* scratch) {
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) v = lane_add(v, off);
  const int wave = threadIdx.x / MI_WAVE, lane = threadIdx.x % MI_WAVE;
  const int n_waves = (blockDim.x + MI_WAVE - 1) / MI_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  A parts[16];
#pragma unroll
  for (int w = 0; w < 16; ++w) parts[w] = scratch[min(w, n_waves - 1)];
  A total = 0;
#pragma unroll
  for (int w = 0; w < 16; ++w)
    if (w < n_waves) total += parts[w];
  return total;
}

__device__ __forceinline__ float inv_root_of(float mean_sq, float eps) { return 1.0f / sqrtf(mean_sq + eps); }
__device__ __forceinline__ double inv_root_of(double mean_sq, double eps) { return 1.0 / sqrt(mean_sq + eps); }

inline bool is_aligned16(const void* p) { return ((uintptr_t)p % 16) == 0; }
inline int threads_for(int rows, int items) { return (rows < 256 && items > 1024) ? 1024 : 256; }

// ---------------------------------------------------------------------------------------------

template <typename T, int VEC>
__global__ __launch_bounds__(256) void embed_pair_hash_kernel(
    const T* __restrict__ table, const T* __restrict__ pairs, const int* __restrict__ ids,
    const int* __restrict__ positions, const int* __restrict__ token_request, const int* __restrict__ cu_seqlens,
    const int* __restrict__ state_slots, int* __restrict__ last_token, int64_t last_stride, int num_slots,
    float* __restrict__ out, T* __restrict__ cast, int hidden, int vocab, int buckets, int mul_prev, int mul_cur) {
  const int t = blockIdx.x;
  const int id = ids[t];
  const int req = token_request[t];
  const int first = cu_seqlens[req];
  int prev = 0;
  if (t > first) {
    prev = ids[t - 1];
  } else {
    // the step's first token of its request: the token before it is what the last step left,
    // and what this step will leave is written by this same block (read first, then written)
    int slot = state_slots[req];
    if (slot < 0 || slot >= num_slots) slot = num_slots;  // nobody's row
    int* kept = last_token + (int64_t)slot * last_stride;
    prev = kept[0];
    __syncthreads();
    const int last = cu_seqlens[req + 1] - 1;
    if (threadIdx.x == 0 && last >= first) kept[0] = ids[last];
  }
  int64_t row = buckets;
  if (positions[t] > 0) row = ((int64_t)prev * mul_prev + (int64_t)id * mul_cur) % buckets;
  if (row < 0) row += buckets;
  const bool known = id >= 0 && id < vocab;
  const T* a = table + (int64_t)(known ? id : 0) * hidden;
  const T* b = pairs + row * hidden;
  float* o = out + (int64_t)t * hidden;
  for (int c = threadIdx.x * VEC; c < hidden; c += blockDim.x * VEC) {
    float x[VEC], y[VEC];
    mi_load_cols<T, VEC>(a + c, x);
    mi_load_cols<T, VEC>(b + c, y);
#pragma unroll
    for (int j = 0; j < VEC; ++j) x[j] = known ? x[j] + y[j] : 0.f;
    mi_store_cols<float, VEC>(o + c, x);
    if (cast != nullptr) mi_store_cols<T, VEC>(cast + (int64_t)t * hidden + c, x);
  }
}

// ---------------------------------------------------------------------------------------------

template <typename T, int VEC>
__global__ __launch_bounds__(1024) void scale_add_norm_kernel(
    float* __restrict__ stream, const T* __restrict__ y, int64_t y_stride, const float* __restrict__ scale,
    const float* __restrict__ factor, const int* __restrict__ rows, T* __restrict__ cast, int hidden, float alpha,
    float eps) {
  using A = typename WideOf<T>::type;
  __shared__ A scratch[16];
  const int t = rows != nullptr ? rows[blockIdx.x] : blockIdx.x;
  float* x = stream + (int64_t)t * hidden;
  const T* add = y != nullptr ? y + (int64_t)t * y_stride : nullptr;
  // a row is at most a few thousand columns: the sums of a thread's columns stay in registers
  // between the two passes where they fit (4 turns), and are made again where they do not
  constexpr int KEPT = 4;
  A kept[KEPT][VEC];
  A squares = 0;
  int turn = 0;
  for (int c = threadIdx.x * VEC; c < hidden; c += blockDim.x * VEC, ++turn) {
    float v[VEC], u[VEC], s[VEC];
    mi_load_cols<float, VEC>(x + c, v);
    if (add != nullptr) {
      mi_load_cols<T, VEC>(add + c, u);
      if (scale != nullptr) mi_load_cols<float, VEC>(scale + c, s);
    }
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      A sum = (A)v[j];
      if (add != nullptr) sum = (A)alpha * (A)v[j] + (scale != nullptr ? (A)s[j] * (A)u[j] : (A)u[j]);
      if (turn < KEPT) kept[turn][j] = sum;
      squares += sum * sum;
    }
  }
  const A inv = inv_root_of(block_add<A>(squares, scratch) / (A)hidden, (A)eps);
  T* narrow = cast != nullptr ? cast + (int64_t)blockIdx.x * hidden : nullptr;
  turn = 0;
  for (int c = threadIdx.x * VEC; c < hidden; c += blockDim.x * VEC, ++turn) {
    float f[VEC], r[VEC];
    mi_load_cols<float, VEC>(factor + c, f);
    if (turn < KEPT) {
#pragma unroll
      for (int j = 0; j < VEC; ++j) r[j] = (float)((kept[turn][j] * inv) * (A)f[j]);
    } else {
      float v[VEC], u[VEC], s[VEC];
      mi_load_cols<float, VEC>(x + c, v);
      if (add != nullptr) {
        mi_load_cols<T, VEC>(add + c, u);
        if (scale != nullptr) mi_load_cols<float, VEC>(scale + c, s);
      }
#pragma unroll
      for (int j = 0; j < VEC; ++j) {
        A sum = (A)v[j];
        if (add != nullptr) sum = (A)alpha * (A)v[j] + (scale != nullptr ? (A)s[j] * (A)u[j] : (A)u[j]);
        r[j] = (float)((sum * inv) * (A)f[j]);
      }
    }
    if (rows == nullptr) mi_store_cols<float, VEC>(x + c, r);
    if (narrow != nullptr) mi_store_cols<T, VEC>(narrow + c, r);
  }
}

// The routed experts' rows of a token (made [pair][width], expert by expert as expert_combine in routed_experts.hip takes them), which
// are added up here instead of there: y[t] = sum_k weights[t, k] * (row of choice k) + shared_gate[t] * shared[t], rounded to T.
struct ExpertRows {
  const void *made, *x, *shared;
  const int* chosen;
  const float *weights, *shared_gate;
  int64_t x_stride, shared_stride;
  int experts, top;
};

// The same norm with the experts' sum made here.  A row is a chain: the choices, their rows, the squares over the block, the factors, the
// result; few rows (decode) are that chain's time.  So the factors are asked for with the columns, and the turns whose columns are kept are
// counted when compiling, so that their loads are in flight together.  Microseconds of expert_combine and the kernel above / of this / of
// this with the loop above: 2 experts a token, 8 rows of 4096 7.9 / 5.5 / 6.6, 1,501 rows of 3072 19.4 / 12.8 / 13.5.  (Without experts the
// loop above is as fast or faster: 8 rows of 1024 2.9 against 3.2, of 4096 4.4 / 4.2, 1,501 float32 rows of 3072 12.3 / 14.4.)
template <typename T, int VEC>
__global__ __launch_bounds__(1024) void experts_add_norm_kernel(
    float* __restrict__ stream, const float* __restrict__ scale, const float* __restrict__ factor, T* __restrict__ cast, int hidden,
    float alpha, float eps, ExpertRows e) {
  using A = typename WideOf<T>::type;
  __shared__ A scratch[16];
  const int t = blockIdx.x;
  float* x = stream + (int64_t)t * hidden;
  auto sum_at = [&](int c, A (&sum)[VEC]) {
    float v[VEC], u[VEC], s[VEC];
    mi_load_cols<float, VEC>(x + c, v);
    A total[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) total[j] = 0;
    for (int k = 0; k < e.top; ++k) {
      const int64_t pair = (int64_t)t * e.top + k;
      const int chosen = e.chosen[pair];
      if (chosen < 0) continue;
      const T* src = chosen >= e.experts ? (const T*)e.x + (int64_t)t * e.x_stride : (const T*)e.made + pair * hidden;
      mi_load_cols<T, VEC>(src + c, u);
      const A weight = e.weights != nullptr ? (A)e.weights[pair] : (A)1;
#pragma unroll
      for (int j = 0; j < VEC; ++j) total[j] += weight * (A)u[j];
    }
    if (e.shared != nullptr) {
      mi_load_cols<T, VEC>((const T*)e.shared + (int64_t)t * e.shared_stride + c, u);
      const A g = e.shared_gate != nullptr ? (A)e.shared_gate[t] : (A)1;
#pragma unroll
      for (int j = 0; j < VEC; ++j) total[j] += g * (A)u[j];
    }
    if (scale != nullptr) mi_load_cols<float, VEC>(scale + c, s);
#pragma unroll
    for (int j = 0; j < VEC; ++j) {
      const float y = to_f32(from_f32<T>((float)total[j]));
      sum[j] = (A)alpha * (A)v[j] + (scale != nullptr ? (A)s[j] * (A)y : (A)y);
    }
  };
  constexpr int KEPT = 4;
  const int each = blockDim.x * VEC;
  A kept[KEPT][VEC];
  float f[KEPT][VEC];
  A squares = 0;
#pragma unroll
  for (int turn = 0; turn < KEPT; ++turn) {
    const int c = threadIdx.x * VEC + turn * each;
    if (c < hidden) {
      mi_load_cols<float, VEC>(factor + c, f[turn]);
      sum_at(c, kept[turn]);
#pragma unroll
      for (int j = 0; j < VEC; ++j) squares += kept[turn][j] * kept[turn][j];
    }
  }
  for (int c = threadIdx.x * VEC + KEPT * each; c < hidden; c += each) {  // (made again below)
    A sum[VEC];
    sum_at(c, sum);
#pragma unroll
    for (int j = 0; j < VEC; ++j) squares += sum[j] * sum[j];
  }
  const A inv = inv_root_of(block_add_at_once<A>(squares, scratch) / (A)hidden, (A)eps);
  T* narrow = cast != nullptr ? cast + (int64_t)t * hidden : nullptr;
  auto write = [&](int c, const A (&sum)[VEC], const float (&factors)[VEC]) {
    float r[VEC];
#pragma unroll
    for (int j = 0; j < VEC; ++j) r[j] = (float)((sum[j] * inv) * (A)factors[j]);
    mi_store_cols<float, VEC>(x + c, r);
    if (narrow != nullptr) mi_store_cols<T, VEC>(narrow + c, r);
  };
#pragma unroll
  for (int turn = 0; turn < KEPT; ++turn) {
    const int c = threadIdx.x * VEC + turn * each;
    if (c < hidden) write(c, kept[turn], f[turn]);
  }
  for (int c = threadIdx.x * VEC + KEPT * each; c < hidden; c += each) {
    A sum[VEC];
    float factors[VEC];
    sum_at(c, sum);
    mi_load_cols<float, VEC>(factor + c, factors);
    write(c, sum, factors);
  }
}

// ---------------------------------------------------------------------------------------------

template <typename T>
__global__ __launch_bounds__(256) void norm_rows_kernel(const T* __restrict__ in, int64_t in_stride,
                                                        const float* __restrict__ weight, T* __restrict__ out,
                                                        int64_t out_stride, int width, float eps) {
  using A = typename WideOf<T>::type;
  __shared__ A scratch[16];
  const T* x = in + (int64_t)blockIdx.x * in_stride;
  A squares = 0;
  for (int c = threadIdx.x; c < width; c += blockDim.x) {
    const A v = (A)to_f32(x[c]);
    squares += v * v;
  }
  const A inv = inv_root_of(block_add<A>(squares, scratch) / (A)width, (A)eps);
  T* o = out + (int64_t)blockIdx.x * out_stride;
  for (int c = threadIdx.x; c < width; c += blockDim.x)
    o[c] = from_f32<T>((float)(((A)to_f32(x[c]) * inv) * (A)weight[c]));
}

}  // namespace

extern "C" int mi_embed_pair_hash(int dtype, const void* table, const void* pairs, const int* ids, const int* positions,
                                  const int* token_request, const int* cu_seqlens, const int* state_slots,
                                  int* last_token, int64_t last_stride, int num_slots, float* out, void* cast,
                                  int num_tokens, int hidden, int vocab, int buckets, int mul_prev, int mul_cur,
                                  hipStream_t stream) {
  MI_REQUIRE(num_tokens >= 0 && hidden > 0 && vocab > 0 && buckets > 0, "embed_pair_hash: bad sizes tokens=%d hidden=%d vocab=%d buckets=%d",
             num_tokens, hidden, vocab, buckets);
  MI_REQUIRE(last_token != nullptr && last_stride > 0 && num_slots > 0, "embed_pair_hash: the requests' state rows are missing");
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "embed_pair_hash: unknown dtype %d", dtype);
  if (num_tokens == 0) return MI_OK;
  const bool vec = hidden % 4 == 0 && is_aligned16(table) && is_aligned16(pairs) && is_aligned16(out) && is_aligned16(cast);
#define MI_PAIR(T, VEC)                                                                                              \
  embed_pair_hash_kernel<T, VEC><<<num_tokens, 256, 0, stream>>>((const T*)table, (const T*)pairs, ids, positions,   \
                                                                 token_request, cu_seqlens, state_slots, last_token, \
                                                                 last_stride, num_slots, out, (T*)cast, hidden,      \
                                                                 vocab, buckets, mul_prev, mul_cur)
  if (dtype == MI_F32) {
    if (vec) MI_PAIR(float, 4);
    else MI_PAIR(float, 1);
  } else {
    if (vec) MI_PAIR(bf16_t, 4);
    else MI_PAIR(bf16_t, 1);
  }
#undef MI_PAIR
  MI_CHECK_LAUNCH("embed_pair_hash");
  return MI_OK;
}

// `y` (and `scale`) may be null: the norm alone.  `rows` (may be null) lists the rows to norm: the
// stream is then left as it is and `cast` [num_rows, hidden] gets the normed rows in list order.
// made (may be null): the sum of routed experts in y's place (ExpertRows above; y is null then, and rows too).
extern "C" int mi_scale_add_norm(int dtype, float* stream_rows, const void* y, int64_t y_stride, const float* scale,
                                 const float* factor, const int* rows, void* cast, int num_rows, int hidden,
                                 float alpha, float eps, const void* made, const int* chosen, const float* weights, const void* x,
                                 int64_t x_stride, const void* shared, int64_t shared_stride, const float* shared_gate, int experts,
                                 int top, hipStream_t stream) {
  MI_REQUIRE(num_rows >= 0 && hidden > 0 && (y == nullptr || y_stride >= hidden), "scale_add_norm: bad sizes rows=%d hidden=%d stride=%lld",
             num_rows, hidden, (long long)y_stride);
  MI_REQUIRE(factor != nullptr && stream_rows != nullptr, "scale_add_norm: the stream and the norm's factors are needed");
  MI_REQUIRE(rows == nullptr || cast != nullptr, "scale_add_norm: rows picked from the stream need a place to go");
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "scale_add_norm: unknown dtype %d", dtype);
  MI_REQUIRE(made == nullptr || (y == nullptr && rows == nullptr && chosen != nullptr && x != nullptr && x_stride >= hidden && experts > 0 &&
                                 top > 0 && (shared == nullptr || shared_stride >= hidden)),
             "scale_add_norm: experts=%d top=%d strides %lld, %lld", experts, top, (long long)x_stride, (long long)shared_stride);
  if (num_rows == 0) return MI_OK;
  const bool vec = hidden % 4 == 0 && y_stride % 4 == 0 && is_aligned16(stream_rows) && is_aligned16(y) && is_aligned16(scale) &&
                   is_aligned16(factor) && is_aligned16(cast) && is_aligned16(made) && is_aligned16(x) && is_aligned16(shared) &&
                   x_stride % 4 == 0 && shared_stride % 4 == 0;
  const int threads = threads_for(num_rows, vec ? hidden / 4 : hidden);
  const ExpertRows e = {made, x, shared, chosen, weights, shared_gate, x_stride, shared_stride, experts, top};
#define MI_POST(T, VEC)                                                                                                    \
  do {                                                                                                                     \
    if (made != nullptr)                                                                                                   \
      experts_add_norm_kernel<T, VEC><<<num_rows, threads, 0, stream>>>(stream_rows, scale, factor, (T*)cast, hidden, alpha, eps, e); \
    else                                                                                                                   \
      scale_add_norm_kernel<T, VEC><<<num_rows, threads, 0, stream>>>(stream_rows, (const T*)y, y_stride, scale, factor,   \
                                                                      rows, (T*)cast, hidden, alpha, eps);                 \
  } while (0)
  if (dtype == MI_F32) {
    if (vec) MI_POST(float, 4);
    else MI_POST(float, 1);
  } else {
    if (vec) MI_POST(bf16_t, 4);
    else MI_POST(bf16_t, 1);
  }
#undef MI_POST
  MI_CHECK_LAUNCH("scale_add_norm");
  return MI_OK;
}

extern "C" int mi_norm_rows(int dtype, const void* in, int64_t in_stride, const float* weight, void* out,
                            int64_t out_stride, int num_rows, int width, float eps, hipStream_t stream) {
  MI_REQUIRE(num_rows >= 0 && width > 0 && in_stride >= width && out_stride >= width, "norm_rows: bad sizes rows=%d width=%d", num_rows, width);
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "norm_rows: unknown dtype %d", dtype);
  if (num_rows == 0) return MI_OK;
  if (dtype == MI_F32)
    norm_rows_kernel<float><<<num_rows, 256, 0, stream>>>((const float*)in, in_stride, weight, (float*)out, out_stride, width, eps);
  else
    norm_rows_kernel<bf16_t><<<num_rows, 256, 0, stream>>>((const bf16_t*)in, in_stride, weight, (bf16_t*)out, out_stride, width, eps);
  MI_CHECK_LAUNCH("norm_rows");
  return MI_OK;
}
