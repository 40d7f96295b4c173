// Recurrences with a matrix state per head, over many tokens of a request, on the matrix cores.
//
//     S_t = a_t S_(t-1) + k_t u_t^T        o_t = S_t^T q_t        (S is dim x vdim, float32)
//
// Tokens are taken CHUNK at a time.  With G_i the product of a chunk's decays up to its token i (all factors below
// are quotients G_i / G_j with j <= i, so at most 1) and S0 the state before it:
//
//     O = G Q S0 + W U            W_ij = (G_i / G_j) (q_i . k_j)   for j <= i
//     S = G_last S0 + K^T (G_last / G) U
//
// where U's rows are the (scaled) values, or, for the gated delta rule,
//
//     U = T w (V - G K S0)        T = (1 + L)^-1,  L_ij = w_i (G_i / G_j) (k_i . k_j) for j < i.
//
// W, T and the factors do not depend on the state: a first launch makes them for all chunks and heads side by side
// (delta_chunks.hip, decay_chunks.hip).  What is left is a walk over the chunks, here: a block keeps 16 columns of a
// head's S, in the layout in which the matrix instruction leaves its results, which is also the layout of its second
// operand with the rows of S in another order; its 4 waves own a quarter of the rows each, their partial K S0 and
// Q S0 meet in LDS (one barrier a chunk), and everything after that is registers.  All operands are float32 and so is
// the matrix instruction (16x16x4, 154 TFLOP/s): nothing is rounded that the token-by-token form keeps.
//
// What bounds it: the chain of one chunk after another.  Measured at 2,048 tokens, one wave a SIMD: 2.3 us a chunk for
// the delta rule (32 heads of 128 x 128: 68 matrix instructions a wave, 35 cycles each, make 1.0 us of it; the rest is
// the way through LDS and back, and 0.4 us that the loads of the next chunk's operands cost beside it), 1.6 us for the
// others.  A block's loads are limited by what the CU's L1 returns, not by their latency, so what all four waves need (W, T,
// the factors, the values) is brought once, a piece a thread, and goes through LDS under the barrier that is there
// anyway: 187 -> 145 us for the delta rule, 83 -> 70 and 81 -> 72 for the others (3B sizes, 1,777 tokens), against each
// wave loading all of it.  Whole calls with the first launch and the norm, token by token before: delta rule 896 -> 184 us,
// decay per head (64 heads of 128 x 64) 717 -> 117, decay per channel (16 heads of 128 x 256) 774 -> 144.  Waiting for
// everything in flight at the barrier cost 2 us a chunk more.  A chunk of 32: at twice that W and T (quadratic) weigh as much
// as the products with the state, and the inverse no longer stays in a wave's registers.
//
// Only finite numbers may be taken like this: the zeros of W and T above the diagonal make NaN of an infinite value, for
// tokens before it, quotients behind a decay of zero are infinity less infinity, and a chunk's decays together may be zero, which
// makes NaN of an infinite state that each by itself leaves infinite.  Whatever is not finite in the state, the values, the
// gates, and (for the delta rule by itself, else through the factors) in queries and keys stays in S to the end: products with
// zero keep it.  So where a block's S does not end finite it leaves the state as it found it and takes its columns again, token by token (walk_by_token).
// (A launch of their own behind the walk for columns that it had flagged: 4.6 us of every call.  Three prompts of 80 tokens, 12 layers, 2,165 / 2,126 us, of
// 67 at 8B widths 4,135 / 4,090, one token beside 144 1,548 / 1,530.)  The barrier at a block's end costs 0.3 us;
// sums of what a chunk adds and of Q S0, the same in all waves and without a barrier, cost more (77.6 us for the 70 of a decay per head).
#pragma once
#include "common.h"

#define CHUNK 32

namespace chunk_scan {

enum { PER_CHANNEL = 0, PER_HEAD = 1, DELTA = 2 };

typedef float f32x4_t __attribute__((ext_vector_type(4)));

// What the first launch leaves, per chunk (a request's chunks lie one after another from `first_chunk` on).
struct Made {
  float* q;       // [chunks][shares][CHUNK][pad]; PER_CHANNEL: times G_i
  float* k;       // the same (DELTA only)
  float* kt;      // [chunks][shares][pad][CHUNK]; PER_CHANNEL: times G_last / G_j
  float* within;  // W [chunks][heads][CHUNK][CHUNK]; PER_HEAD: for U = V, its columns times the step sizes
  float* solve;   // T w, the same (DELTA only)
  float* factor;  // G, and G_last / G (PER_HEAD: times the step sizes, NaN of a token whose query or key is not finite)
                  // [chunks][heads][2][CHUNK]; not PER_CHANNEL
  float* fade;    // G_last: PER_CHANNEL [chunks][heads][pad]; NaN where a query, key or decay of the chunk is not finite
  int shares;     // rows q and k are shared by heads / shares heads
};

// The chunk number of a request's first chunk: requests' chunks never meet, since b + cu[b] / CHUNK grows by at least
// the chunks of request b from one request to the next.
__device__ __forceinline__ int first_chunk(int cu_b, int b) { return cu_b / CHUNK + b; }
static inline int64_t chunk_count(int tokens, int requests) { return (int64_t)tokens / CHUNK + requests; }

// Of a request's only token the first launch leaves what walk_one_token reads and nothing else: row 0 of q and k (without DELTA: k as row 1 of q), the
// first value of W, of T w and of both factors, and the fade.  One thread a channel makes it.
//
// The sums over a block of 256 threads, the same in all of them; `scratch`: 4 * N floats.
template <int N>
__device__ __forceinline__ void sum_of_block(float (&v)[N], float* scratch) {
#pragma unroll
  for (int i = 0; i < N; ++i) {
#pragma unroll
    for (int off = 1; off < MI_WAVE; off <<= 1) v[i] += __shfl_xor(v[i], off, MI_WAVE);
    if (threadIdx.x % MI_WAVE == 0) scratch[threadIdx.x / MI_WAVE * N + i] = v[i];
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] = (scratch[i] + scratch[N + i]) + (scratch[2 * N + i] + scratch[3 * N + i]);
}

// Which request a chunk number belongs to: all threads of the block call this; -1: no request's.
__device__ __forceinline__ int request_of_chunk(int chunk, const int* __restrict__ cu, int requests, int* shared_answer) {
  if (threadIdx.x == 0) *shared_answer = -1;
  __syncthreads();
  for (int b = threadIdx.x; b < requests; b += blockDim.x) {
    const int first = first_chunk(cu[b], b), tokens = cu[b + 1] - cu[b];
    if (chunk >= first && chunk < first + (tokens + CHUNK - 1) / CHUNK) *shared_answer = b;
  }
  __syncthreads();
  return *shared_answer;
}

// N values of a row from `at` on as float32, zeros from `dim` on (or all of them); `eights`: rows lie on 16 bytes in whole 8s.
template <int N>
__device__ __forceinline__ void row_values(const bf16_t* row, int at, int dim, bool eights, bool in, float (&v)[N]) {
  static_assert(N % 8 == 0, "eight values a load");
  if (eights) {
#pragma unroll
    for (int e = 0; e < N; e += 8) {
      const bool has = in && at + e < dim;
      const uint4 got = *reinterpret_cast<const uint4*>(row + (at + e < dim ? at + e : 0));
      const uint32_t keep = has ? ~0u : 0u;
      const uint32_t words[4] = {got.x & keep, got.y & keep, got.z & keep, got.w & keep};
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        v[e + 2 * w] = __uint_as_float(words[w] << 16);
        v[e + 2 * w + 1] = __uint_as_float(words[w] & 0xFFFF0000u);
      }
    }
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) v[e] = in && at + e < dim ? to_f32(row[at + e]) : 0.f;
  }
}
static inline bool in_eights(const void* rows, int64_t stride, int64_t column, int dim) {
  return (uintptr_t)rows % 16 == 0 && stride % 8 == 0 && column % 8 == 0 && dim % 8 == 0;
}

struct WalkArgs {
  Made made;
  const bf16_t* v;  // value rows
  int64_t v_stride;  // under MAX_ROW values: offsets inside a chunk are 32-bit
  int v_col;  // first column of head 0
  const float* skip;  // PER_HEAD: per head, times the value, added to the read-out; may be null
  float* state;       // [slots + 1][heads][vdim][pad]
  int64_t state_stride;
  const int *cu, *slots;
  int num_slots;
  float* out;  // float32 [tokens, heads * vdim]
  int heads, vdim;
};
constexpr int64_t MAX_ROW = 1 << 24;

__device__ __forceinline__ f32x4_t mma(float a, float b, f32x4_t acc) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, acc, 0, 0, 0); }
__device__ __forceinline__ f32x4_t mma4(const float4& a, const f32x4_t& b, f32x4_t acc) {
  acc = mma(a.x, b[0], acc), acc = mma(a.y, b[1], acc), acc = mma(a.z, b[2], acc);
  return mma(a.w, b[3], acc);
}
__device__ __forceinline__ float4 load4(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ f32x4_t scaled(const float4& s, const f32x4_t& v) { return f32x4_t{s.x * v[0], s.y * v[1], s.z * v[2], s.w * v[3]}; }

// A barrier for LDS alone: __syncthreads() would also wait for the next chunk's operands, which are in flight (5.3 us a
// chunk with it).
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One chunk's operands on their way, in a thread's registers.  Rows of S of the wave's own, in the order of the matrix
// instruction's operands: row tiles t of 16 tokens, token 16 t + lane % 16 and four rows of S (or, of kt, a row of S and four
// tokens) side by side.  What all waves read: a piece of it, which goes through LDS.
template <int DT, int MODE>
struct Operands {
  float4 q[2][DT], k[MODE == DELTA ? 2 : 1][DT], kt[2][DT];
  float4 fade[MODE == PER_CHANNEL ? DT : 1];
  float4 within, solve;  // four values of a row of W and of T
  float factor;          // one of the 64 factors
  uint32_t v[2];         // two columns of a token's values, as read
};

// What the block's waves share of a chunk.  (Rows of 36: 16-byte reads of 16 rows fall on different banks.)
constexpr int LDS_ROW = CHUNK + 4;
template <int MODE>
struct Shared {
  float within[CHUNK * LDS_ROW];
  float solve[MODE == DELTA ? CHUNK * LDS_ROW : 4];
  float v[16 * LDS_ROW];  // [column][token]
  float factor[2 * CHUNK];
};

// A request's only token, for G column blocks of 16 at once: bound by the state's bytes, and as a chunk of one token a block had 8 KB of them on the way
// while it brought in 40 KB of operands.  Every wave keeps its rows of S as in the walk.  Steps with single tokens beside a long portion, all of them in chunks
// / so: 34 and 500 of the delta rule with 32 heads of 128 x 128 (12 layers, half of them of the rule) 5,625 / 5,036 us, 25 and 400 with 24 heads 3,278 / 2,902, 34 and 700
// with 64 heads of 128 x 64 8,551 / 7,847 (the long portion's blocks first in both: before that 8,847).
// Returns the column blocks that did not end finite and whose state is as it was, a bit each.
template <int DT, int MODE, int G>
__device__ __forceinline__ int walk_one_token(const WalkArgs& p, float* sums, int b, int first, int head, int block0) {
  constexpr int PAD = 64 * DT;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), lane = threadIdx.x % MI_WAVE;
  const int r = lane % 16, quad = lane / 16, row0 = 16 * DT * wave + 4 * quad;
  const int slot = p.slots[b];
  const bool kept = slot >= 0 && slot < p.num_slots;
  float* state = p.state + (int64_t)(kept ? slot : p.num_slots) * p.state_stride + (int64_t)head * p.vdim * PAD + row0;
  const int64_t chunk = first_chunk(first, b), rows = chunk * p.made.shares + head / (p.heads / p.made.shares), of = chunk * p.heads + head;
  f32x4_t S[G][DT];
  float v[G];
  const bf16_t* v_row = p.v + (int64_t)first * p.v_stride + p.v_col + (int64_t)head * p.vdim;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const int col = min((block0 + g) * 16 + r, p.vdim - 1);  // (past the last column: that one again, not written)
#pragma unroll
    for (int d = 0; d < DT; ++d) S[g][d] = *reinterpret_cast<const f32x4_t*>(state + (int64_t)col * PAD + 16 * d);
    v[g] = to_f32(v_row[col]);
  }
  float4 q[DT], k[DT], fade[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) {
    q[d] = load4(p.made.q + rows * CHUNK * PAD + row0 + 16 * d);
    k[d] = load4((MODE == DELTA ? p.made.k : p.made.q + PAD) + rows * CHUNK * PAD + row0 + 16 * d);
    if constexpr (MODE == PER_CHANNEL) fade[d] = load4(p.made.fade + of * PAD + row0 + 16 * d);
  }
  const float* factor = p.made.factor + of * 2 * CHUNK;
  const float decay = MODE == PER_CHANNEL ? 1.f : factor[0], tail = MODE == PER_CHANNEL ? 1.f : factor[CHUNK];
  const float within = p.made.within[of * CHUNK * CHUNK], solve = MODE == DELTA ? p.made.solve[of * CHUNK * CHUNK] : 1.f;
  const float skip = (MODE == PER_HEAD && p.skip) ? p.skip[head] : 0.f;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    float qs = 0.f, ks = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      qs = fmaf(q[d].x, S[g][d][0], fmaf(q[d].y, S[g][d][1], fmaf(q[d].z, S[g][d][2], fmaf(q[d].w, S[g][d][3], qs))));
      if constexpr (MODE == DELTA) ks = fmaf(k[d].x, S[g][d][0], fmaf(k[d].y, S[g][d][1], fmaf(k[d].z, S[g][d][2], fmaf(k[d].w, S[g][d][3], ks))));
    }
#pragma unroll
    for (int off = 16; off < MI_WAVE; off <<= 1) {
      qs += __shfl_xor(qs, off, MI_WAVE);
      if constexpr (MODE == DELTA) ks += __shfl_xor(ks, off, MI_WAVE);
    }
    if (quad == 0) {
      sums[(wave * G + g) * 32 + r] = qs;
      if constexpr (MODE == DELTA) sums[(wave * G + g) * 32 + 16 + r] = ks;
    }
  }
  __syncthreads();
  int odd = 0;  // column blocks that do not end finite, a bit each
#pragma unroll
  for (int g = 0; g < G; ++g) {
    auto whole = [&](int at) { return (sums[g * 32 + at] + sums[(G + g) * 32 + at]) + (sums[(2 * G + g) * 32 + at] + sums[(3 * G + g) * 32 + at]); };
    float u = v[g];
    if constexpr (MODE == DELTA) u = solve * (u - decay * whole(16 + r));
    const float add = MODE == PER_CHANNEL ? u : tail * u;
    float zeros = 0.f;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if constexpr (MODE == PER_CHANNEL) S[g][d] = scaled(fade[d], S[g][d]);
      else S[g][d] *= decay;
      S[g][d] = f32x4_t{fmaf(k[d].x, add, S[g][d][0]), fmaf(k[d].y, add, S[g][d][1]), fmaf(k[d].z, add, S[g][d][2]), fmaf(k[d].w, add, S[g][d][3])};
#pragma unroll
      for (int e = 0; e < 4; ++e) zeros = fmaf(0.f, S[g][d][e], zeros);
    }
    odd |= (__ballot(!(zeros == 0.f)) != 0) << g;
    const int col = (block0 + g) * 16 + r;
    if (wave * 4 + quad == g && col < p.vdim) {
      float read = fmaf(within, u, decay * whole(r));
      if constexpr (MODE == PER_HEAD) read = fmaf(skip, v[g], read);
      p.out[(int64_t)first * p.heads * p.vdim + (int64_t)head * p.vdim + col] = read;
    }
  }
  __syncthreads();  // (the sums have been read)
  int* odd_of = reinterpret_cast<int*>(sums);
  if (lane == 0) odd_of[wave] = odd;
  __syncthreads();
  odd = (odd_of[0] | odd_of[1]) | (odd_of[2] | odd_of[3]);
  if (kept) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int col = (block0 + g) * 16 + r;
      if (col >= p.vdim || (odd >> g & 1)) continue;
#pragma unroll
      for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4_t*>(state + (int64_t)col * PAD + 16 * d) = S[g][d];
    }
  }
  return odd;
}

// One wave a SIMD walks, so what a chunk costs is what a wave issues: addresses are a base that is the same for the wave plus a lane's offset made
// once, without branches (at the end of one everything in flight would be waited for) and multiplications.
// Returns whether S did not end finite; the state is then as it was.
template <int DT, int MODE>
__device__ __forceinline__ bool walk_portion(const WalkArgs& p, f32x4_t (*parts)[4][MODE == DELTA ? 4 : 2][MI_WAVE], Shared<MODE>* shared, int b, int first, int last,
                                             int head, int block) {
  constexpr int PAD = 64 * DT;
  constexpr int SUMS = MODE == DELTA ? 4 : 2;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), lane = threadIdx.x % MI_WAVE;
  const uint32_t r = lane % 16, quad = lane / 16;
  const int col = block * 16 + r;
  const bool live = col < p.vdim;
  const int slot = p.slots[b];
  const int row0 = 16 * DT * wave;  // of S
  const bool kept = live && slot >= 0 && slot < p.num_slots;  // (without a slot: from the spare row, which stays as it is)
  float* mine = p.state + (int64_t)(kept ? slot : p.num_slots) * p.state_stride + ((int64_t)head * p.vdim + (live ? col : 0)) * PAD + row0 + 4 * quad;
  f32x4_t S[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) S[d] = live ? *reinterpret_cast<const f32x4_t*>(mine + 16 * d) : f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int share = head / (p.heads / p.made.shares);
  const int chunk0 = first_chunk(first, b), chunks = (last - first + CHUNK - 1) / CHUNK;
  const float skip = (MODE == PER_HEAD && p.skip) ? p.skip[head] : 0.f;
  const int out_stride = p.heads * p.vdim;
  // a lane's offsets
  const uint32_t at_row = r * PAD + 4 * quad, at_column = r * CHUNK + 4 * quad, in_lds = r * LDS_ROW + 4 * quad;
  uint32_t out_at[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) out_at[e] = (16 * (wave & 1) + 4 * quad + e) * (uint32_t)out_stride + (uint32_t)col;
  // values a thread brings: token 8 * wave + lane / 8 of the chunk, columns lane % 8 and 8 further
  const uint32_t v_token = 8 * wave + lane / 8, v_at = v_token * (uint32_t)p.v_stride;
  const uint32_t v_first = (uint32_t)min((int)(col - r) + lane % 8, p.vdim - 1), v_second = (uint32_t)min((int)(col - r) + lane % 8 + 8, p.vdim - 1);

  auto fetch = [&](int n, Operands<DT, MODE>& o) {
    const int64_t chunk = chunk0 + n, rows = chunk * p.made.shares + share, of = chunk * p.heads + head;
    const float *q = p.made.q + rows * CHUNK * PAD + row0, *kt = p.made.kt + rows * PAD * CHUNK + row0 * CHUNK;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        o.q[t][d] = load4(q + 16 * t * PAD + 16 * d + at_row);
        o.kt[t][d] = load4(kt + 16 * d * CHUNK + 16 * t + at_column);
      }
    if constexpr (MODE == DELTA) {
      const float* k = p.made.k + rows * CHUNK * PAD + row0;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int d = 0; d < DT; ++d) o.k[t][d] = load4(k + 16 * t * PAD + 16 * d + at_row);
      o.solve = load4(p.made.solve + of * CHUNK * CHUNK + 4 * threadIdx.x);
    }
    o.within = load4(p.made.within + of * CHUNK * CHUNK + 4 * threadIdx.x);
    if constexpr (MODE == PER_CHANNEL) {
      const float* fade = p.made.fade + of * PAD + row0;
#pragma unroll
      for (int d = 0; d < DT; ++d) o.fade[d] = load4(fade + 16 * d + 4 * quad);
    } else {
      o.factor = p.made.factor[of * 2 * CHUNK + lane];
    }
    // (of tokens past the last one the last one's; the rest of the request may be more rows than 32 bits reach over)
    const int t0 = first + n * CHUNK;
    const bf16_t* v = p.v + (int64_t)t0 * p.v_stride + p.v_col + (int64_t)head * p.vdim;
    const uint32_t v_row = min(v_at, (uint32_t)min(CHUNK - 1, last - 1 - t0) * (uint32_t)p.v_stride);
    o.v[0] = *reinterpret_cast<const uint16_t*>(v + (v_row + v_first));
    o.v[1] = *reinterpret_cast<const uint16_t*>(v + (v_row + v_second));
  };
  auto step = [&](int n, const Operands<DT, MODE>& o) {
    const int nt = last - first - n * CHUNK;
    const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
    f32x4_t sum[SUMS];
#pragma unroll
    for (int t = 0; t < SUMS; ++t) sum[t] = zero;
#pragma unroll
    for (int d = 0; d < DT; ++d)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        sum[t] = mma4(o.q[t][d], S[d], sum[t]);
        if constexpr (MODE == DELTA) sum[2 + t] = mma4(o.k[t][d], S[d], sum[2 + t]);
      }
    // (two buffers: a wave that runs ahead writes the other one, and cannot pass the next barrier)
#pragma unroll
    for (int t = 0; t < SUMS; ++t) parts[n & 1][wave][t][lane] = sum[t];
    Shared<MODE>& both = shared[n & 1];
    const int piece = threadIdx.x / 8 * LDS_ROW + threadIdx.x % 8 * 4;
    *reinterpret_cast<float4*>(&both.within[piece]) = o.within;
    if constexpr (MODE == DELTA) *reinterpret_cast<float4*>(&both.solve[piece]) = o.solve;
    if constexpr (MODE != PER_CHANNEL) {
      if (wave == 0) both.factor[lane] = o.factor;
    }
    {  // (of tokens past the last one zeros, by their bits: a choice would be compiled into a branch around the load, and every
       // load waited for by itself)
      const uint32_t keep = (int)v_token < nt ? 0xFFFF0000u : 0u;
      both.v[lane % 8 * LDS_ROW + v_token] = __uint_as_float((o.v[0] << 16) & keep);
      both.v[(lane % 8 + 8) * LDS_ROW + v_token] = __uint_as_float((o.v[1] << 16) & keep);
    }
    lds_barrier();
    f32x4_t v[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) v[t] = *reinterpret_cast<const f32x4_t*>(&both.v[in_lds + 16 * t]);
    float4 g[2], tails[2];
    float g_last = 1.f;
    if constexpr (MODE != PER_CHANNEL) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        g[t] = load4(&both.factor[16 * t + 4 * quad]);
        tails[t] = load4(&both.factor[CHUNK + 16 * t + 4 * quad]);
      }
      g_last = both.factor[CHUNK - 1];
    }
    auto whole = [&](int t) {
      return (parts[n & 1][0][t][lane] + parts[n & 1][1][t][lane]) + (parts[n & 1][2][t][lane] + parts[n & 1][3][t][lane]);
    };
    f32x4_t u[2] = {v[0], v[1]};
    if constexpr (MODE == DELTA) {
#pragma unroll
      for (int t = 0; t < 2; ++t) u[t] -= scaled(g[t], whole(2 + t));
      const f32x4_t upper = mma4(load4(&both.solve[in_lds]), u[0], zero), lower = mma4(load4(&both.solve[16 * LDS_ROW + in_lds]), u[0], zero);
      u[1] = lower + mma4(load4(&both.solve[16 * LDS_ROW + 16 + in_lds]), u[1], zero);
      u[0] = upper;
    }
    f32x4_t tail[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) {
      if constexpr (MODE == PER_CHANNEL) tail[t] = u[t];
      else tail[t] = scaled(tails[t], u[t]);
    }
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      if constexpr (MODE == PER_CHANNEL) S[d] = scaled(o.fade[d], S[d]);
      else S[d] *= g_last;
    }
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int d = 0; d < DT; ++d) S[d] = mma4(o.kt[t][d], tail[t], S[d]);
    if (wave < 2) {
      f32x4_t read = whole(wave);
      if constexpr (MODE != PER_CHANNEL) read = scaled(wave == 1 ? g[1] : g[0], read);
      const float* within = &both.within[16 * wave * LDS_ROW + in_lds];
      read += mma4(load4(within), u[0], zero);
      if (wave == 1) read += mma4(load4(within + 16), u[1], zero);
      if constexpr (MODE == PER_HEAD) read += skip * (wave == 0 ? v[0] : v[1]);
      float* out = p.out + (int64_t)(first + n * CHUNK) * out_stride + (int64_t)head * p.vdim;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if ((int)(16 * wave + 4 * quad + e) < nt && live) out[out_at[e]] = read[e];
    }
  };
  // (two sets of operands: with a third, two chunks ahead, 162 us instead of 145)
  Operands<DT, MODE> even, odd;
  fetch(0, even);
  for (int n = 0; n + 1 < chunks; n += 2) {
    fetch(n + 1, odd);
    step(n, even);
    fetch(min(n + 2, chunks - 1), even);
    step(n + 1, odd);
  }
  if (chunks & 1) step(chunks - 1, even);
  f32x4_t zeros = {0.f, 0.f, 0.f, 0.f};  // unless something is not finite
#pragma unroll
  for (int d = 0; d < DT; ++d) zeros += 0.f * S[d];
  const bool again = __syncthreads_or(!((zeros[0] + zeros[1]) + (zeros[2] + zeros[3]) == 0.f));
  if (kept && !again) {
#pragma unroll
    for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4_t*>(mine + 16 * d) = S[d];
  }
  return again;
}

// 16 columns token by token, for what is not finite: 16 lanes a column, 4 * DT rows a lane, in the arithmetic of the token-by-token kernels.  Tokens go in tiles
// through LDS (`room`, the walk's own), the threads side by side along the channels, and a token's operands are read one token ahead.  The next tile is not
// asked for while one is walked, and few of a tile's values at a time: it is the registers of the whole kernel, and with them the waves on a CU, that this must not
// raise (the next tile in registers: 3 waves a SIMD instead of 4 with a decay per channel of 64).  Microseconds of a scan, 2,048 tokens with a NaN, as a launch of the
// token-by-token kernels behind the walk / here with every lane reading and making its operands itself / so: delta rule, 32 heads of 128 x 128 1,103 / 2,699 / 1,062, 8 of
// 256 x 256 1,606 / 9,342 / 1,722; a decay per head, 48 of 128 x 64 927 / 2,297 / 824; per channel, 12 of 128 x 256 984 / 4,713 / 879, 8 of 256 x 256 1,551 / 13,422 / 1,659.
// TokenRows in the .hip files: what a token's operands are.
template <int CTRL>
__device__ __forceinline__ float lane_moved(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
__device__ __forceinline__ float sum_of_16(float v) {  // (neighbours, pairs, the mirror images inside 8 and inside 16 lanes)
  v += lane_moved<0xB1>(v);
  v += lane_moved<0x4E>(v);
  v += lane_moved<0x141>(v);
  return v + lane_moved<0x140>(v);
}

template <int DT, int MODE>
struct TokenTile {
  static constexpr int TOKENS = 32 / DT;
  float q[TOKENS * 64 * DT], k[TOKENS * 64 * DT], a[MODE == PER_CHANNEL ? TOKENS * 64 * DT : 4];
  float v[TOKENS][16], decay[TOKENS], step[TOKENS];
};

template <int DT, int MODE, typename Rows>
__device__ __forceinline__ void walk_by_token(const WalkArgs& p, const Rows& rows, TokenTile<DT, MODE>& room, int b, int first, int last, int head, int block) {
  constexpr int R = 4 * DT, PAD = 64 * DT, TOKENS = TokenTile<DT, MODE>::TOKENS;
  const int part = threadIdx.x % 16, column = threadIdx.x / 16, col = block * 16 + column, slot = p.slots[b];
  const bool live = col < p.vdim, kept = live && slot >= 0 && slot < p.num_slots;
  float* mine = p.state + (int64_t)(kept ? slot : p.num_slots) * p.state_stride + ((int64_t)head * p.vdim + (live ? col : p.vdim - 1)) * PAD + part * R;
  f32x4_t S[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) S[d] = *reinterpret_cast<const f32x4_t*>(mine + 4 * d);
  const float skip = (MODE == PER_HEAD && p.skip) ? p.skip[head] : 0.f;
  struct Of {
    float4 q[DT], k[DT], a[MODE == PER_CHANNEL ? DT : 1];
    float x, decay, step;
  };
  auto read = [&](int i) {
    Of o;
#pragma unroll
    for (int d = 0; d < DT; ++d) {
      o.q[d] = load4(&room.q[i * PAD + part * R + 4 * d]);
      o.k[d] = load4(&room.k[i * PAD + part * R + 4 * d]);
      if constexpr (MODE == PER_CHANNEL) o.a[d] = load4(&room.a[i * PAD + part * R + 4 * d]);
    }
    o.x = room.v[i][column], o.decay = MODE == PER_CHANNEL ? 1.f : room.decay[i], o.step = MODE == PER_CHANNEL ? 1.f : room.step[i];
    return o;
  };
  for (int t0 = first; t0 < last; t0 += TOKENS) {
    const int n = min(TOKENS, last - t0);
    lds_barrier();  // the last tile, or what stood here before it, has been read
    {
      const int d = threadIdx.x % PAD, from = min(d, rows.width() - 1);  // (past the last channel that one again, as zeros)
#pragma unroll 4
      for (int token = threadIdx.x / PAD; token < TOKENS; token += 256 / PAD) {  // (past the last token that one again)
        const int64_t t = t0 + min(token, n - 1);
        float q, k;
        rows.channel(t, head, p.heads, from, q, k);
        room.q[token * PAD + d] = d == from ? q : 0.f, room.k[token * PAD + d] = d == from ? k : 0.f;
        if constexpr (MODE == PER_CHANNEL) room.a[token * PAD + d] = rows.channel_gate(t, head, from);
      }
      if constexpr (MODE == PER_CHANNEL) {  // (the gates that this thread has left)
        const float bias = rows.channel_bias(head, from);
#pragma unroll 2
        for (int token = threadIdx.x / PAD; token < TOKENS; token += 256 / PAD) {
          const float a = rows.channel_decay(room.a[token * PAD + d] + bias);
          room.a[token * PAD + d] = d == from ? a : 0.f;
        }
      } else if (threadIdx.x < n) {
        rows.head_gates(t0 + threadIdx.x, head, room.decay[threadIdx.x], room.step[threadIdx.x]);
      }
      for (int token = column; token < n; token += 16)
        room.v[token][part] = to_f32(p.v[(int64_t)(t0 + token) * p.v_stride + p.v_col + (int64_t)head * p.vdim + min(block * 16 + part, p.vdim - 1)]);
    }
    lds_barrier();
    if constexpr (MODE == DELTA) {  // unit vectors: 8 * DT lanes a token, 8 channels a lane
      float *q = &room.q[threadIdx.x * 8], *k = &room.k[threadIdx.x * 8], qq = 0.f, kk = 0.f;
#pragma unroll
      for (int i = 0; i < 8; ++i) qq = fmaf(q[i], q[i], qq), kk = fmaf(k[i], k[i], kk);
#pragma unroll
      for (int off = 1; off < 8 * DT; off <<= 1) qq += __shfl_xor(qq, off, MI_WAVE), kk += __shfl_xor(kk, off, MI_WAVE);
      const float q_inv = rsqrtf(qq + 1e-6f) * (1.0f / sqrtf((float)rows.width())), k_inv = rsqrtf(kk + 1e-6f);
#pragma unroll
      for (int i = 0; i < 8; ++i) q[i] *= q_inv, k[i] *= k_inv;
      lds_barrier();
    }
    Of now = read(0);
    for (int i = 0; i < n; ++i) {
      const Of next = read(min(i + 1, n - 1));
      float u = now.step * now.x;
      if constexpr (MODE == DELTA) {
        float seen = 0.f;
#pragma unroll
        for (int d = 0; d < DT; ++d) seen = fmaf(S[d][0], now.k[d].x, fmaf(S[d][1], now.k[d].y, fmaf(S[d][2], now.k[d].z, fmaf(S[d][3], now.k[d].w, seen))));
        u = now.step * (now.x - sum_of_16(seen) * now.decay);
      }
      float out = 0.f;
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const float4 a = MODE == PER_CHANNEL ? now.a[d] : make_float4(now.decay, now.decay, now.decay, now.decay);
        S[d] = f32x4_t{fmaf(now.k[d].x, u, a.x * S[d][0]), fmaf(now.k[d].y, u, a.y * S[d][1]), fmaf(now.k[d].z, u, a.z * S[d][2]), fmaf(now.k[d].w, u, a.w * S[d][3])};
        out = fmaf(S[d][0], now.q[d].x, fmaf(S[d][1], now.q[d].y, fmaf(S[d][2], now.q[d].z, fmaf(S[d][3], now.q[d].w, out))));
      }
      out = sum_of_16(out);
      if constexpr (MODE == PER_HEAD) out = fmaf(skip, now.x, out);
      if (part == 0 && live) p.out[((int64_t)(t0 + i) * p.heads + head) * p.vdim + col] = out;
      now = next;
    }
  }
  if (kept) {
#pragma unroll
    for (int d = 0; d < DT; ++d) *reinterpret_cast<f32x4_t*>(mine + 4 * d) = S[d];
  }
}

// The item-th piece of work of a launch: requests of several tokens first, a piece a head and block of 16 columns (the heads side by side, so that an XCD's
// blocks share their chunk data), then the others, a piece a head and TOGETHER column blocks; each from the last request on, as a step's long portion
// commonly comes last and its chain should not begin when everything else is done (20 single tokens beside 555 of 32 heads of 128 x 64: 55 us, so 38).
// False: there are fewer.  All lanes get the same answer.
struct Piece {
  int b, first, last, head, block;
};
__device__ __forceinline__ bool find_piece(const int* __restrict__ cu, int requests, int heads, int many_each, int one_each, int together, int item, Piece& piece) {
  const int lane = threadIdx.x % MI_WAVE;
  int many = 0, from = 0, first = 0, last = 0;
  auto load = [&](int base) {  // (up to 64 requests: once)
    from = base;
    const int b = requests - 1 - base - lane;
    first = b >= 0 ? cu[b] : 0, last = b >= 0 ? cu[b + 1] : 0;
  };
  load(0);
  auto find = [&](bool of_many, int which) {  // request number `which` of its kind from the last on
    for (int base = 0; base < requests; base += MI_WAVE) {
      if (base != from) load(base);
      const bool is = requests - 1 - base - lane >= 0 && (last - first > 1) == of_many;
      const uint64_t mask = __ballot(is);
      const int count = __popcll(mask);
      if (of_many) many += count;
      if (which < count) {
        const int at = __ffsll(__ballot(is && (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0)) == which)) - 1;
        piece.b = requests - 1 - base - at;
        piece.first = __builtin_amdgcn_readlane(first, at);
        piece.last = __builtin_amdgcn_readlane(last, at);
        return true;
      }
      which -= count;
    }
    return false;
  };
  if (find(true, item / many_each)) {
    piece.head = item % many_each % heads, piece.block = item % many_each / heads;
    return true;
  }
  item -= many * many_each;
  piece.head = item % one_each % heads, piece.block = item % one_each / heads * together;
  return find(false, item / one_each);
}

// 256 threads.  DT: 16-row tiles of S a wave keeps; pad = 64 * DT.  grid: heads * column blocks, requests; or, where most requests are known to bring one
// token (launch_walk), as many blocks as there are pieces of work, of which a block takes every gridDim.x-th.  (Blocks that find nothing to do are not
// free: each waits for the place of one that works.  31 single tokens beside 64, a block for each request / for each piece: a decay per channel, 16 heads of
// 128 x 256 66.5 / 54, 8 heads 62.7 / 41; delta rule, 24 heads of 128 x 128 52.2 / 47.6, 8 of 256 x 256 124 / 64, 32 of 128 x 128 55 / 56; a decay per head, 64
// heads of 128 x 64 43 / 45.  The search costs 1 us.)
template <int DT, int MODE, bool SEARCH, typename Rows>
__global__ __launch_bounds__(256, MODE == DELTA || DT > 2 ? 1 : 2) void walk_kernel(WalkArgs p, Rows rows, int requests) {
  constexpr int TOGETHER = MODE == DELTA ? 8 : 4;
  struct Walked {
    f32x4_t parts[2][4][MODE == DELTA ? 4 : 2][MI_WAVE];
    Shared<MODE> shared[2];
  };
  __shared__ __align__(16) unsigned char room[sizeof(Walked)];
  Walked& walked = *reinterpret_cast<Walked*>(room);
  static_assert(sizeof(walked.parts) >= sizeof(float) * 4 * TOGETHER * 32 && sizeof(TokenTile<DT, MODE>) <= sizeof(Walked), "single tokens' sums and tiles of tokens fit");
  const int blocks = (p.vdim + 15) / 16;
  auto make = [&](const Piece& at) {
    int odd = 0;
    if (at.last - at.first > 1) odd = walk_portion<DT, MODE>(p, walked.parts, walked.shared, at.b, at.first, at.last, at.head, at.block);
    else if (at.last - at.first == 1 && at.block % TOGETHER == 0)
      odd = walk_one_token<DT, MODE, TOGETHER>(p, reinterpret_cast<float*>(room), at.b, at.first, at.head, at.block);
    for (int g = 0; odd >> g != 0; ++g)
      if ((odd >> g & 1) && at.block + g < blocks)
        walk_by_token<DT, MODE>(p, rows, *reinterpret_cast<TokenTile<DT, MODE>*>(room), at.b, at.first, at.last, at.head, at.block + g);
  };
  Piece at;
  if constexpr (SEARCH) {
    const int one_each = p.heads * ((blocks + TOGETHER - 1) / TOGETHER);
    for (int item = blockIdx.x; find_piece(p.cu, requests, p.heads, p.heads * blocks, one_each, TOGETHER, item, at); item += gridDim.x) {
      if (item != (int)blockIdx.x) __syncthreads();  // (the last piece's sums have been read)
      make(at);
    }
  } else {
    at.b = requests - 1 - (int)blockIdx.y, at.head = blockIdx.x % p.heads, at.block = blockIdx.x / p.heads;
    at.first = p.cu[at.b], at.last = p.cu[at.b + 1];
    make(at);
  }
}

template <int MODE, typename Rows>
static int launch_walk(const WalkArgs& p, const Rows& rows, int pad, int tokens, int requests, int longest, hipStream_t stream) {
  constexpr int TOGETHER = MODE == DELTA ? 8 : 4;
  const int blocks = ceil_div(p.vdim, 16), others = requests - 1;
  // requests of several tokens: where every one brings a token those that bring more; not known: as if there were one long portion, with a few
  // rounds of blocks in case there are more
  const int many = longest == 1 ? requests : longest == 0 ? 1 : 1 + max(0, min(others, tokens - longest - others));
  const int64_t all = (int64_t)requests * p.heads * blocks, a_few_rounds = 8 * mi_compute_units();
  const int64_t pieces = (int64_t)p.heads * ((int64_t)many * blocks + (int64_t)(requests - many) * ceil_div(blocks, TOGETHER));
  MI_REQUIRE(all < ((int64_t)1 << 30), "chunk_walk: %d requests of %d heads", requests, p.heads);
  // (a decay per head, and the delta rule where a request has a block for each compute unit, are as fast or up to 5 % faster with a block for each request)
  constexpr bool SEARCHED = MODE != PER_HEAD;
  const bool search = SEARCHED && (MODE == PER_CHANNEL || p.heads * blocks < mi_compute_units()) && many < requests && all > a_few_rounds;
  const dim3 grid = search ? dim3((unsigned)(longest == 0 ? max(pieces, a_few_rounds) : pieces)) : dim3(p.heads * blocks, requests);
#define MI_WALK(DT)                                                                                  \
  do {                                                                                               \
    if (search) walk_kernel<DT, MODE, SEARCHED><<<grid, 256, 0, stream>>>(p, rows, requests);        \
    else walk_kernel<DT, MODE, false><<<grid, 256, 0, stream>>>(p, rows, requests);                  \
  } while (0)
  if (pad == 64) MI_WALK(1);
  else if (pad == 128) MI_WALK(2);
  else MI_WALK(4);
#undef MI_WALK
  MI_CHECK_LAUNCH("chunk_walk");
  return MI_OK;
}

}  // namespace chunk_scan
