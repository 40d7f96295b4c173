// Recurrent mixers whose state is a matrix per head that decays and takes one outer product a
// token:
//
//     S_t = diag(a_t) S_(t-1) + k_t v_t^T          o_t = S_t^T q_t          (S is dim x vdim, float32)
//
//   DECAY_PER_CHANNEL  a_t is a vector over the key channels, a = logistic(z + bias)^(1/tau)
//                      (gated linear attention); q comes times a constant.
//   DECAY_PER_HEAD     a_t is one number per head, a = exp(-exp(rate) * dt), dt = softplus(raw +
//                      bias); the value row enters times dt, and the read-out gets skip * value
//                      added (a state-space layer in its recurrent form: k, q are its B, C rows,
//                      shared by the heads of a group).
//
// A head's state lies in memory transposed and padded, [vdim][dim_pad].  Column j of S is kept
// by L neighbouring lanes, each holding a run of R rows in registers (dim_pad = R * L), so a
// token costs a lane R multiply-adds for the update and R for the read-out, and the partial
// read-outs of a column meet through register moves between its lanes.  Columns never meet, so
// a head's columns are shared out among blocks of 256 / L columns.  Tokens are taken a tile at
// a time: the next tile's rows are asked of memory while this one is walked, all threads
// evaluate decays and step sizes and leave them in LDS as float32; the walk over the tile's
// tokens reads LDS only.
//
//   readout_gate_norm  what follows the read-out: an RMS norm over groups of columns times a
//                      weight, and a gate silu(g), before the norm or after it.
//
// Everything that enters the recurrence is float32 (projections and convolution outputs are read
// in the element type); in the 32-bit engine decays, step sizes, the read-out's sums and the
// norm's statistics are evaluated in 64-bit and rounded once.
#include "common.h"
#include "linear_recurrence.h"

#include <math.h>

#define SCAN_TILE 16  // tokens fetched at once

namespace {

enum { DECAY_PER_CHANNEL = 0, DECAY_PER_HEAD = 1 };

struct ScanArgs {
  const void *q, *k, *v, *gate;  // rows in the element type
  int64_t q_stride, k_stride, v_stride, gate_stride;
  int q_col, k_col, v_col, gate_col;  // first column of head (or group) 0 in a row
  const float* gate_bias;             // per channel [heads * dim] or per head [heads]
  const float* rate;                  // per head (DECAY_PER_HEAD)
  const float* skip;                  // per head (DECAY_PER_HEAD), may be null
  float inv_tau, q_scale;
  float* state;  // [slots + 1][heads][vdim][dim_pad]
  int64_t state_stride;
  const int *cu, *slots;
  int num_slots;
  float* out;  // float32 [tokens, heads * vdim]
  int heads, groups, dim, vdim;
  bool tokens_alone;  // a request's only token goes through decay_token (launch_scan)
};

template <typename T>
struct Wide {
  using type = float;
};
template <>
struct Wide<float> {
  using type = double;
};

// log(logistic(z)), stable on both sides
template <typename A>
__device__ __forceinline__ A log_logistic(A z) {
  if constexpr (sizeof(A) == 8) return z >= 0 ? -log1p(exp(-z)) : z - log1p(exp(z));
  else return z >= 0 ? -log1pf(expf(-z)) : z - log1pf(expf(z));
}

template <typename A>
__device__ __forceinline__ A soft_plus(A z) {
  if constexpr (sizeof(A) == 8) return fmax(z, 0.0) + log1p(exp(-fabs(z)));
  else return fmaxf(z, 0.f) + log1pf(expf(-fabsf(z)));
}

// Sum over the L neighbouring lanes that keep one column (4, 8 or 16, inside a row of 16
// lanes); every lane gets the total.  The exchanges are register moves (DPP): neighbours,
// pairs, then the mirror image inside 8 and inside 16 lanes.
template <int CTRL>
__device__ __forceinline__ float dpp_move(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xF, 0xF, true));
}
template <int L>
__device__ __forceinline__ float lanes_sum(float v) {
  v += dpp_move<0xB1>(v);  // quad_perm [1,0,3,2]
  v += dpp_move<0x4E>(v);  // quad_perm [2,3,0,1]
  if constexpr (L >= 8) v += dpp_move<0x141>(v);   // row_half_mirror
  if constexpr (L >= 16) v += dpp_move<0x140>(v);  // row_mirror
  return v;
}
template <int L>
__device__ __forceinline__ double lanes_sum(double v) {
#pragma unroll
  for (int off = 1; off < L; off <<= 1) v += __shfl_xor(v, off, MI_WAVE);
  return v;
}

// R values of a row from `at` on as float32, zeros from `dim` (a multiple of R) on; the row can be read in pieces of 16 bytes, of all R where those are fewer.
template <typename T, int R>
__device__ __forceinline__ void run_of_row(const T* row, int at, int dim, float (&v)[R]) {
  constexpr int V = sizeof(T) == 2 && R >= 8 ? 8 : 4;
#pragma unroll
  for (int i = 0; i < R; i += V) {
    float some[V];
    if constexpr (V == 8) {
      const uint4 got = *reinterpret_cast<const uint4*>(row + (at < dim ? at + i : 0));
      const uint32_t words[4] = {got.x, got.y, got.z, got.w};
#pragma unroll
      for (int w = 0; w < 4; ++w) some[2 * w] = __uint_as_float(words[w] << 16), some[2 * w + 1] = __uint_as_float(words[w] & 0xFFFF0000u);
    } else {
      mi_load_cols<T, V>(row + (at < dim ? at + i : 0), some);
    }
#pragma unroll
    for (int j = 0; j < V; ++j) v[i + j] = at < dim ? some[j] : 0.f;
  }
}

// One token of a request, a decay per head: bound by reading and writing its state.  Every lane reads what its rows of S need itself, beside the state
// of G times 256 / L columns, which is all asked for at once: with G = 1 a block had 8 KB on the way, and the blocks went in rounds of 4 us each.
// The arithmetic is that of the walk below, term by term.  64 heads of 128 x 64, states from memory, G = 1 / 4: 34 requests 37.8 / 33.7 us, of them in a
// recorded step of 64 57.3 / 40.2, 64 requests 65.6 / 56.8 (4.7 TB/s).  (With a decay per channel, made once a wave and shared through LDS, 34
// requests of 16 heads of 128 x 256 46 us; the walk takes 43.)
template <typename T, int R, int L, int G>
__device__ __forceinline__ void decay_token(const ScanArgs& p, int64_t t, int slot, int head, int col0) {
  using A = typename Wide<T>::type;
  constexpr bool WIDE = sizeof(T) == 4;
  constexpr int DP = R * L, COLS = 256 / L;
  const int part = threadIdx.x % L, at = part * R, grp = head / (p.heads / p.groups);
  const bool kept = slot >= 0 && slot < p.num_slots;  // (else a row that fills a recorded step: from the spare row, which stays as it is)
  float* state = p.state + (int64_t)(kept ? slot : p.num_slots) * p.state_stride + (int64_t)head * p.vdim * DP + at;
  float S[G][R], q[R], k[R], x[G];
  int col[G];
#pragma unroll
  for (int g = 0; g < G; ++g) {
    col[g] = col0 + g * COLS + threadIdx.x / L;
#pragma unroll
    for (int i = 0; i < R; i += 4) {  // (past the last column: that one again, not written)
      const float4 got = *reinterpret_cast<const float4*>(state + (int64_t)min(col[g], p.vdim - 1) * DP + i);
      S[g][i] = got.x, S[g][i + 1] = got.y, S[g][i + 2] = got.z, S[g][i + 3] = got.w;
    }
  }
  run_of_row<T, R>((const T*)p.q + p.q_col + t * p.q_stride + (int64_t)grp * p.dim, at, p.dim, q);
  run_of_row<T, R>((const T*)p.k + p.k_col + t * p.k_stride + (int64_t)grp * p.dim, at, p.dim, k);
  const T* v_row = (const T*)p.v + p.v_col + t * p.v_stride + (int64_t)head * p.vdim;
#pragma unroll
  for (int g = 0; g < G; ++g) x[g] = to_f32(v_row[min(col[g], p.vdim - 1)]);
  const float raw = to_f32(((const T*)p.gate)[p.gate_col + t * p.gate_stride + head]), head_bias = p.gate_bias[head];
  const float skip = p.skip ? p.skip[head] : 0.f;
  float a, dt;
  if constexpr (WIDE) {
    const double step = soft_plus<double>((double)raw + (double)head_bias);
    a = (float)exp(-exp((double)p.rate[head]) * step);
    dt = (float)step;
  } else {
    const float rate = expf(p.rate[head]) * 1.4426950408889634f;
    dt = mi_soft_plus_fast(raw + head_bias);
    a = __builtin_amdgcn_exp2f(-rate * dt);
  }
#pragma unroll
  for (int i = 0; i < R; ++i) q[i] *= p.q_scale;
#pragma unroll
  for (int g = 0; g < G; ++g) {
    const float vv = x[g] * dt;
    A acc = 0;
#pragma unroll
    for (int i = 0; i < R; ++i) {
      S[g][i] = fmaf(k[i], vv, a * S[g][i]);
      if constexpr (WIDE) acc = fma((double)S[g][i], (double)q[i], acc);
      else acc = fmaf(S[g][i], q[i], acc);
    }
    acc = lanes_sum<L>(acc);
    if (col[g] >= p.vdim) continue;
    if (part == 0) {
      if constexpr (WIDE) acc = fma((double)skip, (double)x[g], acc);
      else acc = fmaf(skip, x[g], acc);
      p.out[t * ((int64_t)p.heads * p.vdim) + (int64_t)head * p.vdim + col[g]] = (float)acc;
    }
    if (!kept) continue;
#pragma unroll
    for (int i = 0; i < R; i += 4)
      *reinterpret_cast<float4*>(state + (int64_t)col[g] * DP + i) = make_float4(S[g][i], S[g][i + 1], S[g][i + 2], S[g][i + 3]);
  }
}

// whether a launch may have single tokens go through decay_token (in float32 launch_scan has the walk take them with one column block a block)
template <typename T, int MODE, int R, int L, int G>
constexpr bool MAY_BE_ALONE = MODE == DECAY_PER_HEAD && (sizeof(T) == 2 || (G > 1 && R * L > 64));

// Decoded tokens, short portions and the 32-bit engine; long portions of bfloat16 steps go in chunks (decay_chunks.hip).
// 256 threads keep 256 / L columns of a head's S, L lanes a column, R rows a lane.  Tokens are
// taken SCAN_TILE at a time: a tile's rows are asked of memory while the tile before it is
// walked (they wait in registers), then all threads turn them into float32 q, k, decays and
// step sizes in LDS, and the walk reads LDS only, each token's operands one token ahead.  In LDS
// a lane's run of R entries is followed by four unused ones where runs of 32 or 64 bytes would
// otherwise meet 2 or 4 to a bank in a 16-byte read of all lanes.
template <typename T, int MODE, int R, int L>
__device__ __forceinline__ void decay_scan_columns(const ScanArgs& p, int b, int head, int col0) {
  using A = typename Wide<T>::type;
  constexpr bool WIDE = sizeof(T) == 4;
  constexpr int DP = R * L;  // padded dim
  constexpr int RUN = R == 4 ? 4 : R + 4;
  constexpr int LP = L * RUN;  // a token's row in LDS
  constexpr int COLS = 256 / L;
  constexpr int EACH = SCAN_TILE * DP / 256;       // entries of the tile's q (k, decay) rows a thread prepares
  constexpr int VALUES = SCAN_TILE * COLS / 256;   // of the tile's values
  static_assert(EACH >= 1 && VALUES >= 1, "a tile gives every thread something to prepare");
  __shared__ __align__(16) float q_lds[SCAN_TILE * LP];
  __shared__ __align__(16) float k_lds[SCAN_TILE * LP];
  __shared__ __align__(16) float a_lds[MODE == DECAY_PER_CHANNEL ? SCAN_TILE * LP : SCAN_TILE];
  __shared__ float v_lds[SCAN_TILE * COLS];  // the value rows as read
  __shared__ float dt_lds[SCAN_TILE];

  const int tid = threadIdx.x;
  const int grp = head / (p.heads / p.groups);
  const int part = tid % L, c = tid / L, col = col0 + c;
  const bool live = col < p.vdim;
  const int first = p.cu[b], last = p.cu[b + 1];
  if (last <= first) return;
  const int slot = p.slots[b];
  const bool kept = slot >= 0 && slot < p.num_slots;  // (see decay_token)
  float* mine = p.state + (int64_t)(kept ? slot : p.num_slots) * p.state_stride + ((int64_t)head * p.vdim + (live ? col : 0)) * DP + part * R;
  float S[R];
#pragma unroll
  for (int i = 0; i < R; i += 4) {
    const float4 got = *reinterpret_cast<const float4*>(mine + i);
    S[i] = got.x, S[i + 1] = got.y, S[i + 2] = got.z, S[i + 3] = got.w;
  }
  const T* q_rows = (const T*)p.q + p.q_col + (int64_t)grp * p.dim;
  const T* k_rows = (const T*)p.k + p.k_col + (int64_t)grp * p.dim;
  const T* v_rows = (const T*)p.v + p.v_col + (int64_t)head * p.vdim + col0;
  const T* g_rows = (const T*)p.gate + p.gate_col;
  const float skip = (MODE == DECAY_PER_HEAD && p.skip) ? p.skip[head] : 0.f;
  float rate = 0.f, head_bias = 0.f;
  double rate_wide = 0.0;
  if constexpr (MODE == DECAY_PER_HEAD) {
    head_bias = p.gate_bias[head];
    rate = expf(p.rate[head]) * 1.4426950408889634f;  // (times log2 e: the decay is an exp2)
    rate_wide = exp((double)p.rate[head]);
  }
  float ch_bias[EACH];
  if constexpr (MODE == DECAY_PER_CHANNEL) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int d = (tid + i * 256) % DP;
      ch_bias[i] = d < p.dim ? p.gate_bias[head * p.dim + d] : 0.f;
    }
  }

  float q_raw[EACH], k_raw[EACH], g_raw[MODE == DECAY_PER_CHANNEL ? EACH : 1], v_raw[VALUES];
  auto ask = [&](int t0, int n) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int e = tid + i * 256, tt = e / DP, d = e % DP;
      const bool in = tt < n && d < p.dim;
      const int64_t t = t0 + (in ? tt : 0);
      q_raw[i] = in ? to_f32(q_rows[t * p.q_stride + d]) : 0.f;
      k_raw[i] = in ? to_f32(k_rows[t * p.k_stride + d]) : 0.f;
      if constexpr (MODE == DECAY_PER_CHANNEL) g_raw[i] = in ? to_f32(g_rows[t * p.gate_stride + head * p.dim + d]) : 0.f;
    }
    if constexpr (MODE == DECAY_PER_HEAD) g_raw[0] = tid < n ? to_f32(g_rows[(int64_t)(t0 + tid) * p.gate_stride + head]) : 0.f;
#pragma unroll
    for (int i = 0; i < VALUES; ++i) {
      const int e = tid + i * 256, tt = e / COLS, cc = e % COLS;
      v_raw[i] = (tt < n && col0 + cc < p.vdim) ? to_f32(v_rows[(int64_t)(t0 + tt) * p.v_stride + cc]) : 0.f;
    }
  };
  auto put = [&](int n) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int e = tid + i * 256, tt = e / DP, d = e % DP;
      if (i * 256 >= n * DP) continue;  // (a tile of few tokens: no decays of others)
      const int at = tt * LP + d + (d / R) * (RUN - R);
      q_lds[at] = q_raw[i] * p.q_scale;
      k_lds[at] = k_raw[i];
      if constexpr (MODE == DECAY_PER_CHANNEL) {
        float av = 0.f;
        if (d < p.dim) {
          if constexpr (WIDE) av = (float)exp(log_logistic<double>((double)g_raw[i] + (double)ch_bias[i]) * (double)p.inv_tau);
          else av = mi_channel_decay(g_raw[i] + ch_bias[i], p.inv_tau);
        }
        a_lds[at] = av;
      }
    }
    if constexpr (MODE == DECAY_PER_HEAD) if (tid < SCAN_TILE) {
      if constexpr (WIDE) {
        const double step = soft_plus<double>((double)g_raw[0] + (double)head_bias);
        a_lds[tid] = (float)exp(-rate_wide * step);
        dt_lds[tid] = (float)step;
      } else {
        const float step = mi_soft_plus_fast(g_raw[0] + head_bias);
        a_lds[tid] = __builtin_amdgcn_exp2f(-rate * step);
        dt_lds[tid] = step;
      }
    }
#pragma unroll
    for (int i = 0; i < VALUES; ++i) v_lds[tid + i * 256] = v_raw[i];
  };

  struct Operands {
    float q[R], k[R], a[R], x, dt;
  };
  auto fetch = [&](int tt, Operands& o) {
    const float4* qt = reinterpret_cast<const float4*>(q_lds + tt * LP + part * RUN);
    const float4* kt = reinterpret_cast<const float4*>(k_lds + tt * LP + part * RUN);
#pragma unroll
    for (int i = 0; i < R; i += 4) {
      const float4 q4 = qt[i / 4], k4 = kt[i / 4];
      o.q[i] = q4.x, o.q[i + 1] = q4.y, o.q[i + 2] = q4.z, o.q[i + 3] = q4.w;
      o.k[i] = k4.x, o.k[i + 1] = k4.y, o.k[i + 2] = k4.z, o.k[i + 3] = k4.w;
    }
    if constexpr (MODE == DECAY_PER_CHANNEL) {
      const float4* at = reinterpret_cast<const float4*>(a_lds + tt * LP + part * RUN);
#pragma unroll
      for (int i = 0; i < R; i += 4) {
        const float4 a4 = at[i / 4];
        o.a[i] = a4.x, o.a[i + 1] = a4.y, o.a[i + 2] = a4.z, o.a[i + 3] = a4.w;
      }
      o.dt = 1.f;
    } else {
      o.a[0] = a_lds[tt];
      o.dt = dt_lds[tt];
    }
    o.x = v_lds[tt * COLS + c];
  };

  ask(first, min(SCAN_TILE, last - first));
  float* out_at = p.out + (int64_t)head * p.vdim + (live ? col : 0);
  const int64_t out_stride = (int64_t)p.heads * p.vdim;
  for (int t0 = first; t0 < last; t0 += SCAN_TILE) {
    const int n = min(SCAN_TILE, last - t0);
    __syncthreads();  // the last tile has been walked
    put(n);
    __syncthreads();
    if (t0 + SCAN_TILE < last) ask(t0 + SCAN_TILE, min(SCAN_TILE, last - t0 - SCAN_TILE));  // (waits in registers through the walk)
    auto step = [&](int tt, const Operands& o) {
      const float vv = MODE == DECAY_PER_HEAD ? o.x * o.dt : o.x;
      A acc = 0;
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const float a = MODE == DECAY_PER_HEAD ? o.a[0] : o.a[i];
        S[i] = fmaf(o.k[i], vv, a * S[i]);
        if constexpr (WIDE) acc = fma((double)S[i], (double)o.q[i], acc);
        else acc = fmaf(S[i], o.q[i], acc);
      }
      acc = lanes_sum<L>(acc);
      if (part == 0 && live) {
        if constexpr (WIDE) acc = fma((double)skip, (double)o.x, acc);
        else acc = fmaf(skip, o.x, acc);
        out_at[(int64_t)(t0 + tt) * out_stride] = (float)acc;
      }
    };
    // two tokens a turn, each one's operands read from LDS while the one before it is worked on
    Operands even, odd;
    fetch(0, even);
    for (int tt = 0; tt < n; tt += 2) {
      if (tt + 1 < n) fetch(tt + 1, odd);
      step(tt, even);
      if (tt + 1 < n) {
        if (tt + 2 < n) fetch(tt + 2, even);
        step(tt + 1, odd);
      }
    }
  }
  if (live && kept) {
#pragma unroll
    for (int i = 0; i < R; i += 4) *reinterpret_cast<float4*>(mine + i) = make_float4(S[i], S[i + 1], S[i + 2], S[i + 3]);
  }
}

// Blocks: a request's heads and columns side by side, so that they spread over the XCDs (workgroups are dealt to the 8 of them in turn), and the last
// request first: a step's long portion commonly comes last, and its chain should not begin when everything else is done.  With the requests
// side by side every eighth block was the long portion's where requests come in 8s: 31 single tokens beside 64 of 64 heads of 128 x 64 184 us, so 34;
// 16 heads of 128 x 256 254 / 66.  Heads go round before columns: a head's column blocks then share an XCD's L2 (512 tokens of 64 heads 144 us, 164
// the other way).
// The blocks are the launch's own three dimensions: in one row, divided up by every block, and with decay_token also where none goes through it, small
// ones held up by both, 48 float32 requests of 64 heads of 16 x 64 13.2 us, so 11.2.
// G: column blocks that a block takes, a single token's together, other requests' one after another (launch_scan says where).  With a block for every
// column block, of which a single token's first took four and the others left at once, all work was on a quarter of the compute units with 8 heads:
// 64 requests of 8 heads of 128 x 512 135 us, so 53, as one at a time 59.
template <typename T, int MODE, int R, int L, int G>
__global__ __launch_bounds__(256) void decay_scan_kernel(ScanArgs p, int last_request, int first_col_block) {
  constexpr int COLS = 256 / L;
  const int b = last_request - (int)blockIdx.z, head = blockIdx.x, col0 = (first_col_block + (int)blockIdx.y) * (G * COLS);
  if constexpr (MAY_BE_ALONE<T, MODE, R, L, G>) {
    const int first = p.cu[b];
    if (p.tokens_alone && p.cu[b + 1] - first == 1) {
      decay_token<T, R, L, G>(p, first, p.slots[b], head, col0);
      return;
    }
  }
#pragma unroll 1
  for (int g = 0; g < G && (g == 0 || col0 + g * COLS < p.vdim); ++g) decay_scan_columns<T, MODE, R, L>(p, b, head, col0 + g * COLS);
}

// rows per lane and lanes per column for a head whose keys are `dim` wide
inline void scan_shape(int dim, int* rows, int* lanes) {
  if (dim <= 16) *rows = 4, *lanes = 4;
  else if (dim <= 32) *rows = 8, *lanes = 4;
  else if (dim <= 64) *rows = 8, *lanes = 8;
  else if (dim <= 128) *rows = 8, *lanes = 16;
  else *rows = 16, *lanes = 16;
}

constexpr int MOST_BLOCKS = 65535;  // of a launch's second and third dimension

template <typename T, int MODE>
int launch_scan(ScanArgs p, int tokens, int requests, hipStream_t stream) {
  int rows, lanes;
  scan_shape(p.dim, &rows, &lanes);
  constexpr int TOGETHER = MODE == DECAY_PER_HEAD ? 4 : 1;  // column blocks
  const int col_blocks = ceil_div(p.vdim, 256 / lanes);
  // Single tokens by decay_token: where rows of q and k are read a lane's run at a time, in float32 only four column blocks together and keys of more than 64.
  // Microseconds as in a walk / so, a decay per head, from memory: bfloat16, 64 heads of 128 x 64, 8 / 40 requests 11.5 / 10.1 and 44.9 / 35.9, 48 of 64 x 64 6.0 / 5.4 and
  // 19.8 / 17.0; value by value 64 of 100 x 64 at 8 11.4 / 17.0, 24 of 200 x 256 33.5 / 61.5 and 121 / 183, 64 of 256 x 64 24.1 / 50.2 and 88.8 / 116; float32, 64 of
  // 128 x 64 at 40 49.3 / 37.3, at 8 13.7 / 14.2, beside a portion 46 / 54, 48 of 64 x 64 at 40 19.2 / 22.6, 64 of 256 x 64 at 8 / 40 23.6 / 28.1 and 90.6 / 83.7.
  const int piece = min(16, rows * (int)sizeof(T));
  auto in_pieces = [&](const void* row, int64_t stride, int col) {
    return ((uintptr_t)row + (uintptr_t)col * sizeof(T)) % piece == 0 && stride * sizeof(T) % piece == 0;
  };
  p.tokens_alone = p.dim % rows == 0 && in_pieces(p.q, p.q_stride, p.q_col) && in_pieces(p.k, p.k_stride, p.k_col);
  // Four column blocks together from two rounds of what the CUs hold on; 24 requests of 32 heads of 64 columns, 3,072 blocks, take the same either way.  Beside a long
  // portion, whose chain the larger blocks hold up, one: 38 tokens beside 73, a step of 12 layers 2,910 / 2,928 us.  (A head's last block would read for four
  // whatever it holds: heads of whole fours only.)
  const bool together = TOGETHER > 1 && p.tokens_alone && (sizeof(T) == 2 || p.dim > 64) && tokens <= requests &&
                        (int64_t)requests * p.heads * col_blocks >= 4096 && col_blocks % TOGETHER == 0;
  MI_REQUIRE(p.heads < (1 << 24), "decay_scan: %d heads are too many", p.heads);
  const int each = together ? col_blocks / TOGETHER : col_blocks;
#define MI_SCAN(RR, LL)                                                                                              \
  do {                                                                                                               \
    if (together) decay_scan_kernel<T, MODE, RR, LL, TOGETHER><<<grid, 256, 0, stream>>>(p, requests - 1 - r, c);     \
    else decay_scan_kernel<T, MODE, RR, LL, 1><<<grid, 256, 0, stream>>>(p, requests - 1 - r, c);                     \
  } while (0)
  for (int r = 0; r < requests; r += MOST_BLOCKS) for (int c = 0; c < each; c += MOST_BLOCKS) {
    const dim3 grid(p.heads, min(MOST_BLOCKS, each - c), min(MOST_BLOCKS, requests - r));
    if (rows == 4) MI_SCAN(4, 4);
    else if (rows == 8 && lanes == 4) MI_SCAN(8, 4);
    else if (rows == 8 && lanes == 8) MI_SCAN(8, 8);
    else if (rows == 8 && lanes == 16) MI_SCAN(8, 16);
    else MI_SCAN(16, 16);
  }
#undef MI_SCAN
  MI_CHECK_LAUNCH("decay_scan");
  return MI_OK;
}

// Bound by the rows' bytes.  blockDim.x threads take a group of a row, V columns a thread at once, blockDim.y groups share
// a block.  ONE: the threads hold the whole group (V columns each), which stays in registers from the sum to the
// result; else it is read a second time.  1,777 rows of
// 3,072 beside bfloat16 gates (44 MB, 9.3 us at the rate of a large copy): one group 15.6, 12 groups 12.2;
// nine calls of the former and three of the latter took 18.8 on average when every value was read twice, a block took one
// group and a weight's place a division.
template <typename T, int V, bool ONE>
__global__ __launch_bounds__(1024) void readout_gate_norm_kernel(const float* __restrict__ o, const T* __restrict__ gate,
                                                                 int64_t gate_stride, const float* __restrict__ weight,
                                                                 int weight_period, T* __restrict__ out, int64_t out_stride,
                                                                 int width, int group_width, int gate_first, float eps) {
  using A = typename Wide<T>::type;
  __shared__ A scratch[16];
  const int t = blockIdx.x, groups = width / group_width;
  const int g = blockIdx.y * blockDim.y + threadIdx.y;
  const bool in = g < groups;  // (a block's last groups may be past the row's: of those the last one again, unwritten)
  const int64_t at = (int64_t)(in ? g : groups - 1) * group_width;
  const float* orow = o + (int64_t)t * width + at;
  const T* grow = gate + (int64_t)t * gate_stride + at;
  T* dst = out + (int64_t)t * out_stride + at;
  auto gate_of = [&](float raw) -> A {
    const A z = (A)raw;
    if constexpr (sizeof(A) == 8) return z / (1.0 + exp(-z));
    else return z / (1.f + expf(-z));
  };
  const int c0 = threadIdx.x * V, step = ONE ? group_width : blockDim.x * V;
  A ss = 0;
  float y[V], z[V];
  A gated[V];
  for (int c = c0; c < group_width; c += step) {
    mi_load_cols<float, V>(orow + c, y);
    if (gate_first || ONE) mi_load_cols<T, V>(grow + c, z);
#pragma unroll
    for (int j = 0; j < V; ++j) {
      A v = (A)y[j];
      if (gate_first) v = (A)(float)(v * gate_of(z[j]));
      gated[j] = v;
      ss += v * v;
    }
  }
  // (fixed order: lanes by butterfly, waves one after another)
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) ss += __shfl_xor(ss, off, MI_WAVE);
  const int n_waves = blockDim.x / MI_WAVE;
  A* mine = scratch + threadIdx.y * n_waves;
  if (n_waves > 1) {
    if (threadIdx.x % MI_WAVE == 0) mine[threadIdx.x / MI_WAVE] = ss;
    __syncthreads();
    ss = 0;
    for (int w = 0; w < n_waves; ++w) ss += mine[w];
  }
  if (!in) return;
  A r;
  if constexpr (sizeof(A) == 8) r = 1.0 / sqrt(ss / (double)group_width + (double)eps);
  else r = 1.0f / sqrtf(ss / (float)group_width + eps);
  int first_weight = c0 < group_width ? ((int)at + c0) % weight_period : 0;
  const int weights_on = ONE ? 0 : step % weight_period;
  for (int c = c0; c < group_width; c += step) {
    if constexpr (!ONE) {
      mi_load_cols<float, V>(orow + c, y);
      mi_load_cols<T, V>(grow + c, z);
    }
    float res[V];
    int of_weight = first_weight;  // (one division; the next columns' count on)
    first_weight += weights_on;
    if (first_weight >= weight_period) first_weight -= weight_period;
#pragma unroll
    for (int j = 0; j < V; ++j) {
      const A w = (A)weight[of_weight];
      if (++of_weight == weight_period) of_weight = 0;
      A v = (A)y[j];
      if (gate_first) v = (ONE ? gated[j] : (A)(float)(v * gate_of(z[j]))) * r * w;
      else v = v * r * w * gate_of(z[j]);
      res[j] = (float)v;
    }
    mi_store_cols<T, V>(dst + c, res);
  }
}

}  // namespace

extern "C" int mi_decay_scan_dim_pad(int dim) {
  int rows, lanes;
  scan_shape(dim, &rows, &lanes);
  return rows * lanes;
}

int mi_decay_scan_check(int dtype, int mode, int64_t q_stride, int q_col, int64_t k_stride, int k_col, int64_t v_stride, int v_col,
                        int64_t gate_stride, int gate_col, const float* gate_bias, const float* rate, const float* state,
                        int64_t state_stride, int num_slots, int num_tokens, int num_requests, int heads, int groups, int dim, int vdim) {
  MI_REQUIRE(num_tokens >= 0 && num_requests >= 0 && heads > 0 && groups > 0 && dim > 0 && vdim > 0,
             "decay_scan: bad sizes tokens=%d requests=%d heads=%d groups=%d dim=%d vdim=%d", num_tokens, num_requests, heads,
             groups, dim, vdim);
  MI_REQUIRE(heads % groups == 0, "decay_scan: heads=%d is not a multiple of groups=%d", heads, groups);
  MI_REQUIRE(dim <= 256, "decay_scan: dim=%d is above 256", dim);
  MI_REQUIRE(mode == 0 || mode == 1, "decay_scan: mode %d (0 per channel, 1 per head)", mode);
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "decay_scan: unknown dtype %d", dtype);
  MI_REQUIRE(num_slots >= 1 && num_requests <= 65535 * 32 && heads <= 65535, "decay_scan: bad slot or grid counts");
  MI_REQUIRE(q_stride >= q_col + (int64_t)groups * dim && k_stride >= k_col + (int64_t)groups * dim &&
                 v_stride >= v_col + (int64_t)heads * vdim,
             "decay_scan: row strides shorter than the columns read");
  MI_REQUIRE(gate_stride >= gate_col + (int64_t)heads * (mode == 0 ? dim : 1), "decay_scan: the gates' rows are too short");
  MI_REQUIRE(gate_bias != nullptr && (mode == 0 || rate != nullptr), "decay_scan: missing gate constants");
  MI_REQUIRE(state_stride >= (int64_t)heads * vdim * mi_decay_scan_dim_pad(dim) && ((uintptr_t)state % 16 == 0) &&
                 state_stride % 4 == 0,
             "decay_scan: the state rows are too short or not 16-byte aligned");
  return MI_OK;
}

// mode 0: decay per key channel (gate: [tokens, heads * dim] logits, gate_bias [heads * dim], inv_tau);
// mode 1: decay per head (gate: [tokens, heads] raw step sizes, gate_bias [heads], rate [heads], skip [heads] or null).
// q, k: rows holding `groups` heads of `dim` from q_col / k_col on (head h reads group h / (heads / groups));
// v: rows holding `heads` heads of `vdim` from v_col on.  state float32 [slots + 1][heads][vdim][dim_pad].
// out float32 [tokens, heads * vdim].
extern "C" int mi_decay_scan(int dtype, int mode, const void* q, int64_t q_stride, int q_col, const void* k, int64_t k_stride,
                             int k_col, const void* v, int64_t v_stride, int v_col, const void* gate, int64_t gate_stride,
                             int gate_col, const float* gate_bias, const float* rate, const float* skip, float inv_tau,
                             float q_scale, float* state, int64_t state_stride, const int* cu, const int* slots, int num_slots,
                             float* out, int num_tokens, int num_requests, int heads, int groups, int dim, int vdim,
                             hipStream_t stream) {
  const int bad = mi_decay_scan_check(dtype, mode, q_stride, q_col, k_stride, k_col, v_stride, v_col, gate_stride, gate_col, gate_bias,
                                      rate, state, state_stride, num_slots, num_tokens, num_requests, heads, groups, dim, vdim);
  if (bad != MI_OK) return bad;
  if (num_tokens == 0 || num_requests == 0) return MI_OK;
  ScanArgs p;
  p.q = q, p.k = k, p.v = v, p.gate = gate;
  p.q_stride = q_stride, p.k_stride = k_stride, p.v_stride = v_stride, p.gate_stride = gate_stride;
  p.q_col = q_col, p.k_col = k_col, p.v_col = v_col, p.gate_col = gate_col;
  p.gate_bias = gate_bias, p.rate = rate, p.skip = skip, p.inv_tau = inv_tau, p.q_scale = q_scale;
  p.state = state, p.state_stride = state_stride, p.cu = cu, p.slots = slots, p.num_slots = num_slots, p.out = out;
  p.heads = heads, p.groups = groups, p.dim = dim, p.vdim = vdim, p.tokens_alone = false;
  if (dtype == MI_F32) return mode == 0 ? launch_scan<float, DECAY_PER_CHANNEL>(p, num_tokens, num_requests, stream)
                                        : launch_scan<float, DECAY_PER_HEAD>(p, num_tokens, num_requests, stream);
  return mode == 0 ? launch_scan<bf16_t, DECAY_PER_CHANNEL>(p, num_tokens, num_requests, stream)
                   : launch_scan<bf16_t, DECAY_PER_HEAD>(p, num_tokens, num_requests, stream);
}

// o float32 [tokens, width]; gate [tokens, >= width] in the element type (row stride, from its first column);
// weight float32 [weight_period] (column c takes weight[c % weight_period]); the norm runs over
// groups of `group_width` columns.  gate_first: out = norm(o * silu(g)) * w, else norm(o) * w * silu(g).
extern "C" int mi_readout_gate_norm(int dtype, const float* o, const void* gate, int64_t gate_stride, const float* weight,
                                    int weight_period, void* out, int64_t out_stride, int num_tokens, int width,
                                    int group_width, int gate_first, float eps, hipStream_t stream) {
  MI_REQUIRE(num_tokens >= 0 && width > 0 && group_width > 0 && width % group_width == 0,
             "readout_gate_norm: bad sizes tokens=%d width=%d group=%d", num_tokens, width, group_width);
  MI_REQUIRE(weight_period > 0 && gate_stride >= width && out_stride >= width, "readout_gate_norm: rows or weight too short");
  MI_REQUIRE(width / group_width <= 65535, "readout_gate_norm: too many groups");
  MI_REQUIRE(dtype == MI_F32 || dtype == MI_BF16, "readout_gate_norm: unknown dtype %d", dtype);
  if (num_tokens == 0) return MI_OK;
  const size_t elem = dtype == MI_F32 ? 4 : 2;
  const bool wide = group_width % 4 == 0 && gate_stride % 4 == 0 && out_stride % 4 == 0 && (uintptr_t)o % 16 == 0 &&
                    (uintptr_t)gate % (4 * elem) == 0 && (uintptr_t)out % (4 * elem) == 0;
  const int columns = wide ? 4 : 1, groups = width / group_width;
  const int threads = min(1024, ceil_div(ceil_div(group_width, columns), MI_WAVE) * MI_WAVE);
  const bool one = group_width <= threads * columns;
  const int shared = min(max(1, 256 / threads), groups);  // groups a block
  dim3 grid(num_tokens, ceil_div(groups, shared)), block(threads, shared);
#define MI_READOUT(TT, VV, ONE)                                                                                              \
  readout_gate_norm_kernel<TT, VV, ONE><<<grid, block, 0, stream>>>(o, (const TT*)gate, gate_stride, weight, weight_period,  \
                                                                    (TT*)out, out_stride, width, group_width, gate_first, eps)
#define MI_READOUT_OF(TT)                   \
  if (wide && one) MI_READOUT(TT, 4, true); \
  else if (wide) MI_READOUT(TT, 4, false);  \
  else if (one) MI_READOUT(TT, 1, true);    \
  else MI_READOUT(TT, 1, false)
  if (dtype == MI_F32) {
    MI_READOUT_OF(float);
  } else {
    MI_READOUT_OF(bf16_t);
  }
#undef MI_READOUT_OF
#undef MI_READOUT
  MI_CHECK_LAUNCH("readout_gate_norm");
  return MI_OK;
}
