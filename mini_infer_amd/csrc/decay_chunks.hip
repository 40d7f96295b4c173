// The decaying recurrences over many tokens of a request: see chunk_scan.h for the form, linear_recurrence.hip for
// the recurrences.  The first launch makes, per chunk and head, what does not depend on the state.
#include "chunk_scan.h"
#include "linear_recurrence.h"

#include <math.h>

namespace {

using namespace chunk_scan;

struct RowArgs {
  const bf16_t *q, *k, *gate;
  int64_t q_stride, k_stride, gate_stride;
  int q_col, k_col, gate_col;
  const float *gate_bias, *rate;
  float inv_tau, q_scale;
  const int* cu;
  int requests, heads, groups, dim;
  bool eights;  // rows of q, k (and the channels' gates) lie on 16 bytes in whole 8s
};

// What walk_by_token takes of a token.
template <int MODE>
struct TokenRows {
  RowArgs p;
  __device__ __forceinline__ void channel(int64_t t, int head, int heads, int d, float& q, float& k) const {
    const int64_t at = head / (heads / p.groups) * (int64_t)p.dim + d;
    q = to_f32(p.q[t * p.q_stride + p.q_col + at]) * p.q_scale, k = to_f32(p.k[t * p.k_stride + p.k_col + at]);
  }
  __device__ __forceinline__ float channel_gate(int64_t t, int head, int d) const {
    return to_f32(p.gate[t * p.gate_stride + p.gate_col + (int64_t)head * p.dim + d]);
  }
  __device__ __forceinline__ float channel_bias(int head, int d) const { return p.gate_bias[(int64_t)head * p.dim + d]; }
  __device__ __forceinline__ float channel_decay(float z) const { return mi_channel_decay(z, p.inv_tau); }
  __device__ __forceinline__ void head_gates(int64_t t, int head, float& decay, float& step) const {
    step = mi_soft_plus_fast(to_f32(p.gate[t * p.gate_stride + p.gate_col + head]) + p.gate_bias[head]);
    decay = __builtin_amdgcn_exp2f(-(expf(p.rate[head]) * 1.4426950408889634f) * step);
  }
  __device__ __forceinline__ int width() const { return p.dim; }
};

// a decay per head: one block per (chunk, group of rows, 8 heads of the group), 4 waves
template <int DT>
__global__ __launch_bounds__(256) void head_decay_chunk_kernel(RowArgs p, Made made) {
  constexpr int PAD = 64 * DT, ROW = PAD + 4, EACH = PAD / 8, INNER = CHUNK * (CHUNK + 4);
  __shared__ __align__(16) float q_s[CHUNK * ROW], k_s[CHUNK * ROW], qk_s[INNER];
  __shared__ float zeros_s[CHUNK];
  __shared__ int which;
  const int chunk = blockIdx.x, share = blockIdx.y;
  const int b = request_of_chunk(chunk, p.cu, p.requests, &which);
  if (b < 0) return;
  const int t0 = p.cu[b] + (chunk - first_chunk(p.cu[b], b)) * CHUNK, nt = min(CHUNK, p.cu[b + 1] - t0);
  const int tid = threadIdx.x, wave = tid / MI_WAVE, lane = tid % MI_WAVE;
  if (p.cu[b + 1] - p.cu[b] == 1) {
    if (blockIdx.z > 0) return;
    const int64_t row = t0, at = tid < p.dim ? (int64_t)share * p.dim + tid : -1;
    const float q = at >= 0 ? to_f32(p.q[row * p.q_stride + p.q_col + at]) : 0.f, k = at >= 0 ? to_f32(p.k[row * p.k_stride + p.k_col + at]) : 0.f;
    float sums[2] = {q * p.q_scale * k, fmaf(0.f, k, 0.f * q)};
    sum_of_block(sums, qk_s);
    float* rows = made.q + ((int64_t)chunk * made.shares + share) * CHUNK * PAD;
    if (tid < PAD) rows[tid] = q * p.q_scale, rows[PAD + tid] = k;
    for (int h = share * (p.heads / p.groups) + tid; h < (share + 1) * (p.heads / p.groups); h += 256) {
      const int64_t of = (int64_t)chunk * p.heads + h;
      const float dt = mi_soft_plus_fast(to_f32(p.gate[row * p.gate_stride + p.gate_col + h]) + p.gate_bias[h]);
      const float sum = -(expf(p.rate[h]) * 1.4426950408889634f * dt), whole = __builtin_amdgcn_exp2f(0.f * sum);  // (1, or NaN)
      made.factor[of * 2 * CHUNK] = __builtin_amdgcn_exp2f(sum);
      made.factor[of * 2 * CHUNK + CHUNK] = whole * dt + sums[1];
      made.within[of * CHUNK * CHUNK] = whole * sums[0] * dt;
    }
    return;
  }
  {
    const int token = tid / 8, sub = tid % 8;
    const int64_t row = t0 + min(token, nt - 1);
    const bf16_t *q = p.q + row * p.q_stride + p.q_col + (int64_t)share * p.dim, *k = p.k + row * p.k_stride + p.k_col + (int64_t)share * p.dim;
    float* out = made.q + (((int64_t)chunk * made.shares + share) * CHUNK + token) * PAD + sub * EACH;
    float qv[EACH], kv[EACH];
    row_values(q, sub * EACH, p.dim, p.eights, token < nt, qv);
    row_values(k, sub * EACH, p.dim, p.eights, token < nt, kv);
    float zeros = 0.f;  // unless something is not finite
#pragma unroll
    for (int e = 0; e < EACH; ++e) zeros = fmaf(0.f, kv[e], fmaf(0.f, qv[e], zeros));
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) zeros += __shfl_xor(zeros, off, MI_WAVE);
    if (sub == 0) zeros_s[token] = zeros;
#pragma unroll
    for (int e = 0; e < EACH; e += 4) {
      const float4 q4 = make_float4(qv[e] * p.q_scale, qv[e + 1] * p.q_scale, qv[e + 2] * p.q_scale, qv[e + 3] * p.q_scale);
      *reinterpret_cast<float4*>(&q_s[token * ROW + sub * EACH + e]) = q4;
      *reinterpret_cast<float4*>(&k_s[token * ROW + sub * EACH + e]) = make_float4(kv[e], kv[e + 1], kv[e + 2], kv[e + 3]);
      if (blockIdx.z == 0) *reinterpret_cast<float4*>(out + e) = q4;
    }
  }
  __syncthreads();
  if (blockIdx.z == 0)
    for (int i = tid; i < PAD * (CHUNK / 4); i += 256) {
      const int d = i % PAD, t = i / PAD * 4;
      *reinterpret_cast<float4*>(made.kt + (((int64_t)chunk * made.shares + share) * PAD + d) * CHUNK + t) =
          make_float4(k_s[t * ROW + d], k_s[(t + 1) * ROW + d], k_s[(t + 2) * ROW + d], k_s[(t + 3) * ROW + d]);
    }
  const int r = lane % 16, quad = lane / 16;
  f32x4_t qk = {0.f, 0.f, 0.f, 0.f};
  const int ti = wave / 2, tj = wave % 2;
#pragma unroll
  for (int d = 0; d < PAD; d += 16) {
    const float4 kj = load4(&k_s[(16 * tj + r) * ROW + d + 4 * quad]);
    qk = mma4(load4(&q_s[(16 * ti + r) * ROW + d + 4 * quad]), f32x4_t{kj.x, kj.y, kj.z, kj.w}, qk);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) qk_s[(16 * ti + 4 * quad + e) * (CHUNK + 4) + 16 * tj + r] = qk[e];
  __syncthreads();
  const int group = p.heads / p.groups, i0 = lane % CHUNK;
  for (int g = blockIdx.z * 8 + wave; g < min(group, (int)blockIdx.z * 8 + 8); g += 4) {
    const int h = share * group + g;
    const int64_t of = (int64_t)chunk * p.heads + h;
    // lane i and lane i + 32: token i's step size and the sum of the decays' logarithms (base 2) up to it, in 64-bit
    const float raw = to_f32(p.gate[(int64_t)(t0 + min(i0, nt - 1)) * p.gate_stride + p.gate_col + h]);
    const float dt = i0 < nt ? mi_soft_plus_fast(raw + p.gate_bias[h]) : 0.f;
    double sum = -(double)(expf(p.rate[h]) * 1.4426950408889634f * dt);
#pragma unroll
    for (int off = 1; off < CHUNK; off <<= 1) {
      const double before = __shfl_up(sum, off, CHUNK);
      if (i0 >= off) sum += before;
    }
    if (lane < CHUNK) {
      float* factor = made.factor + of * 2 * CHUNK + lane;
      factor[0] = __builtin_amdgcn_exp2f((float)sum);
      factor[CHUNK] = __builtin_amdgcn_exp2f((float)(__shfl(sum, CHUNK - 1, CHUNK) - sum)) * dt + zeros_s[lane];
    }
    float* within = made.within + of * CHUNK * CHUNK + i0;
#pragma unroll
    for (int n = 0; n < CHUNK / 2; ++n) {
      const int i = 2 * n + lane / CHUNK;
      const double sum_i = __shfl(sum, i, MI_WAVE);
      within[i * CHUNK] = i >= i0 ? __builtin_amdgcn_exp2f((float)(sum_i - sum)) * qk_s[i * (CHUNK + 4) + i0] * dt : 0.f;
    }
  }
}

// a decay per key channel: one block per (chunk, head).  Everything is a running product of decays down the chunk's
// tokens, as in the token-by-token form; W by thread (token j, an eighth of the channels), which carries k_j on from
// token to token and meets every q_i.
template <int DT>
__global__ __launch_bounds__(256) void channel_decay_chunk_kernel(RowArgs p, Made made) {
  constexpr int PAD = 64 * DT, ROW = PAD + 4, EACH = PAD / 8;
  extern __shared__ __align__(16) float channel_lds[];
  float *q_s = channel_lds, *k_s = q_s + CHUNK * ROW, *a_s = k_s + CHUNK * ROW;
  __shared__ int which;
  const int chunk = blockIdx.x, head = blockIdx.y;
  const int b = request_of_chunk(chunk, p.cu, p.requests, &which);
  if (b < 0) return;
  const int t0 = p.cu[b] + (chunk - first_chunk(p.cu[b], b)) * CHUNK, nt = min(CHUNK, p.cu[b + 1] - t0);
  const int tid = threadIdx.x, share = head / (p.heads / p.groups);
  int odd = 0;
  if (p.cu[b + 1] - p.cu[b] == 1) {
    const bool in = tid < p.dim;
    const int64_t row = t0, at = (int64_t)share * p.dim + tid;
    const float q = in ? to_f32(p.q[row * p.q_stride + p.q_col + at]) : 0.f, k = in ? to_f32(p.k[row * p.k_stride + p.k_col + at]) : 0.f;
    const float a = in ? mi_channel_decay(to_f32(p.gate[row * p.gate_stride + p.gate_col + (int64_t)head * p.dim + tid]) + p.gate_bias[(int64_t)head * p.dim + tid],
                                          p.inv_tau) : 1.f;
    odd = __syncthreads_or(!(fmaf(0.f, q, 0.f * k) + 0.f * a == 0.f));
    float sums[1] = {q * p.q_scale * k};
    sum_of_block(sums, channel_lds);
    float* rows = made.q + ((int64_t)chunk * made.shares + head) * CHUNK * PAD;
    if (tid < PAD) {
      rows[tid] = q * p.q_scale * a, rows[PAD + tid] = k;
      made.fade[((int64_t)chunk * p.heads + head) * PAD + tid] = odd ? NAN : a;
    }
    if (tid == 0) made.within[((int64_t)chunk * p.heads + head) * CHUNK * CHUNK] = sums[0];
    return;
  }
  {
    const int token = tid / 8, sub = tid % 8;
    const int64_t row = t0 + min(token, nt - 1);
    const bf16_t *q = p.q + row * p.q_stride + p.q_col + (int64_t)share * p.dim, *k = p.k + row * p.k_stride + p.k_col + (int64_t)share * p.dim;
    const bf16_t* gate = p.gate + row * p.gate_stride + p.gate_col + (int64_t)head * p.dim;
    float qv[EACH], kv[EACH], av[EACH];
    row_values(q, sub * EACH, p.dim, p.eights, token < nt, qv);
    row_values(k, sub * EACH, p.dim, p.eights, token < nt, kv);
    row_values(gate, sub * EACH, p.dim, p.eights, token < nt, av);
    const float* bias = p.gate_bias + (int64_t)head * p.dim;
    float zeros = 0.f;
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
      const int d = sub * EACH + e;
      const float a = mi_channel_decay(av[e] + bias[min(d, p.dim - 1)], p.inv_tau);
      q_s[token * ROW + d] = qv[e] * p.q_scale;
      k_s[token * ROW + d] = kv[e];
      zeros = fmaf(0.f, qv[e], zeros) + 0.f * kv[e] + 0.f * a;
      a_s[token * ROW + d] = token < nt && d < p.dim ? a : 1.f;
    }
    odd = !(zeros == 0.f);
  }
  odd = __syncthreads_or(odd);
  for (int d = tid; d < PAD; d += 256) {
    const int64_t of = (int64_t)chunk * made.shares + head;  // (rows of a head of its own)
    double product = 1.0, tail = 1.0;  // (rounded once, where they are used)
#pragma unroll 8
    for (int i = 0; i < CHUNK; ++i) {
      product *= (double)a_s[i * ROW + d];
      made.q[(of * CHUNK + i) * PAD + d] = (float)((double)q_s[i * ROW + d] * product);
    }
    made.fade[((int64_t)chunk * p.heads + head) * PAD + d] = odd ? NAN : (float)product;
    float four[4];
    float* kt = made.kt + (of * PAD + d) * CHUNK;
#pragma unroll
    for (int j = CHUNK - 1; j >= 0; --j) {
      four[j % 4] = (float)((double)k_s[j * ROW + d] * tail);
      tail *= (double)a_s[j * ROW + d];
      if (j % 4 == 0) *reinterpret_cast<float4*>(kt + j) = make_float4(four[0], four[1], four[2], four[3]);
    }
  }
  const int j = tid / 8, sub = tid % 8;
  float carried[EACH], own[EACH];
#pragma unroll
  for (int e = 0; e < EACH; e += 4) {  // (channels 4 * sub .. of every 32: the eight threads of a token read side by side)
    const float4 k = load4(&k_s[j * ROW + e * 8 + 4 * sub]);
    own[e] = k.x, own[e + 1] = k.y, own[e + 2] = k.z, own[e + 3] = k.w;
    carried[e] = carried[e + 1] = carried[e + 2] = carried[e + 3] = 0.f;
  }
  float* within = made.within + ((int64_t)chunk * p.heads + head) * CHUNK * CHUNK + j;
#pragma unroll 4
  for (int i = 0; i < CHUNK; ++i) {
    float sum4[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int e = 0; e < EACH; e += 4) {
      const int d = e * 8 + 4 * sub;
      const float4 a = load4(&a_s[i * ROW + d]), q = load4(&q_s[i * ROW + d]);
      const float as[4] = {a.x, a.y, a.z, a.w}, qs[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        carried[e + c] = i == j ? own[e + c] : carried[e + c] * as[c];
        sum4[c] = fmaf(qs[c], carried[e + c], sum4[c]);
      }
    }
    float sum = (sum4[0] + sum4[1]) + (sum4[2] + sum4[3]);
    // over the eight threads of token j: neighbours, pairs, and the mirror image inside 8 lanes (register moves)
    sum += lane_moved<0xB1>(sum);
    sum += lane_moved<0x4E>(sum);
    sum += lane_moved<0x141>(sum);
    if (sub == 0) within[i * CHUNK] = sum;
  }
}

int made_shares(int mode, int heads, int groups) { return mode == PER_CHANNEL ? heads : groups; }

}  // namespace

// Floats of scratch that mi_decay_scan_chunks takes; 0: sizes it does not take.
extern "C" int64_t mi_decay_scan_chunks_scratch(int mode, int num_tokens, int num_requests, int heads, int groups, int dim, int vdim) {
  const int pad = mi_decay_scan_dim_pad(dim);
  if (num_tokens <= 0 || num_requests <= 0 || num_requests > 65535 || dim > 256 || pad < 64 || heads <= 0 || heads > 65535 || groups <= 0 || vdim <= 0) return 0;
  return chunk_count(num_tokens, num_requests) * ((int64_t)2 * made_shares(mode, heads, groups) * CHUNK * pad +
                                                  (int64_t)heads * (CHUNK * CHUNK + (mode == PER_CHANNEL ? pad : 2 * CHUNK)));
}

// As mi_decay_scan for bfloat16, with `scratch` on 16 bytes; longest: tokens of the longest portion, 0: not known.
extern "C" int mi_decay_scan_chunks(int mode, const void* q, int64_t q_stride, int q_col, const void* k, int64_t k_stride, int k_col,
                                    const void* v, int64_t v_stride, int v_col, const void* gate, int64_t gate_stride, int gate_col,
                                    const float* gate_bias, const float* rate, const float* skip, float inv_tau, float q_scale,
                                    float* state, int64_t state_stride, const int* cu, const int* slots, int num_slots, float* scratch,
                                    float* out, int num_tokens, int num_requests, int longest, int heads, int groups, int dim, int vdim,
                                    hipStream_t stream) {
  const int bad = mi_decay_scan_check(MI_BF16, mode, q_stride, q_col, k_stride, k_col, v_stride, v_col, gate_stride, gate_col, gate_bias,
                                      rate, state, state_stride, num_slots, num_tokens, num_requests, heads, groups, dim, vdim);
  if (bad != MI_OK) return bad;
  if (num_tokens == 0 || num_requests == 0) return MI_OK;
  MI_REQUIRE(mi_decay_scan_chunks_scratch(mode, num_tokens, num_requests, heads, groups, dim, vdim) > 0, "decay_scan_chunks: sizes it does not take");
  MI_REQUIRE(scratch != nullptr && (uintptr_t)scratch % 16 == 0, "decay_scan_chunks: no scratch");
  const int pad = mi_decay_scan_dim_pad(dim);
  const int64_t chunks = chunk_count(num_tokens, num_requests), rows = chunks * made_shares(mode, heads, groups) * CHUNK * pad;
  MI_REQUIRE(chunks <= 2147483647 && v_stride < MAX_ROW && (int64_t)heads * vdim < MAX_ROW, "decay_scan_chunks: sizes it does not take");
  Made made;
  made.q = scratch, made.kt = made.q + rows, made.within = made.kt + rows;
  made.fade = made.within + chunks * heads * CHUNK * CHUNK;
  made.factor = made.fade + (mode == PER_CHANNEL ? chunks * heads * pad : 0);
  made.k = made.solve = nullptr;
  made.shares = made_shares(mode, heads, groups);
  RowArgs a;
  a.q = (const bf16_t*)q, a.k = (const bf16_t*)k, a.gate = (const bf16_t*)gate;
  a.q_stride = q_stride, a.k_stride = k_stride, a.gate_stride = gate_stride;
  a.q_col = q_col, a.k_col = k_col, a.gate_col = gate_col;
  a.gate_bias = gate_bias, a.rate = rate, a.inv_tau = inv_tau, a.q_scale = q_scale;
  a.cu = cu, a.requests = num_requests, a.heads = heads, a.groups = groups, a.dim = dim;
  a.eights = in_eights(q, q_stride, q_col, dim) && in_eights(k, k_stride, k_col, dim) &&
             (mode != PER_CHANNEL || in_eights(gate, gate_stride, gate_col, dim));
  if (mode == PER_CHANNEL) {
    dim3 grid((unsigned)chunks, heads);
    const size_t lds = sizeof(float) * 3 * CHUNK * (pad + 4);
#define MI_CHANNEL_CHUNKS(DT) channel_decay_chunk_kernel<DT><<<grid, 256, lds, stream>>>(a, made)
    if (pad == 64) MI_CHANNEL_CHUNKS(1);
    else if (pad == 128) MI_CHANNEL_CHUNKS(2);
    else MI_CHANNEL_CHUNKS(4);
#undef MI_CHANNEL_CHUNKS
    MI_CHECK_LAUNCH("channel_decay_chunk");
  } else {
    dim3 grid((unsigned)chunks, groups, ceil_div(heads / groups, 8));
    if (pad == 64) head_decay_chunk_kernel<1><<<grid, 256, 0, stream>>>(a, made);
    else if (pad == 128) head_decay_chunk_kernel<2><<<grid, 256, 0, stream>>>(a, made);
    else head_decay_chunk_kernel<4><<<grid, 256, 0, stream>>>(a, made);
    MI_CHECK_LAUNCH("head_decay_chunk");
  }
  WalkArgs p;
  p.made = made;
  p.v = (const bf16_t*)v, p.v_stride = v_stride, p.v_col = v_col, p.skip = skip;
  p.state = state, p.state_stride = state_stride, p.cu = cu, p.slots = slots, p.num_slots = num_slots;
  p.out = out, p.heads = heads, p.vdim = vdim;
  return mode == PER_CHANNEL ? launch_walk<PER_CHANNEL>(p, TokenRows<PER_CHANNEL>{a}, pad, num_tokens, num_requests, longest, stream)
                             : launch_walk<PER_HEAD>(p, TokenRows<PER_HEAD>{a}, pad, num_tokens, num_requests, longest, stream);
}
