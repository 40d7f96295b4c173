// The gated delta rule over many tokens of a request: see chunk_scan.h for the form, delta_rule.hip for the rule.
// The first launch, one block per (chunk, key/value head): unit q and k rows in float32, their products inside the
// chunk on the matrix cores, and per head the decays' quotients, W, and T by forward substitution.
#include "chunk_scan.h"
#include "delta_rule.h"

#include <math.h>

namespace {

using namespace chunk_scan;

// What walk_by_token takes of a token (it makes the unit vectors).
struct TokenRows {
  const bf16_t *qkv, *proj;
  int64_t qkv_stride, proj_stride;
  int col_b, col_a, kv_heads, dim;
  const float *a_log, *dt_bias;
  __device__ __forceinline__ void channel(int64_t t, int head, int heads, int d, float& q, float& k) const {
    const bf16_t* row = qkv + t * qkv_stride + head / (heads / kv_heads) * dim + d;
    q = to_f32(row[0]), k = to_f32(row[kv_heads * dim]);
  }
  __device__ __forceinline__ void head_gates(int64_t t, int head, float& decay, float& step) const {
    const bf16_t* gates = proj + t * proj_stride + head;
    const float z = to_f32(gates[col_a]) + dt_bias[head];
    decay = expf(-expf(a_log[head]) * (z > 20.f ? z : log1pf(expf(z))));
    step = 1.f / (1.f + expf(-to_f32(gates[col_b])));
  }
  __device__ __forceinline__ int width() const { return dim; }
};

// 256 threads: 8 of them bring one token's q and k rows in and make them unit vectors; then a wave makes a 16 x 16
// tile of each product; then a wave takes a head at a time.  The sums of the decays' logarithms are carried in
// 64-bit: a quotient is the exponential of a difference of two of them, and they grow with the chunk while it may
// be small.
template <int DT>
__global__ __launch_bounds__(256) void delta_chunk_kernel(const bf16_t* __restrict__ qkv, int64_t qkv_stride, const bf16_t* __restrict__ proj,
                                                          int64_t proj_stride, int col_b, int col_a, const float* __restrict__ a_log,
                                                          const float* __restrict__ dt_bias, const int* __restrict__ cu, int requests,
                                                          Made made, int heads, int dim, bool eights) {
  constexpr int PAD = 64 * DT, ROW = PAD + 4, EACH = PAD / 8;
  constexpr int ROWS_FLOATS = 2 * CHUNK * ROW, INNER = CHUNK * (CHUNK + 4);
  __shared__ __align__(16) float lds[ROWS_FLOATS > 6 * INNER ? ROWS_FLOATS : 6 * INNER];
  __shared__ int which;
  float *q_s = lds, *k_s = lds + CHUNK * ROW;                  // rows [CHUNK][ROW]; afterwards:
  float *kk_s = lds, *qk_s = lds + INNER, *l_s = lds + 2 * INNER;  // k . k, q . k, and L per wave, [CHUNK][CHUNK + 4]
  const int chunk = blockIdx.x, share = blockIdx.y, kv_heads = gridDim.y;
  const int b = request_of_chunk(chunk, cu, requests, &which);
  if (b < 0) return;
  const int t0 = cu[b] + (chunk - first_chunk(cu[b], b)) * CHUNK, nt = min(CHUNK, cu[b + 1] - t0);
  const int tid = threadIdx.x, wave = tid / MI_WAVE, lane = tid % MI_WAVE;
  if (cu[b + 1] - cu[b] == 1) {
    const bf16_t* row = qkv + (int64_t)t0 * qkv_stride + share * dim;
    const float q = tid < dim ? to_f32(row[tid]) : 0.f, k = tid < dim ? to_f32(row[kv_heads * dim + tid]) : 0.f;
    float sums[3] = {q * q, k * k, q * k};
    sum_of_block(sums, lds);
    const float q_inv = rsqrtf(sums[0] + 1e-6f) * (1.0f / sqrtf((float)dim)), k_inv = rsqrtf(sums[1] + 1e-6f);
    const int64_t at = ((int64_t)chunk * made.shares + share) * CHUNK * PAD + tid;
    if (tid < PAD) made.q[at] = q * q_inv, made.k[at] = k * k_inv;
    for (int h = share * (heads / kv_heads) + tid; h < (share + 1) * (heads / kv_heads); h += 256) {
      const int64_t of = (int64_t)chunk * heads + h;
      const bf16_t* p = proj + (int64_t)t0 * proj_stride;
      const float z = to_f32(p[col_a + h]) + dt_bias[h];
      const float gate = -(expf(a_log[h]) * (z > 20.f ? z : log1pf(expf(z))));
      made.factor[of * 2 * CHUNK] = expf(gate);
      made.factor[of * 2 * CHUNK + CHUNK] = expf(0.f * gate);
      made.within[of * CHUNK * CHUNK] = expf(0.f * gate) * (sums[2] * q_inv * k_inv);
      made.solve[of * CHUNK * CHUNK] = 1.f / (1.f + expf(-to_f32(p[col_b + h])));
    }
    return;
  }
  {
    const int token = tid / 8, sub = tid % 8;
    const bf16_t* row = qkv + (int64_t)(t0 + min(token, nt - 1)) * qkv_stride + share * dim;
    float q[EACH], k[EACH], qq = 0.f, kk = 0.f;
    row_values(row, sub * EACH, dim, eights, token < nt, q);
    row_values(row + kv_heads * dim, sub * EACH, dim, eights, token < nt, k);
#pragma unroll
    for (int e = 0; e < EACH; ++e) {
      qq = fmaf(q[e], q[e], qq);
      kk = fmaf(k[e], k[e], kk);
    }
#pragma unroll
    for (int off = 1; off < 8; off <<= 1) qq += __shfl_xor(qq, off, MI_WAVE), kk += __shfl_xor(kk, off, MI_WAVE);
    const float q_inv = rsqrtf(qq + 1e-6f) * (1.0f / sqrtf((float)dim)), k_inv = rsqrtf(kk + 1e-6f);
    const int64_t at = (((int64_t)chunk * made.shares + share) * CHUNK + token) * PAD + sub * EACH;
#pragma unroll
    for (int e = 0; e < EACH; e += 4) {
      const float4 q4 = make_float4(q[e] * q_inv, q[e + 1] * q_inv, q[e + 2] * q_inv, q[e + 3] * q_inv);
      const float4 k4 = make_float4(k[e] * k_inv, k[e + 1] * k_inv, k[e + 2] * k_inv, k[e + 3] * k_inv);
      *reinterpret_cast<float4*>(&q_s[token * ROW + sub * EACH + e]) = q4;
      *reinterpret_cast<float4*>(&k_s[token * ROW + sub * EACH + e]) = k4;
      *reinterpret_cast<float4*>(made.q + at + e) = q4;
      *reinterpret_cast<float4*>(made.k + at + e) = k4;
    }
  }
  __syncthreads();
  // k once more with its tokens side by side
  for (int i = tid; i < PAD * (CHUNK / 4); i += 256) {
    const int d = i % PAD, t = i / PAD * 4;
    *reinterpret_cast<float4*>(made.kt + (((int64_t)chunk * made.shares + share) * PAD + d) * CHUNK + t) =
        make_float4(k_s[t * ROW + d], k_s[(t + 1) * ROW + d], k_s[(t + 2) * ROW + d], k_s[(t + 3) * ROW + d]);
  }
  const int r = lane % 16, quad = lane / 16;
  f32x4_t kk = {0.f, 0.f, 0.f, 0.f}, qk = kk;
  const int ti = wave / 2, tj = wave % 2;  // (tile 0, 1 is above the diagonal and is not read)
#pragma unroll
  for (int d = 0; d < PAD; d += 16) {
    const float4 ki = load4(&k_s[(16 * ti + r) * ROW + d + 4 * quad]), kj = load4(&k_s[(16 * tj + r) * ROW + d + 4 * quad]);
    const float4 qi = load4(&q_s[(16 * ti + r) * ROW + d + 4 * quad]);
    const f32x4_t other = {kj.x, kj.y, kj.z, kj.w};
    kk = mma4(ki, other, kk);
    qk = mma4(qi, other, qk);
  }
  __syncthreads();  // the rows have been read
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    kk_s[(16 * ti + 4 * quad + e) * (CHUNK + 4) + 16 * tj + r] = kk[e];
    qk_s[(16 * ti + 4 * quad + e) * (CHUNK + 4) + 16 * tj + r] = qk[e];
  }
  __syncthreads();
  const int group = heads / kv_heads, i0 = lane % CHUNK;
  float* mine = l_s + wave * INNER;
  for (int h = share * group + wave; h < (share + 1) * group; h += 4) {
    const int64_t of = (int64_t)chunk * heads + h;
    // lane i and lane i + 32: token i's gates and the sum of the decays' logarithms up to it
    const bf16_t* p = proj + (int64_t)(t0 + min(i0, nt - 1)) * proj_stride;
    const float z = to_f32(p[col_a + h]) + dt_bias[h];
    const float soft = z > 20.f ? z : log1pf(expf(z));
    const float write = i0 < nt ? 1.f / (1.f + expf(-to_f32(p[col_b + h]))) : 0.f;
    double sum = i0 < nt ? -(double)(expf(a_log[h]) * soft) : 0.0;
#pragma unroll
    for (int off = 1; off < CHUNK; off <<= 1) {
      const double before = __shfl_up(sum, off, CHUNK);
      if (i0 >= off) sum += before;
    }
    const float g = expf((float)sum), tail = expf((float)(__shfl(sum, CHUNK - 1, CHUNK) - sum));
    if (lane < CHUNK) {
      float* factor = made.factor + of * 2 * CHUNK + lane;
      factor[0] = g, factor[CHUNK] = tail;
    }
    // column i0 of W and L, the rows shared out between the wave's halves
    float* within = made.within + of * CHUNK * CHUNK + i0;
#pragma unroll
    for (int n = 0; n < CHUNK / 2; ++n) {
      const int i = 2 * n + lane / CHUNK;
      const double sum_i = __shfl(sum, i, MI_WAVE);
      const float write_i = __shfl(write, i, MI_WAVE);
      const float quotient = i >= i0 ? expf((float)(sum_i - sum)) : 0.f;
      within[i * CHUNK] = i >= i0 ? quotient * qk_s[i * (CHUNK + 4) + i0] : 0.f;
      mine[i * (CHUNK + 4) + i0] = i > i0 ? write_i * quotient * kk_s[i * (CHUNK + 4) + i0] : 0.f;
    }
    // (a wave's own LDS, whose accesses keep their order)
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    // column i0 of T: t_i = (i == i0) - sum over j < i of L_ij t_j
    float t[CHUNK];
    float* solve = made.solve + of * CHUNK * CHUNK + i0;
#pragma unroll
    for (int i = 0; i < CHUNK; ++i) {
      float part[4] = {i == i0 ? 1.f : 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int j = 0; j < i; j += 4) {
        const float4 l = load4(&mine[i * (CHUNK + 4) + j]);
        part[0] = fmaf(-l.x, t[j], part[0]);
        if (j + 1 < i) part[1] = fmaf(-l.y, t[j + 1], part[1]);
        if (j + 2 < i) part[2] = fmaf(-l.z, t[j + 2], part[2]);
        if (j + 3 < i) part[3] = fmaf(-l.w, t[j + 3], part[3]);
      }
      t[i] = (part[0] + part[1]) + (part[2] + part[3]);
      if (lane < CHUNK) solve[i * CHUNK] = t[i] * write;
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  }
}

}  // namespace

// Floats of scratch that mi_gated_delta_chunks takes; 0: sizes it does not take.
extern "C" int64_t mi_gated_delta_chunks_scratch(int num_tokens, int num_requests, int heads, int kv_heads, int dim, int vdim) {
  if (num_tokens <= 0 || num_requests <= 0 || dim > 256 || vdim > 256 || vdim <= 0 || heads <= 0 || kv_heads <= 0 || kv_heads > 65535) return 0;
  const int pad = mi_gated_delta_rows(dim, vdim);
  return chunk_count(num_tokens, num_requests) * ((int64_t)3 * kv_heads * CHUNK * pad + (int64_t)heads * (2 * CHUNK * CHUNK + 2 * CHUNK));
}

// As mi_gated_delta for bfloat16, with `scratch` on 16 bytes; longest: tokens of the longest portion, 0: not known.
extern "C" int mi_gated_delta_chunks(const void* qkv, int64_t qkv_stride, const void* proj, int64_t proj_stride, int col_b, int col_a,
                                     int col_g, const float* a_log, const float* dt_bias, const float* norm_weight, float* state,
                                     int64_t state_stride, const int* cu, const int* slots, float* readout, float* scratch, void* out,
                                     int64_t out_stride, int num_tokens, int num_requests, int longest, int heads, int kv_heads, int dim,
                                     int vdim, int dim_pad, float eps, int num_slots, hipStream_t stream) {
  const int bad = mi_gated_delta_check(qkv_stride, proj_stride, col_b, col_a, col_g, state, state_stride, out_stride, num_requests, heads,
                                       kv_heads, dim, vdim, dim_pad, eps, num_slots);
  if (bad != MI_OK) return bad;
  if (num_requests == 0 || num_tokens == 0) return MI_OK;
  MI_REQUIRE(readout != nullptr && scratch != nullptr && (uintptr_t)scratch % 16 == 0, "gated_delta_chunks: no buffers");
  MI_REQUIRE(mi_gated_delta_chunks_scratch(num_tokens, num_requests, heads, kv_heads, dim, vdim) > 0, "gated_delta_chunks: sizes it does not take");
  const int64_t chunks = chunk_count(num_tokens, num_requests), rows = chunks * kv_heads * CHUNK * dim_pad;
  MI_REQUIRE(chunks <= 2147483647 && qkv_stride < MAX_ROW && (int64_t)heads * vdim < MAX_ROW, "gated_delta_chunks: sizes it does not take");
  Made made;
  made.q = scratch, made.k = made.q + rows, made.kt = made.k + rows;
  made.within = made.kt + rows, made.solve = made.within + chunks * heads * CHUNK * CHUNK;
  made.factor = made.solve + chunks * heads * CHUNK * CHUNK;
  made.fade = nullptr;
  made.shares = kv_heads;
  dim3 grid((unsigned)chunks, kv_heads);
#define MI_DELTA_CHUNKS(DT)                                                                                              \
  delta_chunk_kernel<DT><<<grid, 256, 0, stream>>>((const bf16_t*)qkv, qkv_stride, (const bf16_t*)proj, proj_stride, \
                                                           col_b, col_a, a_log, dt_bias, cu, num_requests, made, heads, dim, \
                                                   in_eights(qkv, qkv_stride, 0, dim))
  if (dim_pad == 64) MI_DELTA_CHUNKS(1);
  else if (dim_pad == 128) MI_DELTA_CHUNKS(2);
  else MI_DELTA_CHUNKS(4);
#undef MI_DELTA_CHUNKS
  MI_CHECK_LAUNCH("delta_chunk");
  WalkArgs p;
  p.made = made;
  p.v = (const bf16_t*)qkv, p.v_stride = qkv_stride, p.v_col = 2 * kv_heads * dim;
  p.skip = nullptr;
  p.state = state, p.state_stride = state_stride, p.cu = cu, p.slots = slots, p.num_slots = num_slots;
  p.out = readout, p.heads = heads, p.vdim = vdim;
  const TokenRows rows_of = {(const bf16_t*)qkv, (const bf16_t*)proj, qkv_stride, proj_stride, col_b, col_a, kv_heads, dim, a_log, dt_bias};
  const int walked = launch_walk<DELTA>(p, rows_of, dim_pad, num_tokens, num_requests, longest, stream);
  if (walked != MI_OK) return walked;
  return mi_delta_readout_norm(MI_BF16, readout, proj, proj_stride, col_g, norm_weight, out, out_stride, num_tokens, heads, vdim, eps, stream);
}
