// Shared helpers of the HIP kernels: element types, wave reductions, error reporting.
// Everything here is written for gfx950 (CDNA4): 64-lane waves, 160 KB LDS per CU.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

typedef __bf16 bf16_t;

#define MI_WAVE 64

// Every entry point returns 0 on success.  On refusal it returns a negative code
// and leaves a message that mi_last_error() returns.
#define MI_OK 0
#define MI_ERR_SHAPE (-1)
#define MI_ERR_LAUNCH (-2)
#define MI_ERR_LIMIT (-3)

void mi_set_error(const char* fmt, ...);

#define MI_REQUIRE(cond, ...)        \
  do {                               \
    if (!(cond)) {                   \
      mi_set_error(__VA_ARGS__);     \
      return MI_ERR_SHAPE;           \
    }                                \
  } while (0)

#define MI_CHECK_LAUNCH(name)                                               \
  do {                                                                      \
    hipError_t mi_err_ = hipGetLastError();                                 \
    if (mi_err_ != hipSuccess) {                                            \
      mi_set_error("%s: launch failed: %s", name, hipGetErrorString(mi_err_)); \
      return MI_ERR_LAUNCH;                                                 \
    }                                                                       \
  } while (0)

// dtype codes shared with the Python side
#define MI_F32 0
#define MI_BF16 1

__device__ __forceinline__ float to_f32(float v) { return v; }
__device__ __forceinline__ float to_f32(bf16_t v) { return (float)v; }

template <typename T>
__device__ __forceinline__ T from_f32(float v);
template <>
__device__ __forceinline__ float from_f32<float>(float v) { return v; }
template <>
__device__ __forceinline__ bf16_t from_f32<bf16_t>(float v) { return (bf16_t)v; }

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8_t;
typedef int int32x4_t __attribute__((ext_vector_type(4)));

// How a weight-streaming product reads its weights ("LINES" in the kernels).  The matrix-core
// operand wants, per k-step (32 elements), 16 bytes of each of 16 weight rows in every 16
// lanes: four lanes a row, 64 bytes, half a cache line; the other half is asked for by the
// next k-step's load.  Whole lines per load run faster, and non-temporal loads (the weights
// are read once) faster again, but only on whole lines.  Measured on MI355X, microseconds for
// 6144 x 4096 / 4096 x 14336 / 28672 x 4096 / 128256 x 4096 at 8 rows, weights not in any
// cache: half lines 13.5 / 30.1 / 46.3 / 192; non-temporal on half lines slower (28672 x
// 4096: 47.5-50.1 in a kernel that only reads); whole lines with every 16 lanes on 8 lines and
// an exchange inside the 16 lanes 14.8 / 27.7 / 42.3 / 168; whole lines with every 8 lanes
// on one line (this) 11.4 / 23.8 / 40.0 / 168.  A long plain read reaches 6.1-6.3 TB/s, a
// non-temporal one 7.0-7.1 TB/s.
// So a load takes 8 rows x 128 bytes (two k-steps): lane l reads 16-byte chunk l % 8 of the
// line of row l / 8 of the tile's lower or upper 8 rows.  Of a pair of such loads (lower rows,
// upper rows) the lanes with chunks 4-7 of the first and those with chunks 0-3 of the second
// change places (inside every 16 lanes: two DPP moves), which sorts the chunks by k-step; then
// every lane fetches its operand's 16 bytes from the lane that holds them (ds_bpermute, which
// moves data between lanes through the LDS crossbar without touching LDS memory).
// Needs: rows of the matrix on 128-byte boundaries, k-steps taken in even-aligned pairs.
__device__ __forceinline__ void lines_to_operands(bf16x8_t& lower_rows, bf16x8_t& upper_rows) {
  int32x4_t lo = __builtin_bit_cast(int32x4_t, lower_rows), hi = __builtin_bit_cast(int32x4_t, upper_rows);
  // operand lane (quad, col) wants row col, chunk quad of its k-step: after the exchange that
  // is lane 8 * (col % 8) + 4 * (col / 8) + quad
  const int lane = threadIdx.x % MI_WAVE, col = lane % 16, quad = lane / 16;
  const int from = 4 * (8 * (col % 8) + 4 * (col / 8) + quad);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const int lo_was = lo[e];
    // row_shr:4 into lanes 4-7 and 12-15 of every 16: the upper rows' chunks 0-3 (first k-step)
    lo[e] = __builtin_amdgcn_update_dpp(lo[e], hi[e], 0x114, 0xF, 0xA, false);
    // row_shl:4 into lanes 0-3 and 8-11: the lower rows' chunks 4-7 (second k-step)
    hi[e] = __builtin_amdgcn_update_dpp(hi[e], lo_was, 0x104, 0xF, 0x5, false);
    lo[e] = __builtin_amdgcn_ds_bpermute(from, lo[e]);
    hi[e] = __builtin_amdgcn_ds_bpermute(from, hi[e]);
  }
  lower_rows = __builtin_bit_cast(bf16x8_t, lo);  // operand of the pair's first k-step
  upper_rows = __builtin_bit_cast(bf16x8_t, hi);  // operand of its second
}

// The row (0..7 of the lower or upper 8) whose line a lane reads, and its 16-byte chunk of
// that line as a byte offset.
__device__ __forceinline__ int line_row_of_lane(int lane) { return lane / 8; }
__device__ __forceinline__ uint32_t line_chunk_of_lane(int lane) { return (uint32_t)(lane % 8) * 16u; }

// One of the loads below by itself.
__device__ __forceinline__ bf16x8_t load_line(const void* matrix, int64_t first_kstep, uint32_t at) {
  using global_bytes = const __attribute__((address_space(1))) char;
  using global_chunk = const __attribute__((address_space(1))) bf16x8_t;
  uint64_t base_bits = reinterpret_cast<uint64_t>(matrix) + (uint64_t)first_kstep * 64u;
  asm("" : "+s"(base_bits));
  asm("" : "+v"(at));
  return __builtin_nontemporal_load((global_chunk*)((global_bytes*)base_bits + at));
}

// The two loads of a pair of k-steps, non-temporal unless other blocks read the same rows (ONCE false): base (uniform, kept in
// scalar registers) + the lane's offsets.
template <bool ONCE = true>
__device__ __forceinline__ void load_line_pair(const void* matrix, int64_t first_kstep, uint32_t lower_at,
                                               uint32_t upper_at, bf16x8_t& lower_rows, bf16x8_t& upper_rows) {
  using global_bytes = const __attribute__((address_space(1))) char;
  using global_chunk = const __attribute__((address_space(1))) bf16x8_t;
  uint64_t base_bits = reinterpret_cast<uint64_t>(matrix) + (uint64_t)first_kstep * 64u;
  asm("" : "+s"(base_bits));  // scalar: the lanes add their 32-bit offsets
  global_bytes* base = (global_bytes*)base_bits;
  // (opaque to the compiler, or it widens the offsets to 64 bits once and for all and adds
  // whole addresses in vector registers for every load)
  asm("" : "+v"(lower_at), "+v"(upper_at));
  if constexpr (ONCE) {
    lower_rows = __builtin_nontemporal_load((global_chunk*)(base + lower_at));
    upper_rows = __builtin_nontemporal_load((global_chunk*)(base + upper_at));
  } else {
    lower_rows = *(global_chunk*)(base + lower_at);
    upper_rows = *(global_chunk*)(base + upper_at);
  }
}

// (float32 elements: evaluated in 64-bit and rounded once; the float32 exponential and two more
// roundings put the result 4.7e-8 away on average, twice what rounding alone costs)
template <typename T>
__device__ __forceinline__ float silu_times(float g, float u) {
  if constexpr (sizeof(T) == 4) return (float)((double)g / (1.0 + exp(-(double)g)) * (double)u);
  else return g / (1.f + expf(-g)) * u;
}

// 1 / (1 + exp(-z)) in float32 on the hardware's exponential and reciprocal (v_exp_f32, v_rcp_f32:
// one ulp each).  The library's expf and an IEEE division cost some 70 instructions per gate,
// and a prompt's gated recurrence was bound by them, not by memory (2,048 x 4,096 gates: 17 us
// of arithmetic).  Every kernel that evaluates a gate of the recurrence uses this one function,
// so a token's state does not depend on which kernel its step ran.
__device__ __forceinline__ float mi_logistic(float z) {
  return __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(z * -1.4426950408889634f));
}

__device__ __forceinline__ float wave_max(float v) {
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, MI_WAVE));
  return v;
}

__device__ __forceinline__ float wave_sum(float v) {
#pragma unroll
  for (int off = MI_WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, MI_WAVE);
  return v;
}

// Sum over a whole block in a fixed order: lanes by butterfly, waves one after another.
// `scratch` holds at least blockDim.x / 64 floats.  All threads get the result.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  v = wave_sum(v);
  const int wave = threadIdx.x / MI_WAVE;
  const int lane = threadIdx.x % MI_WAVE;
  const int n_waves = (blockDim.x + MI_WAVE - 1) / MI_WAVE;
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < n_waves; ++w) total += scratch[w];
  return total;
}

// V columns of a row at once: 16-byte loads of float32, 8-byte loads of bfloat16 for V = 4.
template <typename T, int V>
__device__ __forceinline__ void mi_load_cols(const T* p, float (&v)[V]) {
  if constexpr (V == 1) {
    v[0] = to_f32(p[0]);
  } else if constexpr (sizeof(T) == 4) {
    const float4 got = *reinterpret_cast<const float4*>(p);
    v[0] = got.x, v[1] = got.y, v[2] = got.z, v[3] = got.w;
  } else {
    const uint2 got = *reinterpret_cast<const uint2*>(p);
    v[0] = __uint_as_float(got.x << 16), v[1] = __uint_as_float(got.x & 0xFFFF0000u);
    v[2] = __uint_as_float(got.y << 16), v[3] = __uint_as_float(got.y & 0xFFFF0000u);
  }
}

template <typename T, int V>
__device__ __forceinline__ void mi_store_cols(T* p, const float (&v)[V]) {
  if constexpr (V == 1) {
    p[0] = from_f32<T>(v[0]);
  } else if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
  } else {
    union {
      bf16_t h[4];
      uint2 bits;
    } packed;
#pragma unroll
    for (int j = 0; j < 4; ++j) packed.h[j] = from_f32<bf16_t>(v[j]);
    *reinterpret_cast<uint2*>(p) = packed.bits;
  }
}

// Transposed value pages keep a dim's slots side by side.  Where a step's tokens fill a whole page in order (a prompt's
// portion) a dim's row of the page is written at once, 16 bytes a store, and the page's tokens share the (head, dim)
// rows among them, each taking one page_size-th: all of them on the page's first token measured 18.1 us for 2,048
// tokens of 8 heads of 128, shared out 11 us.  (Norm, mixing and writing of 1,501 tokens of 24 query and 8 key/value heads
// of 128: 19.9 us an element a store, 11.5 so.)
//
// Looking costs a dependent read of the slots, 0.2 to 0.4 us a launch, so where a few decoded tokens cannot fill a page and the kernel
// has nothing to wait for beside it only steps from MI_LOOK_FOR_PAGES tokens on look (norm and writing of 24 query and 8 key/value
// heads of 128, microseconds without and with: 30 decoded tokens 3.6, 4.0; 128 tokens in order 4.4, 3.9; 300 7.2, 4.6).
constexpr int MI_LOOK_FOR_PAGES = 128;

// Whether token t, whose slot is page * page_size + off, lies in such a page.  Called by whole waves.
__device__ __forceinline__ bool mi_fills_page(const int* slot_mapping, int t, int page, int off, int page_size, int num_tokens) {
  const int lead = t - off;
  if (page_size % 8 != 0 || lead < 0 || lead + page_size > num_tokens) return false;
  bool differs = false;
  for (int i = threadIdx.x % MI_WAVE; i < page_size; i += MI_WAVE) differs = differs || slot_mapping[lead + i] != page * page_size + i;
  return __ballot(differs) == 0;
}

// Token t's share of its page's rows (pages on 16 bytes): value_of(token, e) is the float32 value of (head, dim) e = head * v_dim + dim of a
// token.  first, stride: of the threads that share the work of token t.
template <typename T, typename F>
__device__ __forceinline__ void mi_write_page_rows(T* v_pages, int t, int page, int off, int page_size, int kv_heads, int v_dim,
                                                   int first, int stride, F value_of) {
  const int lead = t - off, rows = kv_heads * v_dim, rows_each = (rows + page_size - 1) / page_size;
  const int e_end = min((off + 1) * rows_each, rows);
  for (int e = off * rows_each + first; e < e_end; e += stride) {
    T* dst = v_pages + ((int64_t)page * rows + e) * page_size;
    for (int i0 = 0; i0 < page_size; i0 += 8) {
      float x[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) x[i] = value_of(lead + i0 + i, e);
      alignas(16) T out[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) out[i] = from_f32<T>(x[i]);
#pragma unroll
      for (int i = 0; i < (int)sizeof(out) / 16; ++i) reinterpret_cast<uint4*>(dst + i0)[i] = reinterpret_cast<const uint4*>(out)[i];
    }
  }
}

// The two elements of a head that are rotated together.  Each is one product, rounded, and one fused multiply-add; which of an element's two products
// is rounded shows in its last bit, and left to the compiler that differed from kernel to kernel.
__device__ __forceinline__ void mi_rotate(float x0, float x1, float c, float s, float& y0, float& y1) {
  y0 = __builtin_fmaf(x0, c, -(x1 * s));
  y1 = __builtin_fmaf(x1, c, x0 * s);
}

static __host__ __device__ inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
static inline int64_t ceil_div64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Compute units of the current device (asked once per device).
static inline int mi_compute_units() {
  static int cached[64] = {0};
  int device = 0;
  if (hipGetDevice(&device) != hipSuccess || device < 0 || device >= 64) return 0;
  if (cached[device] == 0) {
    int count = 0;
    if (hipDeviceGetAttribute(&count, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess) return 0;
    cached[device] = count;
  }
  return cached[device];
}
