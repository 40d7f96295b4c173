// True float32 matrix product for the 32-bit path: C[M,N] = A[M,K] * W[N,K]^T.
// No reduced-precision matrix mode: float32 values are widened to 64-bit (exactly) and
// multiplied and summed by the matrix cores' 64-bit instruction, and the sum is rounded to
// float32 once, when it is written: an output differs from the exact product of its float32
// operands by that one rounding (relative 2.5e-8 on average), whatever K is.  (Float32 sums
// in 16-deep slices added up with compensation measured 8e-8 at K = 4,096, a plain float32
// sum 2.7e-6; over 32 layers such errors are what the logits show.)
//
// Every output is summed in one fixed order that depends on K alone, in both kernels here, so
// a row gives the same bits however many other rows its step has and wherever its tile lies:
// K is cut into SEGMENTS runs of whole 32-value slices; inside a run one accumulator takes,
// slice by slice, the slice's lower and then upper 16 values, of these the values 0, 4, 8, 12
// first, then 1, 5, 9, 13 and so on (a lane of the matrix instruction's operand holds four
// values that lie side by side, one of them per instruction); the runs' sums are added in
// order.  Values past K are zeros and add nothing, exactly.
//
// What bounds it: the 64-bit matrix instruction (16x16x4) takes 64 cycles a SIMD, 76 TFLOP/s on
// the whole part (the vector pipe's 64-bit multiply-add reached 51, and needs a widened operand
// in registers for every one of them; the instruction shares it among 16 products).
#include "gemm_f32_lines.h"

#define BN 64

// four values of a row from `at` on, zeros past its end
template <bool ALIGNED>
__device__ __forceinline__ float4 four_of_row(const float* row, int at, int k) {
  if constexpr (ALIGNED) return at < k ? *reinterpret_cast<const float4*>(row + at) : make_float4(0.f, 0.f, 0.f, 0.f);
  return make_float4(at < k ? row[at] : 0.f, at + 1 < k ? row[at + 1] : 0.f, at + 2 < k ? row[at + 2] : 0.f,
                     at + 3 < k ? row[at + 3] : 0.f);
}

// What lies between the matrices of one head and the next where a launch makes the products of several side by side (elements).
struct Heads {
  int64_t a, w, c;
};

// Many rows: a block of 4 waves owns BM x 64 outputs, STAGE slices of both operands in LDS, the next ones in
// flight in registers.  With 64 cycles an instruction the LDS is idle most of the time, so small tiles cost
// nothing.  BM = 64 (a wave 32 x 32), one slice a stage, where there are at least four blocks a CU to cover one
// another's barriers and loads; else BM = 32 (a wave 32 x 16): twice the blocks, four slices a stage where a run is whole stages, else one.
// ALIGNED: 16-byte loads (K, both row strides multiples of 4 values, both matrices on 16 bytes).
template <int BM, int STAGE, bool ALIGNED>
__global__ __launch_bounds__(256) void gemm_f32_kernel(const float* __restrict__ a, int64_t lda,
                                                       const float* __restrict__ w, int64_t ldw,
                                                       float* __restrict__ c, int64_t ldc, int m, int n, int k, Heads heads) {
  constexpr int LDS_ROW = STAGE * SLICE + 4;  // floats: 16-byte reads of 16 rows fall on different banks
  constexpr int CT = BM == 64 ? 2 : 1;  // 16-column tiles of a wave (it has two tiles of rows)
  constexpr int AL = STAGE * BM / 32, WL = STAGE * BN / 32;  // 16-byte pieces a thread stages
  __shared__ __attribute__((aligned(16))) float a_s[BM][LDS_ROW];
  __shared__ __attribute__((aligned(16))) float w_s[BN][LDS_ROW];
  a += (int64_t)blockIdx.z * heads.a, w += (int64_t)blockIdx.z * heads.w, c += (int64_t)blockIdx.z * heads.c;
  const int tid = threadIdx.x, wave = tid / MI_WAVE, lane = tid % MI_WAVE;
  const int row0 = blockIdx.y * BM, col0 = blockIdx.x * BN;
  const int wave_row = BM == 64 ? wave / 2 * 32 : 0, wave_col = BM == 64 ? wave % 2 * 32 : wave * 16;
  const int r = lane % 16, quad = lane / 16;
  constexpr int LANES = STAGE * SLICE / 4, ROWS = 256 / LANES;  // threads a row, rows a pass of the block's loads
  const int l_row = tid / LANES, l_k = tid % LANES * 4;

  // (rows past the last one repeat it and are not written: no branch around a load but one for the whole block, where K
  // ends inside a stage; with a branch around each load 509 x 2048 x 2048 took 91 us instead of 87)
  const float *a_row[AL], *w_row[WL];
#pragma unroll
  for (int i = 0; i < AL; ++i) a_row[i] = a + (int64_t)min(row0 + l_row + ROWS * i, m - 1) * lda + (ALIGNED ? l_k : 0);
#pragma unroll
  for (int i = 0; i < WL; ++i) w_row[i] = w + (int64_t)min(col0 + l_row + ROWS * i, n - 1) * ldw + (ALIGNED ? l_k : 0);
  float4 a_next[AL], w_next[WL];
  auto fetch = [&](int k0) {
    if (ALIGNED && k0 + STAGE * SLICE <= k) {
#pragma unroll
      for (int i = 0; i < AL; ++i) a_next[i] = *reinterpret_cast<const float4*>(a_row[i] + k0);
#pragma unroll
      for (int i = 0; i < WL; ++i) w_next[i] = *reinterpret_cast<const float4*>(w_row[i] + k0);
    } else {
#pragma unroll
      for (int i = 0; i < AL; ++i) a_next[i] = four_of_row<ALIGNED>(a_row[i] - (ALIGNED ? l_k : 0), k0 + l_k, k);
#pragma unroll
      for (int i = 0; i < WL; ++i) w_next[i] = four_of_row<ALIGNED>(w_row[i] - (ALIGNED ? l_k : 0), k0 + l_k, k);
    }
  };
  f64x4_t total[2][CT], acc[2][CT];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) total[i][j] = acc[i][j] = f64x4_t{0.0, 0.0, 0.0, 0.0};

  const int run = segment_slices(k), slices = ceil_div(k, SLICE);
  int left = run;  // slices until the run's sum is complete
  fetch(0);
  for (int slice0 = 0; slice0 < slices; slice0 += STAGE) {
    __syncthreads();  // the last slices' reads are done
#pragma unroll
    for (int i = 0; i < AL; ++i) *reinterpret_cast<float4*>(&a_s[l_row + ROWS * i][l_k]) = a_next[i];
#pragma unroll
    for (int i = 0; i < WL; ++i) *reinterpret_cast<float4*>(&w_s[l_row + ROWS * i][l_k]) = w_next[i];
    __syncthreads();
    if (slice0 + STAGE < slices) fetch((slice0 + STAGE) * SLICE);
#pragma unroll
    for (int slice = 0; slice < STAGE; ++slice) {  // (a slice past the last one is zeros)
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int at = SLICE * slice + 16 * half + 4 * quad;
        float av[2][4], wv[CT][4];
#pragma unroll
        for (int i = 0; i < 2; ++i)
          *reinterpret_cast<float4*>(av[i]) = *reinterpret_cast<const float4*>(&a_s[wave_row + 16 * i + r][at]);
#pragma unroll
        for (int j = 0; j < CT; ++j)
          *reinterpret_cast<float4*>(wv[j]) = *reinterpret_cast<const float4*>(&w_s[wave_col + 16 * j + r][at]);
#pragma unroll
        for (int s = 0; s < 4; ++s)
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < CT; ++j) acc[i][j] = mma(av[i][s], wv[j][s], acc[i][j]);
      }
    }
    // (runs are whole stages: looked at after every slice, the sums went through other registers and back each time, with
    // the matrix pipe drained: 87 us instead of 82 at 509 x 2048 x 2048)
    left -= STAGE;
    if (left == 0) {
      left = run;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) {
          total[i][j] += acc[i][j];
          acc[i][j] = f64x4_t{0.0, 0.0, 0.0, 0.0};
        }
    }
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) total[i][j] += acc[i][j];  // (the last run may be short)
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        // (the 64-bit instruction's result: register e of a lane is row 4 * e + lane / 16)
        const int row = row0 + wave_row + 16 * i + 4 * e + quad, col = col0 + wave_col + 16 * j + r;
        if (row < m && col < n) c[(int64_t)row * ldc + col] = (float)total[i][j][e];
      }
}

// The same without a branch around the load, for loads that stay in flight (the row's first values where it has ended, masked).
template <bool ALIGNED>
__device__ __forceinline__ float4 four_in_flight(const float* row, int at, int k) {
  uint32_t bits[4];
  if constexpr (ALIGNED) {
    const uint4 got = *reinterpret_cast<const uint4*>(row + (at < k ? at : 0));
    bits[0] = got.x, bits[1] = got.y, bits[2] = got.z, bits[3] = got.w;
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) bits[e] = __float_as_uint(row[at + e < k ? at + e : 0]);
  }
#pragma unroll
  for (int e = 0; e < 4; ++e) bits[e] &= at + e < k ? ~0u : 0u;
  return make_float4(__uint_as_float(bits[0]), __uint_as_float(bits[1]), __uint_as_float(bits[2]), __uint_as_float(bits[3]));
}

// Up to a few hundred rows (those that gemm_f32_few_kernel does not take): bound by the matrix instruction, or by what a CU brings in where there are few
// rows.  A block owns 16 * RT rows and 16 * FT features, as many as leave a block for every CU (f32_micros); its 8 waves take
// one run of K each (the order above), every wave streams its part of the weights from memory, two slices ahead,
// and the runs' sums meet in LDS.  LINES: whole lines of W, non-temporal, brought into operand order by lane
// exchanges (common.h): rows of W on 128 bytes, K a multiple of 32, A on 16 bytes.  PIECES: 16 bytes a load in operand order
// (K and both strides in whole 4s, both matrices on 16 bytes); VALUES: single ones.
// Rows past m and features past n repeat the last one and are not written.
enum { VALUES = 0, PIECES = 1, LINES = 2 };

template <int RT, int FT, int FORM>
__global__ __launch_bounds__(SEGMENTS * MI_WAVE) void gemm_f32_rows_kernel(const float* __restrict__ a, int64_t lda,
                                                            const float* __restrict__ w, int64_t ldw,
                                                            float* __restrict__ c, int64_t ldc, int m, int n, int k, int row_tiles, int total, Heads heads) {
  constexpr int AT_ONCE = RT * FT < 4 ? RT * FT : 4;  // tiles whose runs' sums meet in LDS at a time
  __shared__ double sums[SEGMENTS][AT_ONCE][16][17];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), lane = threadIdx.x % MI_WAVE;
  // (consecutive places go to one XCD: the row tiles that read the same rows of W run at the same time behind one L2)
  const int place = row_tiles > 1 ? (int)(blockIdx.x % 8 * (gridDim.x / 8) + blockIdx.x / 8) : (int)blockIdx.x;
  if (place >= total) return;
  const int row0 = place % row_tiles * (16 * RT), col0 = place / row_tiles * (16 * FT);
  a += (int64_t)blockIdx.y * heads.a + (int64_t)row0 * lda, w += (int64_t)blockIdx.y * heads.w, c += (int64_t)blockIdx.y * heads.c + (int64_t)row0 * ldc;
  m -= row0;
  const int r = lane % 16, quad = lane / 16;
  const float* a_row[RT];
  f64x4_t acc[RT][FT];
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    a_row[i] = a + (int64_t)min(16 * i + r, m - 1) * lda;
#pragma unroll
    for (int f = 0; f < FT; ++f) acc[i][f] = f64x4_t{0.0, 0.0, 0.0, 0.0};
  }
  const int run = segment_slices(k), slices = ceil_div(k, SLICE);
  const int first = min(wave * run, slices), last = min(first + run, slices);

  if constexpr (FORM == LINES) {
    // (offsets from the first of the block's rows: at most 32 rows of at most 2^26 bytes)
    uint32_t lower[FT], upper[FT];
#pragma unroll
    for (int f = 0; f < FT; ++f) {
      const int row = 16 * f + line_row_of_lane(lane), most = n - 1 - col0;
      lower[f] = (uint32_t)min(row, most) * (uint32_t)(ldw * 4) + line_chunk_of_lane(lane);
      upper[f] = (uint32_t)min(row + 8, most) * (uint32_t)(ldw * 4) + line_chunk_of_lane(lane);
    }
    lines_product<RT, FT>(w + (int64_t)col0 * ldw, lower, upper, a_row, first, last, acc);
  } else {
    constexpr int AHEAD = 2;
    const float* w_row[FT];
#pragma unroll
    for (int f = 0; f < FT; ++f) w_row[f] = w + (int64_t)min(col0 + 16 * f + r, n - 1) * ldw;
    float4 wv[AHEAD][FT][2], xv[AHEAD][RT][2];
    auto fetch = [&](int slot, int slice) {
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int at = slice * SLICE + 16 * half + 4 * quad;
#pragma unroll
        for (int f = 0; f < FT; ++f) wv[slot][f][half] = four_in_flight<FORM == PIECES>(w_row[f], at, k);
#pragma unroll
        for (int i = 0; i < RT; ++i) xv[slot][i][half] = four_in_flight<FORM == PIECES>(a_row[i], at, k);
      }
    };
#pragma unroll
    for (int s = 0; s < AHEAD; ++s)
      if (first + s < last) fetch(s, first + s);
    for (int at = first; at < last; at += AHEAD) {
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) {
        if (at + s < last) {
          float ws[FT][2][4], xs[RT][2][4];
          __builtin_memcpy(ws, wv[s], sizeof(ws));
          __builtin_memcpy(xs, xv[s], sizeof(xs));
          if (at + s + AHEAD < last) fetch(s, at + s + AHEAD);
#pragma unroll
          for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int i = 0; i < RT; ++i)
#pragma unroll
                for (int f = 0; f < FT; ++f) acc[i][f] = mma(xs[i][half][e], ws[f][half][e], acc[i][f]);
        }
      }
    }
  }
#pragma unroll
  for (int t0 = 0; t0 < RT * FT; t0 += AT_ONCE) {
    if (t0 > 0) __syncthreads();
#pragma unroll
    for (int t = t0; t < t0 + AT_ONCE; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) sums[wave][t - t0][4 * e + quad][r] = acc[t / FT][t % FT][e];
    __syncthreads();
    for (int at = threadIdx.x; at < 256 * AT_ONCE; at += SEGMENTS * MI_WAVE) {
      const int tile = t0 + at / 256, row = tile / FT * 16 + at / 16 % 16, col = col0 + tile % FT * 16 + at % 16;
      double whole = 0.0;
#pragma unroll
      for (int s = 0; s < SEGMENTS; ++s) whole += sums[s][at / 256][at / 16 % 16][at % 16];
      if (row < m && col < n) c[(int64_t)row * ldc + col] = (float)whole;
    }
  }
}

// The same for up to 4 * G rows, of which the instruction above would leave most of its 16 idle: the 64-bit instruction of
// four 4x4 products (4x4x4) takes a quarter of its time and keeps W where it has it (a lane's feature is lane % 16, its piece of K lane / 16; a
// row of A is lane % 4), and sums in the same order, so a row gives the same bits.  Rows of A go through LDS, a wave's own run of them
// CHUNK slices at a time: read from memory like W, they were a load for every one of W's (gate|up at 3 rows without them 27 -> 25 us, without
// the products 21).  Form LINES only.  A block owns FEATURES features and all of K, eight waves a run each; 8 features where 16 would
// leave half of the CUs without a block (the upper eight of the operand then repeat the lower ones and are not written).
//
// Deeper prefetch is no better (the output head at 8 slices 192 us, 151 at 2 and 4): blocks beside one another on a CU cover the
// waits.  Microseconds at 3 rows (1B sizes), before -> after: q|k|v 3072 x 2048 9.3 -> 7.9, o 2048 x 2048 8.8 -> 7.0, down 2048 x 8192
// 28.4 -> 20.4, gate|up 16384 x 2048 30.4 -> 22.6, head 128256 x 2048 180 -> 151 (6.9 TB/s); at 7 rows (two slices ahead) 9.1 -> 8.8, 8.9 -> 8.7,
// 30.7 -> 25.7, 184 -> 180, and above 16 slices a run no better than with one 16 x 16 product (2048 x 8192 29.1 against 28.5, 4096 x 14336
// 48.8 / 47.6), so those stay.
//
// GATED: W is [gate; up], n features each; a block's operand holds the gate rows of 8 features and the up rows of the same, and
// silu(gate) * up is written, both products rounded to float32 first, as silu_mul takes them (the same bits, a launch less: 1B with 3 requests
// decoding 1,688 -> 1,658 us a step).
//
// FEW_ROPE: q|k|v, rotated and written where they belong; a block holds 8 features of the first half of a head and the 8 that they are turned with.
// 1B with 3 requests decoding 1,656 -> 1,619 us a step.  (With the norms in the products around them too, their factors applied to the 64-bit sums,
// 1,571, but that rounds elsewhere than the norm's launch in front of more rows: a request's logits changed when a fifth one joined.  The
// factor first, its sum in the order of that launch, has every block add up all rows' squares: o, norm and gate|up of 3 rows at those sizes 33.6 ->
// 38.6 us.)
enum { FEW_PLAIN = 0, FEW_GATED = 1, FEW_ROPE = 2, FEW_HEADS = 3 };  // (FEW_HEADS: plain, a product a head)

struct FewRows {  // what FEW_ROPE has beside the product (see the entry)
  const float *cos_t, *sin_t;  // [m][half]
  const int* slots;
  float *k_pages, *v_pages;
  int q_heads, kv_heads, head_dim, page_size, v_transposed;
};

template <int G, int FEATURES, int KIND = FEW_PLAIN>
__global__ __launch_bounds__(SEGMENTS * MI_WAVE) void gemm_f32_few_kernel(const float* __restrict__ a, int64_t lda,
                                                           const float* __restrict__ w, int64_t ldw,
                                                           float* __restrict__ c, int64_t ldc, int m, int n, int k, int chunk, FewRows with, Heads heads) {
  if constexpr (KIND == FEW_HEADS) a += (int64_t)blockIdx.y * heads.a, w += (int64_t)blockIdx.y * heads.w, c += (int64_t)blockIdx.y * heads.c;
  extern __shared__ __attribute__((aligned(16))) float4 staged[];  // [wave][slice of the chunk][group of rows][half][piece of K][row]
  __shared__ double sums[SEGMENTS][G][MI_WAVE];
  constexpr int AHEAD = G == 1 ? 4 : 2;
  constexpr bool PAIRED = KIND == FEW_GATED || KIND == FEW_ROPE;  // the operand's upper 8 features belong to its lower 8
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE), lane = threadIdx.x % MI_WAVE;
  static_assert(!PAIRED || FEATURES == 16, "a block's operand holds both features of a pair");
  const int half_dim = KIND == FEW_ROPE ? with.head_dim / 2 : 0;
  const int rope_head = KIND == FEW_ROPE ? (int)(blockIdx.x * 8) / half_dim : 0, rope_dim = KIND == FEW_ROPE ? (int)(blockIdx.x * 8) % half_dim : 0;
  const int col0 = KIND == FEW_ROPE ? rope_head * with.head_dim + rope_dim : blockIdx.x * (PAIRED ? 8 : FEATURES);
  const int most = n - 1 - col0;
  const int run = segment_slices(k), slices = ceil_div(k, SLICE);
  const int first = min(wave * run, slices), last = min(first + run, slices);
  const uint32_t lower = (uint32_t)min(line_row_of_lane(lane), most) * (uint32_t)(ldw * 4) + line_chunk_of_lane(lane);
  const uint32_t upper = PAIRED ? lower + (uint32_t)(KIND == FEW_ROPE ? half_dim : n) * (uint32_t)(ldw * 4)
                         : FEATURES == 8 ? lower
                                         : (uint32_t)min(line_row_of_lane(lane) + 8, most) * (uint32_t)(ldw * 4) + line_chunk_of_lane(lane);
  const float* w_block = w + (int64_t)col0 * ldw;
  const int row = wave * 4 + lane / 16, f = lane % 16;  // (the instruction's result: row lane / 16, feature lane % 16)
  const bool written = wave < G && row < m && f < (PAIRED ? 8 : FEATURES) && f <= most;
  float* const to = c + (int64_t)row * ldc + col0 + f;
  bf16x8_t lo[AHEAD], hi[AHEAD];  // 16-byte pieces; what they hold is float32
  auto fetch = [&](int slot, int slice) {
    if constexpr (FEATURES == 8) lo[slot] = load_line(w_block, 2 * (int64_t)slice, lower);
    else load_line_pair(w_block, 2 * (int64_t)slice, lower, upper, lo[slot], hi[slot]);
  };
  float4* mine = staged + wave * chunk * (32 * G);
  auto stage = [&](int from, int upto) {
    const int piece = lane % 16, row = lane / 16;  // two slices a load
    for (int s = from; s < upto; s += 2) {
      if (s + piece / 8 < upto) {
#pragma unroll
        for (int g = 0; g < G; ++g)
          mine[((s - from + piece / 8) * G + g) * 32 + piece % 8 * 4 + row] =
              *reinterpret_cast<const float4*>(a + (int64_t)min(g * 4 + row, m - 1) * lda + (int64_t)s * SLICE + piece * 4);
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");  // (nobody else reads them: no barrier)
  };
  double acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g) acc[g] = 0.0;
#pragma unroll
  for (int s = 0; s < AHEAD; ++s)
    if (first + s < last) fetch(s, first + s);
  const float4* from = mine + lane / 16 * 4 + lane % 4;
  for (int begin = first; begin < last; begin += chunk) {
    const int end = min(begin + chunk, last);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    stage(begin, end);
    for (int at = begin; at < end; at += AHEAD) {
#pragma unroll
      for (int s = 0; s < AHEAD; ++s) {
        if (at + s < end) {
          float wv[2][4], xv[G][2][4];
          if constexpr (FEATURES == 8) hi[s] = lo[s];
          lines_to_operands(lo[s], hi[s]);
          __builtin_memcpy(wv[0], &lo[s], 16);
          __builtin_memcpy(wv[1], &hi[s], 16);
#pragma unroll
          for (int g = 0; g < G; ++g)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
              const float4 x = from[((at + s - begin) * G + g) * 32 + half * 16];
              __builtin_memcpy(xv[g][half], &x, 16);
            }
          if (at + s + AHEAD < last) fetch(s, at + s + AHEAD);
#pragma unroll
          for (int half = 0; half < 2; ++half)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
              for (int g = 0; g < G; ++g)
                acc[g] = __builtin_amdgcn_mfma_f64_4x4x4f64((double)xv[g][half][e], (double)wv[half][e], acc[g], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int g = 0; g < G; ++g) sums[wave][g][lane] = acc[g];
  __syncthreads();
  if (wave < G) {
    double total = 0.0;
#pragma unroll
    for (int s = 0; s < SEGMENTS; ++s) total += sums[s][wave][lane];
    if constexpr (KIND == FEW_GATED) {
      const float up = __shfl_down((float)total, 8, MI_WAVE);
      if (written) *to = silu_times<float>((float)total, up);
    } else if constexpr (KIND == FEW_ROPE) {
      const float x0 = (float)total, x1 = __shfl_down(x0, 8, MI_WAVE);
      if (written) {
        const int d = rope_dim + f;
        const bool is_value = rope_head >= with.q_heads + with.kv_heads;
        float y0 = x0, y1 = x1;
        if (!is_value) {
          const float cj = with.cos_t[(int64_t)row * half_dim + d], sj = with.sin_t[(int64_t)row * half_dim + d];
          mi_rotate(x0, x1, cj, sj, y0, y1);
        }
        if (rope_head < with.q_heads) {
          to[0] = y0;
          to[half_dim] = y1;
        } else {
          const int slot = with.slots[row];
          if (slot >= 0) {
            const int head = rope_head - with.q_heads - (is_value ? with.kv_heads : 0);
            const int64_t page = (int64_t)(slot / with.page_size) * with.kv_heads + head;
            const int at = slot % with.page_size;
            const bool turned = is_value && with.v_transposed;  // values as [dim][slot]
            float* at_head = (is_value ? with.v_pages : with.k_pages) + page * with.page_size * with.head_dim;
            at_head[turned ? (int64_t)d * with.page_size + at : (int64_t)at * with.head_dim + d] = y0;
            at_head[turned ? (int64_t)(d + half_dim) * with.page_size + at : (int64_t)at * with.head_dim + d + half_dim] = y1;
          }
        }
      }
    } else {
      if (written) *to = (float)total;
    }
  }
}

template <int BM, int STAGE>
static void launch_tiles(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n,
                         int k, bool aligned, int count, const Heads& heads, hipStream_t stream) {
  dim3 grid(ceil_div(n, BN), ceil_div(m, BM), count);
  if (aligned) gemm_f32_kernel<BM, STAGE, true><<<grid, 256, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k, heads);
  else gemm_f32_kernel<BM, STAGE, false><<<grid, 256, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k, heads);
}

template <int G, int FEATURES, int KIND = FEW_PLAIN>
static void launch_few(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n, int k,
                       hipStream_t stream, const FewRows& with = FewRows(), int count = 1, const Heads& heads = Heads()) {
  const int chunk = min(segment_slices(k), 16 / G);
  const int blocks = KIND == FEW_ROPE ? (with.q_heads + 2 * with.kv_heads) * (with.head_dim / 16) : ceil_div(n, KIND == FEW_GATED ? 8 : FEATURES);
  gemm_f32_few_kernel<G, FEATURES, KIND><<<dim3(blocks, count), SEGMENTS * MI_WAVE, SEGMENTS * chunk * G * 32 * sizeof(float4), stream>>>(
      a, lda, w, ldw, c, ldc, m, n, k, chunk, with, heads);
}

// A launch of a kind for one or two groups of four rows.
template <int FEATURES, int KIND>
static void launch_few_of(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n, int k,
                          hipStream_t stream, const FewRows& with = FewRows()) {
  if (m > 4) launch_few<2, FEATURES, KIND>(a, lda, w, ldw, c, ldc, m, n, k, stream, with);
  else launch_few<1, FEATURES, KIND>(a, lda, w, ldw, c, ldc, m, n, k, stream, with);
}

template <int RT, int FT>
static void launch_rows(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n,
                        int k, int form, int count, const Heads& heads, hipStream_t stream) {
  const int row_tiles = ceil_div(m, 16 * RT), total = row_tiles * ceil_div(n, 16 * FT), block = SEGMENTS * MI_WAVE;
  dim3 grid(row_tiles > 1 ? ceil_div(total, 8) * 8 : total, count);
  if (form == LINES) gemm_f32_rows_kernel<RT, FT, LINES><<<grid, block, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k, row_tiles, total, heads);
  else if (form == PIECES) gemm_f32_rows_kernel<RT, FT, PIECES><<<grid, block, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k, row_tiles, total, heads);
  else gemm_f32_rows_kernel<RT, FT, VALUES><<<grid, block, 0, stream>>>(a, lda, w, ldw, c, ldc, m, n, k, row_tiles, total, heads);
}

// Whether gemm_f32_few_kernel is the faster one (figures there).
static bool few_rows_take(int m, int k) { return m <= (segment_slices(k) <= 16 ? 8 : 4); }

// Whole lines of W, rows of A on 16 bytes; the streaming loads' offsets reach over `rows` rows of W in 32 bits.
static bool whole_lines(const float* a, int64_t lda, const float* w, int64_t ldw, int k, int64_t rows) {
  return lda % 4 == 0 && (uintptr_t)a % 16 == 0 && k % SLICE == 0 && ldw % 32 == 0 && (uintptr_t)w % 128 == 0 && rows * ldw < (1 << 29);
}

// silu(a * gate^T) * (a * up^T) of a few rows, w = [gate; up] of n rows each.
extern "C" int mi_gemm_f32_swiglu_takes(const float* a, int64_t lda, const float* w, int64_t ldw, int m, int n, int k) {
  return m >= 1 && n >= 1 && k >= 1 && lda >= k && ldw >= k && few_rows_take(m, k) && whole_lines(a, lda, w, ldw, k, (int64_t)n + 8) ? 1 : 0;
}

extern "C" int mi_gemm_f32_swiglu(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n, int k,
                                  hipStream_t stream) {
  MI_REQUIRE(mi_gemm_f32_swiglu_takes(a, lda, w, ldw, m, n, k) && ldc >= n, "gemm_f32_swiglu: m=%d n=%d k=%d lda=%lld ldw=%lld ldc=%lld is not taken", m,
             n, k, (long long)lda, (long long)ldw, (long long)ldc);
  launch_few_of<16, FEW_GATED>(a, lda, w, ldw, c, ldc, m, n, k, stream);
  MI_CHECK_LAUNCH("gemm_f32_swiglu");
  return MI_OK;
}

extern "C" int mi_gemm_f32_rope_takes(const float* a, int64_t lda, const float* w, int64_t ldw, int m, int k, int head_dim) {
  return m >= 1 && k >= 1 && lda >= k && ldw >= k && head_dim >= 16 && head_dim % 16 == 0 && head_dim <= 4096 && few_rows_take(m, k) &&
                 whole_lines(a, lda, w, ldw, k, (int64_t)head_dim) ? 1 : 0;
}

// The stacked q|k|v product of a few rows, whole heads rotated in half pairing (cos_t, sin_t [m][head_dim / 2]): queries to q_out, keys and
// values to their slots (kv_heads = 0: queries alone; a slot below 0 is not written).
extern "C" int mi_gemm_f32_rope(const float* a, int64_t lda, const float* w, int64_t ldw, float* q_out, int64_t ldq, const float* cos_t,
                                const float* sin_t, const int* slots, float* k_pages, float* v_pages, int m, int k, int q_heads, int kv_heads,
                                int head_dim, int page_size, int num_pages, int v_transposed, hipStream_t stream) {
  MI_REQUIRE(mi_gemm_f32_rope_takes(a, lda, w, ldw, m, k, head_dim) && q_heads >= 1 && kv_heads >= 0 && q_out && cos_t && sin_t &&
                 ldq >= (int64_t)q_heads * head_dim && ((int64_t)q_heads + 2 * (int64_t)kv_heads) * head_dim < (1ll << 31),
             "gemm_f32_rope: m=%d k=%d lda=%lld ldw=%lld heads %d and %d of %d is not taken", m, k, (long long)lda, (long long)ldw, q_heads, kv_heads, head_dim);
  MI_REQUIRE(kv_heads == 0 || (slots && k_pages && v_pages && page_size > 0 && num_pages > 0), "gemm_f32_rope: keys and values need pages and slots");
  FewRows with = {};
  with.cos_t = cos_t;
  with.sin_t = sin_t;
  with.slots = slots;
  with.k_pages = k_pages;
  with.v_pages = v_pages;
  with.q_heads = q_heads;
  with.kv_heads = kv_heads;
  with.head_dim = head_dim;
  with.page_size = page_size;
  with.v_transposed = v_transposed;
  launch_few_of<16, FEW_ROPE>(a, lda, w, ldw, q_out, ldq, m, (q_heads + 2 * kv_heads) * head_dim, k, stream, with);
  MI_CHECK_LAUNCH("gemm_f32_rope");
  return MI_OK;
}

// Before the 64-bit matrix instruction (64-bit multiply-adds on the vector pipe, 4 x 4 outputs a thread), microseconds at rows x N x K, weights from
// memory: 20 x 2048 x 2048 317, 60 x 16384 x 2048 355, 509 x 16384 x 2048 1060 -> 580 (59 TFLOP/s, where the vendor library's 64-bit product
// reaches 64), 509 x 2048 x 8192 1340 -> 316.  Rows off whole lines, 16-byte pieces (single values waited for one
// by one before): 1 x 128256 x 2052 684 -> 267, 32 rows 1,410 -> 509; 16 x 4096 x 4096, rows not on a line, 66 -> 23; single values, 8 x
// 32000 x 4095 415 -> 218.

// The kernels that a call may take: the 16s of rows and of features that a block of gemm_f32_rows_kernel makes, then the others.
#define F32_ROWS_FORMS(X) X(0, 1, 1) X(1, 1, 2) X(2, 2, 1) X(3, 2, 2) X(4, 4, 1) X(5, 4, 2)
enum { F32_ROWS = 6, F32_FEW = 6, F32_TILES_32 = 7, F32_TILES_64 = 8, F32_FORMS = 9 };

// Microseconds that a form is expected to take, for operands that are read value by value, in pieces and in lines.  The rows' kernel: a launch; for every
// two rounds of its blocks over the compute units (two of them are on one at a time) the loads of a wave's slices one after another; for every round a block's
// slices on one matrix pipe (waves w and w + 4 share one) with its 16 x 16 products and their operands, and what its sums and its end take.  The tiles: a launch and for
// every slice a first round and the others.  Fitted to 3,110 products of 1 to 600 rows, 16 to 20,000 features and K 32 to 9,000, each in every form: half of the times are
// within 6 % (11 % value by value) for the rows' kernel and 4 % for the tiles.
struct RowsCost {
  double launch, trip, round, tile, product, operand;
};
struct TilesCost {
  double launch, only, each, rest;
};
static double f32_micros(int form, int how, int m, int n, int k, int count, int cus) {
  static const RowsCost rows_cost[3] = {{2.08, 0.557, 0, 0.0466, 0.0546, 0.0849}, {2.41, 0.139, 0.0215, 0.0994, 0.0678, 0.0238}, {2.58, 0.0654, 0.117, 0.139, 0.0653, 0.0144}};
  static const TilesCost tiles_64[3] = {{3.04, 1.83, 1.41, 0.396}, {3.18, 1.43, 1.29, 0}, {2.89, 1.45, 1.17, 0.246}};
  static const TilesCost tiles_32[3][2] = {  // one slice a stage, four
      {{2.67, 1.18, 0.779, 0.286}, {5.89, 1.12, 0.803, 0}}, {{2.75, 0.893, 0.67, 0.14}, {5.01, 0.749, 0.559, 0.127}}, {{2.62, 0.897, 0.627, 0.285}, {4.59, 0.741, 0.553, 0.127}}};
  const int slices = ceil_div(k, SLICE);
  auto rounds = [&](int rows, int features) { return (double)ceil_div64((int64_t)ceil_div(m, rows) * ceil_div(n, features) * count, cus); };
  if (form == F32_TILES_32 || form == F32_TILES_64) {
    const TilesCost& c = form == F32_TILES_64 ? tiles_64[how] : tiles_32[how][segment_slices(k) % 4 == 0];
    const double r = rounds(form == F32_TILES_64 ? 64 : 32, BN);
    return c.launch + slices * (r > 1 ? c.each * r + c.rest : c.only);
  }
  constexpr int of[F32_ROWS][2] = {
#define X(I, RT, FT) {RT, FT},
      F32_ROWS_FORMS(X)
#undef X
  };
  const RowsCost& c = rows_cost[how];
  const int rt = of[form][0], ft = of[form][1], run = segment_slices(k), on_a_pipe = ceil_div(slices, run) > 4 ? 2 * run : run;
  const double r = rounds(16 * rt, 16 * ft);
  const double t = c.launch + ceil(r / 2) * run * c.trip + r * (c.round + c.tile * rt * ft + 4 * on_a_pipe * (c.product * rt * ft + c.operand * (rt + ft)));
  return r > 1 && run <= 4 && rt * ft >= 4 ? 1.15 * t : t;  // (large blocks in several rounds end and begin more than they multiply)
}

// The form of m rows for which the four-row products are not taken: the one that is expected to be the fastest.  (All give the same bits.)  Over the
// products that the times are fitted to, as geometric means of the fastest form's time, in lines / in pieces / value by value: all rows a block up to 32 rows, or 64 with
// less than 8,192 features, and tiles above 1.35 / 1.23 / 1.16; by times that know neither a tile's launch nor how operands are read 1.08 / 1.14 / 1.13 (13 x 512
// x 160 6.8 for 3.5 us, 2 x 1024 x 145 8.2 / 4.0, 232 x 6418 x 1024 value by value 167 / 116); so 1.008 / 1.013 / 1.010.  In lines, weights from memory,
// before forms in blocks of rows / so:
//     rows            25             64             96             128            256
//     2048 x 2048     15.1 / 9.6     27.5 / 15.0    50.9 / 22.3    51.3 / 23.6    51.8 / 43.7
//     3072 x 2048     15.8 / 15.3    28.3 / 22.4    51.1 / 32.8    51.3 / 36.2    82.1 / 67.2
//     16384 x 2048    51.4 / 50.3    89.4 / 87.6    123 / 122      161 / 160      303 / 303
//     2048 x 8192     50.1 / 31.5    91.0 / 51.5    195 / 77.7     196 / 83.5     199 / 148
static int f32_form(int how, int m, int n, int k, int count, int cus) {
  int best = F32_TILES_64;
  if (m > 32 * 65535) return best;
  double least = f32_micros(best, how, m, n, k, count, cus);
  for (int form = 0; form < F32_FORMS; ++form) {
    if (form == F32_FEW || form == F32_TILES_64) continue;
    const double t = f32_micros(form, how, m, n, k, count, cus);
    if (t < least) least = t, best = form;
  }
  return best;
}

// `count` products side by side, `heads` apart; only: a form, or -1.
static int gemm_f32(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n, int k, int count, const Heads& heads,
                    int only, hipStream_t stream) {
  MI_REQUIRE(m >= 0 && n > 0 && k > 0 && count >= 1 && count <= 65535, "gemm_f32: bad sizes m=%d n=%d k=%d, %d of them", m, n, k, count);
  MI_REQUIRE(lda >= k && ldw >= k && ldc >= n, "gemm_f32: a row stride is shorter than its row");
  MI_REQUIRE(ceil_div(m, 64) <= 65535, "gemm_f32: m=%d is too large for one call", m);
  if (m == 0) return MI_OK;
  const bool a16 = lda % 4 == 0 && (uintptr_t)a % 16 == 0 && (count == 1 || heads.a % 4 == 0), w16 = ldw % 4 == 0 && (uintptr_t)w % 16 == 0 && (count == 1 || heads.w % 4 == 0);
  const bool lines = whole_lines(a, lda, w, ldw, k, 32) && (count == 1 || (heads.a % 4 == 0 && heads.w % 32 == 0));
  const bool few = lines && few_rows_take(m, k);
  const bool aligned = a16 && w16 && k % 4 == 0;
  const int how = lines ? LINES : aligned ? PIECES : VALUES;
  const int form = only >= 0 ? only : few ? (int)F32_FEW : f32_form(how, m, n, k, count, max(8, mi_compute_units()));
  MI_REQUIRE(form < F32_FORMS && (form != F32_FEW || few), "gemm_f32: form %d does not take m=%d k=%d", form, m, k);
  if (form == F32_FEW) {
    const bool half_empty = (int64_t)ceil_div(n, 16) * count <= 128;
#define MI_FEW(FEATURES, KIND)                                                                                          \
  do {                                                                                                                  \
    if (m > 4) launch_few<2, FEATURES, KIND>(a, lda, w, ldw, c, ldc, m, n, k, stream, FewRows(), count, heads);         \
    else launch_few<1, FEATURES, KIND>(a, lda, w, ldw, c, ldc, m, n, k, stream, FewRows(), count, heads);               \
  } while (0)
    if (count > 1 && half_empty) MI_FEW(8, FEW_HEADS);
    else if (count > 1) MI_FEW(16, FEW_HEADS);
    else if (half_empty) MI_FEW(8, FEW_PLAIN);
    else MI_FEW(16, FEW_PLAIN);
#undef MI_FEW
  } else if (form == F32_TILES_64) {
    launch_tiles<64, 1>(a, lda, w, ldw, c, ldc, m, n, k, aligned, count, heads, stream);
  } else if (form == F32_TILES_32) {
    if (segment_slices(k) % 4 == 0) launch_tiles<32, 4>(a, lda, w, ldw, c, ldc, m, n, k, aligned, count, heads, stream);
    else launch_tiles<32, 1>(a, lda, w, ldw, c, ldc, m, n, k, aligned, count, heads, stream);
  }
#define X(I, RT, FT) \
  else if (form == I) launch_rows<RT, FT>(a, lda, w, ldw, c, ldc, m, n, k, how, count, heads, stream);
  F32_ROWS_FORMS(X)
#undef X
  MI_CHECK_LAUNCH("gemm_f32");
  return MI_OK;
}

extern "C" int mi_gemm_f32(const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n, int k, hipStream_t stream) {
  return gemm_f32(a, lda, w, ldw, c, ldc, m, n, k, 1, {}, -1, stream);
}

// The same in one of its forms (those that do not take the sizes refuse them).
extern "C" int mi_gemm_f32_as(int form, const float* a, int64_t lda, const float* w, int64_t ldw, float* c, int64_t ldc, int m, int n, int k,
                              hipStream_t stream) {
  MI_REQUIRE(form >= 0, "gemm_f32: form %d", form);
  return gemm_f32(a, lda, w, ldw, c, ldc, m, n, k, 1, {}, form, stream);
}

// A product a head: a, w and c of head h lie h times a_head, w_head and c_head elements further on.
extern "C" int mi_gemm_f32_heads(const float* a, int64_t lda, int64_t a_head, const float* w, int64_t ldw, int64_t w_head, float* c, int64_t ldc,
                                 int64_t c_head, int m, int n, int k, int heads, hipStream_t stream) {
  return gemm_f32(a, lda, w, ldw, c, ldc, m, n, k, heads, {a_head, w_head, c_head}, -1, stream);
}
