// A tile of C = A * W^T in bfloat16 for many rows, made by two groups of four waves that take turns: while one group multiplies, the
// other reads its operands from LDS and asks for later ones.
//
// What bounds such a tile is the matrix cores, as long as something keeps them fed: a wave alone, or eight in step (tile_product.h),
// issue loads, read operands and multiply one after the other.  Each SIMD holds one wave of either group, and a barrier between
// turns keeps the groups half a step apart, so that one of the two always multiplies.  On 2048 x 8192 x 8192 tiles of 256 x 256 then take
// 2,205 cycles a step of 64 of K, of which 2,048 are matrix instructions (in step 1.2 times that), and the card's power
// sets the pace: it lowers the clock to 1.4 GHz and the library's kernel and this one take the same time.
//
// Both operands go straight from memory into LDS, 64 of K at a time, in a ring of STAGES; a row of a stage is 128 bytes (a whole cache
// line: half lines, 32 of K at a time, hold as many lines up for half the bytes, 433 against 376 us for 2048 x 28672 x 4096), eight
// chunks of 16, chunk c of row r at place c ^ (r % 8), so that the lanes that are served together find their pieces in
// different banks.  Sums run over K from its beginning, 32 at a time: the order of one wave alone, so all tile shapes give the same bits, and
// the vendor library's kernels that do not cut K give them too (`turns_keep_the_order` in ops/kernels.py).
#pragma once

#include "gated_tile.h"

typedef float f32x4_u __attribute__((ext_vector_type(4)));

// WM x WN = 8 waves: WM along the rows of A, WN along the rows of W; MT x NT: a wave's tiles of 16 rows of A and of W.
//   STAGES >= 3: a turn is 64 of K.  Operands of a turn are read, then the stage after the last one on its way is asked for, into the place that
//     both groups are done with; a wave waits for its own loads of the next stage before the barrier that ends its turn.
//   STAGES == 2, for tiles whose stages fill LDS: a turn is half of a wave's rows of A.  W and the first half are read in the one turn,
//     the second half in the other, and each place is filled anew as soon as it has been read: all of a stage is on its way for
//     a whole step.
template <int WM_, int WN_, int MT_, int NT_, int STAGES_>
struct TurnsProduct {
  static constexpr int WM = WM_, WN = WN_, MT = MT_, NT = NT_, STAGES = STAGES_;
  static constexpr int WAVES = 8, THREADS = WAVES * MI_WAVE;
  static constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
  static constexpr int STEP_K = 64;
  static constexpr int STAGE = (BM + BN) * STEP_K, RING = STAGES * STAGE;  // elements
  static constexpr bool HALVES = STAGES == 2;
  static constexpr int LO = HALVES ? MT / 2 : MT;                       // row tiles of the first half
  static constexpr int LOADS = (BM + BN) / 8;                           // of 8 rows x 128 bytes
  static constexpr int FIRST = HALVES ? BN / 8 + WM * LO * 2 : LOADS;   // of W and the first half of A; then the second half
  static constexpr int EACH = LOADS / WAVES, REST = LOADS % WAVES, MOST = EACH + (REST > 0);  // a wave makes EACH, the first REST one more
  static constexpr int OF_FIRST = FIRST / WAVES, OF_SECOND = MOST - OF_FIRST;                // (HALVES)
  static_assert(WM * WN == WAVES && RING * 2 <= 163840, "eight waves, and the ring fits LDS");
  static_assert(!HALVES || (MT % 2 == 0 && FIRST % WAVES == 0 && REST == 0), "halves take whole rounds of loads");
  static_assert(MOST * (STAGES - 1) < 64, "outstanding loads are counted in six bits");

  int wave, lane, col, quad, wm, wn;
  f32x4_u acc[NT][MT];

  __device__ __forceinline__ TurnsProduct() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE);
    lane = threadIdx.x % MI_WAVE;
    col = lane % 16;
    quad = lane / 16;
    wn = wave % WN;
    wm = wave / WN;
  }

  template <int N>
  static __device__ __forceinline__ void outstanding() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
  }
  // Waits until at most `newer` stages' loads of this wave are outstanding.
  template <int R = STAGES - 2>
  __device__ __forceinline__ void wait_for(int newer) const {
    if constexpr (R <= 0) {
      outstanding<0>();
    } else {
      if (newer >= R) {
        if (REST > 0 && wave < REST) outstanding<R * MOST>();
        else outstanding<R * EACH>();
      } else {
        wait_for<R - 1>(newer);
      }
    }
  }
  static __device__ __forceinline__ void meet() {
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  // Operands are in registers: what they were read from may be written once all waves have met.
  static __device__ __forceinline__ void have_read() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

  // Row of the tile's A (below BM) or W (from BM on) that lies in row i of a stage.  STAGES >= 3: A, then W; HALVES: W, then the waves' first
  // halves of A, then their second halves.
  static __device__ __forceinline__ int row_in(int i) {
    if constexpr (!HALVES) return i;
    if (i < BN) return BM + i;
    constexpr int HALF = LO * 16;
    const int j = i - BN, second = j / (WM * HALF), rest = j % (WM * HALF);
    return rest / HALF * (MT * 16) + second * HALF + rest % HALF;
  }

  // acc = the tile's sums over `steps` (at least one) times 64 of K; a_row(r) and w_row(r) give the first of them of the tile's row r,
  // 0 <= r < BM, BN, on 16 bytes and readable.  Nothing of `ring` may be written before the block has met once more.  ONCE: nobody else reads
  // these rows of W (they are then read past the caches).
  template <bool ONCE = false, typename RowA, typename RowW>
  __device__ __forceinline__ void run(bf16_t* ring, int steps, RowA a_row, RowW w_row) {
    const bf16_t* src[MOST];
    const int chunk = ((lane % 8) ^ (lane / 8)) * 8;
    constexpr int BORDER = HALVES ? BN : BM;  // rows of a stage before it are one operand's, known when compiling for most loads
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
      const int i = min(wave + j * WAVES, LOADS - 1) * 8 + lane / 8;  // (a load that a wave does not make: another's row)
      const int r = row_in(i);
      const bool before = (j + 1) * WAVES * 8 <= BORDER ? true : j * WAVES * 8 >= BORDER ? false : i < BORDER;
      src[j] = (before != HALVES ? a_row(r) : w_row(r - BM)) + chunk;
    }
    using global_void = const __attribute__((address_space(1))) void;
    using lds_void = __attribute__((address_space(3))) void;
    auto fetch = [&](int from, int to, int slot) {  // of this wave's loads those of the next stage that has not been asked for
      bf16_t* at = ring + slot * STAGE + wave * 512;
#pragma unroll
      for (int j = from; j < to; ++j) {
        const bool of_w = HALVES ? (j + 1) * WAVES * 8 <= BN : j * WAVES * 8 >= BM;
        if (j < EACH || wave < REST) {
          if (ONCE && of_w) __builtin_amdgcn_global_load_lds((global_void*)src[j], (lds_void*)(at + j * (WAVES * 512)), 16, 0, 2);
          else __builtin_amdgcn_global_load_lds((global_void*)src[j], (lds_void*)(at + j * (WAVES * 512)), 16, 0, 0);
        }
        src[j] += STEP_K;
      }
    };
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_u{0.f, 0.f, 0.f, 0.f};
    bf16x8_t wf[2][NT], af[2][LO];
    const int place[2] = {(quad ^ (col % 8)) * 8, ((4 + quad) ^ (col % 8)) * 8};
    const bf16_t* w_at = ring + ((HALVES ? 0 : BM) + wn * NT * 16 + col) * STEP_K;
    const bf16_t* a_at = ring + ((HALVES ? BN : 0) + wm * LO * 16 + col) * STEP_K;
    auto read_w = [&](int slot) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int n = 0; n < NT; ++n) wf[h][n] = *reinterpret_cast<const bf16x8_t*>(w_at + slot * STAGE + n * 16 * STEP_K + place[h]);
    };
    auto read_a = [&](int slot, int half) {
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < LO; ++m)
          af[h][m] = *reinterpret_cast<const bf16x8_t*>(a_at + slot * STAGE + (half * WM * LO + m) * 16 * STEP_K + place[h]);
    };
    auto multiply = [&](int half) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int m = 0; m < LO; ++m)
#pragma unroll
          for (int n = 0; n < NT; ++n) {
            f32x4_u& c = acc[n][half * LO + m];
            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[h][n], af[h][m], c, 0, 0, 0);
          }
      __builtin_amdgcn_s_setprio(0);
    };
    const bool late = wave >= WAVES / 2;  // the group that is half a step behind
    if constexpr (HALVES) {
      fetch(0, OF_FIRST, 0);
      fetch(OF_FIRST, MOST, 0);
      if (steps > 1) {
        fetch(0, OF_FIRST, 1);
        outstanding<MOST>();
      } else {
        outstanding<OF_SECOND>();
      }
      meet();
      if (late) meet();
      auto step = [&](int slot, auto after) {  // after: steps behind this one, counted up to two
        constexpr int AFTER = decltype(after)::value;
        read_w(slot);
        read_a(slot, 0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (AFTER >= 1) fetch(OF_FIRST, MOST, slot ^ 1);
        outstanding<AFTER >= 1 ? MOST : 0>();  // this step's second half is there
        have_read();
        meet();
        multiply(0);
        meet();
        read_a(slot, 1);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (AFTER >= 2) fetch(0, OF_FIRST, slot);
        if constexpr (AFTER >= 1) outstanding<AFTER >= 2 ? MOST : OF_SECOND>();  // W and the first half of the next step are
        have_read();
        meet();
        multiply(1);
        meet();
      };
      int s = 0;
      for (; s + 2 < steps; ++s) step(s & 1, Count<2>{});
      if (steps > 1) step(s++ & 1, Count<1>{});
      step(s & 1, Count<0>{});
    } else {
#pragma unroll
      for (int s = 0; s < STAGES - 1; ++s)
        if (s < steps) fetch(0, MOST, s);
      wait_for(steps - 1);
      meet();
      if (late) meet();
      int slot = 0, into = STAGES - 1, s = 0;
      for (; s + STAGES - 1 < steps; ++s) {
        read_w(slot);
        read_a(slot, 0);
        __builtin_amdgcn_sched_barrier(0);
        fetch(0, MOST, into);
        into = slot;
        slot = slot + 1 == STAGES ? 0 : slot + 1;
        if (REST > 0 && wave < REST) outstanding<(STAGES - 2) * MOST>();
        else outstanding<(STAGES - 2) * EACH>();
        have_read();
        meet();
        multiply(0);
        meet();
      }
      for (; s < steps; ++s) {
        read_w(slot);
        read_a(slot, 0);
        slot = slot + 1 == STAGES ? 0 : slot + 1;
        wait_for(steps - 2 - s);
        have_read();
        meet();
        multiply(0);
        meet();
      }
    }
    if (!late) meet();
  }

  template <int N>
  struct Count {
    static constexpr int value = N;
  };

  // The sums, each as value_of(sum, row of the tile) rounded to bfloat16, as rows of the tile in `ring`, MADE elements apart; all threads see them
  // afterwards.  What follows reads them in a loop: written from registers, the last steps of 32 little tiles are 60 KB of instructions, which
  // every launch fetches anew (2048 x 6144 x 4096 86 us alone, 101 in a kernel with four sizes of tiles).
  static constexpr int MADE = BN + 8;
  static_assert(BM * MADE <= 79872, "the tile fits the largest ring");
  template <typename F>
  __device__ __forceinline__ void leave(bf16_t* ring, F value_of) {
    meet();  // (the group that is ahead does not write what the other still reads)
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int r = (wm * MT + m) * 16 + col;
#pragma unroll
      for (int n = 0; n < NT; ++n) {
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = value_of(acc[n][m][j], r);
        mi_store_cols<bf16_t, 4>(ring + r * MADE + (wn * NT + n) * 16 + quad * 4, v);
      }
    }
    __syncthreads();
  }
  using Pairs = GatedTile<NT>;  // where the tile holds gate and up rows
};

// The tiles that launches choose among, rows of A x rows of W, and the microseconds that a step of 64 of K takes one.
// X(number, rows, rows of W, gate and up rows side by side?, microseconds a step, shape)
#define TURNS_FORMS_OF(X) \
  X(0, 64, 256, true, 0.556f, 2, 4, 2, 4, 3) \
  X(1, 128, 256, true, 0.814f, 2, 4, 4, 4, 3) \
  X(2, 160, 256, true, 0.943f, 2, 4, 5, 4, 3) \
  X(3, 256, 256, true, 1.286f, 2, 4, 8, 4, 2) \
  X(4, 64, 128, true, 0.345f, 2, 4, 2, 2, 4) \
  X(5, 128, 128, true, 0.486f, 4, 2, 2, 4, 4) \
  X(6, 160, 128, true, 0.603f, 2, 4, 5, 2, 4) \
  X(7, 192, 128, true, 0.674f, 2, 4, 6, 2, 3) \
  X(8, 256, 128, true, 0.786f, 4, 2, 4, 4, 3) \
  X(9, 128, 192, false, 0.668f, 2, 4, 4, 3, 3) \
  X(10, 192, 192, false, 0.847f, 2, 4, 6, 3, 3)
constexpr int TURNS_K = 64;
constexpr int TURNS_FORMS = 11;
template <int F>
struct TurnsOf;
#define X(I, ROWS, FEATURES, GATED, MICROS, ...)                                                                 \
  template <>                                                                                                    \
  struct TurnsOf<I> {                                                                                            \
    using type = TurnsProduct<__VA_ARGS__>;                                                                      \
    static_assert(type::BM == ROWS && type::BN == FEATURES && type::RING <= 79872 && (!GATED || type::NT % 2 == 0)); \
  };
TURNS_FORMS_OF(X)
#undef X
constexpr int TURNS_RING = TurnsOf<2>::type::RING;  // the largest
struct TurnsForm {
  int rows, features;
  bool gated;
  float step_micros;
};
__host__ __device__ constexpr TurnsForm turns_form(int i) {
  constexpr TurnsForm forms[TURNS_FORMS] = {
#define X(I, ROWS, FEATURES, GATED, MICROS, ...) {ROWS, FEATURES, GATED, MICROS},
      TURNS_FORMS_OF(X)
#undef X
  };
  return forms[i];
}

// Microseconds of the rounds that `tiles` tiles of form f take on `each` compute units (of one XCD): the last one, where it does not fill them, is a
// little shorter, because the card's power then lets the clock rise.  And of the bytes of n rows of W of k elements that `blocks` tiles read.  (The
// microseconds of a step in the table above and these rates were fitted to profiles/turns_tiles_forms_times.txt.)
__host__ __device__ inline float turns_rounds_micros(int f, int tiles, int each, int k) {
  if (tiles == 0) return 0.f;
  const int rounds = (tiles + each - 1) / each, idle = rounds * each - tiles;
  return ((float)rounds - 0.29f * (float)idle / (float)each) * ((float)(k / TURNS_K) * turns_form(f).step_micros + 3.4f);
}
__host__ __device__ inline float turns_bytes_micros(int f, int64_t blocks, int n, int k) {
  return 2.33e-7f * (float)n * (float)k * 2.f + 0.73e-7f * (float)blocks * (float)k * ((float)turns_form(f).features * 2.f);
}
