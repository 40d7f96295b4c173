// A tile of C = A * W^T in bfloat16 on the matrix cores, both operands streamed through a ring in LDS.
//
// What bounds such a product of some tens to some hundreds of rows is what a CU can bring in: its 32 KB of vector cache are
// all that is ever outstanding, and what comes from a cache waits in order behind what comes from memory, so that a CU gets
// 53 KB a microsecond from memory while the others are idle, 24 while all 256 read (6.2 TB/s), 40 when half of the bytes
// hit L2, 147 when all do; neither more waves, nor more bytes asked for at once, nor a wave that only fetches, nor another
// order over K, nor whole lines of several steps side by side changed that (64 rows of A and of W a block, 16384 x 3072:
// 25.3 us with 3 or 8 stages in flight; 25.2 with the matrix instructions left out; 12 with W from L2).  So a tile is as
// near to square as the sizes allow, and a launch cuts K where that gives every CU a tile; gemm_tiles_bf16.hip chooses.
//
// Both operands go straight from memory into LDS (no registers between), 64 of K at a time, STAGES stages in a ring; a wave waits
// for its own loads of a stage, then all meet, then the place that was read last is filled anew.  A row of a stage is 128
// bytes, eight chunks of 16; chunk c of row r lies at place c ^ (r % 8), so that the eight lanes that are served together
// find their pieces in different banks.  Operands are read from LDS one piece of 32 of K ahead of their products.
#pragma once

#include "common.h"

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;
typedef const __attribute__((address_space(1))) void global_void;

// WM x WN x WK waves: WM along the rows of A, WN along the rows of W, WK (1 or 2) along the K of a stage (two waves then
// sum the halves of every 64, and their sums meet at the end); MT x NT: a wave's tiles of 16 rows of A and of W.
template <int WM_, int WN_, int WK_, int MT_, int NT_, int STAGES_>
struct TileProduct {
  static constexpr int WM = WM_, WN = WN_, WK = WK_, MT = MT_, NT = NT_, STAGES = STAGES_;
  static constexpr int WAVES = WM * WN * WK, THREADS = WAVES * MI_WAVE;
  static constexpr int BM = WM * MT * 16, BN = WN * NT * 16;
  static constexpr int STEP_K = 64;
  static constexpr int STAGE = (BM + BN) * STEP_K;  // elements
  static constexpr int EXCHANGE = WK == 1 ? 0 : WM * WN * NT * MT * MI_WAVE * 8;  // elements: float32 sums that change hands
  static constexpr int MADE = BN + 8;  // elements from one row that `leave` leaves to the next
  static constexpr int WORK = STAGES * STAGE > EXCHANGE ? STAGES * STAGE : EXCHANGE;
  static constexpr int RING = WORK > BM * MADE ? WORK : BM * MADE;
  static constexpr int LOADS = (BM + BN) / 8;  // of 8 rows x 128 bytes
  static constexpr int EACH = LOADS / WAVES, REST = LOADS % WAVES;  // a wave makes EACH, the first REST one more
  static constexpr int MOST = EACH + (REST > 0);
  static constexpr int FIRST_M = (MT + 1) / 2;  // with WK == 2: row tiles that the first half of the waves ends up with
  static_assert(MOST * (STAGES - 1) < 64, "outstanding loads are counted in six bits");

  int wave, lane, col, quad, wm, wn, wk;
  f32x4_t acc[NT][MT];

  __device__ __forceinline__ TileProduct() {
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x / MI_WAVE);
    lane = threadIdx.x % MI_WAVE;
    col = lane % 16;
    quad = lane / 16;
    wn = wave % WN;
    wm = wave / WN % WM;
    wk = wave / (WN * WM);
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

  // acc = the tile's sums over `halves` pieces of 32 of K (at least one); a_row(r) and w_row(r) give the first of them of the tile's
  // row r, 0 <= r < BM, BN, on 16 bytes and readable.  ONCE: nobody else reads these rows of W (they are then read past the
  // caches: 4 % at 64 rows; not where several row tiles share them).  ODD: `halves` may be odd.  ROUND: begin at the step (of 64) `begin`, after the last
  // one step 0 follows; not with ODD.  (All known when
  // compiling: a branch in the loop for either of the first two cost 5 to 20 %, going round 1 % of a step of 271 tokens at 3072 wide that does not.)
  template <bool ONCE, bool ODD, bool ROUND = false, typename RowA, typename RowW>
  __device__ __forceinline__ void run(bf16_t* ring, int halves, RowA a_row, RowW w_row, int begin = 0) {
    const int steps = ODD ? (halves + 1) / 2 : halves / 2;
    const bf16_t* src[MOST];
    const int row_of = lane / 8;
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
      const int load = wave + j * WAVES;
      const int r = load * 8 + row_of;
      const int chunk = (lane % 8) ^ (r % 8);
      if (load * 8 < BM) src[j] = a_row(r) + chunk * 8;
      else if (load < LOADS) src[j] = w_row(r - BM) + chunk * 8;
      else src[j] = nullptr;  // (not fetched)
    }
    int fetched = 0, left = steps - begin;
    if constexpr (ROUND) {
#pragma unroll
      for (int j = 0; j < MOST; ++j) src[j] += begin * STEP_K;
    }
    auto fetch = [&](int slot) {
      if (ODD && ++fetched == steps && halves % 2 != 0) {  // the last 32 of K have no other half: the first one again, not multiplied
#pragma unroll
        for (int j = 0; j < MOST; ++j)
          if (((lane % 8) ^ ((wave + j * WAVES) * 8 + row_of) % 8) >= 4) src[j] -= STEP_K / 2;
      }
      bf16_t* to = ring + slot * STAGE + wave * 512;
      const int add = ROUND && --left == 0 ? STEP_K - steps * STEP_K : STEP_K;
#pragma unroll
      for (int j = 0; j < MOST; ++j) {
        if (j < EACH || wave < REST) {
          if (ONCE && (wave + j * WAVES) * 8 >= BM) __builtin_amdgcn_global_load_lds((global_void*)src[j], (lds_void*)(to + j * (WAVES * 512)), 16, 0, 2);
          else __builtin_amdgcn_global_load_lds((global_void*)src[j], (lds_void*)(to + j * (WAVES * 512)), 16, 0, 0);
        }
        src[j] += add;
      }
    };
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < steps) fetch(s);
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};

    bf16x8_t wf[2][NT], af[2][MT];  // operands of the piece of 32 of K that is worked on, and of the next one
    const bf16_t* a_at = ring + (wm * MT * 16 + col) * STEP_K;
    const bf16_t* w_at = ring + (BM + wn * NT * 16 + col) * STEP_K;
    auto read = [&](int set, int slot, int half) {
      const int at = slot * STAGE + ((half * 4 + quad) ^ (col % 8)) * 8;
#pragma unroll
      for (int n = 0; n < NT; ++n) wf[set][n] = *reinterpret_cast<const bf16x8_t*>(w_at + n * 16 * STEP_K + at);
#pragma unroll
      for (int m = 0; m < MT; ++m) af[set][m] = *reinterpret_cast<const bf16x8_t*>(a_at + m * 16 * STEP_K + at);
    };
    auto multiply = [&](int set) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][n], af[set][m], acc[n][m], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
    // stage `step` is in LDS for all waves, and nobody reads the one before it any more: its place is filled anew
    auto advance = [&](int step, int before) {
      wait_for(steps - 1 - step);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (step - 1 + STAGES < steps) fetch(before);
    };
    constexpr int PIECES = 2 / WK;  // of 32 of K that a wave multiplies of a stage, from wk * PIECES on
    int slot = 0;
    auto next = [&]() { slot = slot + 1 == STAGES ? 0 : slot + 1; };
    wait_for<STAGES - 1>(steps - 1);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0, wk * PIECES);
    for (int step0 = 0; step0 < steps; step0 += PIECES == 1 ? 2 : 1) {
#pragma unroll
      for (int p = 0; p < (PIECES == 1 ? 2 : PIECES); ++p) {
        const int step = step0 + (PIECES == 1 ? p : 0);
        if (PIECES == 1 && step >= steps) break;
        if (PIECES > 1 && p + 1 < PIECES) {
          read((p + 1) % 2, slot, wk * PIECES + p + 1);
        } else {
          const int before = slot;
          next();
          if (step + 1 < steps) {
            advance(step + 1, before);
            read((p + 1) % 2, slot, wk * PIECES);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        if (!ODD || step + 1 < steps || halves % 2 == 0 || (PIECES == 1 ? wk == 0 : p == 0)) multiply(p % 2);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (WK == 2) {
      __syncthreads();
      f32x4_t* to = reinterpret_cast<f32x4_t*>(ring) + ((wm * WN + wn) * NT * MT) * MI_WAVE + lane;
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          if ((m < FIRST_M) != (wk == 0)) to[(n * MT + m) * MI_WAVE] = acc[n][m];
      __syncthreads();
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          if ((m < FIRST_M) == (wk == 0)) acc[n][m] += to[(n * MT + m) * MI_WAVE];
    }
  }

  // The same sums as eight waves that take an eighth of K each and add theirs in order: halves % 16 == 0.  Of the two waves along K one takes the even
  // eighths, one the odd: a place in the ring holds 64 of K of an even one and the 64 as far into the one behind it.  W is read past the caches.
  // ROUND: begin at pair of eighths `begin` (of 4).  Two eighths at a time, as a wave that sums all of them has twice the reads and products between two
  // barriers: [16384 x 3072 | 2048] at 32 rows so 20.9 and 15.1 us, with waves that sum whole eighths in turn 21.0 and 17.2, in the order of `run` 19.5 and 14.2.
  template <bool ROUND, typename RowA, typename RowW>
  __device__ __forceinline__ void run_eighths(bf16_t* ring, int halves, RowA a_row, RowW w_row, int begin) {
    static_assert(WK == 2 && STAGES % 2 == 0 && WM * WN * 4 * NT * MT * MI_WAVE * 8 <= RING, "the sums that change hands fit");
    constexpr int PLACES = STAGES / 2;
    const int each = halves / 16, rounds = 4 * each;  // steps of 64 of an eighth, of two eighths in turn
    const bf16_t* src[MOST];
    const int row_of = lane / 8;
#pragma unroll
    for (int j = 0; j < MOST; ++j) {
      const int r = (wave + j * WAVES) * 8 + row_of;
      const int chunk = (lane % 8) ^ (r % 8);
      if ((wave + j * WAVES) * 8 < BM) src[j] = a_row(r) + chunk * 8;
      else if (wave + j * WAVES < LOADS) src[j] = w_row(r - BM) + chunk * 8;
      else src[j] = nullptr;  // (not fetched)
      if (ROUND) src[j] += begin * each * (2 * STEP_K);
    }
    int left = each, pair = ROUND ? begin : 0;  // of what is fetched
    auto fetch = [&](int place) {
      bf16_t* to = ring + place * (2 * STAGE) + wave * 512;
      int add = STEP_K;
      if (--left == 0) {
        left = each;
        add += each * STEP_K;
        if (ROUND && ++pair == 4) pair = 0, add -= 8 * each * STEP_K;
      }
#pragma unroll
      for (int j = 0; j < MOST; ++j) {
        if (j < EACH || wave < REST) {
#pragma unroll
          for (int odd = 0; odd < 2; ++odd) {
            if ((wave + j * WAVES) * 8 >= BM) __builtin_amdgcn_global_load_lds((global_void*)(src[j] + odd * each * STEP_K), (lds_void*)(to + odd * STAGE + j * (WAVES * 512)), 16, 0, 2);
            else __builtin_amdgcn_global_load_lds((global_void*)(src[j] + odd * each * STEP_K), (lds_void*)(to + odd * STAGE + j * (WAVES * 512)), 16, 0, 0);
          }
        }
        src[j] += add;
      }
    };
    // waits until at most `newer` (PLACES - 1 or fewer) places' loads of this wave are outstanding
    auto wait_places = [&](int newer) {
      if (newer >= 2) {
        if (REST > 0 && wave < REST) outstanding<2 * 2 * MOST>();
        else outstanding<2 * 2 * EACH>();
      } else if (newer == 1) {
        if (REST > 0 && wave < REST) outstanding<2 * MOST>();
        else outstanding<2 * EACH>();
      } else {
        outstanding<0>();
      }
    };
    static_assert(PLACES == 3, "as wait_places counts");
#pragma unroll
    for (int s = 0; s < PLACES; ++s)
      if (s < rounds) fetch(s);
    f32x4_t sums[4][NT][MT];  // of this wave's eighths
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    bf16x8_t wf[2][NT], af[2][MT];
    const bf16_t* a_at = ring + wk * STAGE + (wm * MT * 16 + col) * STEP_K;
    const bf16_t* w_at = ring + wk * STAGE + (BM + wn * NT * 16 + col) * STEP_K;
    auto read = [&](int set, int place, int half) {
      const int at = place * (2 * STAGE) + ((half * 4 + quad) ^ (col % 8)) * 8;
#pragma unroll
      for (int n = 0; n < NT; ++n) wf[set][n] = *reinterpret_cast<const bf16x8_t*>(w_at + n * 16 * STEP_K + at);
#pragma unroll
      for (int m = 0; m < MT; ++m) af[set][m] = *reinterpret_cast<const bf16x8_t*>(a_at + m * 16 * STEP_K + at);
    };
    auto multiply = [&](int set) {
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[set][n], af[set][m], acc[n][m], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
    };
    int place = 0, done = ROUND ? begin : 0, part_left = each;
    wait_places(min(rounds, PLACES) - 1);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read(0, 0, 0);
    for (int round = 0; round < rounds; ++round) {
      read(1, place, 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(0);
      __builtin_amdgcn_sched_barrier(0);
      const int before = place;
      place = place + 1 == PLACES ? 0 : place + 1;
      if (round + 1 < rounds) {  // the next place is in LDS for all waves, and nobody reads this one any more: it is filled anew
        wait_places(min(rounds - 2 - round, PLACES - 2));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (round + PLACES < rounds) fetch(before);
        read(0, place, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
      multiply(1);
      __builtin_amdgcn_sched_barrier(0);
      if (--part_left == 0) {
        part_left = each;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (done == i) {
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
              for (int m = 0; m < MT; ++m) sums[i][n][m] = acc[n][m];
          }
        done = done == 3 ? 0 : done + 1;
#pragma unroll
        for (int n = 0; n < NT; ++n)
#pragma unroll
          for (int m = 0; m < MT; ++m) acc[n][m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
      }
    }
    __syncthreads();
    f32x4_t* to = reinterpret_cast<f32x4_t*>(ring) + ((wm * WN + wn) * 4 * NT * MT) * MI_WAVE + lane;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          if (!mine(m)) to[((i * NT + n) * MT + m) * MI_WAVE] = sums[i][n][m];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int m = 0; m < MT; ++m)
          if (mine(m)) {
            const f32x4_t other = to[((i * NT + n) * MT + m) * MI_WAVE];
            acc[n][m] += wk == 0 ? sums[i][n][m] : other;
            acc[n][m] += wk == 0 ? other : sums[i][n][m];
          }
  }

  // The sums rounded to bfloat16 as rows of the tile in `ring`, MADE elements apart; all threads see them afterwards.
  __device__ __forceinline__ void leave(bf16_t* ring) {
    __syncthreads();
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (mine(m)) {
#pragma unroll
        for (int n = 0; n < NT; ++n) {
          const float v[4] = {acc[n][m][0], acc[n][m][1], acc[n][m][2], acc[n][m][3]};
          mi_store_cols<bf16_t, 4>(ring + row(m) * MADE + feature(n), v);
        }
      }
    __syncthreads();
  }

  // Whether row tile m's sums are this wave's to write.
  __device__ __forceinline__ bool mine(int m) const { return WK == 1 || (m < FIRST_M) == (wk == 0); }
  // Where they lie in the tile: acc[n][m][j] is row `row(m)`, row of W `feature(n) + j`.
  __device__ __forceinline__ int row(int m) const { return (wm * MT + m) * 16 + col; }
  __device__ __forceinline__ int feature(int n) const { return (wn * NT + n) * 16 + quad * 4; }
};
