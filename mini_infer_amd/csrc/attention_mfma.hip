// Launches of the matrix-core attention (attention_mfma.h): prefill portions and decode tokens, each with a launch of its own.
#include "attention_mfma.h"

// OCC: waves per SIMD the registers are budgeted for.
template <int D, int WAVES, int KW, int RG, int OCC, bool SHARED, int PS, int VD = D, bool ANYV = false>
__global__ __launch_bounds__(64 * WAVES * KW, OCC) void attn_mfma_kernel(
    const bf16_t* __restrict__ q, int64_t q_row_stride, const bf16_t* __restrict__ k_pages,
    const bf16_t* __restrict__ vt_pages, const int* __restrict__ block_table, int max_blocks,
    const int* __restrict__ cu_seqlens_q, const int* __restrict__ positions, int num_requests,
    bf16_t* __restrict__ out, int64_t out_row_stride, float* __restrict__ part_acc,
    float* __restrict__ part_ml, int q_heads, int kv_heads, int page_size_arg, unsigned page_magic, float scale_log2,
    int window, int num_splits, int heads_per_block, int tokens_per_tile, int one_tile_per_request,
    int pair_group, int first_token, int has_sink, float sink_log2, int mask_chunk,
    const float* __restrict__ sinks, const float* __restrict__ slopes, float softcap, int v_dim_arg,
    const bf16_t* __restrict__ gate, int64_t gate_row_stride) {
  attn_mfma_block<D, WAVES, KW, RG, SHARED, PS, VD, ANYV>(
      blockIdx.x, gridDim.x, blockIdx.z, false, 0, q, q_row_stride, k_pages, vt_pages, block_table, max_blocks, cu_seqlens_q, positions,
      num_requests, out, out_row_stride, part_acc, part_ml, q_heads, kv_heads, page_size_arg, page_magic, scale_log2, window, num_splits,
      heads_per_block, tokens_per_tile, one_tile_per_request, pair_group, first_token, has_sink, sink_log2, mask_chunk, sinks, slopes,
      softcap, v_dim_arg, gate, gate_row_stride);
}

extern "C" int mi_attn_mfma_tokens_per_tile(int q_heads, int kv_heads, int shape) {
  if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) return 0;
  const int rows = rows_of_shape(shape);
  const int hb = heads_per_block_for(q_heads / kv_heads, rows);
  const int t = rows / hb;
  return t < 1 ? 1 : t;
}

extern "C" int mi_attn_mfma_supported(int head_dim, int page_size) {
  const bool d_ok = head_dim == 32 || head_dim == 64 || head_dim == 96 || head_dim == 128 ||
                    head_dim == 192 || head_dim == 256;
  return (d_ok && page_size > 0 && page_size % 16 == 0) ? 1 : 0;
}

// Value heads of a width of their own: which pairs of widths have a kernel (pages of 16 slots only).
extern "C" int mi_attn_mfma_values_supported(int head_dim, int v_dim, int page_size) {
  if (!mi_attn_mfma_supported(head_dim, page_size)) return 0;
  if (v_dim == head_dim) return 1;
  return (head_dim == 64 || head_dim == 96 || head_dim == 128 || head_dim == 192) && page_size == 16 && v_dim > 0 &&
                 v_dim % 16 == 0 && v_dim <= 128 ? 1 : 0;
}

// `num_tiles` = sum over requests of ceil(q_len / tokens_per_tile), computed by the
// caller from the host copy of cu_seqlens_q (a larger number is harmless).
// `one_tile_per_request` = 1 promises that no request has more than tokens_per_tile
// tokens in this step, 2 that every request has exactly one (then cu_seqlens_q is not
// read); in both cases num_tiles must be num_requests.
// The requests may be a run out of a larger step: cu_seqlens_q and block_table then point
// at the run's first request, while q, out, positions and the partial buffers stay
// those of the whole step (cu_seqlens_q holds token numbers of the whole step);
// `first_token` is the run's first token and `num_tokens` the run's token count.
// With num_splits > 1, part_acc holds (first_token+num_tokens)*q_heads*num_splits*head_dim
// floats (v_dim floats where value heads have a width of their own) and part_ml
// (first_token+num_tokens)*q_heads*num_splits*2; `combine` = 0 leaves the
// key ranges' results there for the caller's next kernel to combine (`out` is not written).
// `gate` (bfloat16, row t at t * gate_row_stride, one number per query head; may be null): head h's
// result for token t is multiplied by logistic(gate[t][h]).
extern "C" int mi_attn_mfma(const void* q, int64_t q_row_stride, const void* k_pages,
                            const void* vt_pages, const int* block_table, int max_blocks,
                            const int* cu_seqlens_q, const int* positions, int num_requests,
                            int num_tokens, int num_tiles, void* out, int64_t out_row_stride,
                            float* part_acc, float* part_ml, int q_heads, int kv_heads,
                            int head_dim, int page_size, int num_pages, float scale, int window,
                            int num_splits, int shape, int one_tile_per_request,
                            int first_token, int combine, int has_sink, float sink_logit, int mask_chunk,
                            const float* sinks, const float* slopes, float softcap, int v_dim, const void* gate,
                            int64_t gate_row_stride, hipStream_t stream) {
  MI_REQUIRE(mi_attn_mfma_values_supported(head_dim, v_dim, page_size),
             "attn_mfma: value heads of %d beside key heads of %d in pages of %d are not taken", v_dim, head_dim, page_size);
  MI_REQUIRE(gate == nullptr || (gate_row_stride >= q_heads && (num_splits == 1 || combine)),
             "attn_mfma: a gate has one number per query head and goes with combined results");
  MI_REQUIRE(sinks == nullptr || has_sink, "attn_mfma: per-head sink logits come with has_sink");
  MI_REQUIRE(softcap >= 0.f, "attn_mfma: softcap=%g must be 0 (none) or positive", (double)softcap);
  MI_REQUIRE(mask_chunk >= 0, "attn_mfma: mask_chunk=%d must be 0 (none) or positive", mask_chunk);
  MI_REQUIRE(first_token >= 0, "attn_mfma: first_token=%d is negative", first_token);
  MI_REQUIRE(num_tokens >= 0 && num_requests >= 0 && num_tiles >= 0,
             "attn_mfma: bad sizes tokens=%d requests=%d tiles=%d", num_tokens, num_requests, num_tiles);
  MI_REQUIRE(q_heads > 0 && kv_heads > 0 && q_heads % kv_heads == 0,
             "attn_mfma: q_heads=%d is not a multiple of kv_heads=%d", q_heads, kv_heads);
  MI_REQUIRE(mi_attn_mfma_supported(head_dim, page_size),
             "attn_mfma: head_dim=%d (32, 64, 96, 128, 192 or 256) or page_size=%d (multiple of 16) not taken",
             head_dim, page_size);
  MI_REQUIRE(num_pages > 0 && max_blocks > 0, "attn_mfma: bad page counts num_pages=%d max_blocks=%d",
             num_pages, max_blocks);
  MI_REQUIRE((uintptr_t)k_pages % 128 == 0 && (uintptr_t)vt_pages % 128 == 0,
             "attn_mfma: the pages must begin on a 128-byte boundary (they are read in whole cache lines)");
  MI_REQUIRE(window >= 0, "attn_mfma: window=%d must be 0 (none) or positive", window);
  MI_REQUIRE(scale > 0.f, "attn_mfma: the score scale must be positive, got %g", (double)scale);
  MI_REQUIRE(num_splits >= 1 && num_splits <= 64, "attn_mfma: num_splits=%d must be 1..64", num_splits);
  MI_REQUIRE(num_splits == 1 || (part_acc && part_ml), "attn_mfma: split keys need partial buffers");
  MI_REQUIRE(q_row_stride >= (int64_t)q_heads * head_dim && out_row_stride >= (int64_t)q_heads * v_dim,
             "attn_mfma: row strides shorter than q_heads*head_dim");
  MI_REQUIRE(q_row_stride % 8 == 0 && out_row_stride % 4 == 0,
             "attn_mfma: row strides must keep 16-byte (q) and 8-byte (out) alignment");
  MI_REQUIRE(one_tile_per_request >= 0 && one_tile_per_request <= 2, "attn_mfma: one_tile_per_request is 0, 1 or 2");
  MI_REQUIRE(one_tile_per_request != 2 || num_tokens == num_requests,
             "attn_mfma: one token per request needs num_tokens == num_requests");
  MI_REQUIRE(!one_tile_per_request || num_tiles == num_requests,
             "attn_mfma: one tile per request needs num_tiles == num_requests");
  if (num_tokens == 0 || num_tiles == 0) return MI_OK;

  MI_REQUIRE(shape == MI_SHAPE_PREFILL || shape == MI_SHAPE_DECODE || (shape == MI_SHAPE_PREFILL_WIDE && head_dim <= 128),
             "attn_mfma: shape %d (0 prefill, 1 decode, 2 wide prefill for head sizes up to 128)", shape);
  const bool decode_only = shape == MI_SHAPE_DECODE;
  const int group = q_heads / kv_heads;
  const int rows = rows_of_shape(shape);
  const int hb = heads_per_block_for(group, rows);
  const int tq = mi_attn_mfma_tokens_per_tile(q_heads, kv_heads, shape);
  const int head_blocks = ceil_div(group, hb);
  MI_REQUIRE((int64_t)num_tiles * kv_heads * head_blocks < (1ll << 31), "attn_mfma: too many tiles x heads");
  MI_REQUIRE(num_splits <= 65535, "attn_mfma: too many splits");
  dim3 grid((unsigned)(num_tiles * kv_heads * head_blocks), 1, num_splits);
  const float scale_log2 = scale * LOG2E;
  // prefill blocks run two to a CU: see the tile order in the kernel (8 XCDs share the CUs evenly)
  int pair_group = 0;
  if (shape == MI_SHAPE_PREFILL && MI_PREFILL_OCC(head_dim) == 2) {
    int device = 0, cus = 0;
    if (hipGetDevice(&device) == hipSuccess &&
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess)
      pair_group = cus / 8;
  }
  // keys reach max_blocks*page_size + 32 at most; the multiply-high division is exact below 2^32/page_size
  MI_REQUIRE(((int64_t)max_blocks * page_size + 64) * page_size < (1ll << 32),
             "attn_mfma: block table of %d pages of %d is too long for this kernel", max_blocks, page_size);
  const unsigned page_magic = (unsigned)((1ull << 32) / (unsigned)page_size) + 1u;

#define MI_LAUNCH_V(DD, WW, KK, RR, OO, SS, PP, VV, AA)                                                \
  attn_mfma_kernel<DD, WW, KK, RR, OO, SS, PP, VV, AA><<<grid, 64 * WW * KK, 0, stream>>>(            \
      (const bf16_t*)q, q_row_stride, (const bf16_t*)k_pages, (const bf16_t*)vt_pages,            \
      block_table, max_blocks, cu_seqlens_q, positions, num_requests, (bf16_t*)out,               \
      out_row_stride, part_acc, part_ml, q_heads, kv_heads, page_size, page_magic, scale_log2,    \
      window,                                                                                     \
      num_splits, hb, tq, one_tile_per_request, pair_group, first_token, has_sink, sink_logit * LOG2E, mask_chunk, \
      sinks, slopes, softcap, v_dim, (const bf16_t*)gate, gate_row_stride)
#define MI_LAUNCH(DD, WW, KK, RR, OO, SS, PP) MI_LAUNCH_V(DD, WW, KK, RR, OO, SS, PP, DD, false)
// (head sizes above 128 have no wide shape and were refused above: their cases name the 128 kernel,
// so that nothing is compiled for them)
#define MI_LAUNCH_P(DD, PP)                                                                       \
  if (decode_only) MI_LAUNCH(DD, 1, MI_DECODE_KW, 1, 2, false, PP);                               \
  else if (shape == MI_SHAPE_PREFILL_WIDE) MI_LAUNCH((DD <= 128 ? DD : 128), MI_WIDE_WAVES, 1, MI_PREFILL_RG, 2, true, PP); \
  else MI_LAUNCH(DD, MI_PREFILL_WAVES, 1, MI_PREFILL_RG, MI_PREFILL_OCC(DD), true, PP)
#define MI_LAUNCH_D(DD)                 \
  if (page_size == 16) {                \
    MI_LAUNCH_P(DD, 16);                \
  } else {                              \
    MI_LAUNCH_P(DD, 0);                 \
  }
// value heads of a width of their own: rounded up to 64, 96 or 128
#define MI_LAUNCH_DV(DD, VV)                                                                               \
  if (decode_only) MI_LAUNCH_V(DD, 1, MI_DECODE_KW, 1, 2, false, 16, VV, true);                            \
  else if (shape == MI_SHAPE_PREFILL_WIDE)                                                                 \
    MI_LAUNCH_V((DD <= 128 ? DD : 128), MI_WIDE_WAVES, 1, MI_PREFILL_RG, 2, true, 16, VV, true);           \
  else MI_LAUNCH_V(DD, MI_PREFILL_WAVES, 1, MI_PREFILL_RG, MI_PREFILL_OCC(DD), true, 16, VV, true)
#define MI_LAUNCH_ANYV(DD)                          \
  if (v_dim <= 64) { MI_LAUNCH_DV(DD, 64); }        \
  else if (v_dim <= 96) { MI_LAUNCH_DV(DD, 96); }   \
  else { MI_LAUNCH_DV(DD, 128); }
  if (v_dim != head_dim) {
    switch (head_dim) {
      case 64: MI_LAUNCH_ANYV(64); break;
      case 96: MI_LAUNCH_ANYV(96); break;
      case 128: MI_LAUNCH_ANYV(128); break;
      default: MI_LAUNCH_ANYV(192); break;
    }
  } else {
    switch (head_dim) {
      case 32: MI_LAUNCH_D(32); break;
      case 64: MI_LAUNCH_D(64); break;
      case 96: MI_LAUNCH_D(96); break;
      case 128: MI_LAUNCH_D(128); break;
      case 192: MI_LAUNCH_D(192); break;
      default: MI_LAUNCH_D(256); break;
    }
  }
#undef MI_LAUNCH_ANYV
#undef MI_LAUNCH_DV
#undef MI_LAUNCH_D
#undef MI_LAUNCH_P
#undef MI_LAUNCH
#undef MI_LAUNCH_V
  MI_CHECK_LAUNCH("attn_mfma");
  if (num_splits > 1 && combine) {
    const int64_t first_slot = (int64_t)first_token * q_heads * num_splits;
    return mi_attn_reduce_bf16(part_acc + first_slot * v_dim, part_ml + first_slot * 2,
                               (bf16_t*)out + (int64_t)first_token * out_row_stride, out_row_stride,
                               num_tokens, q_heads, v_dim, num_splits, 0, 1, has_sink, sink_logit, sinks,
                               gate ? (const bf16_t*)gate + (int64_t)first_token * gate_row_stride : nullptr,
                               gate_row_stride, stream);
  }
  return MI_OK;
}
