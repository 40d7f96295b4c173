// The matrix-core attention (attention_mfma.h) of a step that brings portions of prompts beside single tokens, as one launch: some
// blocks are of the prefill shape, the others of the decode shape, and one combining launch serves both.
//
// What bounds it: neither part fills the GPU (15 single tokens and a portion of 256 at 24 heads of 128 over 8: 240 blocks that read
// their keys once, and 56 of 128 rows), so launched one after the other each waited for the other's tail, and each had a combining
// launch of its own.  That step's attention at 3B widths (single tokens at up to 1,500 positions), a layer: 43.1 us (17.0 + 6.0 for the
// single tokens, 14.0 + 6.0 for the portion, which was cut by the longest request's keys into more ranges than it has) -> 24.1 us (20.2 +
// 3.9); the whole step 4,934 -> 4,350 us, two launches a layer fewer for the host.   In a
// recorded step every single token stood in a tile of 128 rows of its own.
// The prefill blocks come first, as the longer ones, and the decode blocks fill the CUs beside them.
#include "attention_mfma.h"

namespace {

struct MixedPart {  // see attn_mfma_block
  unsigned blocks;
  int num_splits, heads_per_block, tokens_per_tile, one_tile_per_request, slot_token, num_requests;
  int64_t slots;  // partial results that lie before this part's
};

template <int D>
__global__ __launch_bounds__(64 * MI_PREFILL_WAVES, MI_PREFILL_OCC(D)) void attn_mixed_kernel(
    const bf16_t* __restrict__ q, int64_t q_row_stride, const bf16_t* __restrict__ k_pages, const bf16_t* __restrict__ vt_pages,
    const int* __restrict__ block_table, int max_blocks, const int* __restrict__ cu_seqlens_q, const int* __restrict__ positions,
    bf16_t* __restrict__ out, int64_t out_row_stride, float* __restrict__ part_acc, float* __restrict__ part_ml, int q_heads, int kv_heads,
    float scale_log2, int window, int pair_group, int singles, int has_sink, float sink_log2, int mask_chunk,
    const float* __restrict__ sinks, const float* __restrict__ slopes, float softcap, const bf16_t* __restrict__ gate,
    int64_t gate_row_stride, MixedPart tiles, MixedPart single) {
  static_assert(MI_PREFILL_WAVES == MI_DECODE_KW, "blocks of both shapes have the same threads");
  const unsigned of_tiles = tiles.blocks * (unsigned)tiles.num_splits;
  if (blockIdx.x < of_tiles) {
    const int lead = max(singles, 0);
    attn_mfma_block<D, MI_PREFILL_WAVES, 1, MI_PREFILL_RG, true, 16>(
        blockIdx.x % tiles.blocks, tiles.blocks, blockIdx.x / tiles.blocks, singles < 0, tiles.slot_token, q, q_row_stride, k_pages, vt_pages,
        block_table + (int64_t)lead * max_blocks, max_blocks, cu_seqlens_q + lead, positions, tiles.num_requests, out, out_row_stride,
        part_acc + tiles.slots * D, part_ml + tiles.slots * 2, q_heads, kv_heads, 16, 0u, scale_log2, window, tiles.num_splits,
        tiles.heads_per_block, tiles.tokens_per_tile, tiles.one_tile_per_request, pair_group, 0, has_sink, sink_log2, mask_chunk, sinks,
        slopes, softcap, D, gate, gate_row_stride);
  } else {
    const unsigned at = blockIdx.x - of_tiles;
    attn_mfma_block<D, 1, MI_DECODE_KW, 1, false, 16>(
        at % single.blocks, single.blocks, at / single.blocks, false, single.slot_token, q, q_row_stride, k_pages, vt_pages, block_table,
        max_blocks, cu_seqlens_q, positions, single.num_requests, out, out_row_stride, part_acc + single.slots * D,
        part_ml + single.slots * 2, q_heads, kv_heads, 16, 0u, scale_log2, window, single.num_splits, single.heads_per_block,
        single.tokens_per_tile, single.one_tile_per_request, 0, 0, has_sink, sink_log2, mask_chunk, sinks, slopes, softcap, D, gate,
        gate_row_stride);
  }
}

}  // namespace

extern "C" int mi_attn_mixed_supported(int head_dim, int v_dim, int page_size) {
  return (head_dim == 64 || head_dim == 128) && v_dim == head_dim && page_size == 16 ? 1 : 0;
}

// Arguments as mi_attn_mfma, over a whole step of num_requests requests.  singles >= 0: the first `singles` requests bring one token
// each (the first tokens of the step), and num_tiles counts the tiles of the others; singles < 0: which requests bring a single token is found on the device (a recorded
// step), num_tiles is at least the tiles of all the others, and both parts have the same number of key ranges.
// part_acc holds the partial results of the tokens whose keys are cut: (singles * single_splits + (num_tokens - singles) * tile_splits) *
// q_heads * head_dim floats, less the half whose number of ranges is 1 (singles < 0: num_tokens * tile_splits * q_heads * head_dim);
// part_ml the same with 2 in place of head_dim.
extern "C" int mi_attn_mixed(const void* q, int64_t q_row_stride, const void* k_pages, const void* vt_pages, const int* block_table,
                             int max_blocks, const int* cu_seqlens_q, const int* positions, int num_requests, int num_tokens, int singles,
                             int num_tiles, void* out, int64_t out_row_stride, float* part_acc, float* part_ml, int q_heads, int kv_heads,
                             int head_dim, int page_size, int num_pages, float scale, int window, int single_splits, int tile_splits,
                             int has_sink, float sink_logit, int mask_chunk, const float* sinks, const float* slopes, float softcap,
                             const void* gate, int64_t gate_row_stride, hipStream_t stream) {
  MI_REQUIRE(mi_attn_mixed_supported(head_dim, head_dim, page_size), "attn_mixed: heads of %d in pages of %d are not taken", head_dim, page_size);
  MI_REQUIRE(q_heads > 0 && kv_heads > 0 && q_heads % kv_heads == 0, "attn_mixed: q_heads=%d is not a multiple of kv_heads=%d", q_heads, kv_heads);
  MI_REQUIRE(num_tokens > 0 && num_requests > 0 && singles < num_requests && singles < num_tokens && num_tiles > 0,
             "attn_mixed: tokens=%d requests=%d singles=%d tiles=%d", num_tokens, num_requests, singles, num_tiles);
  MI_REQUIRE(gate == nullptr || gate_row_stride >= q_heads, "attn_mixed: a gate has one number per query head");
  MI_REQUIRE(sinks == nullptr || has_sink, "attn_mixed: per-head sink logits come with has_sink");
  MI_REQUIRE(softcap >= 0.f && mask_chunk >= 0 && window >= 0 && scale > 0.f, "attn_mixed: softcap=%g mask_chunk=%d window=%d scale=%g",
             (double)softcap, mask_chunk, window, (double)scale);
  MI_REQUIRE(num_pages > 0 && max_blocks > 0 && ((int64_t)max_blocks * page_size + 64) * page_size < (1ll << 32),
             "attn_mixed: bad page counts num_pages=%d max_blocks=%d", num_pages, max_blocks);
  MI_REQUIRE((uintptr_t)k_pages % 128 == 0 && (uintptr_t)vt_pages % 128 == 0, "attn_mixed: the pages must begin on a 128-byte boundary");
  MI_REQUIRE(single_splits >= 1 && single_splits <= 64 && tile_splits >= 1 && tile_splits <= 64 && (singles >= 0 || single_splits == tile_splits),
             "attn_mixed: key ranges %d and %d", single_splits, tile_splits);
  MI_REQUIRE((single_splits == 1 && tile_splits == 1) || (part_acc && part_ml), "attn_mixed: split keys need partial buffers");
  MI_REQUIRE(q_row_stride >= (int64_t)q_heads * head_dim && out_row_stride >= (int64_t)q_heads * head_dim && q_row_stride % 8 == 0 &&
                 out_row_stride % 4 == 0,
             "attn_mixed: row strides %lld and %lld", (long long)q_row_stride, (long long)out_row_stride);
  const int group = q_heads / kv_heads;
  const bool known = singles >= 0;
  auto part = [&](int shape, int splits, int units) {
    MixedPart p;
    p.heads_per_block = heads_per_block_for(group, rows_of_shape(shape));
    p.tokens_per_tile = max(1, rows_of_shape(shape) / p.heads_per_block);
    p.blocks = (unsigned)((int64_t)units * kv_heads * ceil_div(group, p.heads_per_block));
    p.num_splits = splits;
    p.slot_token = 0;
    p.slots = 0;
    return p;
  };
  MI_REQUIRE(((int64_t)num_tiles + num_requests) * q_heads * 64 < (1ll << 31), "attn_mixed: too many tiles x heads");
  MixedPart tiles = part(MI_SHAPE_PREFILL, tile_splits, num_tiles), single = part(MI_SHAPE_DECODE, single_splits, known ? singles : num_requests);
  tiles.one_tile_per_request = 0;
  tiles.num_requests = num_requests - max(singles, 0);
  single.one_tile_per_request = known ? 2 : 3;
  single.num_requests = known ? singles : num_requests;
  if (known) {
    tiles.slot_token = singles;
    if (single_splits > 1) tiles.slots = (int64_t)singles * q_heads * single_splits;  // (tokens that are not cut have no partial results)
  }
  int device = 0, cus = 0, pair_group = 0;  // (see the tile order in the kernel)
  if (hipGetDevice(&device) == hipSuccess && hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) == hipSuccess)
    pair_group = cus / 8;
  const unsigned grid = tiles.blocks * (unsigned)tile_splits + single.blocks * (unsigned)single_splits;
  const auto kernel = head_dim == 64 ? attn_mixed_kernel<64> : attn_mixed_kernel<128>;
  kernel<<<grid, 64 * MI_PREFILL_WAVES, 0, stream>>>(
      (const bf16_t*)q, q_row_stride, (const bf16_t*)k_pages, (const bf16_t*)vt_pages, block_table, max_blocks, cu_seqlens_q, positions,
      (bf16_t*)out, out_row_stride, part_acc, part_ml, q_heads, kv_heads, scale * LOG2E, window, pair_group, singles, has_sink,
      sink_logit * LOG2E, mask_chunk, sinks, slopes, softcap, (const bf16_t*)gate, gate_row_stride, tiles, single);
  MI_CHECK_LAUNCH("attn_mixed");
  // the tokens whose results lie in pieces
  const int first = known && single_splits == 1 ? singles : 0;
  const int last = known && tile_splits == 1 ? singles : num_tokens;
  if (first >= last || (single_splits == 1 && tile_splits == 1)) return MI_OK;
  const int lead = known && first == 0 ? singles : 0;
  return mi_attn_reduce_bf16(part_acc + (first > 0 ? tiles.slots * head_dim : 0), part_ml + (first > 0 ? tiles.slots * 2 : 0),
                             (bf16_t*)out + (int64_t)first * out_row_stride, out_row_stride, last - first, q_heads, head_dim, tile_splits, lead,
                             single_splits, has_sink, sink_logit, sinks,
                             gate ? (const bf16_t*)gate + (int64_t)first * gate_row_stride : nullptr, gate_row_stride, stream);
}
