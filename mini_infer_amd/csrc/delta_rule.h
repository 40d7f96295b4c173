// What the two forms of the gated delta rule share (delta_rule.hip, delta_chunks.hip).
#pragma once
#include "common.h"

extern "C" int mi_gated_delta_rows(int dim, int vdim);  // rows of a head's S as kept: dim rounded up

// Refuses sizes, strides and columns that do not fit one another.
int mi_gated_delta_check(int64_t qkv_stride, int64_t proj_stride, int col_b, int col_a, int col_g, const float* state,
                         int64_t state_stride, int64_t out_stride, int num_requests, int heads, int kv_heads, int dim, int vdim,
                         int dim_pad, float eps, int num_slots);

// The token-by-token recurrence over a step's bfloat16 rows, sizes checked, for the columns whose flag in `again` (one for 16
// columns, [requests][heads][ceil(vdim / 16)]) is set.
int mi_delta_again(const void* qkv, int64_t qkv_stride, const void* proj, int64_t proj_stride, int col_b, int col_a, const float* a_log,
                   const float* dt_bias, float* state, int64_t state_stride, const int* cu, const int* slots, float* readout,
                   const int* again, int num_requests, int heads, int kv_heads, int dim, int vdim, int num_slots, hipStream_t stream);

// The read-outs' norm and gate, the last launch of both.
int mi_delta_readout_norm(int dtype, const float* readout, const void* proj, int64_t proj_stride, int col_g, const float* norm_weight,
                          void* out, int64_t out_stride, int num_tokens, int heads, int vdim, float eps, hipStream_t stream);
