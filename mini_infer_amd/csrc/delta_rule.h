// What the two forms of the gated delta rule share (delta_rule.hip, delta_chunks.hip).
#pragma once
#include "common.h"

extern "C" int mi_gated_delta_rows(int dim, int vdim);  // rows of a head's S as kept: dim rounded up

// Refuses sizes, strides and columns that do not fit one another.
int mi_gated_delta_check(int64_t qkv_stride, int64_t proj_stride, int col_b, int col_a, int col_g, const float* state,
                         int64_t state_stride, int64_t out_stride, int num_requests, int heads, int kv_heads, int dim, int vdim,
                         int dim_pad, float eps, int num_slots);

// The read-outs' norm and gate, the last launch of both.
int mi_delta_readout_norm(int dtype, const float* readout, const void* proj, int64_t proj_stride, int col_g, const float* norm_weight,
                          void* out, int64_t out_stride, int num_tokens, int heads, int vdim, float eps, hipStream_t stream);
