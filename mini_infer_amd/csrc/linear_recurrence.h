// What the two forms of the decaying recurrences share (linear_recurrence.hip, decay_chunks.hip).
#pragma once
#include "common.h"

extern "C" int mi_decay_scan_dim_pad(int dim);  // rows of a head's S as kept: dim rounded up

// Refuses sizes, strides and columns that do not fit one another.
int mi_decay_scan_check(int dtype, int mode, int64_t q_stride, int q_col, int64_t k_stride, int k_col, int64_t v_stride, int v_col,
                        int64_t gate_stride, int gate_col, const float* gate_bias, const float* rate, const float* state,
                        int64_t state_stride, int num_slots, int num_tokens, int num_requests, int heads, int groups, int dim, int vdim);

// log(1 + e) for 0 <= e <= 1 on the hardware's logarithm (one ulp), with the series where 1 + e
// would round e away
__device__ __forceinline__ float mi_log1p_small(float e) {
  return e < 1e-3f ? e * (1.f - e * (0.5f - e * 0.33333334f)) : 0.6931471805599453f * __builtin_amdgcn_logf(1.f + e);
}
// log(logistic(z)) = -softplus(-z), and softplus, float32 on the hardware's exponential and logarithm
__device__ __forceinline__ float mi_soft_plus_fast(float z) {
  return fmaxf(z, 0.f) + mi_log1p_small(__builtin_amdgcn_exp2f(-fabsf(z) * 1.4426950408889634f));
}
// logistic(z)^(1/tau)
__device__ __forceinline__ float mi_channel_decay(float z, float inv_tau) {
  return __builtin_amdgcn_exp2f(-mi_soft_plus_fast(-z) * (inv_tau * 1.4426950408889634f));
}
