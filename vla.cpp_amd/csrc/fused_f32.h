// Launches that the host layer takes beside the C ABI (plain C++, no device types).
#pragma once

#include "vla_kernels.h"

namespace vk {

// fp32: rms_norm(x) * norm_w and the projection behind it as one launch, for the few rows that the narrow tiles take.
// Arguments as vla_attn_qkv_rope and vla_glu_linear take them (W is not folded).  VLA_K_ERR_SHAPE, launching nothing,
// where the shape is not one of theirs: the caller then runs the norm as a launch of its own.
int f32_rmsnorm_attn_qkv_rope(const float* x, const float* norm_w, float eps, const float* W, const float* bias, int M, int K, int S,
                              int n_q_heads, int n_kv_heads, int has_k, int has_v, int head_dim, const float* cos_tab,
                              const float* sin_tab, void* q_out, void* k_cache, void* vt_cache, int t_max, int tok_offset,
                              vla_stream_t stream);
int f32_rmsnorm_glu_linear(const float* x, const float* norm_w, float eps, const float* W_gate_up, void* y, int M, int I, int K, int act,
                           vla_stream_t stream);

}  // namespace vk
