#pragma once

#include "gemm_common.h"

namespace vk {

constexpr int F32_NORM_MAX_K = 2048;  // K of a projection with the norm inside: its weight stays in LDS

// A projection of fp32 rows on narrow tiles of 16 << plan rows x 16 columns (plan 0, 2); QKV and GLU with norm_eps >= 0: of
// their RMSNorm with weight norm_w.
template <int kEpi>
void launch_narrow_f32(const GemmArgs& a, int plan, hipStream_t st);

}  // namespace vk
