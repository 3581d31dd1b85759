#pragma once

#include "gemm_common.h"

namespace vk {

// A projection of fp32 rows on narrow tiles of 16 << plan rows x 16 columns (plan 0, 1, 2).
template <int kEpi>
void launch_narrow_f32(const GemmArgs& a, int plan, hipStream_t st);

}  // namespace vk
