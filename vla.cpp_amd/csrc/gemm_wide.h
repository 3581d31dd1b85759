#pragma once

#include <type_traits>

#include "gemm_common.h"

namespace vk {

// A bf16 projection on tile `tile` of the wide-tile kernel; false, launching nothing, when the grid is too large for it.
template <int kEpi>
bool launch_wide(const GemmArgs& a, int tile, hipStream_t st);

}  // namespace vk
