// Internal interface of the any-length GEMV (gemv.hip) for the Q8_0 entry points.
#pragma once
#include "tsp_common.hpp"

namespace tsp {

// One token row against raw GGUF Q8_0 rows; *taken says whether the shape is one the kernel takes (nothing is launched otherwise).
int gemv_q8_row(const void* matrix, const float* x, float* y, uint32_t columns, uint32_t rows, uint32_t* error_word, hipStream_t stream, bool* taken);

}  // namespace tsp
