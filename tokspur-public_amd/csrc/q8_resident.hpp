// Internal interface of the Q8_0 product that keeps its token rows in registers (q8_resident.hip).
#pragma once
#include "tsp_common.hpp"

namespace tsp {

// x token-major [width, columns], y token-major [width, rows], width <= 16; columns a multiple of 256 up to 2560 (q8_lanes_v1 rows: 2560), 16-byte aligned
// matrix and activations. f32: the activations as the floats they are, always so beyond 2048 columns; else 22 significant bits of each row's largest
int q8_resident(bool lanes, bool f32, const void* matrix, const float* x, float* y, uint32_t columns, uint32_t rows, uint32_t width, uint32_t* error_word, hipStream_t stream);

}  // namespace tsp
