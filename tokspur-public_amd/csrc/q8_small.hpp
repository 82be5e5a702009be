// Internal interface of the Q8_0 product for few token rows against matrices too small for the persistent kernel (q8_small.hip).
#pragma once
#include "tsp_common.hpp"

namespace tsp {

// y[t, r] = sum_k W[r, k] x[t, k] for any number of token rows, sixteen (eight) at a time, raw GGUF rows of a multiple of 64 columns, rows any distance apart that
// 16 bytes (x) resp. 4 bytes (y) divide.
bool q8_small_takes(const void* matrix, const float* x, uint64_t x_stride_bytes, uint32_t columns, uint32_t rows);
int q8_small(const void* matrix, const float* x, uint64_t x_stride_bytes, float* y, uint64_t y_stride_bytes, uint32_t columns, uint32_t rows, uint32_t tokens,
             uint32_t* error_word, hipStream_t stream);

}  // namespace tsp
