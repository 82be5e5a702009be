// Internal interface of the dense Q4_K GEMM over raw GGUF rows (dense_tile.hip), any number of activation rows whose halves stay
// under 4 GiB.
#pragma once
#include "tsp_common.hpp"

namespace tsp {

struct DenseTileArgs {
    const _Float16* a;   // activation rows as halves (bf16 values), a_stride halves apart, columns of every eight in the order
                         // (0, 2, 1, 3, 4, 6, 5, 7): the order in which a word of nibbles unpacks two at a time
    uint32_t a_stride;
    const _Float16* sx;  // per row and 256-column super-block: the eight 32-column sums as high halves, then their residuals
    const uint8_t* w;    // [n rows][k / 256 blocks of 144 B], under 4 GiB
    uint32_t m, n, k;
    uint32_t band;       // set by the launch
    void* out;           // f32 or bf16 rows, out_stride bytes apart
    uint64_t out_stride;
    int out_bf16;
    uint32_t* error_word;
};

int launch_dense_tile(const DenseTileArgs& a, hipStream_t stream);

}  // namespace tsp
