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

// Each XCD fetches the activation rows and the weight rows that its run of tiles touches into an L2 of its own: the band (of row tiles) that
// makes the run touch the fewest bytes.
inline uint32_t dense_band(uint32_t m_tiles, uint32_t n_tiles, uint32_t tile_m, uint32_t tile_n) {
    const uint32_t run = (m_tiles * n_tiles + 7) / 8;
    uint64_t least = ~0ull;
    uint32_t best = 1;
    for (uint32_t band = 1; band <= m_tiles; ++band) {
        const uint32_t wide = n_tiles < (run + band - 1) / band ? n_tiles : (run + band - 1) / band, rounds = run / (band * n_tiles), high = band * (rounds ? rounds : 1);
        const uint64_t bytes = uint64_t(high) * tile_m * 32 + uint64_t(wide) * tile_n * 9;
        if (bytes < least) { least = bytes; best = band; }
    }
    return best;
}

// Few rows are multiplied by exact integer factors, more by weights rounded once to half.
inline bool dense_exact(uint32_t m, uint32_t n) { return m < 512 || n < 256; }

// The kernel for few tiles (dense_fragments.hip): how many waves a workgroup takes, 0 where launch_dense_tile is the faster one.
// It wants `a` and `sx` in fragment order: 32 rows at a time (fewer at the end) from where plain rows would put the first of them, then 16-byte pieces
// [16 columns or, for the sums, a super-block][k-half][row].
uint32_t dense_fragments_waves(uint32_t m, uint32_t n, uint32_t k);
int launch_dense_fragments(DenseTileArgs a, uint32_t waves, hipStream_t stream);

}  // namespace tsp
