// Q8_0 GEMV for 1, 2, 4 or 8 token rows (LM head / MTP verify): each weight byte is read once
// and decoded once for all token rows.
//
// Raw GGUF Q8_0 rows are 34-byte blocks (f16 scale + 32 int8), so blocks are only 2-byte aligned,
// but a row of K columns is K*17/16 bytes: a whole number of dwords whenever K % 64 == 0. The
// kernel therefore streams a row as a flat dword array, lane i taking dwords i, i+64, ... (fully
// coalesced), and works out per dword which block it lies in. A dword holds up to four quants of
// ONE block (the two bytes of a scale field that may share the dword are masked to a neutral
// code). The scale of that block is fetched with a 2-byte load that hits the same cache lines.
//
//   sum_k d*q_k*x_k with q_k = u_k - 128 (u = q ^ 0x80) = d * (sum_k u_k*x_k - 128 * sum_k x_k)
//
// so the four bytes convert with v_cvt_f32_ubyte0..3 and a masked byte (u = 0x80) contributes 0.
#include "decode.hpp"
#include "gemv.hpp"
#include "q8_mfma.hpp"
#include "q8_small.hpp"

using namespace tsp;

namespace {

struct Q8Args {
    const uint8_t* matrix;
    const float* x;   // token-major [M, columns]
    float* y;         // token-major [M, rows]
    uint32_t columns, rows;
    uint32_t* error_word;
};

__device__ __forceinline__ float ubf(uint32_t w, int i) { return float((w >> (8 * i)) & 0xffu); }

// M token rows; activations live in LDS as [M][columns + 4] with two zero floats either side so the
// neutral positions of a straddling dword read in-bounds, finite values.
template <int M>
__global__ __launch_bounds__(256) void q8_flat(Q8Args a) {
    extern __shared__ float lds[];
    const uint32_t stride = a.columns + 4;
    for (uint32_t i = threadIdx.x; i < M * stride; i += blockDim.x) {
        const uint32_t m = i / stride, c = i % stride;
        lds[i] = (c >= 2 && c < a.columns + 2) ? a.x[m * a.columns + (c - 2)] : 0.0f;
    }
    __syncthreads();

    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t row_dwords = a.columns / 32 * 34 / 4;
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    for (uint32_t row = blockIdx.x * (blockDim.x / kWave) + wave; row < a.rows; row += waves) {
        const uint8_t* data = a.matrix + uint64_t(row) * row_dwords * 4;
        float acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = 0;
        for (uint32_t dw = lane; dw < row_dwords; dw += kWave) {
            const uint32_t w = *reinterpret_cast<const uint32_t*>(data + dw * 4);
            const uint32_t byte0 = dw * 4, block = byte0 / 34, pos = byte0 - block * 34;  // pos even, 0..32
            // bytes of this dword that are quants of `block`: pos == 0 -> bytes 2,3; pos == 32 -> bytes 0,1
            const uint32_t vmask = pos == 0 ? 0xffff0000u : pos == 32 ? 0x0000ffffu : 0xffffffffu;
            const uint32_t u = ((w ^ 0x80808080u) & vmask) | (0x80808080u & ~vmask);
            const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(data + block * 34));
            // element index of byte 0 within the row, shifted by the two leading pad floats
            const uint32_t e0 = block * 32 + pos;  // = (block*32 + pos - 2) + 2
            const float u0 = ubf(u, 0), u1 = ubf(u, 1), u2 = ubf(u, 2), u3 = ubf(u, 3);
#pragma unroll
            for (int m = 0; m < M; ++m) {
                const float* xs = lds + m * stride + e0;
                const float x0 = xs[0], x1 = xs[1], x2 = xs[2], x3 = xs[3];
                float t = -128.0f * ((x0 + x1) + (x2 + x3));
                t = __builtin_fmaf(u0, x0, t);
                t = __builtin_fmaf(u1, x1, t);
                t = __builtin_fmaf(u2, x2, t);
                t = __builtin_fmaf(u3, x3, t);
                acc[m] = __builtin_fmaf(d, t, acc[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float total = wave_sum(acc[m]);
            if (lane == 0) {
                if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
                a.y[uint64_t(m) * a.rows + row] = total;
            }
        }
    }
}

// q8_lanes_v1 rows: [f16 scale x blocks][runs of 16 blocks x 512 B, byte = index*width + block%16].
// One lane takes the `width` bytes of one (run, index): element `index` of up to 16 blocks.
template <int M>
__global__ __launch_bounds__(256) void q8_lanes(Q8Args a) {
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t blocks = a.columns / 32, row_bytes = blocks * 34, runs = (blocks + 15) / 16;
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    for (uint32_t row = blockIdx.x * (blockDim.x / kWave) + wave; row < a.rows; row += waves) {
        const uint8_t* data = a.matrix + uint64_t(row) * row_bytes;
        float acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = 0;
        for (uint32_t item = lane; item < runs * 32; item += kWave) {
            const uint32_t run = item / 32, index = item % 32;
            const uint32_t width = blocks - run * 16 < 16 ? blocks - run * 16 : 16;
            const uint8_t* q = data + blocks * 2 + run * 512 + index * width;
            for (uint32_t b = 0; b < width; ++b) {
                const uint32_t block = run * 16 + b;
                const float wv = half_bits_to_float(ld16(data + block * 2)) * float(int(int8_t(q[b])));
#pragma unroll
                for (int m = 0; m < M; ++m) acc[m] = __builtin_fmaf(wv, a.x[uint64_t(m) * a.columns + block * 32 + index], acc[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float total = wave_sum(acc[m]);
            if (lane == 0) {
                if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
                a.y[uint64_t(m) * a.rows + row] = total;
            }
        }
    }
}

// Any K (multiple of 32) and any alignment: wave per row, lane per block.
template <int M>
__global__ __launch_bounds__(256) void q8_blocks(Q8Args a) {
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t blocks = a.columns / 32;
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);
    for (uint32_t row = blockIdx.x * (blockDim.x / kWave) + wave; row < a.rows; row += waves) {
        const uint8_t* data = a.matrix + uint64_t(row) * blocks * 34;
        float acc[M];
#pragma unroll
        for (int m = 0; m < M; ++m) acc[m] = 0;
        for (uint32_t b = lane; b < blocks; b += kWave) {
            const uint8_t* block = data + b * 34;
            const float d = half_bits_to_float(ld16(block));
            for (uint32_t i = 0; i < 32; ++i) {
                const float wv = d * float(int(int8_t(block[2 + i])));
#pragma unroll
                for (int m = 0; m < M; ++m) acc[m] = __builtin_fmaf(wv, a.x[uint64_t(m) * a.columns + b * 32 + i], acc[m]);
            }
        }
#pragma unroll
        for (int m = 0; m < M; ++m) {
            const float total = wave_sum(acc[m]);
            if (lane == 0) {
                if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
                a.y[uint64_t(m) * a.rows + row] = total;
            }
        }
    }
}

template <int M>
int launch(uint32_t layout, const Q8Args& a, hipStream_t stream) {
    const uint32_t grid = (a.rows + 3) / 4 > 4096 ? 4096 : (a.rows + 3) / 4;
    if (layout == TSP_LAYOUT_Q8_LANES_V1) {
        TSP_LAUNCH("q8_lanes", stream, q8_lanes<M><<<grid, 256, 0, stream>>>(a));
        return launch_status("q8_lanes");
    }
    const uint64_t lds_bytes = uint64_t(M) * (a.columns + 4) * 4;
    if (a.columns % 64 == 0 && reinterpret_cast<uintptr_t>(a.matrix) % 4 == 0 && lds_bytes <= 96 * 1024) {
        static std::atomic<uint64_t> raised{0};  // one per instantiation (M)
        int device = 0;
        if (lds_bytes > 48 * 1024 && setup_pending(raised, &device)) {
            TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_flat<M>), hipFuncAttributeMaxDynamicSharedMemorySize, 96 * 1024));
            setup_done(raised, device);
        }
        TSP_LAUNCH("q8_flat", stream, q8_flat<M><<<grid, 256, lds_bytes, stream>>>(a));
        return launch_status("q8_flat");
    }
    TSP_LAUNCH("q8_blocks", stream, q8_blocks<M><<<grid, 256, 0, stream>>>(a));
    return launch_status("q8_blocks");
}

// Two and more token rows against raw rows: workgroups of 16 matrix rows and 16 token rows (q8_small.hip), all in one launch, or up to sixteen at a time a persistent
// kernel (q8_resident.hip; q8_mfma.hip for up to ten token rows of more than 2048 columns). The latter starts slowly, with five to ten microseconds whatever the
// rows; the former goes up by a step for every 4096 matrix rows, with nine to sixteen token rows a larger one, as many workgroups as there are compute units. us a call,
// small and persistent:
//   up to eight token rows: on either side of three steps. Eight by 12 001 x 2048 12.8 and 13.4, 13 000 16.3 and 13.6; x 1280 10.0 and 11.7, 12.5 and 11.9; x 256 7.5 and 7.5.
//   nine to sixteen: nine by 6001 x 2048 11.9 and 10.3, 9000 17.0 and 13.3; sixteen by 7000 x 1792 11.1 and 11.4, 9000 15.8 and 13.9; 6001 x 512 7.5 and 7.6.
//   more: passes of the persistent kernel, each of which goes up with every 8192 matrix rows, against all steps together. 64 by 8100 x 1536 37.4 and 40.6, 9400 45.6 and 49.5, 11 350 54.4
//   and 50.3; 200 by 8100 113.0 and 129.8, 11 350 158.2 and 158.5, 12 650 175.5 and 159.3. At 2048 columns passes are cheaper (32 by 6150 23.4 and 22.9; 200 by 7450 131.3 and 144.8,
//   8100 142.5 and 145.1, 9400 163.5 and 174.6, 11 350 199.2 and 177.3), up to 768 dearer (64 by 11 350 x 512 30.4 and 32.8, 200 by 12 500 97.8 and 105.7, 13 950 106.7 and 105.8), above
//   2048 dearer still (64 by 9400 x 2560 66.5 and 89.9, 13 900 91.2 and 95.4, 17 850 119.8 and 114.9; 32 by 12 500 47.3 and 51.8).
//   more than 2048 columns: up to ten token rows (five where columns are no two halves) 27 and 35 at 24 576 x 2560, 37 and 36 at 32 000; more, all in
//   registers, eight by 20 000 x 2304 24.1 and 25.2, 22 000 29.2 and 26.4; sixteen by 12 000 x 2560 21.8 and 23.5, 16 000 28.2 and 24.8.
// Widths that the persistent kernels refuse all go to the former.
bool small_rows(const void* matrix, const float* x, uint64_t x_stride_bytes, uint32_t columns, uint32_t rows, uint32_t tokens) {
    if (!q8_small_takes(matrix, x, x_stride_bytes, columns, rows)) return false;
    if (x_stride_bytes != uint64_t(columns) * 4 || !q8_mfma_supported(matrix, x, columns, rows)) return true;
    if (tokens > 16) {
        const uint32_t tiles = (tokens + 15) / 16, steps = ((rows + 15) / 16 * tiles + 255) / 256, stretches = (rows + 8191) / 8192;
        const uint32_t pass = columns > 2048 ? 17 + 9 * stretches : columns == 2048 ? 14 + 5 * stretches : columns > 768 ? 12 + 8 * stretches : 11 + 10 * stretches;  // tenths of a step
        return 10 * steps <= pass * tiles;
    }
    if (columns > 2048) {
        if (tokens > (columns % 512 == 0 ? 10u : 5u)) return tokens > 8 ? rows < 13000 : rows <= 20480;
        return rows < (tokens > 8 ? 22000u : 31000u);
    }
    return tokens > 8 ? rows < 6000 : rows <= 12288;
}

}  // namespace

extern "C" int tsp_q8_matvec_many(uint32_t layout, const void* matrix, uint64_t matrix_bytes, const float* x, float* y,
                                  uint32_t columns, uint32_t rows, uint32_t width, uint32_t* error_word, void* stream) {
    TSP_REQUIRE(columns && columns <= 65536 && columns % 32 == 0 && rows && rows <= 1000000 &&
                    (width == 1 || width == 2 || width == 4 || width == 8),
                "unsupported Q8-many projection shape");
    TSP_REQUIRE(layout == TSP_LAYOUT_GGUF || layout == TSP_LAYOUT_Q8_LANES_V1, "Q8-many layout");
    TSP_REQUIRE(uint64_t(columns / 32) * rows * 34 == matrix_bytes, "Q8-many matrix byte span mismatch");
    TSP_REQUIRE(matrix && x && y && error_word, "null device pointer");
    const uint64_t x_span = uint64_t(columns) * width * 4, y_span = uint64_t(rows) * width * 4;
    TSP_REQUIRE(!ranges_overlap(y, y_span, matrix, matrix_bytes) && !ranges_overlap(y, y_span, x, x_span), "Q8-many output overlaps an input");
    const Q8Args a{static_cast<const uint8_t*>(matrix), x, y, columns, rows, error_word};
    const auto s = static_cast<hipStream_t>(stream);
    if (layout == TSP_LAYOUT_GGUF && width > 1 && small_rows(matrix, x, uint64_t(columns) * 4, columns, rows, width))
        return q8_small(matrix, x, uint64_t(columns) * 4, y, uint64_t(rows) * 4, columns, rows, width, error_word, s);
    // One row against a matrix of less than 100 MB, or of a width the persistent matrix-core kernels do not take: those start slowly, and this one by and by has too few
    // bytes on their way (46 000 x 2048, 100 MB, 27.5 us here and 25.8 there; 92 000 x 1024 25.8 and 24.3; 36 770 x 2560 26.9 and 37.7)
    if (layout == TSP_LAYOUT_GGUF && width == 1 && (matrix_bytes < 100000000 || !q8_mfma_supported(matrix, x, columns, rows))) {
        bool taken = false;
        const int rc = gemv_q8_row(matrix, x, y, columns, rows, error_word, s, &taken);
        if (taken) return rc;
    }
    if (layout == TSP_LAYOUT_GGUF && q8_mfma_supported(matrix, x, columns, rows)) return q8_mfma(matrix, x, y, columns, rows, width, error_word, s);
    if (layout == TSP_LAYOUT_Q8_LANES_V1 && q8_lanes_mfma_supported(matrix, x, columns, rows))
        return q8_lanes_mfma(matrix, x, y, columns, rows, width, error_word, s);
    switch (width) {
    case 1: return launch<1>(layout, a, s);
    case 2: return launch<2>(layout, a, s);
    case 4: return launch<4>(layout, a, s);
    default: return launch<8>(layout, a, s);
    }
}

extern "C" int tsp_dense_mm_q8(uint32_t layout, const void* matrix, uint64_t matrix_bytes, const float* input, uint64_t input_stride_bytes,
                               float* output, uint64_t output_stride_bytes, uint32_t tokens, uint32_t columns, uint32_t rows,
                               uint32_t* error_word, void* stream) {
    TSP_REQUIRE(tokens && tokens <= 65536 && input_stride_bytes % 4 == 0 && output_stride_bytes % 4 == 0 &&
                    input_stride_bytes >= uint64_t(columns) * 4 && output_stride_bytes >= uint64_t(rows) * 4,
                "dense Q8_0 GEMM row geometry mismatch");
    TSP_REQUIRE(input && output, "null device pointer");
    const uint64_t in_span = uint64_t(tokens - 1) * input_stride_bytes + uint64_t(columns) * 4;
    const uint64_t out_span = uint64_t(tokens - 1) * output_stride_bytes + uint64_t(rows) * 4;
    TSP_REQUIRE(!ranges_overlap(output, out_span, matrix, matrix_bytes) && !ranges_overlap(output, out_span, input, in_span),
                "dense Q8_0 GEMM output overlaps an input");
    // Sixteen token rows, of some q8_lanes_v1 matrices eight, go through a matrix-core kernel in one pass over the weights;
    // where none does and the rows lie back to back they go eight, four, two, one at a time (the width sequence of
    // src/q8_many.cpp:20-29), and one by one where there is padding between them.
    const bool packed = input_stride_bytes == uint64_t(columns) * 4 && output_stride_bytes == uint64_t(rows) * 4;
    const bool whole = matrix && error_word && columns && columns % 32 == 0 && rows && rows <= 1000000 && uint64_t(columns / 32) * rows * 34 == matrix_bytes;
    const bool lanes = layout == TSP_LAYOUT_Q8_LANES_V1, raw = layout == TSP_LAYOUT_GGUF;
    const bool eight = whole && packed && (raw ? q8_mfma_supported(matrix, input, columns, rows) : lanes && q8_lanes_mfma_supported(matrix, input, columns, rows));
    const bool sixteen = eight && (raw || q8_lanes_mfma_supported_16(matrix, input, columns, rows));
    for (uint32_t done = 0; done < tokens;) {
        const uint32_t left = tokens - done;
        const float* const from = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(input) + uint64_t(done) * input_stride_bytes);
        float* const to = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(output) + uint64_t(done) * output_stride_bytes);
        const auto s = static_cast<hipStream_t>(stream);
        const uint32_t most = left < 16 ? left : 16;
        if (left > 1 && whole && raw && small_rows(matrix, input, input_stride_bytes, columns, rows, left)) {
            return q8_small(matrix, from, input_stride_bytes, to, output_stride_bytes, columns, rows, left, error_word, s);  // all that is left
        }
        if (eight && left > 1) {
            const uint32_t width = sixteen ? most : left < 8 ? left : 8;
            const int rc = (lanes ? q8_lanes_mfma : q8_mfma)(matrix, from, to, columns, rows, width, error_word, s);
            if (rc != TSP_OK) return rc;
            done += width;
            continue;
        }
        uint32_t width = 1;
        if (packed) tsp_q8_many_width(tokens - done, &width);
        const int rc = tsp_q8_matvec_many(layout, matrix, matrix_bytes, from, to, columns, rows, width, error_word, stream);
        if (rc != TSP_OK) return rc;
        done += width;
    }
    return TSP_OK;
}
