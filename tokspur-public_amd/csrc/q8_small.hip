// A Q8_0 matrix of a few megabytes against up to sixteen token rows (a sublayer's shared expert at draft verify, a short prompt):
// y[t, r] = sum over blocks b of d[r, b] * sum_{k in b} q[r, k] * x[t, k].
//
// The persistent kernel (q8_resident.hip) has tiles of 32 matrix rows for its workgroups, so a matrix of 640 rows is twenty of them on the
// whole chip. Here a workgroup is ONE tile of 16 matrix rows and its sixteen waves take the columns in turns of 64, so that 640 x 2560 is 640 waves that each ask for at most three pieces. A piece is read as it lies (17
// dwords of each weight row, 256 bytes of each token row, neighbouring lanes at neighbouring addresses: asking for fragments
// directly, sixteen rows by 8 bytes at a time, took 12 us where this takes 5.4) and put into fragment order through LDS that belongs
// to the wave alone, so no barrier stands between a piece's arrival and its multiplication. A token row is three bf16 pieces that are the
// float exactly (mfma_quant.hpp), each against the same quants. The waves' sums meet in LDS in wave order. Bound by latency: launch,
// one round trip to memory, the sum.
#include "q8_small.hpp"

#include "mfma_quant.hpp"

using namespace tsp;

namespace {

constexpr uint32_t kWaves = 16, kThreads = kWaves * kWave, kTile = 16, kBlocks = 2, kStep = kBlocks * 32;
constexpr uint32_t kPieceDwords = kBlocks * 34 / 4;                             // 17: odd, so sixteen rows start in different banks
constexpr uint32_t kPieceLoads = (kTile * kPieceDwords + kWave - 1) / kWave;    // 5, the last a quarter used
constexpr uint32_t kRowStride = kStep + 8;                                      // bf16 values between operand rows: 36 dwords

struct Q8SmallArgs {
    const uint8_t* matrix;
    const float* x;
    uint64_t x_stride;  // bytes
    float* y;
    uint64_t y_stride;
    uint32_t columns, rows, tokens;
    uint32_t* error_word;
};

// WIDE: nine to sixteen token rows, an operand each of their first, second and third pieces; else one operand whose rows 0..7 are the
// first pieces and 8..15 the second pieces of up to eight token rows, and one with the third pieces and eight rows of zeros.
template <bool WIDE>
__global__ __launch_bounds__(kThreads) void q8_small_kernel(Q8SmallArgs a) {
    constexpr uint32_t kTokens = WIDE ? 16 : 8, kOperandRows = 3 * kTokens + (WIDE ? 0 : 1), kTokenLoads = kTokens / 4;
    struct WaveLds {
        float back[kTokens];  // what undoes the scale of a token row's part of the piece at hand
        uint32_t weights[kPieceLoads * kWave];
        __bf16 tokens[kOperandRows * kRowStride];  // kTokens rows each of first, second and third pieces, a row of zeros
    };
    __shared__ __attribute__((aligned(16))) WaveLds lds[kWaves];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid / kWave))), n16 = lane % 16, kq = lane / 16;
    const uint32_t token0 = blockIdx.y * kTokens;  // more token rows than that: the grid's second dimension
    const uint32_t row0 = blockIdx.x * kTile, row_bytes = a.columns / 32 * 34, steps = a.columns / kStep;
    const uint8_t* const w = a.matrix + uint64_t(row0) * row_bytes;
    const uint8_t* const x = reinterpret_cast<const uint8_t*>(a.x) + token0 * a.x_stride;
    uint32_t* const weights = lds[wave].weights;
    __bf16* const tokens = lds[wave].tokens;
    float* const back = lds[wave].back;
    uint32_t bad = 0;
    if (!WIDE && lane < kStep / 4) *reinterpret_cast<uint2*>(tokens + 3 * kTokens * kRowStride + lane * 4) = uint2{0, 0};
    const uint32_t third_row = WIDE ? 32 + n16 : n16 < 8 ? 16 + n16 : 24;

    // rows past the end repeat the last one, lanes past the piece its last dword
    uint32_t w_at[kPieceLoads], x_at[kTokenLoads];
#pragma unroll
    for (uint32_t t = 0; t < kPieceLoads; ++t) {
        uint32_t id = t * kWave + lane;
        id = id < kTile * kPieceDwords ? id : kTile * kPieceDwords - 1;
        const uint32_t row = row0 + id / kPieceDwords < a.rows ? id / kPieceDwords : a.rows - 1 - row0;
        w_at[t] = row * row_bytes + id % kPieceDwords * 4;
    }
#pragma unroll
    for (uint32_t t = 0; t < kTokenLoads; ++t) {
        const uint32_t token = token0 + t * 4 + kq < a.tokens ? token0 + t * 4 + kq : a.tokens - 1;
        x_at[t] = uint32_t((token - token0) * a.x_stride) + n16 * 16;
    }
    struct Piece { uint32_t w[kPieceLoads]; f32x4 x[kTokenLoads]; };
    auto fetch = [&](uint32_t s) {
        Piece p;
#pragma unroll
        for (uint32_t t = 0; t < kTokenLoads; ++t) p.x[t] = *reinterpret_cast<const f32x4*>(x + uint64_t(s) * (kStep * 4) + x_at[t]);
#pragma unroll
        for (uint32_t t = 0; t < kPieceLoads; ++t) p.w[t] = *reinterpret_cast<const uint32_t*>(w + uint64_t(s) * (kBlocks * 34) + w_at[t]);
        return p;
    };
    f32x4 acc{};
    uint32_t s = wave < steps ? wave : steps - 1;
    Piece next = fetch(s);
    for (s = wave; s < steps; s += kWaves) {
        const Piece now = next;
        next = fetch(s + kWaves < steps ? s + kWaves : s);
#pragma unroll
        for (uint32_t t = 0; t < kTokenLoads; ++t) {
            // sixteen lanes hold a row's 64 columns
            uint32_t largest = 0;  // as bits, where infinities and NaNs come out on top
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t bits = __float_as_uint(now.x[t][e]) & 0x7fffffffu;
                largest = bits > largest ? bits : largest;
            }
            largest = row16_largest_bits(largest);
            if (largest >= 0x7f800000u) bad = TSP_ERRBIT_NONFINITE;
            const int shift = row_lift(__uint_as_float(largest));
            const float scale = power_of_two(shift);
            const Pieces p[4] = {three_pieces(now.x[t][0] * scale), three_pieces(now.x[t][1] * scale), three_pieces(now.x[t][2] * scale), three_pieces(now.x[t][3] * scale)};
            __bf16* at = tokens + (t * 4 + kq) * kRowStride + n16 * 4;
            *reinterpret_cast<uint2*>(at) = uint2{two_tops(p[0].hi, p[1].hi), two_tops(p[2].hi, p[3].hi)};
            *reinterpret_cast<uint2*>(at + kTokens * kRowStride) = uint2{two_tops(p[0].mid, p[1].mid), two_tops(p[2].mid, p[3].mid)};
            *reinterpret_cast<uint2*>(at + 2 * kTokens * kRowStride) = uint2{two_tops(p[0].lo, p[1].lo), two_tops(p[2].lo, p[3].lo)};
            back[t * 4 + kq] = power_of_two(-shift);
        }
#pragma unroll
        for (uint32_t t = 0; t < kPieceLoads; ++t) weights[t * kWave + lane] = now.w[t];
        __builtin_amdgcn_wave_barrier();
        const f32x4 undo = *reinterpret_cast<const f32x4*>(back + (4 * kq) % kTokens);  // of operand rows 4 kq .. 4 kq + 3
        const uint32_t* const mine = weights + n16 * kPieceDwords;
#pragma unroll
        for (uint32_t b = 0; b < kBlocks; ++b) {
            // block b of the piece starts at byte 34 b: its scale, then the quants, 2 bytes past a dword in the even block
            const uint32_t* const q = mine + (34 * b + 2) / 4 + kq * 2;
            uint32_t w0 = q[0], w1 = q[1];
            float d;
            if (b % 2 == 0) {
                const uint32_t w2 = q[2];
                w0 = __builtin_amdgcn_alignbyte(w1, w0, 2);
                w1 = __builtin_amdgcn_alignbyte(w2, w1, 2);
                d = half_bits_to_float(uint16_t(mine[34 * b / 4]));
            } else {
                d = half_bits_to_float(uint16_t(mine[34 * b / 4] >> 16));
            }
            const bf16x8 quants = quants8_bf16(w0, w1);
            auto operand = [&](uint32_t row) { return *reinterpret_cast<const bf16x8*>(tokens + row * kRowStride + b * 32 + kq * 8); };
            f32x4 part{};
            part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand(third_row), quants, part, 0, 0, 0);
            if constexpr (WIDE) part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand(16 + n16), quants, part, 0, 0, 0);
            part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(operand(n16), quants, part, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(d * undo[v], part[v], acc[v]);
        }
        __builtin_amdgcn_wave_barrier();
    }
    // accumulator v of lane (n, kq) is operand row 4 kq + v, matrix row n of the tile; the sums lie over the pieces of their own wave
    float* const sums = reinterpret_cast<float*>(weights);
#pragma unroll
    for (int v = 0; v < 4; ++v) sums[(4 * kq + v) * 16 + n16] = acc[v];
    __syncthreads();
    constexpr uint32_t kValues = WIDE ? 256 : 128;
    if (tid < kValues) {
        const uint32_t t = token0 + tid / 16, r = row0 + n16;
        float value = 0;
#pragma unroll
        for (uint32_t q = 0; q < kWaves; ++q) {
            const float* const other = reinterpret_cast<const float*>(lds[q].weights);
            value += WIDE ? other[tid] : other[tid] + other[tid + 128];
        }
        if (t < a.tokens && r < a.rows) {
            if (nonfinite(value)) bad = TSP_ERRBIT_NONFINITE;
            reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.y) + t * a.y_stride)[r] = value;
        }
    }
    publish_error(bad, a.error_word);
}

}  // namespace

namespace tsp {

bool q8_small_takes(const void* matrix, const float* x, uint64_t x_stride_bytes, uint32_t columns, uint32_t rows) {
    return columns % kStep == 0 && rows >= 1 && reinterpret_cast<uintptr_t>(matrix) % 4 == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && x_stride_bytes % 16 == 0 &&
           x_stride_bytes <= (1u << 26);
}

int q8_small(const void* matrix, const float* x, uint64_t x_stride_bytes, float* y, uint64_t y_stride_bytes, uint32_t columns, uint32_t rows, uint32_t tokens,
             uint32_t* error_word, hipStream_t s) {
    const Q8SmallArgs a{static_cast<const uint8_t*>(matrix), x, x_stride_bytes, y, y_stride_bytes, columns, rows, tokens, error_word};
    const dim3 grid((rows + kTile - 1) / kTile, tokens > 8 ? (tokens + 15) / 16 : 1);
    if (tokens > 8) TSP_LAUNCH("q8_small", s, q8_small_kernel<true><<<grid, kThreads, 0, s>>>(a));
    else TSP_LAUNCH("q8_small", s, q8_small_kernel<false><<<grid, kThreads, 0, s>>>(a));
    return launch_status("q8_small");
}

}  // namespace tsp
