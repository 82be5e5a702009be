// The router projection of a prefill chunk as one f32 GEMM: logits[token, expert] = sum_k W[expert, k] * x[token, k].
//
// Replaces the engine's `graph_moe_router_f32_batch` (kernels/moe_router_f32_batch.metal:13-50: 32x32x32 f32 tiles,
// full-precision multiply-accumulate, operands never narrowed) and its windowed sibling for up to 2048 tokens.
// Both operands stay f32 from memory to the accumulator: the products run on the f32 matrix-core instruction
// (v_mfma_f32_32x32x2_f32), which rounds once per fused multiply-add like the scalar code does.
//
// Many tokens: one workgroup of eight waves owns a 64 token x 64 expert tile. Per 64-column step both 64 x 64 operand tiles go
// global -> registers -> LDS (rows padded to 68 floats so that the 16-byte fragment reads of a wave spread over all
// banks), double buffered with one barrier per step; waves 0-3 multiply the first 32 columns of the step, waves 4-7 the
// last 32, so every SIMD holds two waves that hide each other's LDS latency. The two halves are added in a fixed order
// at the end (deterministic). Consecutive tiles of one token block go to one XCD so that its L2 serves the x rows.
#include "tsp_common.hpp"

using namespace tsp;

namespace {

constexpr uint32_t kTile = 64;                          // tokens and experts per workgroup
constexpr uint32_t kStep = 64;                          // columns per LDS stage
constexpr uint32_t kPitch = 68;                         // floats per LDS row
constexpr uint32_t kStageFloats = 2 * kTile * kPitch;   // x tile, then W tile
constexpr uint32_t kLdsBytes = 2 * kStageFloats * 4;    // 69 632

typedef float acc16 __attribute__((ext_vector_type(16)));

struct RouterArgs {
    const float* weights;
    const float* input;
    float* output;
    uint64_t input_stride, output_stride;  // floats
    uint32_t columns, experts, tokens;
    uint32_t expert_tiles, tiles, tiles_per_xcd;
    uint32_t* error_word;
};

__global__ __launch_bounds__(512) void router_f32_gemm(RouterArgs a) {
    extern __shared__ __align__(16) float lds[];
    // blockIdx % 8 names the XCD; each XCD takes a contiguous run of tiles (all expert tiles of a token block together)
    const uint32_t tile = (blockIdx.x % 8) * a.tiles_per_xcd + blockIdx.x / 8;
    if (tile >= a.tiles || blockIdx.x / 8 >= a.tiles_per_xcd) return;
    const uint32_t token0 = (tile / a.expert_tiles) * kTile, expert0 = (tile % a.expert_tiles) * kTile;
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const uint32_t half = wave / 4, wt = (wave % 4) / 2, we = wave % 2;

    // staging: thread t moves float4 number t and t + 512 of each 64 x 64 tile (row = n / 16, 16-byte column = n % 16)
    const float* xrow[2];
    const float* wrow[2];
    uint32_t slot[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const uint32_t n = tid + i * 512, row = n / 16, c4 = n % 16;
        const uint32_t token = min(token0 + row, a.tokens - 1), expert = min(expert0 + row, a.experts - 1);  // tails re-read a valid row
        xrow[i] = a.input + uint64_t(token) * a.input_stride + c4 * 4;
        wrow[i] = a.weights + uint64_t(expert) * a.columns + c4 * 4;
        slot[i] = row * kPitch + c4 * 4;
    }
    const uint32_t c4 = tid % 16;
    float4 rx[2], rw[2];
    auto fetch = [&](uint32_t step) {
        const uint32_t k = step * kStep;
        const bool inside = k + c4 * 4 < a.columns;  // columns is a multiple of 32: a last half step reads zeros
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            rx[i] = inside ? *reinterpret_cast<const float4*>(xrow[i] + k) : float4{0, 0, 0, 0};
            rw[i] = inside ? *reinterpret_cast<const float4*>(wrow[i] + k) : float4{0, 0, 0, 0};
        }
    };
    auto stash = [&](uint32_t stage) {
        float* base = lds + stage * kStageFloats;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<float4*>(base + slot[i]) = rx[i];
            *reinterpret_cast<float4*>(base + kTile * kPitch + slot[i]) = rw[i];
        }
    };

    // fragments of v_mfma_f32_32x32x2_f32: lane holds A[lane % 32][lane / 32] and B[lane / 32][lane % 32]. A 16-byte read
    // gives a lane four columns; the same four go to A and B, so the order in which columns meet does not matter.
    const uint32_t frag_x = (wt * 32 + lane % 32) * kPitch + half * 32 + (lane / 32) * 4;
    const uint32_t frag_w = kTile * kPitch + (we * 32 + lane % 32) * kPitch + half * 32 + (lane / 32) * 4;
    acc16 acc = {};
    const uint32_t steps = (a.columns + kStep - 1) / kStep;
    fetch(0);
    stash(0);
    if (steps > 1) fetch(1);
    __syncthreads();
    for (uint32_t s = 0; s < steps; ++s) {
        const float* base = lds + (s & 1) * kStageFloats;
        float4 fx[4], fw[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            fx[q] = *reinterpret_cast<const float4*>(base + frag_x + q * 8);
            fw[q] = *reinterpret_cast<const float4*>(base + frag_w + q * 8);
        }
        if (s + 1 < steps) stash((s + 1) & 1);   // the other stage: every wave left it before the last barrier
        if (s + 2 < steps) fetch(s + 2);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[q].x, fw[q].x, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[q].y, fw[q].y, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[q].z, fw[q].z, acc, 0, 0, 0);
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fx[q].w, fw[q].w, acc, 0, 0, 0);
        }
        __syncthreads();
    }
    // second column half -> LDS -> added by the wave that owns the same 32 x 32 block
    float* sums = lds + (wave % 4) * 1024;
    if (half == 1) {
#pragma unroll
        for (int v = 0; v < 16; ++v) sums[v * 64 + lane] = acc[v];
    }
    __syncthreads();
    if (half == 0) {
        uint32_t bad = 0;
        const uint32_t expert = expert0 + we * 32 + lane % 32;
#pragma unroll
        for (int v = 0; v < 16; ++v) {
            const float value = acc[v] + sums[v * 64 + lane];
            const uint32_t token = token0 + wt * 32 + (v / 4) * 8 + (lane / 32) * 4 + v % 4;  // D[i][j]: j = lane % 32
            if (token < a.tokens && expert < a.experts) {
                bad |= nonfinite(value) ? TSP_ERRBIT_NONFINITE : 0u;
                a.output[uint64_t(token) * a.output_stride + expert] = value;
            }
        }
        publish_error(bad, a.error_word);
    }
}

// Fewer tokens than fill the chip with 64 x 64 tiles (eight of them for a draft's tokens): a workgroup owns ET * 16 experts x
// TT * 16 tokens, its eight waves a slice of the columns each, and the eight partial tiles are added in LDS in wave order.
// Operands go straight from memory into the fragments of v_mfma_f32_16x16x4_f32: lane l holds four consecutive columns of
// row l % 16 of either operand, one column per instruction, so no LDS round trip stands between a wave's requests and its
// products and all a wave needs is in flight a batch of kUnits steps ahead. Bound by the latency of one trip to memory and the matrix
// rate of f32 (4 x 32 cycles per 16 columns and tile pair) at eight waves per tile. 512 experts x
// 2048 columns: 203 tokens 42.6 -> 12.8, 400 tokens 42.9 -> 17.2.
constexpr uint32_t kSlices = 8;
typedef float acc4 __attribute__((ext_vector_type(4)));

template <int ET, int TT>
__global__ __launch_bounds__(512) void router_f32_sliced(RouterArgs a) {
    __shared__ __attribute__((aligned(16))) float sums[kSlices * ET * TT * 256];
    const uint32_t token0 = (blockIdx.x / a.expert_tiles) * (TT * 16), expert0 = (blockIdx.x % a.expert_tiles) * (ET * 16);
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64;
    const uint32_t r16 = lane % 16, k4 = lane / 16;
    const float* xrow[TT];
    const float* wrow[ET];
#pragma unroll
    for (int t = 0; t < TT; ++t) xrow[t] = a.input + uint64_t(min(token0 + t * 16 + r16, a.tokens - 1)) * a.input_stride + k4 * 4;
#pragma unroll
    for (int e = 0; e < ET; ++e) wrow[e] = a.weights + uint64_t(min(expert0 + e * 16 + r16, a.experts - 1)) * a.columns + k4 * 4;
    acc4 acc[ET][TT] = {};
    // 16-column units of this wave's slice
    const uint32_t units = a.columns / 16, per_wave = (units + kSlices - 1) / kSlices;
    const uint32_t first = wave * per_wave, last = min(first + per_wave, units);
    constexpr uint32_t kUnits = 8 / (ET * TT > 2 ? 2 : 1);
    for (uint32_t u0 = first; u0 < last; u0 += kUnits) {
        acc4 fx[kUnits][TT], fw[kUnits][ET];
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            const uint32_t k = min(u0 + j, last - 1) * 16;  // past the slice: its last unit again, not multiplied
#pragma unroll
            for (int t = 0; t < TT; ++t) fx[j][t] = *reinterpret_cast<const acc4*>(xrow[t] + k);
#pragma unroll
            for (int e = 0; e < ET; ++e) fw[j][e] = *reinterpret_cast<const acc4*>(wrow[e] + k);
        }
#pragma unroll
        for (uint32_t j = 0; j < kUnits; ++j) {
            if (u0 + j >= last) break;  // uniform over the wave
#pragma unroll
            for (int c = 0; c < 4; ++c)
#pragma unroll
                for (int e = 0; e < ET; ++e)
#pragma unroll
                    for (int t = 0; t < TT; ++t) acc[e][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(fx[j][t][c], fw[j][e][c], acc[e][t], 0, 0, 0);
        }
    }
#pragma unroll
    for (int e = 0; e < ET; ++e)
#pragma unroll
        for (int t = 0; t < TT; ++t) *reinterpret_cast<acc4*>(sums + ((wave * ET + e) * TT + t) * 256 + lane * 4) = acc[e][t];
    __syncthreads();
    uint32_t bad = 0;
    for (uint32_t i = tid; i < ET * TT * 256; i += 512) {  // value i: register i % 4 of lane (i / 4) % 64 of tile i / 256
        float value = sums[i];
#pragma unroll
        for (uint32_t s = 1; s < kSlices; ++s) value += sums[s * ET * TT * 256 + i];
        const uint32_t l = i / 4 % 64, t = i / 256 % TT, e = i / 256 / TT;
        const uint32_t token = token0 + t * 16 + (l / 16) * 4 + i % 4, expert = expert0 + e * 16 + l % 16;  // D[i][j]: j = lane % 16
        if (token < a.tokens && expert < a.experts) {
            bad |= nonfinite(value) ? TSP_ERRBIT_NONFINITE : 0u;
            a.output[uint64_t(token) * a.output_stride + expert] = value;
        }
    }
    publish_error(bad, a.error_word);
}

// A draft's tokens: sixteen rows of tokens would be half empty, and 32 tiles of sixteen experts leave most of the chip idle. A workgroup
// owns two experts, its eight waves every eighth piece of 256 columns, a lane four columns of every token and both experts: at
// 2048 columns one trip to memory, all of it requested at once. Bound by that trip and the launch. 512 experts, 8 tokens: 2048 columns
// 10.1 -> 4.3 us, 2560 columns 11.8 -> 5.8 (5 tokens).
template <uint32_t TOKENS>
__global__ __launch_bounds__(512) void router_f32_pairs(RouterArgs a) {
    constexpr uint32_t E = 2, kPiece = 64, kStep = kSlices * kPiece;
    __shared__ float sums[kSlices][E * TOKENS];
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = tid / 64, expert0 = blockIdx.x * E, quads = a.columns / 4;
    const acc4* w[E];
    const acc4* x[TOKENS];
#pragma unroll
    for (uint32_t e = 0; e < E; ++e) w[e] = reinterpret_cast<const acc4*>(a.weights + uint64_t(min(expert0 + e, a.experts - 1)) * a.columns);
#pragma unroll
    for (uint32_t t = 0; t < TOKENS; ++t) x[t] = reinterpret_cast<const acc4*>(a.input + uint64_t(min(t, a.tokens - 1)) * a.input_stride);
    acc4 acc[E][TOKENS] = {};
    for (uint32_t q0 = wave * kPiece; q0 < quads; q0 += kStep) {
        const uint32_t q = min(q0 + lane, quads - 1);  // past the end: the last piece again, not multiplied
        acc4 fw[E], fx[TOKENS];
#pragma unroll
        for (uint32_t e = 0; e < E; ++e) fw[e] = w[e][q];
#pragma unroll
        for (uint32_t t = 0; t < TOKENS; ++t) fx[t] = x[t][q];
        if (q0 + lane < quads)
#pragma unroll
            for (uint32_t t = 0; t < TOKENS; ++t)
#pragma unroll
                for (uint32_t e = 0; e < E; ++e)
#pragma unroll
                    for (int c = 0; c < 4; ++c) acc[e][t][c] = __builtin_fmaf(fw[e][c], fx[t][c], acc[e][t][c]);
    }
#pragma unroll
    for (uint32_t e = 0; e < E; ++e)
#pragma unroll
        for (uint32_t t = 0; t < TOKENS; ++t) {
            const float sum = wave_sum((acc[e][t][0] + acc[e][t][1]) + (acc[e][t][2] + acc[e][t][3]));
            if (lane == 0) sums[wave][e * TOKENS + t] = sum;
        }
    __syncthreads();
    uint32_t bad = 0;
    if (tid < E * TOKENS) {
        float value = sums[0][tid];
#pragma unroll
        for (uint32_t s = 1; s < kSlices; ++s) value += sums[s][tid];
        const uint32_t token = tid % TOKENS, expert = expert0 + tid / TOKENS;
        if (token < a.tokens && expert < a.experts) {
            bad |= nonfinite(value) ? TSP_ERRBIT_NONFINITE : 0u;
            a.output[uint64_t(token) * a.output_stride + expert] = value;
        }
    }
    publish_error(bad, a.error_word);
}

template <uint32_t TOKENS>
void launch_pairs(const RouterArgs& a, hipStream_t s) {
    TSP_LAUNCH("router_f32_gemm", s, router_f32_pairs<TOKENS><<<(a.experts + 1) / 2, 512, 0, s>>>(a));
}

template <int ET, int TT>
void launch_sliced(RouterArgs a, hipStream_t s) {
    a.expert_tiles = (a.experts + ET * 16 - 1) / (ET * 16);
    const uint32_t tiles = a.expert_tiles * ((a.tokens + TT * 16 - 1) / (TT * 16));
    TSP_LAUNCH("router_f32_gemm", s, router_f32_sliced<ET, TT><<<tiles, 512, 0, s>>>(a));
}

std::atomic<uint64_t> g_lds_raised{0};

}  // namespace

extern "C" int tsp_router_f32_batch(const float* weights, const float* input, uint64_t input_stride_bytes, float* output,
                                    uint64_t output_stride_bytes, uint32_t columns, uint32_t experts, uint32_t tokens,
                                    uint32_t* error_word, void* stream) {
    TSP_REQUIRE(weights && input && output && error_word, "null device pointer");
    TSP_REQUIRE(columns && columns % 32 == 0 && columns <= 65536 && experts && experts <= 65536 && tokens && tokens <= 65536,
                "router f32 batch geometry (columns in multiples of 32)");
    TSP_REQUIRE(input_stride_bytes >= uint64_t(columns) * 4 && output_stride_bytes >= uint64_t(experts) * 4 && input_stride_bytes % 16 == 0 &&
                    output_stride_bytes % 16 == 0 && input_stride_bytes <= (1ull << 32) && output_stride_bytes <= (1ull << 32),
                "router f32 batch stride");
    TSP_REQUIRE(reinterpret_cast<uintptr_t>(weights) % 16 == 0 && reinterpret_cast<uintptr_t>(input) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(output) % 4 == 0,
                "router f32 batch alignment (16 bytes for the operands)");
    const uint64_t in_span = uint64_t(tokens - 1) * input_stride_bytes + uint64_t(columns) * 4;
    const uint64_t out_span = uint64_t(tokens - 1) * output_stride_bytes + uint64_t(experts) * 4;
    const uint64_t w_span = uint64_t(columns) * experts * 4;
    TSP_REQUIRE(!ranges_overlap(output, out_span, input, in_span) && !ranges_overlap(output, out_span, weights, w_span),
                "router f32 batch output overlaps an input");
    int device = 0;
    if (setup_pending(g_lds_raised, &device)) {
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(router_f32_gemm), hipFuncAttributeMaxDynamicSharedMemorySize, int(kLdsBytes)));
        setup_done(g_lds_raised, device);
    }
    RouterArgs a{};
    a.weights = weights; a.input = input; a.output = output;
    a.input_stride = input_stride_bytes / 4; a.output_stride = output_stride_bytes / 4;
    a.columns = columns; a.experts = experts; a.tokens = tokens;
    a.expert_tiles = (experts + kTile - 1) / kTile;
    a.tiles = a.expert_tiles * ((tokens + kTile - 1) / kTile);
    a.tiles_per_xcd = (a.tiles + 7) / 8;
    a.error_word = error_word;
    const auto s = static_cast<hipStream_t>(stream);
    // The sliced form as long as one round of its tiles (256 compute units) covers the product, on the smallest tile for which
    // that holds: 16 x 16 (9 us a round at 2048 columns), 16 experts x 32 tokens (13 us), 32 x 32 (17 us); two rounds of the
    // largest (35 us, 1024 tokens of 512 experts) still beat the 43 us that the 64 x 64 form takes up to a full round of its own.
    const auto tiles = [&](uint32_t e, uint32_t t) { return uint64_t((experts + e - 1) / e) * ((tokens + t - 1) / t); };
    // Up to eight tokens: two experts per workgroup, while the chip takes them in two rounds.
    if (tokens <= 8 && experts <= 1024) tokens <= 2 ? launch_pairs<2>(a, s) : tokens <= 4 ? launch_pairs<4>(a, s) : launch_pairs<8>(a, s);
    else if (tiles(16, 16) <= 256) launch_sliced<1, 1>(a, s);
    else if (tiles(16, 32) <= 256) launch_sliced<1, 2>(a, s);
    else if (tiles(32, 32) <= 512) launch_sliced<2, 2>(a, s);
    else TSP_LAUNCH("router_f32_gemm", s, router_f32_gemm<<<a.tiles_per_xcd * 8, 512, kLdsBytes, s>>>(a));
    return launch_status("router_f32_gemm");
}
