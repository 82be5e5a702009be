// The router projection of a prefill chunk as one f32 GEMM: logits[token, expert] = sum_k W[expert, k] * x[token, k].
//
// Replaces the engine's `graph_moe_router_f32_batch` (kernels/moe_router_f32_batch.metal:13-50: 32x32x32 f32 tiles,
// full-precision multiply-accumulate, operands never narrowed) and its windowed sibling for up to 2048 tokens.
// Few tokens run on the f32 matrix instructions or the vector ALUs, with operands that stay whole floats from memory to the accumulator.
//
// Many tokens: a workgroup of eight waves owns 64 tokens x 64 experts, each wave an eighth of the columns; the partial tiles are added in
// LDS in wave order (deterministic). A float is its three bf16 pieces (mfma_quant.hpp) and a product of two floats the sum of
// eight products of pieces, all exact, in f32 accumulators: v_mfma_f32_32x32x16_bf16 does in 8 x 32 cycles what v_mfma_f32_32x32x2_f32
// does in 512. What is left out, last piece by last piece, is 2^-30 of a product and less. The matrix instruction cuts its sum off where an f32 addition
// rounds, so the products of two first pieces, sixteen bits each, have an accumulator of their own and meet the others in one rounding: a
// logit that is one product is that product rounded once, as in f32 arithmetic (one accumulator and six products: off by 2^-21). Error against 64-bit
// sums, 2-norm, 2048 x 2560 by 512 experts: 1.1e-7 (one accumulator 2.8e-7, f32 products in two column halves 6.5e-7). Bound by the matrix pipe and
// the splitting (6.5 vector instructions a float, in every tile anew) beside it. 512 experts, 2048 tokens: 2560 columns 59 us with f32 products, 40 now
// (34 with six products in one accumulator), 2048 columns 46 and 33 (28).
#include "mfma_quant.hpp"

#include <type_traits>

using namespace tsp;

namespace {

constexpr uint32_t kTile = 64;                          // tokens and experts per workgroup
constexpr uint32_t kLdsBytes = 8 * kTile * kTile * 4;    // the eight waves' partial tiles

// Operands are split 2^24 times their size: a float below 2^-109 would lose bits of its last piece, the smallest one all of it, and against a large
// operand on the other side that shows. Nothing is lost so; products come out 2^48 times theirs.
constexpr float kLift = 0x1p24f, kLower = 0x1p-48f;

// Eight floats as three fragments of bf16 pieces (mfma_quant.hpp)
__device__ __forceinline__ void pieces8(const f32x4 (&v)[2], bf16x8 (&out)[3]) {
    u32x4 hi, mid, lo;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const Pieces p = three_pieces(v[i / 2][2 * (i % 2)] * kLift), q = three_pieces(v[i / 2][2 * (i % 2) + 1] * kLift);
        hi[i] = two_tops(p.hi, q.hi); mid[i] = two_tops(p.mid, q.mid); lo[i] = two_tops(p.lo, q.lo);
    }
    out[0] = __builtin_bit_cast(bf16x8, hi); out[1] = __builtin_bit_cast(bf16x8, mid); out[2] = __builtin_bit_cast(bf16x8, lo);
}

struct RouterArgs {
    const float* weights;
    const float* input;
    float* output;
    uint64_t input_stride, output_stride;  // floats
    uint32_t columns, experts, tokens;
    uint32_t expert_tiles, tiles, tiles_per_xcd;
    uint32_t* error_word;
};

// What f32 arithmetic makes of one product of rows, for results that the pieces cannot give: those that are not finite (an operand of 2^104 or a sum
// of 2^80 is too large once lifted), and those so small that products of pieces may have vanished beside them. By a whole wave.
__device__ __noinline__ float plain_dot(const float* w, const float* x, uint32_t columns) {
    f32x4 sum{};
    for (uint32_t k = threadIdx.x % kWave * 4; k < columns; k += kWave * 4) {
        const f32x4 a = *reinterpret_cast<const f32x4*>(w + k), b = *reinterpret_cast<const f32x4*>(x + k);
#pragma unroll
        for (int c = 0; c < 4; ++c) sum[c] = __builtin_fmaf(a[c], b[c], sum[c]);
    }
    return wave_sum((sum[0] + sum[1]) + (sum[2] + sum[3]));
}

__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) void router_f32_gemm(RouterArgs a) {
    extern __shared__ __align__(16) float lds[];
    // blockIdx % 8 names the XCD; each XCD takes a contiguous run of tiles (all expert tiles of a token block together)
    const uint32_t tile = (blockIdx.x % 8) * a.tiles_per_xcd + blockIdx.x / 8;
    if (tile >= a.tiles || blockIdx.x / 8 >= a.tiles_per_xcd) return;
    const uint32_t token0 = (tile / a.expert_tiles) * kTile, expert0 = (tile % a.expert_tiles) * kTile;
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    // Requests, 32 columns of the tile's 64 + 64 rows at a time into 16 KB of LDS of the wave's own (nobody else's: no barrier):
    // instruction q takes rows 8 q .. 8 q + 7, eight neighbouring lanes one whole line, and position p of row r holds the row's 16-byte
    // chunk p ^ (r / 2) % 8, so that sixteen consecutive lanes of the reads below touch every bank once.
    const uint8_t* const x0 = reinterpret_cast<const uint8_t*>(a.input + uint64_t(token0) * a.input_stride);
    const uint8_t* const w0 = reinterpret_cast<const uint8_t*>(a.weights + uint64_t(expert0) * a.columns);
    uint32_t xat[8], wat[8];  // the launch has checked that 64 rows of either span less than 4 GiB
#pragma unroll
    for (uint32_t q = 0; q < 8; ++q) {  // tails re-read a valid row
        const uint32_t chunk = ((lane % 8) ^ (4 * (q % 2) + lane / 16)) * 16;
        xat[q] = min(q * 8 + lane / 8, a.tokens - 1 - token0) * uint32_t(a.input_stride * 4) + chunk;
        wat[q] = min(q * 8 + lane / 8, a.experts - 1 - expert0) * (a.columns * 4) + chunk;
    }
    uint8_t* const mine = reinterpret_cast<uint8_t*>(lds) + wave * 16384;
    const uint32_t mine_lds = __builtin_amdgcn_readfirstlane(lds_address(mine));
    const uint32_t n = lane % 32, khalf = lane / 32;
    f32x16 acc[2][2] = {}, small[2][2] = {};  // [expert half][token half]: the products of two first pieces, and the others
    // 32-column units of this wave's slice, two groups of sixteen columns each
    const uint32_t units = a.columns / 32, first = uint32_t(uint64_t(units) * wave / 8), last = uint32_t(uint64_t(units) * (wave + 1) / 8);
    auto request = [&](uint32_t unit) {
        unit = min(unit, last - 1);  // every request unconditional: past the end the last unit again, unused
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) load_to_lds_16(x0 + uint64_t(unit) * 128, xat[q], mine_lds + q * 1024);
#pragma unroll
        for (uint32_t q = 0; q < 8; ++q) load_to_lds_16(w0 + uint64_t(unit) * 128, wat[q], mine_lds + 8192 + q * 1024);
    };
    struct Operands { bf16x8 x[2][3], w[2][3]; };
    struct Rows { f32x4 v[4][2]; };  // x rows 0..31, 32..63, w rows 0..31, 32..63
    auto read_rows = [&](uint32_t group) {  // a lane's eight columns of a fragment: chunks 4 group + 2 khalf and the next of row n
        Rows r;
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) r.v[i][j] = *reinterpret_cast<const f32x4*>(mine + i * 4096 + n * 128 + (((4 * group + 2 * khalf + j) ^ (n / 2 % 8)) * 16));
        return r;
    };
    auto split = [&](const Rows& r, Operands& o) {
#pragma unroll
        for (int i = 0; i < 2; ++i) { pieces8(r.v[i], o.x[i]); pieces8(r.v[2 + i], o.w[i]); }
    };
    // One group: its products, and between them the next group's pieces (a 32 x 32 product leaves half of its cycles to the vector ALUs,
    // a 16 x 16 one none).
    auto group_of = [&](uint32_t unit, auto parity, const Operands& now, Operands& next) {
        constexpr uint32_t P = decltype(parity)::value;
        __builtin_amdgcn_sched_barrier(0);
        if (P == 1) wait_all_loads();  // the next unit's rows
        const Rows rows = read_rows(P ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        auto add = [&](int i, int j) {
            auto& sum = i + j ? small : acc;
#pragma unroll
            for (int e = 0; e < 2; ++e)
#pragma unroll
                for (int t = 0; t < 2; ++t) sum[e][t] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(now.x[t][i], now.w[e][j], sum[e][t], 0, 0, 0);
        };
        // the small products first; that of the two last pieces, below 2^-30 of the whole, is left out
        add(2, 1);
        __builtin_amdgcn_sched_barrier(0);
        if (P == 0) {  // the whole unit is in registers: the next one goes there
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            request(unit + 1);
            __builtin_amdgcn_sched_barrier(0);
        }
        split(rows, next);
        add(1, 2); add(2, 0); add(1, 1); add(0, 2); add(1, 0); add(0, 1); add(0, 0);
#pragma unroll
        for (int g = 0; g < 28; ++g) {
            __builtin_amdgcn_sched_group_barrier(0x2, 8, 0);  // eight vector instructions
            __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);  // and a matrix instruction in turn
        }
    };
    if (first < last) {
        Operands even, odd;
        request(first);
        wait_all_loads();
        split(read_rows(0), even);
        for (uint32_t u = first; u < last; ++u) {
            group_of(u, std::integral_constant<uint32_t, 0>{}, even, odd);
            group_of(u, std::integral_constant<uint32_t, 1>{}, odd, even);
        }
        wait_all_loads();  // requests that nobody reads: they must have landed before the stages are reused
    }
    __syncthreads();
    // the eight slices, added in wave order
    f32x4* const sums = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        f32x4 quad;
#pragma unroll
        for (int r = 0; r < 4; ++r) quad[r] = acc[i / 8][i / 4 % 2][i % 4 * 4 + r] + small[i / 8][i / 4 % 2][i % 4 * 4 + r];
        sums[(wave * 16 + i) * 64 + lane] = quad;
    }
    __syncthreads();
    uint32_t bad = 0;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const uint32_t i = tid + j * 512, l = i % 64, b = i / 64 % 4, t = i / 256 % 2, e = i / 512;  // registers 4 b .. 4 b + 3 of lane l of tile (e, t)
        f32x4 value = sums[i];
#pragma unroll
        for (int s = 1; s < 8; ++s) value += sums[s * 1024 + i];
        const uint32_t expert = expert0 + e * 32 + l % 32;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t token = token0 + t * 32 + b * 8 + (l / 32) * 4 + r;  // D[i][j]: j = lane % 32
            const bool live = token < a.tokens && expert < a.experts;
            float v = value[r] * kLower;
            for (uint64_t again = __builtin_amdgcn_ballot_w64(live && (nonfinite(v) || (v != 0.0f && fabsf(v) < 0x1p-64f))); again; again &= again - 1) {
                const uint32_t which = __builtin_ctzll(again);
                const uint32_t row = __builtin_amdgcn_readlane(expert, which), column = __builtin_amdgcn_readlane(token, which);
                const float plain = plain_dot(a.weights + uint64_t(row) * a.columns, a.input + uint64_t(column) * a.input_stride, a.columns);
                if (lane == which) v = plain;
            }
            if (live) {
                bad |= nonfinite(v) ? TSP_ERRBIT_NONFINITE : 0u;
                a.output[uint64_t(token) * a.output_stride + expert] = v;
            }
        }
    }
    publish_error(bad, a.error_word);
}

// Fewer tokens than fill the chip with 64 x 64 tiles (eight of them for a draft's tokens): a workgroup owns ET * 16 experts x
// TT * 16 tokens, its eight waves a slice of the columns each, and the eight partial tiles are added in LDS in wave order.
// Operands come in whole lines, 32 columns of the tile's rows at a time, into LDS of the wave's own (nobody else's: no barrier in the
// loop), two to four such units ahead, and are read as the fragments of v_mfma_f32_16x16x4_f32: lane l holds four consecutive
// columns of row l % 16 of either operand, one column per instruction. (Loaded from memory in that order every request touches 64
// separate pieces and keeps the address unit busy for some 70 cycles, three times as long as whole lines do, which is what bound this
// form.) Bound by the matrix rate of f32 (4 x 32 cycles per 16 columns and tile pair) and, at 32 x 32, by what the unit's lines
// take beside it. 2048 columns, 512 experts: 9 tokens 7.8 -> 5.7 us, 100 9.4 -> 6.2, 203 13.0 -> 8.8, 400 18.2 -> 14.2; 128 experts:
// 300 tokens 9.6 -> 6.1, 1400 18.9 -> 13.9.
constexpr uint32_t kSlices = 8;
typedef float acc4 __attribute__((ext_vector_type(4)));

// Units of 32 columns in flight per wave: what 144 KB of LDS hold for eight waves.
constexpr int sliced_depth(int et, int tt) { return 9 / (et + tt); }
constexpr uint32_t sliced_lds(int et, int tt) { return kSlices * sliced_depth(et, tt) * (et + tt) * 2048; }

template <int ET, int TT>
__global__ __launch_bounds__(512) void router_f32_sliced(RouterArgs a) {
    constexpr int kTiles = ET + TT, kDepth = sliced_depth(ET, TT);
    constexpr uint32_t kUnitBytes = kTiles * 2048;
    extern __shared__ __attribute__((aligned(16))) float sums[];  // [wave][unit in flight][tile][16 rows][128 bytes], then the partial tiles
    // more tokens than experts: an XCD (blockIdx % 8) takes a run of token blocks with all their experts, so that the tokens pass one
    // L2 each (1024 columns, 64 experts, 2048 tokens: 7.6 -> 5.8 us)
    const uint32_t tile = a.tokens > a.experts ? (blockIdx.x % 8) * a.tiles_per_xcd + blockIdx.x / 8 : blockIdx.x;
    if (tile >= a.tiles) return;
    const uint32_t token0 = (tile / a.expert_tiles) * (TT * 16), expert0 = (tile % a.expert_tiles) * (ET * 16);
    const uint32_t tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const uint32_t r16 = lane % 16, k4 = lane / 16;
    uint8_t* const mine = reinterpret_cast<uint8_t*>(sums) + wave * (kDepth * kUnitBytes);
    const uint32_t mine_lds = __builtin_amdgcn_readfirstlane(lds_address(mine));
    // request q takes rows 8 q .. 8 q + 7 of the tiles (tokens first), eight neighbouring lanes a whole line; position p of row r holds chunk
    // p ^ (r / 2) % 8. Tails re-read a valid row.
    const float* from[2 * kTiles];
#pragma unroll
    for (uint32_t q = 0; q < 2 * kTiles; ++q) {
        const uint32_t row = q * 8 + lane / 8, chunk = (lane % 8) ^ (4 * (q % 2) + lane / 16);
        from[q] = (q < 2 * TT ? a.input + uint64_t(min(token0 + row, a.tokens - 1)) * a.input_stride
                              : a.weights + uint64_t(min(expert0 + row - 16 * TT, a.experts - 1)) * a.columns) + chunk * 4;
    }
    acc4 acc[ET][TT] = {};
    // 32-column units of this wave's slice
    const uint32_t units = a.columns / 32, per_wave = (units + kSlices - 1) / kSlices;
    const uint32_t first = min(wave * per_wave, units), last = min(first + per_wave, units);
    auto request = [&](uint32_t unit, uint32_t slot) {  // every request unconditional: past the end the last unit again, unused
        const uint32_t column = min(unit, last - 1) * 32;
#pragma unroll
        for (uint32_t q = 0; q < 2 * kTiles; ++q) load_to_lds_16(from[q] + column, mine_lds + slot * kUnitBytes + q * 1024);
    };
    if (first < last) {
#pragma unroll
        for (uint32_t d = 0; d < kDepth; ++d) request(first + d, d);
        uint32_t slot = 0;
        for (uint32_t u = first; u < last; ++u) {
            wait_after_loads<2 * kTiles * (kDepth - 1)>();
            acc4 f[2][kTiles];
#pragma unroll
            for (uint32_t g = 0; g < 2; ++g)
#pragma unroll
                for (uint32_t i = 0; i < kTiles; ++i)
                    f[g][i] = *reinterpret_cast<const acc4*>(mine + slot * kUnitBytes + i * 2048 + r16 * 128 + (((4 * g + k4) ^ (r16 / 2)) * 16));
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the unit is in registers: another one goes there
            request(u + kDepth, slot);
            slot = slot + 1 == kDepth ? 0 : slot + 1;
#pragma unroll
            for (int g = 0; g < 2; ++g)
#pragma unroll
                for (int c = 0; c < 4; ++c)
#pragma unroll
                    for (int e = 0; e < ET; ++e)
#pragma unroll
                        for (int t = 0; t < TT; ++t) acc[e][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[g][t][c], f[g][TT + e][c], acc[e][t], 0, 0, 0);
        }
        wait_all_loads();  // requests that nobody reads: they must have landed before the stages are reused
    }
    __syncthreads();
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
    a.tiles = a.expert_tiles * ((a.tokens + TT * 16 - 1) / (TT * 16));
    a.tiles_per_xcd = (a.tiles + 7) / 8;
    TSP_LAUNCH("router_f32_gemm", s, router_f32_sliced<ET, TT><<<a.tiles_per_xcd * 8, 512, sliced_lds(ET, TT), s>>>(a));
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
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&router_f32_sliced<1, 1>), hipFuncAttributeMaxDynamicSharedMemorySize, int(sliced_lds(1, 1))));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&router_f32_sliced<1, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, int(sliced_lds(1, 2))));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&router_f32_sliced<2, 2>), hipFuncAttributeMaxDynamicSharedMemorySize, int(sliced_lds(2, 2))));
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
    // that holds: 16 x 16 (6 us a round at 2048 columns), 16 experts x 32 tokens (9 us), 32 x 32 (14 us; two rounds of it would take
    // 28 us, the 64 x 64 form takes 21 at 600 tokens of 512 experts and 28 for a full round of its own). Rows so far apart that 64 of
    // them span 4 GiB stay with the sliced form's 64-bit addresses.
    const bool near = 64 * input_stride_bytes < (1ull << 32);
    const auto tiles = [&](uint32_t e, uint32_t t) { return uint64_t((experts + e - 1) / e) * ((tokens + t - 1) / t); };
    // Up to eight tokens: two experts per workgroup, while the chip takes them in two rounds.
    if (tokens <= 8 && experts <= 1024) tokens <= 2 ? launch_pairs<2>(a, s) : tokens <= 4 ? launch_pairs<4>(a, s) : launch_pairs<8>(a, s);
    else if (tiles(16, 16) <= 256) launch_sliced<1, 1>(a, s);
    else if (tiles(16, 32) <= 256) launch_sliced<1, 2>(a, s);
    else if (tiles(32, 32) <= 256 || !near) launch_sliced<2, 2>(a, s);
    else TSP_LAUNCH("router_f32_gemm", s, router_f32_gemm<<<a.tiles_per_xcd * 8, 512, kLdsBytes, s>>>(a));
    return launch_status("router_f32_gemm");
}
