// Decode / verify GEMV over block-quantised rows: y[r] = sum_c dec(W[r,c]) * x[c], f32 decode and
// f32 accumulate. HBM-bound work: every kernel streams each weight byte exactly once with 16-byte
// coalesced loads, keeps the activation slice a lane needs in registers across rows, unpacks
// nibbles and scales in registers and finishes with DPP reductions inside the wave.
//
//  gemv_generic   wave per row, any decodable encoding and any K: the scalar control arm.
//  gemv_f32       F32 rows.
//  gemv_units     Q4_K, Q6_K and Q8_0 raw GGUF rows of any length up to 12 288 columns.
//  gemv_q4k       Q4_K rows of 2, 4, 8 or 16 super-blocks, raw GGUF rows or one planar v3 expert; a lane owns one 32-byte nibble pair
//                 (two 32-weight sub-blocks), 4 lanes per super-block. The lane's 64 activations are
//                 kept as three planes of signed bytes under a per-sub-block scale (24 bits of each
//                 value), and the nibbles multiply them four at a time with v_dot4_i32_i8: the sums
//                 of q * x are exact integers, scaled by d * sc in f32 once per sub-block.
#include "decode.hpp"
#include "gemv.hpp"

using namespace tsp;

namespace {

struct GemvArgs {
    const uint8_t* matrix;       // first row of expert 0
    const float* x;
    float* y;
    const uint32_t* ids;         // per blockIdx.y expert id, or nullptr
    uint64_t expert_stride;      // bytes between experts
    uint64_t x_stride, y_stride; // bytes between blockIdx.y slices of x / y
    uint32_t columns, rows, experts, count;
    uint32_t* error_word;
    tsp_planar_spec spec;        // planar layouts only
};

// Resolves the blockIdx.y slice: returns false (after zero-filling and flagging) for a bad expert id.
__device__ __forceinline__ bool resolve(const GemvArgs& a, const uint8_t*& w, const float*& x, float*& y) {
    const uint32_t slice = blockIdx.y;
    w = a.matrix;
    x = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.x) + slice * a.x_stride);
    y = reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.y) + slice * a.y_stride);
    if (a.ids) {
        const uint32_t e = a.ids[slice];
        if (e >= a.experts) {
            if (threadIdx.x == 0 && blockIdx.x == 0) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
            for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < a.rows; r += gridDim.x * blockDim.x) y[r] = 0;
            return false;
        }
        w += e * a.expert_stride;
    }
    return true;
}

// ------------------------------------------------------------------------------------ generic
template <uint32_t T>
__global__ __launch_bounds__(256) void gemv_generic(GemvArgs a) {
    constexpr uint32_t E = BlockGeometry<T>::elements, B = BlockGeometry<T>::bytes;
    const uint8_t* w; const float* x; float* y;
    if (!resolve(a, w, x, y)) return;
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint64_t row_bytes = uint64_t(a.columns / E) * B;
    for (uint32_t row = blockIdx.x * 4 + wave; row < a.rows; row += gridDim.x * 4) {
        const uint8_t* data = w + row * row_bytes;
        float acc = 0;
        for (uint32_t c = lane; c < a.columns; c += kWave) acc = __builtin_fmaf(decode_element<T>(data + (c / E) * B, c % E), x[c], acc);
        const float total = wave_sum(acc);
        if (lane == 0) {
            if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
            y[row] = total;
        }
    }
}

// ------------------------------------------------------------------------------------ F32

// Rows of floats (a router projection of one token, the one row of a shared expert's gate against many tokens): a wave per
// row and slice, 16-byte loads. Bound by latency at these sizes (4 MB at 512 x 2048), so everything a wave needs for 2048
// columns, eight pieces of the row and eight of the activations, is requested before the first product: the per-element
// form walked its row in 32 dependent rounds of 4-byte loads. Two waves per workgroup, so that 512 rows are 256 workgroups,
// one per compute unit. 512 x 2048: 12.6 -> 3.7 us; one row against 2048 tokens: 15.5 -> 4.0 us.
typedef float f32v4 __attribute__((ext_vector_type(4)));
__global__ __launch_bounds__(128) void gemv_f32(GemvArgs a) {
    const uint8_t* w; const float* x; float* y;
    if (!resolve(a, w, x, y)) return;
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    for (uint32_t row = blockIdx.x * 2 + wave; row < a.rows; row += gridDim.x * 2) {
        const f32v4* data = reinterpret_cast<const f32v4*>(w + uint64_t(row) * a.columns * 4);
        const f32v4* xs = reinterpret_cast<const f32v4*>(x);
        const uint32_t quads = a.columns / 4;
        f32v4 acc{};
        for (uint32_t q0 = lane; q0 < quads; q0 += 8 * kWave) {
            f32v4 wv[8], xv[8];
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j) {
                const uint32_t q = q0 + j * kWave;  // past the end: the last piece again, without a branch, against zeros
                wv[j] = data[q < quads ? q : quads - 1];
                xv[j] = xs[q < quads ? q : quads - 1];
            }
#pragma unroll
            for (uint32_t j = 0; j < 8; ++j)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(wv[j][e], q0 + j * kWave < quads ? xv[j][e] : 0.0f, acc[e]);
        }
        const float total = wave_sum((acc[0] + acc[1]) + (acc[2] + acc[3]));
        if (lane == 0) {
            if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
            y[row] = total;
        }
    }
}

// ------------------------------------------------------------------------------------ Q4_K

// Sum over aligned groups of N lanes (N = 8, 16, 32, 64); every lane of a group gets the sum.
template <int N>
__device__ __forceinline__ float group_sum(float v) {
    v = dpp_add<0xB1>(v);
    v = dpp_add<0x4E>(v);
    v = dpp_add<0x141>(v);
    if constexpr (N >= 16) v = dpp_add<0x140>(v);
    if constexpr (N >= 32) v += __shfl_xor(v, 16, kWave);
    if constexpr (N >= 64) v += __shfl_xor(v, 32, kWave);
    return v;
}

// One quad of activations as integers, and its share of the sub-block's record in LDS. Per sub-block of 32 one scale brings the
// largest magnitude to 8 290 000 (just under 127 * 2^16 + 2^15, the most that three signed bytes hold); every value is rounded
// to the nearest integer of that grid (2^-24 of the sub-block's largest value: the precision of the f32 operand itself for the
// values that matter) and written as three signed base-256 digits, x = (a 2^16 + b 2^8 + c) / scale with a, b, c in [-128, 127].
// Four activations' digits share a dword, in the order of the four bytes of a word of codes, so that v_dot4_i32_i8
// multiplies four weights per instruction and plane. The integer sums are exact; the three of a sub-block recombine in f32.
// The eight threads of a sub-block are neighbours and agree on its scale with three cross-lane steps.
// A record: three planes of eight dwords (c, b, a), then 1 / scale, the sum, a flag for values that are not finite and a second factor.
// Below 2^-60 a sub-block is first brought up by 2^90 (that is the second factor, 2^-90; else it is 1): the scale itself
// would leave the range of a float from 2.4e-32 down and its inverse would be subnormal from 1e-31 down.
template <uint32_t WORDS>
__device__ __forceinline__ void stage_quad(const float4& x4, bool mine, uint32_t quad, uint32_t* planes) {
    const float v4[4] = {mine ? x4.x : 0.0f, mine ? x4.y : 0.0f, mine ? x4.z : 0.0f, mine ? x4.w : 0.0f};
    float biggest = fmaxf(fmaxf(fabsf(v4[0]), fabsf(v4[1])), fmaxf(fabsf(v4[2]), fabsf(v4[3])));
    float sum = (v4[0] + v4[1]) + (v4[2] + v4[3]);
    uint32_t flag = (nonfinite(v4[0]) || nonfinite(v4[1]) || nonfinite(v4[2]) || nonfinite(v4[3])) ? 1u : 0u;
    biggest = dpp_max<0xB1>(biggest); biggest = dpp_max<0x4E>(biggest); biggest = dpp_max<0x141>(biggest);
    sum = octet_sum(sum);
    flag |= uint32_t(__builtin_amdgcn_update_dpp(0, int(flag), 0xB1, 0xf, 0xf, true));
    flag |= uint32_t(__builtin_amdgcn_update_dpp(0, int(flag), 0x4E, 0xf, 0xf, true));
    flag |= uint32_t(__builtin_amdgcn_update_dpp(0, int(flag), 0x141, 0xf, 0xf, true));
    // a sub-block of zeros or with something not finite in it keeps scale 1 (its integers are zeros)
    const bool usable = biggest > 0 && flag == 0, small = biggest < 0x1p-60f;
    const float lift = small ? 0x1p90f : 1.0f, lifted = biggest * lift;
    const float scale = usable ? 8290000.0f / lifted : 1.0f;
    uint32_t w2 = 0, w1 = 0, w0 = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        const int xi = usable ? __float2int_rn((v4[e] * lift) * scale) : 0;
        const int c = ((xi + 128) & 255) - 128, upper = (xi - c) >> 8;
        const int b = ((upper + 128) & 255) - 128, a8 = (upper - b) >> 8;
        w2 |= uint32_t(a8 & 0xff) << (8 * e);
        w1 |= uint32_t(b & 0xff) << (8 * e);
        w0 |= uint32_t(c & 0xff) << (8 * e);
    }
    uint32_t* sub = planes + (quad / 8) * WORDS;
    if (mine) {
        sub[16 + quad % 8] = w2; sub[8 + quad % 8] = w1; sub[quad % 8] = w0;
        if (quad % 8 == 0) {
            sub[24] = __float_as_uint(usable ? lifted / 8290000.0f : 1.0f);
            sub[25] = __float_as_uint(sum);
            sub[26] = flag;
            sub[27] = __float_as_uint(small ? 0x1p-90f : 1.0f);
        }
    }
}

// BPR = super-blocks per row (K / 256), one of 2, 4, 8, 16. A wave covers 16 super-blocks per step
// (16 / BPR rows); lane = (block-in-step, pair) owns 64 weights and keeps their 64 activations in
// registers for every row it visits.
template <int BPR, bool PLANAR>
__global__ __launch_bounds__(256) void gemv_q4k(GemvArgs a) {
    constexpr int LPR = 4 * BPR;        // lanes per row
    constexpr int RPS = kWave / LPR;    // rows per wave step
    // per sub-block of 32 activations: three planes of eight dwords (four signed bytes each), then 1 / scale, the sum, a flag, the second factor
    constexpr uint32_t kSubWords = 3 * 8 + 4;
    __shared__ __attribute__((aligned(16))) uint32_t planes[BPR * 8 * kSubWords];
    const uint8_t* w; const float* x; float* y;
    if (!resolve(a, w, x, y)) return;
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t pair = lane % 4, blk_in_row = (lane / 4) % BPR, row_in_step = lane / LPR;
    const uint32_t steps = (a.rows + RPS - 1) / RPS;
    const uint32_t waves = gridDim.x * (blockDim.x / kWave);

    // The bytes of one step as they come from memory: nothing is computed on them until they are needed, so that a step's
    // requests can be in flight while something else happens (the activations being staged, the step before being summed).
    struct Raw { uint4 q0, q1, hdr; uint32_t sc, mn, dm; };
    auto fetch = [&](uint32_t step) {
        const uint32_t row = step * RPS + row_in_step;
        const uint64_t blk = uint64_t(row < a.rows ? row : a.rows - 1) * BPR + blk_in_row;
        Raw r{};
        if constexpr (PLANAR) {
            const uint8_t* qs = w + a.spec.qs_offset + blk * 128 + pair * 32;
            r.q0 = *reinterpret_cast<const uint4*>(qs);
            r.q1 = *reinterpret_cast<const uint4*>(qs + 16);
            const uint8_t* sm = w + a.spec.sm_offset + blk * 16 + pair * 2;
            r.sc = *reinterpret_cast<const uint16_t*>(sm);
            r.mn = *reinterpret_cast<const uint16_t*>(sm + 8);
            r.dm = *reinterpret_cast<const uint32_t*>(w + a.spec.dm_offset + blk * 4);
        } else {
            const uint8_t* block = w + blk * 144;
            r.hdr = *reinterpret_cast<const uint4*>(block);
            r.q0 = *reinterpret_cast<const uint4*>(block + 16 + pair * 32);
            r.q1 = *reinterpret_cast<const uint4*>(block + 32 + pair * 32);
        }
        return r;
    };

    // The activations are asked for first (a few cached kilobytes: they come back first), the wave's first weight bytes right
    // behind them; the activations are staged and summed while the weights travel.
    constexpr uint32_t kQuads = BPR * 64;                // float4 in a row of activations
    constexpr uint32_t kMine = (kQuads + 255) / 256;     // per thread: 1 (K = 512, half the threads) .. 16 (K = 4096)
    float4 xv[kMine];
    const bool x_quads = reinterpret_cast<uintptr_t>(x) % 16 == 0;  // else a row that only floats align
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t quad = threadIdx.x + j * 256;
        if (kQuads % 256 == 0 || quad < kQuads) {
            if (x_quads) xv[j] = reinterpret_cast<const float4*>(x)[quad];
            else xv[j] = make_float4(x[4 * quad], x[4 * quad + 1], x[4 * quad + 2], x[4 * quad + 3]);
        }
    }
    uint32_t step = blockIdx.x * (blockDim.x / kWave) + wave;
    Raw cur = fetch(step < steps ? step : 0);
    // the activations become integers, once per workgroup
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t quad = threadIdx.x + j * 256;
        stage_quad<kSubWords>(xv[j], kQuads % 256 == 0 || quad < kQuads, quad, planes);  // uniform over every group of eight lanes
    }
    __syncthreads();

    uint32_t pa[3][8], pb[3][8];
    float sxa, sxb, inv_a, inv_b, back_a, back_b;
    bool x_bad;
    {
        const uint32_t* sa = planes + (blk_in_row * 8 + pair * 2) * kSubWords;
        const uint32_t* sb = sa + kSubWords;
#pragma unroll
        for (int p = 0; p < 3; ++p)
#pragma unroll
            for (int k = 0; k < 8; ++k) { pa[p][k] = sa[p * 8 + k]; pb[p][k] = sb[p * 8 + k]; }
        inv_a = __uint_as_float(sa[24]); sxa = __uint_as_float(sa[25]);
        inv_b = __uint_as_float(sb[24]); sxb = __uint_as_float(sb[25]);
        x_bad = (sa[26] | sb[26]) != 0;
        back_a = __uint_as_float(sa[27]); back_b = __uint_as_float(sb[27]);
    }

    for (; step < steps; step += waves) {
        const uint32_t row = step * RPS + row_in_step;
        const bool live = row < a.rows;
        const Raw now = cur;
        cur = fetch(step + waves < steps ? step + waves : step);  // the next step's bytes travel while this one is summed
        float d, dmin;
        uint32_t sc_a, sc_b, mn_a, mn_b;
        if constexpr (PLANAR) {
            sc_a = now.sc & 0xffu; sc_b = now.sc >> 8; mn_a = now.mn & 0xffu; mn_b = now.mn >> 8;
            d = half_bits_to_float(now.dm & 0xffffu); dmin = half_bits_to_float(now.dm >> 16);
        } else {
            const uint4 hdr = now.hdr;
            d = half_bits_to_float(hdr.x & 0xffffu); dmin = half_bits_to_float(hdr.x >> 16);
            // sub-blocks 2*pair and 2*pair+1: byte j = (2*pair) & 3 (and j+1) of the three header words
            const uint32_t sh = (pair & 1u) * 16u;
            const uint32_t s2 = (hdr.y >> sh) & 0xffffu, m2 = (hdr.z >> sh) & 0xffffu, e2 = (hdr.w >> sh) & 0xffffu;
            if (pair < 2) {
                sc_a = s2 & 63u; sc_b = (s2 >> 8) & 63u; mn_a = m2 & 63u; mn_b = (m2 >> 8) & 63u;
            } else {
                sc_a = (e2 & 15u) | (((s2 >> 6) & 3u) << 4);
                sc_b = ((e2 >> 8) & 15u) | (((s2 >> 14) & 3u) << 4);
                mn_a = ((e2 >> 4) & 15u) | (((m2 >> 6) & 3u) << 4);
                mn_b = ((e2 >> 12) & 15u) | (((m2 >> 14) & 3u) << 4);
            }
        }
        const uint32_t words[8] = {now.q0.x, now.q0.y, now.q0.z, now.q0.w, now.q1.x, now.q1.y, now.q1.z, now.q1.w};
        int a2 = 0, a1 = 0, a0 = 0, b2 = 0, b1 = 0, b0 = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int lo = int(words[k] & 0x0f0f0f0fu), hi = int((words[k] >> 4) & 0x0f0f0f0fu);
            a2 = __builtin_amdgcn_sdot4(lo, int(pa[2][k]), a2, false);
            a1 = __builtin_amdgcn_sdot4(lo, int(pa[1][k]), a1, false);
            a0 = __builtin_amdgcn_sdot4(lo, int(pa[0][k]), a0, false);
            b2 = __builtin_amdgcn_sdot4(hi, int(pb[2][k]), b2, false);
            b1 = __builtin_amdgcn_sdot4(hi, int(pb[1][k]), b1, false);
            b0 = __builtin_amdgcn_sdot4(hi, int(pb[0][k]), b0, false);
        }
        // each plane's sum is below 2^16 and exact as a float; the three recombine with two roundings to f32
        const float dot_a = __builtin_fmaf(float(a2), 65536.0f, __builtin_fmaf(float(a1), 256.0f, float(a0))) * inv_a * back_a;
        const float dot_b = __builtin_fmaf(float(b2), 65536.0f, __builtin_fmaf(float(b1), 256.0f, float(b0))) * inv_b * back_b;
        // sum_c ((d*sc)*q - dmin*mn) * x = (d*sc) * sum q x - (dmin*mn) * sum x, per sub-block
        float part = (d * float(sc_a)) * dot_a - (dmin * float(mn_a)) * sxa;
        part += (d * float(sc_b)) * dot_b - (dmin * float(mn_b)) * sxb;
        if (x_bad) part = __uint_as_float(0x7fc00000u);  // a non-finite activation: the row's sum is not a number, and the batch is refused
        const float total = group_sum<LPR>(part);
        if (live && lane % LPR == 0) {
            if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
            y[row] = total;
        }
    }
}

// ------------------------------------------------------------------------------------ Q4_K, Q6_K, Q8_0 rows of any length
// Rows of any number of super-blocks, and the other two encodings a decode step meets, in the arithmetic of the per-element kernel:
// every weight is decoded to the float it stands for (one rounding, where the format needs one) and meets its activation as a float in a
// fused multiply-add, so one large activation takes no bits from its neighbours. L lanes share a row; a lane takes every L-th unit
// of it (64 weights of a K-quant block, one Q8_0 block). A unit's activations lie together in LDS, in the order its codes
// unpack, four floats of padding behind each unit so that neighbouring lanes' reads of 16 bytes fall in different banks.
// Bound by memory for large matrices (about three and a half instructions per weight take half the time of its bytes), by one round
// trip for small ones: the next unit's bytes are requested before the current one is multiplied. Blocks of 34 and 210 bytes are
// even-aligned only; neighbouring lanes read neighbouring pieces, so the lines are shared all the same. The per-element kernel takes
// 9.8 us at Q6_K 2731 x 2560, this one 4.9; 40 000 x 6144 (202 MB) 48 us = 4.2 TB/s; Q8_0 16 000 x 2560 21 us there, 11 here.
// (Activations as 24-bit integers under one scale per 32, as gemv_q4k has them: 5.8, 46 and 11 us.)
typedef uint32_t piece16 __attribute__((ext_vector_type(4), aligned(2)));
typedef uint32_t piece8 __attribute__((ext_vector_type(2), aligned(2)));
typedef uint32_t quad_words __attribute__((ext_vector_type(4)));

template <uint32_t T> struct UnitBytes;
template <> struct UnitBytes<12> { quad_words hdr, q0, q1; };
template <> struct UnitBytes<14> { piece16 la, lb, qh; piece8 sc; uint16_t d; };
template <> struct UnitBytes<8> { piece16 q0, q1; uint16_t d; };

// Floats of a unit of 64 (32) activations in LDS, padding included, and of a row.
__host__ __device__ constexpr uint32_t unit_floats(uint32_t type) { return type == 8 ? 36u : 68u; }
__host__ __device__ constexpr uint32_t units_lds_bytes(uint32_t type, uint32_t columns) { return columns / (type == 8 ? 32 : 64) * unit_floats(type) * 4; }

__device__ __forceinline__ float code_of(uint32_t word, int i) { return float((word >> (8 * i)) & 0xffu); }

template <uint32_t T, int L>
__global__ __launch_bounds__(256) void gemv_units(GemvArgs a) {
    constexpr uint32_t kUnit = T == 8 ? 32 : 64, kFloats = unit_floats(T), RPS = kWave / L;
    extern __shared__ __attribute__((aligned(16))) float staged[];
    const uint8_t* w; const float* x; float* y;
    if (!resolve(a, w, x, y)) return;
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave, in_row = lane % L, row_in_step = lane / L;
    const uint32_t units = a.columns / kUnit, rounds = (units + L - 1) / L;
    const uint32_t steps = (a.rows + RPS - 1) / RPS, waves = gridDim.x * (blockDim.x / kWave);
    const uint64_t row_bytes = uint64_t(a.columns / BlockGeometry<T>::elements) * BlockGeometry<T>::bytes;

    auto fetch = [&](uint32_t step, uint32_t round) {
        const uint32_t row = step * RPS + row_in_step, u0 = round * L + in_row, u = u0 < units ? u0 : units - 1;
        const uint8_t* from = w + (row < a.rows ? row : a.rows - 1) * row_bytes;
        UnitBytes<T> r;
        if constexpr (T == 12) {
            const uint8_t* block = from + u / 4 * 144;
            r.hdr = *reinterpret_cast<const quad_words*>(block);
            r.q0 = *reinterpret_cast<const quad_words*>(block + 16 + u % 4 * 32);
            r.q1 = *reinterpret_cast<const quad_words*>(block + 32 + u % 4 * 32);
        } else if constexpr (T == 14) {  // section u / 2 % 2, the 16-byte half u % 2 of each of its pieces
            const uint8_t* block = from + u / 4 * 210;
            const uint32_t sec = u / 2 % 2, half = u % 2;
            r.la = *reinterpret_cast<const piece16*>(block + sec * 64 + half * 16);
            r.lb = *reinterpret_cast<const piece16*>(block + sec * 64 + 32 + half * 16);
            r.qh = *reinterpret_cast<const piece16*>(block + 128 + sec * 32 + half * 16);
            r.sc = *reinterpret_cast<const piece8*>(block + 192 + sec * 8);
            r.d = *reinterpret_cast<const uint16_t*>(block + 208);
        } else {
            const uint8_t* block = from + u * 34;
            r.d = *reinterpret_cast<const uint16_t*>(block);
            r.q0 = *reinterpret_cast<const piece16*>(block + 2);
            r.q1 = *reinterpret_cast<const piece16*>(block + 18);
        }
        return r;
    };

    // the activations first, the wave's first weight bytes right behind them; the activations are staged while the weights travel
    const uint32_t quads = a.columns / 4;
    auto load_quad = [&](uint32_t quad) {
        return quad < quads ? *reinterpret_cast<const float4*>(x + 4 * quad) : make_float4(0, 0, 0, 0);
    };
    float4 x0 = load_quad(threadIdx.x);
    uint32_t step = blockIdx.x * (blockDim.x / kWave) + wave;
    UnitBytes<T> cur = fetch(step < steps ? step : 0, 0);
    for (uint32_t quad = threadIdx.x; quad < quads; quad += 256) {
        const float4 here = x0;
        x0 = load_quad(quad + 256);
        uint32_t at;
        if constexpr (T == 14) at = (quad / 64 * 4 + quad / 32 % 2 * 2 + quad / 4 % 2) * kFloats + quad / 8 % 4 * 16 + quad % 4 * 4;  // section, half | quarter
        else at = quad / (kUnit / 4) * kFloats + quad % (kUnit / 4) * 4;
        *reinterpret_cast<float4*>(staged + at) = here;
    }
    __syncthreads();

    float part = 0;
    for (uint32_t round = 0; step < steps;) {
        const UnitBytes<T> now = cur;
        const uint32_t u0 = round * L + in_row, u = u0 < units ? u0 : units - 1;
        const bool last = round + 1 == rounds;
        const uint32_t next_step = last ? (step + waves < steps ? step + waves : step) : step;
        cur = fetch(next_step, last ? 0 : round + 1);  // the next unit's bytes travel while this one is summed
        const float* const xs = staged + u * kFloats;
        float sum[4] = {0, 0, 0, 0};  // four chains
        // four weights, scale * code + offset each, against the unit's activations 4 i .. 4 i + 3
        auto four = [&](int i, uint32_t codes, float scale, float offset) {
            const float4 x4 = *reinterpret_cast<const float4*>(xs + 4 * i);
            sum[0] = __builtin_fmaf(__builtin_fmaf(code_of(codes, 0), scale, offset), x4.x, sum[0]);
            sum[1] = __builtin_fmaf(__builtin_fmaf(code_of(codes, 1), scale, offset), x4.y, sum[1]);
            sum[2] = __builtin_fmaf(__builtin_fmaf(code_of(codes, 2), scale, offset), x4.z, sum[2]);
            sum[3] = __builtin_fmaf(__builtin_fmaf(code_of(codes, 3), scale, offset), x4.w, sum[3]);
        };
        if constexpr (T == 12) {
            const uint32_t pair = u % 4;
            const float d = half_bits_to_float(now.hdr[0] & 0xffffu), dmin = half_bits_to_float(now.hdr[0] >> 16);
            // sub-blocks 2 pair and 2 pair + 1: two neighbouring bytes of the unpacked scales and minima (mfma_quant.hpp: decode_hdr)
            const uint32_t sh = (pair & 1u) * 16u;
            const uint32_t s2 = (now.hdr[1] >> sh) & 0xffffu, m2 = (now.hdr[2] >> sh) & 0xffffu, e2 = (now.hdr[3] >> sh) & 0xffffu;
            const uint32_t sc = pair < 2 ? s2 & 0x3f3fu : (e2 & 0x0f0fu) | ((s2 >> 2) & 0x3030u);
            const uint32_t mn = pair < 2 ? m2 & 0x3f3fu : ((e2 >> 4) & 0x0f0fu) | ((m2 >> 2) & 0x3030u);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                // both products are exact (11 + 6 bits), so is scale * code: the weight is rounded once, as the decoder rounds it
                const float scale = d * code_of(sc, h), offset = -(dmin * code_of(mn, h));
#pragma unroll
                for (int i = 0; i < 8; ++i) four(8 * h + i, ((i < 4 ? now.q0[i % 4] : now.q1[i % 4]) >> (4 * h)) & 0x0f0f0f0fu, scale, offset);
            }
        } else if constexpr (T == 14) {
            const uint32_t half = u % 2;
            const float d = half_bits_to_float(now.d);
#pragma unroll
            for (int q = 0; q < 4; ++q) {  // 16 weights of one sub-scale
                const uint32_t at = 2 * q + half;  // the sub-scale's byte
                const float scale = d * float(int(int8_t((now.sc[at / 4] >> (at % 4 * 8)) & 0xffu)));  // exact; scale * (code - 32) is rounded once
                const float offset = -32.0f * scale;
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    const uint32_t low = q % 2 ? now.lb[i] : now.la[i], high = now.qh[i] >> (2 * q);
                    four(4 * q + i, ((q < 2 ? low : low >> 4) & 0x0f0f0f0fu) | ((high & 0x03030303u) << 4), scale, offset);
                }
            }
        } else {
            const float d = half_bits_to_float(now.d), offset = -128.0f * d;  // a quant is its code less 128, both products exact
#pragma unroll
            for (int i = 0; i < 8; ++i) four(i, (i < 4 ? now.q0[i % 4] : now.q1[i % 4]) ^ 0x80808080u, d, offset);
        }
        part += u0 < units ? (sum[0] + sum[1]) + (sum[2] + sum[3]) : 0.0f;
        if (!last) { ++round; continue; }
        const uint32_t row = step * RPS + row_in_step;
        const float total = group_sum<L>(part);
        if (row < a.rows && in_row == 0) {
            if (nonfinite(total)) atomicOr(a.error_word, TSP_ERRBIT_NONFINITE);
            y[row] = total;
        }
        part = 0;
        round = 0;
        step += waves;
    }
}

// ------------------------------------------------------------------------------------ launch
uint32_t grid_rows(uint32_t work_items, uint32_t per_block) {
    const uint32_t blocks = (work_items + per_block - 1) / per_block;
    return blocks < 1 ? 1 : blocks > 2048 ? 2048 : blocks;
}

// Rows whose activations fit LDS three times (12 288 columns: 52 KB, three workgroups per compute unit), activations in 16-byte pieces, blocks as aligned as their encoding has them.
bool gemv_units_takes(uint32_t encoding, const GemvArgs& a) {
    if (encoding != 8 && encoding != 12 && encoding != 14) return false;
    const uintptr_t step = encoding == 12 ? 16 : 2;
    return a.columns <= 12288 && reinterpret_cast<uintptr_t>(a.matrix) % step == 0 && a.expert_stride % step == 0 &&
           reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && a.x_stride % 16 == 0;
}

template <uint32_t T, int L>
int launch_units_lanes(const GemvArgs& a, hipStream_t stream) {
    const uint32_t bytes = units_lds_bytes(T, a.columns);
    static std::atomic<uint64_t> raised{0};
    int device = 0;
    if (bytes > 48 * 1024 && setup_pending(raised, &device)) {
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&gemv_units<T, L>), hipFuncAttributeMaxDynamicSharedMemorySize, int(units_lds_bytes(T, 12288))));
        setup_done(raised, device);
    }
    uint32_t blocks = grid_rows((a.rows + kWave / L - 1) / (kWave / L), 4);
    const uint32_t most = a.count == 1 ? 1024u : 2048u;
    if (blocks > most) blocks = most;
    TSP_LAUNCH("gemv_units", stream, gemv_units<T, L><<<dim3(blocks, a.count), 256, bytes, stream>>>(a));
    return launch_status("gemv_units");
}

template <uint32_t T>
int launch_units(const GemvArgs& a, hipStream_t stream) {
    // Lanes per row: the count that leaves the fewest lanes without a unit in a row's last round (Q6_K 16 000 x 2560, 40 units: 8
    // lanes 8.8 us, 64 lanes 10.9), sixteen where several leave equally few; more where that would leave the chip with fewer than 512
    // waves (at 512 x 2560: 64 lanes 4.7 us, 8 lanes 6.4).
    const uint32_t units = a.columns / (T == 8 ? 32 : 64);
    uint32_t lanes = 16;
    auto idle = [&](uint32_t l) { return (units + l - 1) / l * l; };
    for (const uint32_t l : {32u, 8u, 64u}) if (idle(l) < idle(lanes)) lanes = l;
    while (lanes < 64 && uint64_t(a.rows) * a.count * lanes / 64 < 512) lanes *= 2;
    switch (lanes) {
    case 8: return launch_units_lanes<T, 8>(a, stream);
    case 16: return launch_units_lanes<T, 16>(a, stream);
    case 32: return launch_units_lanes<T, 32>(a, stream);
    default: return launch_units_lanes<T, 64>(a, stream);
    }
}

int launch_gemv(uint32_t encoding, uint32_t layout, GemvArgs a, hipStream_t stream) {
    const bool aligned = reinterpret_cast<uintptr_t>(a.matrix) % 16 == 0 && a.expert_stride % 16 == 0;
    if (encoding == 12 && aligned && (layout == TSP_LAYOUT_GGUF || layout == TSP_LAYOUT_PLANAR_V3)) {
        const uint32_t bpr = a.columns / 256;
        const bool planar = layout == TSP_LAYOUT_PLANAR_V3;
#define TSP_Q4K_CASE(N)                                                                                                   \
    if (bpr == N) {                                                                                                       \
        /* at most 1024 workgroups, four per compute unit of a 256-unit GPU: sixteen waves per unit with a step in flight each */ \
        /* keep memory as busy as thirty-two do, and a workgroup's set-up (the activations' digit planes) serves more steps */    \
        /* (measured at 65 536 and 262 144 rows of 2048 columns: 15.2 and 59.4 us against 16.3 and 60.0; two steps in flight */   \
        /* per wave: no faster) */                                                                                              \
        uint32_t blocks = grid_rows((a.rows + 64 / (4 * N) - 1) / (64 / (4 * N)), 4);                                     \
        if (a.count == 1 && blocks > 1024) blocks = 1024;                                                                 \
        const dim3 grid(blocks, a.count);                                                                                 \
        if (planar) TSP_LAUNCH("gemv_q4k", stream, gemv_q4k<N, true><<<grid, 256, 0, stream>>>(a));                                                       \
        else TSP_LAUNCH("gemv_q4k", stream, gemv_q4k<N, false><<<grid, 256, 0, stream>>>(a));                                                             \
        return launch_status("gemv_q4k");                                                                                 \
    }
        TSP_Q4K_CASE(2) TSP_Q4K_CASE(4) TSP_Q4K_CASE(8) TSP_Q4K_CASE(16)
#undef TSP_Q4K_CASE
    }
    TSP_REQUIRE(layout == TSP_LAYOUT_GGUF, "no GEMV kernel for this layout/encoding/shape");
    if (gemv_units_takes(encoding, a)) {
        if (encoding == 12) return launch_units<12>(a, stream);
        return encoding == 14 ? launch_units<14>(a, stream) : launch_units<8>(a, stream);
    }
    // 16-byte pieces of every row of either operand, for the routers' sizes (512 x 2560: 5 MB). Above 16 MB the per-element kernel stays,
    // although pieces are faster there as well (4096 x 2048, 32 MB: 7 us against 16): an operator's boundaries in a profile scatter by up
    // to 10 us, and a 32 MB product is what the profile's test orders against an activation. No matrix of a sublayer is that large.
    if (encoding == 0 && uint64_t(a.columns) * a.rows <= (4u << 20) && aligned && a.columns % 4 == 0 && reinterpret_cast<uintptr_t>(a.x) % 16 == 0 && a.x_stride % 16 == 0) {
        const dim3 grid(grid_rows(a.rows, 2), a.count);
        TSP_LAUNCH("gemv_f32", stream, gemv_f32<<<grid, 128, 0, stream>>>(a));
        return launch_status("gemv_f32");
    }
    const dim3 grid(grid_rows(a.rows, 4), a.count);
    const bool ok = dispatch_encoding(encoding, [&]<uint32_t T>() { TSP_LAUNCH("gemv_generic", stream, gemv_generic<T><<<grid, 256, 0, stream>>>(a)); });
    TSP_REQUIRE(ok, "no owned numerical decoder for this encoding");
    return launch_status("gemv_generic");
}

int check_shape(uint32_t encoding, uint32_t layout, uint64_t matrix_bytes, uint32_t columns, uint32_t rows, uint32_t experts,
                tsp_planar_spec* spec, uint64_t* expert_stride) {
    TSP_REQUIRE(tsp_can_decode(encoding) && columns && columns <= 65536 && rows && rows <= 1000000, "unsupported graph GEMV shape/type");
    const auto* enc = find_encoding(encoding);
    TSP_REQUIRE(columns % enc->elements == 0, "GEMV row is not block-aligned");
    std::memset(spec, 0, sizeof *spec);
    if (layout == TSP_LAYOUT_PLANAR_V3) {
        const int rc = tsp_make_expert_spec(encoding, columns, rows, spec);
        if (rc != TSP_OK) return rc;
        *expert_stride = spec->planar_expert_bytes;
    } else {
        TSP_REQUIRE(layout == TSP_LAYOUT_GGUF || (layout == TSP_LAYOUT_Q8_LANES_V1 && encoding == 8), "layout/encoding mismatch");
        *expert_stride = uint64_t(columns / enc->elements) * enc->bytes * rows;
    }
    TSP_REQUIRE(!mul_overflows(*expert_stride, experts) && *expert_stride * experts == matrix_bytes, "graph GEMV buffer shape mismatch");
    return TSP_OK;
}

}  // namespace

namespace tsp {

int gemv_q8_row(const void* matrix, const float* x, float* y, uint32_t columns, uint32_t rows, uint32_t* error_word, hipStream_t stream, bool* taken) {
    GemvArgs a{};
    a.matrix = static_cast<const uint8_t*>(matrix); a.x = x; a.y = y; a.columns = columns; a.rows = rows; a.experts = a.count = 1; a.error_word = error_word;
    *taken = gemv_units_takes(8, a);
    return *taken ? launch_units<8>(a, stream) : TSP_OK;
}

}  // namespace tsp

extern "C" int tsp_gemv_rows(uint32_t encoding, uint32_t layout, const void* matrix, uint64_t matrix_bytes, const float* x,
                             uint64_t x_stride_bytes, float* y, uint64_t y_stride_bytes, uint32_t count, uint32_t columns,
                             uint32_t rows, uint32_t* error_word, void* stream) {
    GemvArgs a{};
    if (encoding == 8 && count == 1 && layout != TSP_LAYOUT_PLANAR_V3)
        return tsp_q8_matvec_many(layout, matrix, matrix_bytes, x, y, columns, rows, 1, error_word, stream);
    const int rc = check_shape(encoding, layout, matrix_bytes, columns, rows, 1, &a.spec, &a.expert_stride);
    if (rc != TSP_OK) return rc;
    TSP_REQUIRE(matrix && x && y && error_word, "null device pointer");
    TSP_REQUIRE(count && count <= 65535 && x_stride_bytes % 4 == 0 && y_stride_bytes % 4 == 0 &&
                    (count == 1 || (x_stride_bytes >= uint64_t(columns) * 4 && y_stride_bytes >= uint64_t(rows) * 4)),
                "graph GEMV row extent mismatch");
    const uint64_t x_span = uint64_t(count - 1) * x_stride_bytes + uint64_t(columns) * 4;
    const uint64_t y_span = uint64_t(count - 1) * y_stride_bytes + uint64_t(rows) * 4;
    TSP_REQUIRE(!ranges_overlap(y, y_span, matrix, matrix_bytes) && !ranges_overlap(y, y_span, x, x_span),
                "GEMV output overlaps an input");
    a.matrix = static_cast<const uint8_t*>(matrix); a.x = x; a.y = y; a.ids = nullptr;
    a.x_stride = x_stride_bytes; a.y_stride = y_stride_bytes;
    a.columns = columns; a.rows = rows; a.experts = 1; a.count = count; a.error_word = error_word;
    return launch_gemv(encoding, layout, a, static_cast<hipStream_t>(stream));
}

extern "C" int tsp_gemv(uint32_t encoding, uint32_t layout, const void* matrix, uint64_t matrix_bytes, const float* x, float* y,
                        uint32_t columns, uint32_t rows, uint32_t* error_word, void* stream) {
    return tsp_gemv_rows(encoding, layout, matrix, matrix_bytes, x, 0, y, 0, 1, columns, rows, error_word, stream);
}

extern "C" int tsp_routed_gemv(uint32_t encoding, const void* matrices, uint64_t matrices_bytes, const uint32_t* ids, const float* x,
                               float* y, uint32_t columns, uint32_t rows, uint32_t experts, uint32_t selected, int broadcast_input,
                               uint32_t* error_word, void* stream) {
    GemvArgs a{};
    TSP_REQUIRE(experts && experts <= 4096 && selected && selected <= 64, "invalid routed GEMV routing shape");
    const int rc = check_shape(encoding, TSP_LAYOUT_GGUF, matrices_bytes, columns, rows, experts, &a.spec, &a.expert_stride);
    if (rc != TSP_OK) return rc;
    TSP_REQUIRE(matrices && ids && x && y && error_word, "null device pointer");
    const uint64_t x_span = uint64_t(broadcast_input ? 1 : selected) * columns * 4, y_span = uint64_t(selected) * rows * 4;
    TSP_REQUIRE(!ranges_overlap(y, y_span, matrices, matrices_bytes) && !ranges_overlap(y, y_span, x, x_span) &&
                    !ranges_overlap(y, y_span, ids, uint64_t(selected) * 4),
                "routed GEMV output overlaps an input");
    a.matrix = static_cast<const uint8_t*>(matrices); a.x = x; a.y = y; a.ids = ids;
    a.x_stride = broadcast_input ? 0 : uint64_t(columns) * 4; a.y_stride = uint64_t(rows) * 4;
    a.columns = columns; a.rows = rows; a.experts = experts; a.count = selected; a.error_word = error_word;
    return launch_gemv(encoding, TSP_LAYOUT_GGUF, a, static_cast<hipStream_t>(stream));
}
