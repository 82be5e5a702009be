// Q8_0 matrix times up to sixteen token rows (LM head, verify), raw rows and q8_lanes_v1 rows: y[m, r] = sum_k d[r, k/32] * q[r, k] * x[m, k].
//
// A wave owns 256 columns, eight blocks, and keeps the token rows' part of them in registers for all of the launch, as matrix operands;
// a workgroup's waves are a whole row of the matrix and take one tile of 32 weight rows after the other. So every tile is work for every
// wave, the matrix is read once for any number of token rows, and LDS holds nothing but the tile's bytes on their way into lane order and the
// waves' sums, which meet there once per tile, in the order of the columns.
//
// A Q8_0 block is one 16x16x32 matrix instruction per 16 weight rows and piece of the activations: lane (n, kq) supplies the eight quants 8 kq .. 8 kq + 7 of
// weight row n, exact bf16 or halves, on the other side are the token rows; the block's scale multiplies the f32 result. F32: each activation as its three bf16 pieces
// (mfma_quant.hpp: the f32 product, whatever else is in the row); else hi + lo halves under a power of two per token row, 22 significant bits of the row's largest.
//
// Bound by the matrix's bytes from some 60 000 rows on (151 936 x 2048: 65 us, 5.1 TB/s), below that by the first bytes' trip as well. What it replaced gave a wave all of a tile's
// columns, so that few tiles were few waves, and nine token rows half of the columns at a time, sums meeting by atomic additions in an output cleared by
// a launch of its own. Calls with the top-64 behind, before and now, by 2048 columns: eight token rows x 32 000 34.2 -> 28.9 us, 45 000 36.9 -> 35.1, 90 000
// 56.5 -> 54.7 (64 001 42.5 and 43.5: where it is the slower way such calls stay, rows_by_waves in q8_mfma.hip); sixteen x 64 001 49.5 -> 45.9, 151 936 94.0 -> 89.0; by 1024, twelve x 64 001 36.0 -> 28.9; by 2560, twelve x 33 000 69 -> 46, 151 936 200 -> 118 (two
// passes before). Without the top-64: nine x 16 000 x 2048 22.6 -> 14.0 (a workgroup per sixteen rows before), eight 16.7 -> 14.1.
// Of q8_lanes_v1 rows a wave has half of each run, 8 bytes of every 16, so two waves fetch each line: only where it saves a pass.
#include "q8_resident.hpp"

#include <type_traits>

#include "mfma_quant.hpp"

using namespace tsp;

namespace {

constexpr uint32_t kTileRows = 32, kMostTokens = 16, kGroupBytes = 272;  // of a row: eight blocks, or their scales and quants
constexpr uint32_t kStageBytes = 9 * 1024, kSumBytes = kTileRows * kMostTokens * 4;
constexpr uint32_t kNowhere = 0x7fffffffu;  // past the end of any buffer here

struct Q8ResidentArgs {
    const uint8_t* matrix;
    const float* x;  // token-major [m, columns]
    float* y;        // token-major [m, rows]
    uint32_t columns, rows, m;
    uint32_t* error_word;
};

// LANES: q8_lanes_v1 rows. DEPTH tiles of a wave's bytes are on their way while one is multiplied.
template <bool LANES, uint32_t WAVES, bool F32, int DEPTH>
__global__ __launch_bounds__(WAVES * kWave) __attribute__((amdgpu_waves_per_eu(WAVES > 8 ? 3 : 2, WAVES > 8 ? 3 : 2))) void q8_resident_kernel(Q8ResidentArgs a) {
    using Frag = std::conditional_t<F32, bf16x8, f16x8>;
    constexpr int PIECES = F32 ? 3 : 2;
    // three waves to a SIMD: 168 registers, and eleven more in scratch (40 bytes a lane), which raw rows use before and behind the tile loop only; of q8_lanes_v1 rows four are read again for each tile
    constexpr bool kTight = WAVES > 8;
    constexpr uint32_t kRounds = (kTileRows * kMostTokens + WAVES * kWave - 1) / (WAVES * kWave);
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // the waves' stages, then two sets of DEPTH tiles' sums [wave][16-row half][lane][4]
    __shared__ float largest[WAVES][kMostTokens];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t n16 = lane % 16, kq = lane / 16;
    const uint32_t blocks = a.columns / 32, row_bytes = blocks * 34, tiles = (a.rows + kTileRows - 1) / kTileRows;
    uint8_t* const stage = lds + wave * kStageBytes;
    float* const sums = reinterpret_cast<float*>(lds + WAVES * kStageBytes);

    // ---- the token rows' part: asked for first
    struct Eight { float4 v[2]; };
    auto token_piece = [&](int b) {
        Eight e{};
        if (n16 < a.m) {
            const float4* const from = reinterpret_cast<const float4*>(a.x + uint64_t(n16) * a.columns + wave * 256 + b * 32 + kq * 8);
            e.v[0] = from[0];
            e.v[1] = from[1];
        }
        return e;
    };
    Eight xv[8];
#pragma unroll
    for (int b = 0; b < 8; ++b) xv[b] = token_piece(b);

    // ---- a tile's bytes: of raw rows a wave has 17 pieces of 16 bytes per row side by side, sixteen lanes to a row and the last pieces by themselves; of
    // lanes rows half of each 16-byte run of one quant index, 32 pieces of 8 bytes per row, and a piece of scales, in LDS in front of them
    typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
    constexpr int kLoads = LANES ? 16 : 8, kRowsAtOnce = LANES ? 2 : 4;
    const uint32_t piece_row = LANES ? lane / 32 : lane / 16, piece = LANES ? lane % 32 : lane % 16;
    const uint32_t pieces_at = piece_row * row_bytes + (LANES ? 2 * blocks + wave / 2 * 512 + wave % 2 * 8 : wave * kGroupBytes) + piece * 16;
    const uint32_t others_at = lane < kTileRows ? lane * row_bytes + (LANES ? wave * 16 : wave * kGroupBytes + 256) : kNowhere;
    struct Bytes { std::conditional_t<LANES, u32x2, u32x4> v[kLoads]; u32x4 others; };
    Bytes bytes[DEPTH];
    auto fetch = [&](uint32_t tile, auto set_tag) {  // rows past the matrix, and tiles past the last, have no bytes: nothing travels
        Bytes& into = bytes[decltype(set_tag)::value];
        const uint32_t row0 = tile * kTileRows, there = tile < tiles ? (a.rows - row0 < kTileRows ? a.rows - row0 : kTileRows) * row_bytes : 0;
        const auto from = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(a.matrix + (tile < tiles ? uint64_t(row0) * row_bytes : 0)), 0, int(there), 0x00020000);
        uint32_t here = pieces_at;
        asm volatile("" : "+v"(here));  // an addition per piece, not a register
#pragma unroll
        for (uint32_t t = 0; t < kLoads; ++t) {
            const uint32_t at = here + t * (kRowsAtOnce * row_bytes);
            if constexpr (LANES) into.v[t] = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(from, at, 0, 0));
            else into.v[t] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(from, at, 0, 0));
        }
        into.others = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(from, others_at, 0, 0));
    };
    uint8_t* const pieces_to = stage + piece_row * kGroupBytes + (LANES ? 16 + piece * 8 : piece * 16);
    uint8_t* const others_to = stage + (lane % kTileRows) * kGroupBytes + (LANES ? 0 : 256);
    const uint32_t step = gridDim.x;
    fetch(blockIdx.x, std::integral_constant<int, 0>{});
    if constexpr (DEPTH == 2) fetch(blockIdx.x + step, std::integral_constant<int, 1>{});
    __builtin_amdgcn_sched_barrier(0);  // every request above is out before the first wait below

    // ---- the activations' pieces
    uint32_t bad = 0;
    float mine = 0;
#pragma unroll
    for (int b = 0; b < 8; ++b)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 v = xv[b].v[h];
            if (nonfinite(v.x) || nonfinite(v.y) || nonfinite(v.z) || nonfinite(v.w)) bad = TSP_ERRBIT_NONFINITE;
            mine = fmaxf(mine, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
    mine = fmaxf(mine, __shfl_xor(mine, 16, kWave));
    mine = fmaxf(mine, __shfl_xor(mine, 32, kWave));
    if (lane < kMostTokens) largest[wave][lane] = mine;
    __syncthreads();
    float biggest = 0;  // of token row n16
    for (uint32_t w = 0; w < WAVES; ++w) biggest = fmaxf(biggest, largest[w][n16]);
    const int exponent = int((__float_as_uint(biggest) >> 23) & 0xffu) - 127;
    const int shift = F32 ? row_lift(biggest) : !(biggest > 0) || nonfinite(biggest) ? 0 : exponent < -87 ? 100 : 13 - exponent;
    const float scale = power_of_two(shift);
    __syncthreads();  // `largest` has been read: its first row becomes what undoes the scales
    if (tid < kMostTokens) largest[0][tid] = power_of_two(-shift);
    Frag act[8][PIECES];  // the smallest pieces first
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        if constexpr (kTight) {  // asked for again: beside the pieces and a tile's bytes still more would not fit the registers
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            xv[b] = token_piece(b);
        }
        const float4 lo4 = xv[b].v[0], hi4 = xv[b].v[1];
        const float v[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
        if constexpr (F32) {
            Pieces p[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) p[e] = three_pieces(v[e] * scale);
            auto operand = [&](float Pieces::*piece) {
                return __builtin_bit_cast(bf16x8, u32x4{two_tops(p[0].*piece, p[1].*piece), two_tops(p[2].*piece, p[3].*piece), two_tops(p[4].*piece, p[5].*piece),
                                                        two_tops(p[6].*piece, p[7].*piece)});
            };
            act[b][0] = operand(&Pieces::lo);
            act[b][1] = operand(&Pieces::mid);
            act[b][2] = operand(&Pieces::hi);
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const float sv = v[e] * scale;
                act[b][1][e] = _Float16(sv);
                act[b][0][e] = _Float16(sv - float(act[b][1][e]));
            }
        }
    }

    const auto out = __builtin_amdgcn_make_buffer_rsrc(a.y, 0, int(a.m * a.rows * 4), 0x00020000);
    uint32_t parity = 0;
    auto item = [&](uint32_t tile, auto set_tag) {
        const Bytes& now = bytes[decltype(set_tag)::value];
        // the tile before has been read out of the stage: LDS serves a wave in order
#pragma unroll
        for (uint32_t t = 0; t < kLoads; ++t) *reinterpret_cast<std::remove_cvref_t<decltype(now.v[0])>*>(pieces_to + t * (kRowsAtOnce * kGroupBytes)) = now.v[t];
        if (lane < kTileRows) *reinterpret_cast<u32x4*>(others_to) = now.others;
        __builtin_amdgcn_sched_barrier(0);
        fetch(tile + DEPTH * step, set_tag);
        __builtin_amdgcn_wave_barrier();
        f32x4 acc[2] = {};
        auto product = [&](int nt, int b, uint32_t w0, uint32_t w1, float d) {
            f32x4 part{};
            if constexpr (F32) {
                const bf16x8 q = quants8_bf16(w0, w1);
#pragma unroll
                for (int p = 0; p < PIECES; ++p) part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(act[b][p], q, part, 0, 0, 0);
            } else {
                const f16x8 q = quants8(w0, w1);
#pragma unroll
                for (int p = 0; p < PIECES; ++p) part = __builtin_amdgcn_mfma_f32_16x16x32_f16(act[b][p], q, part, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[nt][v] = __builtin_fmaf(d, part[v], acc[nt][v]);
        };
        if constexpr (LANES) {
#pragma unroll
            for (int nt = 0; nt < 2; ++nt) {
                if constexpr (kTight) __builtin_amdgcn_sched_barrier(0);
                const uint8_t* const row = stage + (nt * 16 + n16) * kGroupBytes;
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    if constexpr (kTight) __builtin_amdgcn_sched_barrier(0);
                    const u32x2 s = *reinterpret_cast<const u32x2*>(row + m * 8);
                    uint32_t q[8];  // q[j]: quant 8 kq + j of four blocks, one byte per block
#pragma unroll
                    for (int j = 0; j < 8; ++j) q[j] = *reinterpret_cast<const uint32_t*>(row + 16 + (8 * kq + j) * 8 + m * 4);
                    // 4 x 4 squares of bytes turned over: pairs of quants interleaved for blocks 0, 1 (lo) and 2, 3 (hi), then pairs of pairs
                    uint32_t lo[4], hi[4];
#pragma unroll
                    for (int p = 0; p < 4; ++p) {
                        lo[p] = __builtin_amdgcn_perm(q[2 * p + 1], q[2 * p], 0x05010400u);
                        hi[p] = __builtin_amdgcn_perm(q[2 * p + 1], q[2 * p], 0x07030602u);
                    }
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const uint32_t* const from = b < 2 ? lo : hi;
                        const uint32_t select = b % 2 ? 0x07060302u : 0x05040100u;
                        const uint32_t w0 = __builtin_amdgcn_perm(from[1], from[0], select), w1 = __builtin_amdgcn_perm(from[3], from[2], select);
                        product(nt, 4 * m + b, w0, w1, half_bits_to_float((s[b / 2] >> (16 * (b % 2))) & 0xffffu));
                    }
                }
            }
        } else {
            const uint8_t* const mine = stage + n16 * kGroupBytes;
            auto block = [&](auto b_tag) {
                // the lane's eight quants are bytes 34 B + 2 + 8 kq .. + 8 of the row: dword aligned for odd B, 2 bytes past a dword for even B
                constexpr int B = decltype(b_tag)::value;
                constexpr uint32_t Q_AT = 34 * B + 2, ALIGNED = Q_AT & ~3u;
                if constexpr (kTight) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) {
                    const uint8_t* const row = mine + nt * 16 * kGroupBytes;
                    uint32_t w0 = *reinterpret_cast<const uint32_t*>(row + kq * 8 + ALIGNED), w1 = *reinterpret_cast<const uint32_t*>(row + kq * 8 + ALIGNED + 4);
                    if constexpr (Q_AT % 4 != 0) {
                        const uint32_t w2 = *reinterpret_cast<const uint32_t*>(row + kq * 8 + ALIGNED + 8);
                        w0 = __builtin_amdgcn_alignbyte(w1, w0, 2);
                        w1 = __builtin_amdgcn_alignbyte(w2, w1, 2);
                    }
                    product(nt, B, w0, w1, half_bits_to_float(*reinterpret_cast<const uint16_t*>(row + 34 * B)));
                }
            };
            [&]<int... B>(std::integer_sequence<int, B...>) { (block(std::integral_constant<int, B>{}), ...); }(std::make_integer_sequence<int, 8>{});
        }
        float* const to = sums + ((parity * DEPTH + decltype(set_tag)::value) * WAVES + wave) * (kSumBytes / 4);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) *reinterpret_cast<f32x4*>(to + (nt * kWave + lane) * 4) = acc[nt];
    };
    // The sums of the tiles at hand, DEPTH of them. There are two sets: whoever writes the next one has passed the barrier behind which this one's
    // predecessor was read.
    auto finish = [&](uint32_t tile) {
        lds_barrier();
        const float* const set = sums + parity * (DEPTH * WAVES * (kSumBytes / 4));
        parity ^= 1;
        // Stores from every lane, to nowhere where there is no result: what a wave has under way is then the same each time round, and the wait for the
        // next tile's bytes is for these alone.
#pragma unroll
        for (uint32_t d = 0; d < DEPTH; ++d)
#pragma unroll
            for (uint32_t round = 0; round < kRounds; ++round) {
                // token row m = 4 kq + v of accumulator v, weight row 16 nt + n16
                const uint32_t u = tid + round * (WAVES * kWave), m = u / kTileRows % kMostTokens, r = u % kTileRows, from = ((r / 16) * kWave + (m / 4) * 16 + r % 16) * 4 + m % 4;
                float part[WAVES];
#pragma unroll
                for (uint32_t w = 0; w < WAVES; ++w) part[w] = set[(d * WAVES + w) * (kSumBytes / 4) + from];  // all on their way at once
                double total = part[0];  // rounded once: the pieces of a block's product, which meet in one accumulator, are rounded once more than by themselves
#pragma unroll
                for (uint32_t w = 1; w < WAVES; ++w) total += part[w];
                const float sum = float(total) * largest[0][m];
                const uint32_t row = (tile + d * step) * kTileRows + r;
                const bool there = u < kTileRows * a.m && row < a.rows;
                if (there && nonfinite(sum)) bad = TSP_ERRBIT_NONFINITE;
                __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(sum), out, there ? (m * a.rows + row) * 4 : kNowhere, 0, 0);
            }
    };
    __syncthreads();
    for (uint32_t tile = blockIdx.x; tile < tiles; tile += DEPTH * step) {
        item(tile, std::integral_constant<int, 0>{});
        if constexpr (DEPTH == 2) {
            if (tile + step >= tiles) {  // the other half of the set is old sums, of rows past the matrix
                finish(tile);
                break;
            }
            item(tile + step, std::integral_constant<int, 1>{});
        }
        finish(tile);
    }
    publish_error(bad, a.error_word);
}

template <bool LANES, uint32_t WAVES, bool F32, int DEPTH>
int launch(const Q8ResidentArgs& a, hipStream_t s) {
    constexpr uint32_t kLds = WAVES * (kStageBytes + 2 * DEPTH * kSumBytes);
    static_assert(kLds * (WAVES > 4 ? 1 : 8 / WAVES) <= 160 * 1024 - 1024, "the workgroups of a compute unit");
    static std::atomic<uint64_t> raised{0};
    static int units_of[64] = {};
    int device = 0;
    if (setup_pending(raised, &device)) {
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_resident_kernel<LANES, WAVES, F32, DEPTH>), hipFuncAttributeMaxDynamicSharedMemorySize, int(kLds)));
        TSP_HIP(hipDeviceGetAttribute(&units_of[device], hipDeviceAttributeMultiprocessorCount, device));
        setup_done(raised, device);
    }
    const uint32_t units = uint32_t(units_of[device] > 0 ? units_of[device] : 256), tiles = (a.rows + kTileRows - 1) / kTileRows;
    const uint32_t groups = units * (WAVES > 4 ? 1 : 8 / WAVES);
    TSP_LAUNCH("q8_resident", s, (q8_resident_kernel<LANES, WAVES, F32, DEPTH><<<groups < tiles ? groups : tiles, WAVES * kWave, kLds, s>>>(a)));
    return launch_status("q8_resident");
}

}  // namespace

namespace tsp {

int q8_resident(bool lanes, bool f32, const void* matrix, const float* x, float* y, uint32_t columns, uint32_t rows, uint32_t width, uint32_t* error_word, hipStream_t s) {
    const Q8ResidentArgs a{static_cast<const uint8_t*>(matrix), x, y, columns, rows, width, error_word};
    if (lanes) return launch<true, 10, true, 1>(a, s);
    switch (columns / 256) {
    case 1: return f32 ? launch<false, 1, true, 2>(a, s) : launch<false, 1, false, 2>(a, s);
    case 2: return f32 ? launch<false, 2, true, 2>(a, s) : launch<false, 2, false, 2>(a, s);
    case 3: return f32 ? launch<false, 3, true, 2>(a, s) : launch<false, 3, false, 2>(a, s);
    case 4: return f32 ? launch<false, 4, true, 2>(a, s) : launch<false, 4, false, 2>(a, s);
    case 5: return f32 ? launch<false, 5, true, 2>(a, s) : launch<false, 5, false, 2>(a, s);
    case 6: return f32 ? launch<false, 6, true, 2>(a, s) : launch<false, 6, false, 2>(a, s);
    case 7: return f32 ? launch<false, 7, true, 2>(a, s) : launch<false, 7, false, 2>(a, s);
    case 8: return f32 ? launch<false, 8, true, 2>(a, s) : launch<false, 8, false, 2>(a, s);
    case 9: return launch<false, 9, true, 1>(a, s);
    default: return launch<false, 10, true, 1>(a, s);
    }
}

}  // namespace tsp
