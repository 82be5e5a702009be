// Dense Q4_K GEMM over raw GGUF rows with few tiles to go round: out[m, n] = sum_k x[m, k] * w[n, k], activations in fragment order.
//
// With few tiles the chip is not short of bandwidth or of matrix cores but of time: a launch, a trip to memory, and then each wave's chain of
// instructions. So nothing is shared and nothing is waited for but the loads themselves:
//   * The row conversion stores the activations as the matrix instruction takes them, 1 KB of neighbouring lanes per 32 rows x 16 columns: a
//     fragment is one load from memory (or L2) into registers, without LDS, barriers or addresses to keep.
//   * A wave owns 32 activation rows, 32 weight rows and a stretch of the super-blocks, and requests a whole super-block, 88 registers,
//     before it touches any of it; a register is refilled for the next super-block as soon as it has been used.
//   * The waves of a workgroup are the stretches of one tile; their sums meet once, in LDS, in the order of the columns.
// The arithmetic is dense_tile.hip's for either EXACT. Bound by a launch (1.6 us), the trip to memory and a wave's instructions, some 350 a super-block: 62 x 1196
// x 2560 9.3 -> 6.6 us where dense_tile.hip's smallest tiles went through LDS step by step, 12 x 700 x 512 5.5 -> 4.2, 107 x 1649 x 1792 7.7 -> 5.9, 37 x
// 6100 x 2560 10.8 -> 8.8. Tried: deeper rings and weights further ahead in the tiles that go through LDS (no gain: requests were not what they waited for);
// 64 rows to a wave (37 x 6100 x 2560 10.1, 62 x 1196 x 2560 9.5); each lane its own weight row's pieces, without LDS (0.2 us less with one
// workgroup per compute unit, 0.6 more at 37 x 6100).
#include "dense_tile.hpp"

#include <algorithm>

#include "mfma_quant.hpp"

using namespace tsp;

namespace {

constexpr uint32_t kMostWaves = 4, kWPieces = 5, kStageBytes = kWPieces * kWave * 16;
static_assert(kStageBytes >= 32 * 32 * 4, "a wave's sums take its stage's place");

template <bool EXACT>
__global__ __launch_bounds__(64 * kMostWaves) __attribute__((amdgpu_waves_per_eu(3, 3))) void dense_fragments_kernel(DenseTileArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // the waves' super-blocks of weights, then their sums
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave), waves = blockDim.x / kWave;
    const uint32_t col = lane % 32, khalf = lane / 32;

    // ---- the workgroup's tile, as in dense_tile.hip: XCD x takes the x-th run of tiles, bands of a.band row tiles, row tiles fastest
    const uint32_t n_tiles = (a.n + 31) / 32, m_tiles = (a.m + 31) / 32, tiles = n_tiles * m_tiles, per_xcd = (tiles + 7) / 8;
    const uint32_t logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || logical >= tiles) return;
    const uint32_t in_band = a.band * n_tiles, band = logical / in_band, height = m_tiles - band * a.band < a.band ? m_tiles - band * a.band : a.band;
    const uint32_t m_tile = band * a.band + logical % in_band % height, m0 = m_tile * 32, n0 = (logical % in_band / height) * 32;
    const uint32_t bpr = a.k / 256, first = bpr * wave / waves, end = bpr * (wave + 1) / waves;

    // ---- requests: uniform base and step, a lane's part fixed; lanes past the last row repeat it
    const uint32_t rows = a.m - m0 < 32 ? a.m - m0 : 32;
    const uint32_t a_lane = (khalf * rows + (col < rows ? col : rows - 1)) * 16, a_pitch = rows * 32, a_base = m_tile * (64 * a.k), s_base = m_tile * (32 * 32 * bpr);
    // weights: nine neighbouring lanes per row's 144 bytes, turned through LDS
    uint32_t w_lane[kWPieces];
#pragma unroll
    for (uint32_t q = 0; q < kWPieces; ++q) {
        const uint32_t u = q * kWave + lane, c = u < 288 ? u : 287, row = n0 + c / 9 < a.n ? n0 + c / 9 : a.n - 1;
        w_lane[q] = row * (bpr * 144) + c % 9 * 16;
    }
    uint8_t* const stage = lds + wave * kStageBytes;
    const uint8_t* const mine = stage + col * 144;  // 36 words: sixteen lanes' 16 bytes meet all banks once
    auto buffer = [](const void* p, uint64_t bytes) { return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, int(uint32_t(bytes)), 0x00020000); };
    auto load = [](__amdgpu_buffer_rsrc_t from, uint32_t lane_offset, uint32_t offset) { return __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(from, lane_offset, offset, 0)); };

    u32x4 staged[kWPieces];
    f16x8 af[16], sums;
    // What is requested past the wave's last super-block comes from the beginning of buffers without bytes: nothing travels. (From the beginning: whether
    // a scalar offset counts when the hardware compares with a buffer's size is nothing to rely on.)
    struct Sources { __amdgpu_buffer_rsrc_t w, a, s; uint32_t w_at, a_at, a_step, s_at; };
    auto sources = [&](uint32_t b) {
        const bool live = b < end;
        return Sources{buffer(a.w, live ? uint64_t(a.n) * bpr * 144 : 0), buffer(a.a, live ? uint64_t(a.m) * a.k * 2 : 0), buffer(a.sx, live ? uint64_t(a.m) * bpr * 32 : 0),
                       live ? b * 144 : 0, live ? a_base + b * 16 * a_pitch : 0, live ? a_pitch : 0, live ? s_base + b * a_pitch : 0};
    };
    auto request_weights = [&](const Sources& s) {
#pragma unroll
        for (uint32_t q = 0; q < kWPieces; ++q) staged[q] = load(s.w, w_lane[q], s.w_at);
    };
    auto request_rows = [&](const Sources& s, int f) { af[f] = __builtin_bit_cast(f16x8, load(s.a, a_lane, s.a_at + f * s.a_step)); };
    auto request_sums = [&](const Sources& s) { sums = __builtin_bit_cast(f16x8, load(s.s, a_lane, s.s_at)); };

    {
        const Sources s = sources(first);
        request_weights(s);
#pragma unroll
        for (int f = 0; f < 16; ++f) request_rows(s, f);
        if constexpr (EXACT) request_sums(s);
    }
    __builtin_amdgcn_sched_barrier(0);

    f32x16 acc{}, blk;
    const Q4Masks masks = q4_masks();
    const Q4ScaleConsts q4s = q4_scale_consts();
    for (uint32_t b = first; b < end; ++b) {
        const Sources next = sources(b + 1);
#pragma unroll
        for (uint32_t q = 0; q < kWPieces; ++q) *reinterpret_cast<u32x4*>(stage + (q * kWave + lane) * 16) = staged[q];
        __builtin_amdgcn_sched_barrier(0);
        request_weights(next);
        __builtin_amdgcn_wave_barrier();  // the wave's own LDS, served in order
        RawHdrQ4 words;
        words.words = *reinterpret_cast<const uint4*>(mine);
        words.dm = 0;
        const HdrQ4 hdr = decode_hdr_q4k<B_Q4K_RAW>(words);
        auto step = [&](auto p_tag) {
            constexpr int P = decltype(p_tag)::value;
            const u32x4 raw = *reinterpret_cast<const u32x4*>(mine + 16 + P * 32 + khalf * 16);
            f16x2 ps;
            float scale[2], offset[2];
            if constexpr (EXACT) {
                ps = q4_pair_scale<P>(hdr.sc[0], hdr.sc[1], q4s);
            } else {
                constexpr int B = (P % 2) * 2;
                scale[0] = (hdr.d * byte_as_float<B>(hdr.sc[P / 2])) * 16777216.0f;
                scale[1] = (hdr.d * byte_as_float<B + 1>(hdr.sc[P / 2])) * 1048576.0f;
                offset[0] = -(hdr.dmin * byte_as_float<B>(hdr.mn[P / 2]));
                offset[1] = -(hdr.dmin * byte_as_float<B + 1>(hdr.mn[P / 2]));
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {  // (low, high nibbles) x (first, second eight columns of the lane's sixteen)
                const int hi = g / 2, ff = g % 2, f = P * 4 + g;
                __builtin_amdgcn_sched_barrier(0);  // fragments unpacked ahead of their products would not fit the registers
                f16x8 w;
                if constexpr (EXACT) {
                    w = hi ? scaled8_q4_swapped<1>(raw[2 * ff], raw[2 * ff + 1], f16x2{ps[1], ps[1]}, masks)
                           : scaled8_q4_swapped<0>(raw[2 * ff], raw[2 * ff + 1], f16x2{ps[0], ps[0]}, masks);
                    const f32x16 zero{};
                    blk = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[f], w, f == 0 ? zero : blk, 0, 0, 0);
                } else {
                    w = weights8_q4_swapped(raw[2 * ff], raw[2 * ff + 1], hi ? masks.hi : masks.lo, scale[hi], offset[hi]);
                    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[f], w, acc, 0, 0, 0);
                }
                request_rows(next, f);
            }
        };
        step(std::integral_constant<int, 0>{});
        step(std::integral_constant<int, 1>{});
        step(std::integral_constant<int, 2>{});
        step(std::integral_constant<int, 3>{});
        if constexpr (EXACT) {
            // acc += d * blk - dmin * sum_s Sx(hi + lo)[m, s] * mn[n, s]
            __builtin_amdgcn_sched_barrier(0);
            const f32x16 zero{};
            float d = hdr.d * kQ4Lift, dmin = hdr.dmin;
            asm volatile("" : "+v"(d), "+v"(dmin));  // as floats in registers: as halves they make every multiply-add a mixed-precision one, half as fast
            const f32x16 low = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, minima_frag(hdr), zero, 0, 0, 0);
            request_sums(next);
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] = __builtin_fmaf(-dmin, low[v], __builtin_fmaf(d, blk[v], acc[v]));
        }
    }

    // ---- accumulator v: row 8 (v / 4) + 4 khalf + v % 4, weight row col. A thread adds up four rows of a column, in the order of the columns.
    __syncthreads();  // every wave has left its stage
    float* const parts = reinterpret_cast<float*>(lds);  // [wave][4][lane][4]
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<f32x4*>(parts + ((wave * 4 + q) * kWave + lane) * 4) = f32x4{acc[4 * q], acc[4 * q + 1], acc[4 * q + 2], acc[4 * q + 3]};
    __syncthreads();
    uint32_t biggest = 0;  // the largest result's bits without the sign: anything not finite shows at the end
    for (uint32_t u = tid; u < 256; u += blockDim.x) {
        f32x4 sum = *reinterpret_cast<const f32x4*>(parts + u * 4);
        for (uint32_t w = 1; w < waves; ++w) sum += *reinterpret_cast<const f32x4*>(parts + (w * 256 + u) * 4);
        const uint32_t n = n0 + u % 32;
        if (n >= a.n) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t row = m0 + u / 64 * 8 + u / 32 % 2 * 4 + e;
            if (row >= a.m) continue;
            const uint32_t vb = __float_as_uint(sum[e]), magnitude = vb & 0x7fffffffu;
            biggest = biggest > magnitude ? biggest : magnitude;
            uint8_t* const out = static_cast<uint8_t*>(a.out) + uint64_t(row) * a.out_stride;
            if (a.out_bf16) reinterpret_cast<uint16_t*>(out)[n] = uint16_t((vb + 0x7fffu + ((vb >> 16) & 1u)) >> 16);
            else reinterpret_cast<float*>(out)[n] = sum[e];
        }
    }
    publish_error(biggest >= 0x7f800000u ? uint32_t(TSP_ERRBIT_NONFINITE) : 0u, a.error_word);
}

}  // namespace

namespace tsp {

// As long as three workgroups per compute unit, what their registers allow, nearly hold all tiles at once. Kernels alone, against dense_tile.hip's best: 512
// tiles 33 x 8192 x 2560 11.4 -> 9.8 us, 64 x 8192 x 512 5.8 -> 5.7, 1000 x 512 x 2048 11.8 -> 9.8; 658 tiles 200 x 3000 x 2560 13.7 -> 13.1, x 512 6.4 ->
// 6.1; 704 tiles 700 x 1000 x 1280 10.7 -> 9.8; 752 tiles 1500 x 512 x 1536 10.2 -> 10.7, 500 x 1500 x 2560 13.8 -> 14.0; 1024 tiles 2048 x 512 x 1024
// 8.5 -> 9.8, 500 x 8192 x 512 (4096) 11.8 -> 18.4: fragments are fetched once per tile, and some 14 TB/s is what the L2s give. Four waves: with two
// a chain is as long as before (9 x 1500 x 2560 7.5 us, with three 7.1, four 6.6, five 6.7), and of five only two workgroups fit (33 x 8192 x 2560 12.2).
uint32_t dense_fragments_waves(uint32_t m, uint32_t n, uint32_t k) {
    const uint64_t tiles = uint64_t((m + 31) / 32) * ((n + 31) / 32);
    return tiles <= 704 ? std::min(k / 256, kMostWaves) : 0;
}

int launch_dense_fragments(DenseTileArgs a, uint32_t waves, hipStream_t s) {
    const uint32_t m_tiles = (a.m + 31) / 32, n_tiles = (a.n + 31) / 32, groups = (m_tiles * n_tiles + 7) / 8 * 8;
    a.band = dense_band(m_tiles, n_tiles, 32, 32);
    if (dense_exact(a.m, a.n)) TSP_LAUNCH("gemm_dense_fragments", s, (dense_fragments_kernel<true><<<groups, waves * kWave, waves * kStageBytes, s>>>(a)));
    else TSP_LAUNCH("gemm_dense_fragments", s, (dense_fragments_kernel<false><<<groups, waves * kWave, waves * kStageBytes, s>>>(a)));
    return launch_status("dense_fragments");
}

}  // namespace tsp
