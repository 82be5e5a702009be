// Dense Q4_K GEMM over raw GGUF rows: out[m, n] = sum_k x[m, k] * w[n, k] (include/tokspur/graph.hpp:753 `grouped_mm` with one
// expert), activations as halves (bf16 values), products on v_mfma_f32_32x32x16_f16.
//
// Two arithmetics, the engine's for these row counts:
//   EXACT (below 512 rows): the integers sc * q as exact halves, one super-block of 256 columns at a time; d multiplies its f32 sum, and
//     the minima are one more MFMA against the activations' sub-block sums (hi + lo halves). Nothing is rounded.
//   else: a weight is the f32 value d * sc * q - dmin * mn rounded once to half: the code q, masked out where it sits, is the subnormal
//     half q * 2^-24, and one mixed-precision fused multiply-add per weight evaluates (d * sc * 2^24) * that - dmin * mn.
//
// A wave owns RT x 32 activation rows and 32 weight rows. Its workgroup is a tile of WM x WN such waves, times GROUPS: with few tiles
// the waves of a workgroup also share out the columns, group g taking the g-th part of the super-blocks, and the groups' sums meet
// in LDS at the end, added in the order of the columns. 64 columns are a step:
//   * Activations: the tile's rows x 128 bytes go global -> LDS directly, three steps ahead, into a ring of three slabs. 16-byte chunk
//     c of row r sits at position c ^ ((r / 2) % 8): a 16-byte read by sixteen consecutive lanes covers all 64 banks once.
//   * Weights: a super-block of the tile's rows, 144 bytes each, travels the same way once per four steps, as it lies: nine
//     neighbouring lanes per row (32 bytes per row and step took three times as long in the address unit). A lane takes the
//     header and its nibbles of all four steps into registers at the super-block's end, and the place is free again.
//   * Requests go out one at a time between MFMAs (a wave whose request finds the address unit busy stands still), unconditional and
//     from every thread (rows past the end repeat the last row), so that each wave waits with an exact count. One barrier per
//     step, before its last group of MFMAs: by then a wave has read all of the step's slab, and the next step's has landed.
// With 128 x 128 tiles bound by the way into LDS (450 x 8192 x 2560: 22 of 34 us are left with the arithmetic taken out, 21 with only
// the arithmetic), with 256 x 256 tiles by the matrix pipe (63 of 67 us at 2048 x 8192 x 2048).
#include "dense_tile.hpp"

#include <algorithm>
#include <atomic>
#include <type_traits>
#include <utility>

#include "mfma_quant.hpp"

using namespace tsp;

namespace {

// A pointer that is the same in every lane, moved to scalar registers (the base operand of a direct-to-LDS request has to be one).
__device__ __forceinline__ const uint8_t* uniform_pointer(const uint8_t* p) {
    const uint64_t bits = reinterpret_cast<uint64_t>(p);
    const uint32_t lo = uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(bits))), hi = uint32_t(__builtin_amdgcn_readfirstlane(uint32_t(bits >> 32)));
    return reinterpret_cast<const uint8_t*>(uint64_t(hi) << 32 | lo);
}

// 16 bytes per lane from base + lane_offset to LDS at lds_base + AT (uniform) + 16 * lane
template <int AT>
__device__ __forceinline__ void to_lds(const uint8_t* base, uint32_t lane_offset, uint32_t lds_base) {
    asm volatile("s_add_u32 m0, %0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(lane_offset), "s"(base), "n"(AT) : "memory", "m0", "scc");
}

constexpr int kStepK = 64, kRing = 3;

// TN: weight rows of a tile (TN / 32 waves side by side).
template <int RT, int WAVES, int TN, int GROUPS, bool EXACT>
struct Shape {
    static constexpr int kGroupWaves = WAVES / GROUPS, kThreadsT = 64 * kGroupWaves, WN = TN / 32, WM = kGroupWaves / WN, kTileM = WM * RT * 32;
    static constexpr int kSlabBytes = kTileM * kStepK * 2, kSxBytes = EXACT ? kTileM * 32 : 0;
    static_assert(WM >= 1 && WN * WM * GROUPS == WAVES && (RT % GROUPS == 0 || GROUPS % RT == 0));
    static constexpr int kSlabPieces = kSlabBytes / (kThreadsT * 16), kSxPieces = (kSxBytes + kThreadsT * 16 - 1) / (kThreadsT * 16);
    static_assert(kSlabBytes % (kThreadsT * 16) == 0);
    static constexpr int kChunks = TN * 9, kWPieces = (kChunks + kThreadsT - 1) / kThreadsT;  // 16-byte pieces of a super-block of the tile's weight rows
    static constexpr int kWAt = kRing * kSlabBytes, kSxAt = kWAt + kWPieces * kThreadsT * 16, kGroupBytes = kSxAt + 2 * kSxBytes;
    static constexpr int kOwn = RT >= GROUPS ? RT / GROUPS : 1, kShares = RT / kOwn;  // row tiles of the wave's results that a group stores, and groups that store
    static constexpr int kParts = GROUPS == 1 ? 0 : GROUPS * kShares * kThreadsT * kOwn * 64, kRegion = 12 * 1024;
    static constexpr int kLds = std::max(GROUPS * kGroupBytes, std::max(kParts, WAVES * kRegion));
    // Where one workgroup of four waves fills a compute unit the LDS is sized at the launch: knowing its size the compiler would keep sums in
    // accumulator registers and move them out again to scale them.
    static constexpr bool kAtLaunch = WAVES == 4 && kLds > 80 * 1024;
    static_assert(kLds * (kAtLaunch ? 1 : 8 / WAVES) <= 160 * 1024, "the workgroups of a compute unit share 160 KB");
};

template <int RT, int WAVES, int TN, int GROUPS, bool EXACT>
__global__ __launch_bounds__(64 * WAVES) __attribute__((amdgpu_waves_per_eu(2, 2))) void dense_tile_kernel(DenseTileArgs a) {
    using S = Shape<RT, WAVES, TN, GROUPS, EXACT>;
    constexpr int kGroupWaves = S::kGroupWaves, kThreadsT = S::kThreadsT, WN = S::WN, kTileM = S::kTileM, kSlabBytes = S::kSlabBytes, kSxBytes = S::kSxBytes;
    constexpr int kSlabPieces = S::kSlabPieces, kSxPieces = S::kSxPieces, kChunks = S::kChunks, kWPieces = S::kWPieces, kWAt = S::kWAt, kSxAt = S::kSxAt;
    constexpr int kGroupBytes = S::kGroupBytes, kOwn = S::kOwn, kShares = S::kShares, kRegion = S::kRegion;
    __shared__ __attribute__((aligned(16))) uint8_t lds_sized[S::kAtLaunch ? 16 : S::kLds];
    extern __shared__ __attribute__((aligned(16))) uint8_t lds_at_launch[];
    uint8_t* const lds_all = S::kAtLaunch ? lds_at_launch : lds_sized;

    const uint32_t group = GROUPS == 1 ? 0 : uint32_t(__builtin_amdgcn_readfirstlane(int(threadIdx.x / kThreadsT)));
    uint8_t* const lds_raw = lds_all + group * kGroupBytes;
    const uint32_t tid = threadIdx.x % kThreadsT, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t col = lane % 32, khalf = (lane / 32) & 1;
    const uint32_t wm = wave / WN, wn = wave % WN;

    // ---- the workgroup's tile: XCD x (workgroup id % 8) takes the x-th run of consecutive tiles
    const uint32_t n_tiles = (a.n + TN - 1) / TN, m_tiles = (a.m + kTileM - 1) / kTileM;
    const uint32_t tiles = n_tiles * m_tiles, per_xcd = (tiles + 7) / 8;
    const uint32_t logical = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || logical >= tiles) return;
    // the run is a stretch of a band of a.band row tiles, row tiles fastest
    const uint32_t in_band = a.band * n_tiles, band = logical / in_band, height = m_tiles - band * a.band < a.band ? m_tiles - band * a.band : a.band;
    const uint32_t m0 = (band * a.band + logical % in_band % height) * kTileM, n0 = (logical % in_band / height) * TN;
    const uint32_t bpr = a.k / 256, row_bytes = bpr * 144;
    // the group's super-blocks: `first` on, `count` of them; the last group may have fewer, or none, and multiplies the matrix's last one with factors of zero
    const uint32_t count = (bpr + GROUPS - 1) / GROUPS, first = group * count;

    // ---- per-thread parts of the request addresses. Activations: request i of thread t fills 16-byte position t + T i of the slab
    // (T threads) = slot t % 8 of row (t + T i) / 8; weights: chunk u % 9 of row u / 9; sums: half u % 2 of row u / 2.
    uint32_t a_lane[kSlabPieces], w_lane[kWPieces], sx_lane[kSxPieces ? kSxPieces : 1];
#pragma unroll
    for (int i = 0; i < kSlabPieces; ++i) {
        const uint32_t r = (tid + kThreadsT * i) / 8, row = m0 + r < a.m ? m0 + r : a.m - 1;
        a_lane[i] = (row * a.a_stride + (((tid % 8) ^ ((r >> 1) & 7)) * 8)) * 2;
    }
#pragma unroll
    for (int q = 0; q < kWPieces; ++q) {
        const uint32_t u = tid + kThreadsT * q, c = u < kChunks ? u : kChunks - 1, row = n0 + c / 9 < a.n ? n0 + c / 9 : a.n - 1;
        w_lane[q] = row * row_bytes + c % 9 * 16;
    }
#pragma unroll
    for (int q = 0; q < kSxPieces; ++q) {
        const uint32_t u = (tid + kThreadsT * q) % (kTileM * 2), row = m0 + u / 2 < a.m ? m0 + u / 2 : a.m - 1;
        sx_lane[q] = row * bpr * 32 + (u % 2) * 16;
    }
    const uint32_t lds0 = uint32_t(__builtin_amdgcn_readfirstlane(lds_address(lds_all))) + group * kGroupBytes;
    const uint32_t my_bulk = lds0 + wave * 1024;
    constexpr uint32_t kSxWaves = kSxBytes / 1024 ? kSxBytes / 1024 : 1;
    const uint32_t my_sx = lds0 + kSxAt + (wave % kSxWaves) * 1024;

    auto block_at = [&](uint32_t b) { b += first; return b < bpr ? b : bpr - 1; };  // b: counted from the group's first
    auto a_block = [&](uint32_t b) { return uniform_pointer(reinterpret_cast<const uint8_t*>(a.a) + uint64_t(block_at(b)) * 512); };
    auto w_block = [&](uint32_t b) { return uniform_pointer(a.w + uint64_t(block_at(b)) * 144); };
    auto sx_block = [&](uint32_t b) { return uniform_pointer(reinterpret_cast<const uint8_t*>(a.sx) + uint64_t(block_at(b)) * 32); };
    // piece I of a step's activations
    auto request_a = [&]<int I>(const uint8_t* base, uint32_t slot, std::integral_constant<int, I>) { to_lds<I * (kThreadsT * 16)>(base, a_lane[I], my_bulk + slot); };
    auto request_w = [&]<int I>(const uint8_t* base, const uint8_t* sums, uint32_t b, std::integral_constant<int, I>) {
        if constexpr (I < kWPieces) to_lds<kWAt + I * (kThreadsT * 16)>(base, w_lane[I], my_bulk);
        else to_lds<(I - kWPieces) * (kThreadsT * 16)>(sums, sx_lane[I - kWPieces], my_sx + (b % 2) * kSxBytes);
    };
    constexpr int kHead = kWPieces + kSxPieces;

    f32x16 acc[RT], blk[EXACT ? RT : 1];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][v] = 0.0f;

    const uint32_t a_row_at = (wm * (RT * 32) + col) * 128, a_swz = (col >> 1) & 7, w_r = wn * 32 + col;
    uint32_t a_at[4];  // the lane's fragment of group g, row tile 0
#pragma unroll
    for (int g = 0; g < 4; ++g) a_at[g] = a_row_at + ((4 * (g / 2) + 2 * khalf + (g % 2)) ^ a_swz) * 16;
    const uint32_t w_at = kWAt + w_r * 144;
    const uint32_t sx_at = kSxAt + (wm * (RT * 32) + col) * 32 + khalf * 16;

    const Q4Masks masks = q4_masks();
    // Rounded weights: masks in scalar registers. Two mixed-precision multiply-adds follow each and here, so its rate is not what they wait for, and with the registers left to
    // other values the loop's order comes out the better one (in vector registers 2048 x 8192 x 2048 takes 70.9 us for 70.3, 1500 x 8192 x 2560 75.0 for 74.3).
    Q4Masks rounded_masks{0x000f000fu, 0x00f000f0u};
    asm volatile("" : "+s"(rounded_masks.lo), "+s"(rounded_masks.hi));
    const Q4ScaleConsts q4s = q4_scale_consts();
    HdrQ4 hdr{};   // of the super-block at hand: a lane holds one weight row
    u32x4 raw[4];  // the lane's nibbles of the super-block's four steps
    f16x8 af[RT];  // a fragment serves one MFMA, and its register is refilled for the next group right behind it

    auto read_header = [&](uint32_t b) {
        RawHdrQ4 words;
        words.words = *reinterpret_cast<const uint4*>(lds_raw + w_at);
        words.dm = 0;
#pragma unroll
        for (int p = 0; p < 4; ++p) raw[p] = *reinterpret_cast<const u32x4*>(lds_raw + w_at + 16 + p * 32 + khalf * 16);
        hdr = decode_hdr_q4k<B_Q4K_RAW>(words);
        if (GROUPS > 1 && first + b >= bpr) { hdr.d = 0.0f; hdr.dmin = 0.0f; }
    };

    uint32_t slot_now = 0, slot_next = kSlabBytes, slot_last = 2 * kSlabBytes;  // of the step at hand and the two after it
    auto step_fn = [&]<int P>(uint32_t b, const uint8_t* a_now, const uint8_t* a_next, const uint8_t* w_next, const uint8_t* sx_next, std::integral_constant<int, P>) {
        const uint8_t* const a_from = P == 0 ? a_now + 3 * 128 : a_next + (P - 1) * 128;
        f16x2 ps;
        float scale[2], offset[2];
        const float fold_d = hdr.d * kQ4Lift, fold_dmin = hdr.dmin;
        f16x8 minima;
        if constexpr (EXACT) {
            ps = q4_pair_scale<P>(hdr.sc[0], hdr.sc[1], q4s);
            if (P == 3) minima = minima_frag(hdr);
        } else {
            constexpr int B = (P % 2) * 2;
            scale[0] = (hdr.d * byte_as_float<B>(hdr.sc[P / 2])) * 16777216.0f;
            scale[1] = (hdr.d * byte_as_float<B + 1>(hdr.sc[P / 2])) * 1048576.0f;
            offset[0] = -(hdr.dmin * byte_as_float<B>(hdr.mn[P / 2]));
            offset[1] = -(hdr.dmin * byte_as_float<B + 1>(hdr.mn[P / 2]));
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // (low, high nibbles) x (first, second eight columns of the lane's sixteen)
            const int hi = g / 2, ff = g % 2;
            if (g == 3) {
                // The activations of the next step were requested two steps ago; younger are those of the step after it and, at P == 1 and
                // 2, the next super-block's weights and sums.
                lds_barrier_after_loads<kSlabPieces + (P == 1 || P == 2 ? kHead : 0)>();
            }
            f16x8 w;
            if constexpr (EXACT) {
                w = hi ? scaled8_q4_swapped<1>(raw[P][2 * ff], raw[P][2 * ff + 1], f16x2{ps[1], ps[1]}, masks)
                       : scaled8_q4_swapped<0>(raw[P][2 * ff], raw[P][2 * ff + 1], f16x2{ps[0], ps[0]}, masks);
            } else {
                w = weights8_q4_swapped(raw[P][2 * ff], raw[P][2 * ff + 1], hi ? rounded_masks.hi : rounded_masks.lo, scale[hi], offset[hi]);
            }
            if (g == 3 && P == 3) read_header(b + 1);
            uint32_t from = a_at[(g + 1) % 4] + (g < 3 ? slot_now : slot_next);
            asm volatile("" : "+v"(from));
            auto row_tile = [&]<int I>(std::integral_constant<int, I>) {
                constexpr int i = I;
                if constexpr (EXACT) {
                    const f32x16 zero{};
                    blk[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], w, P == 0 && g == 0 ? zero : blk[i], 0, 0, 0);
                } else {
                    acc[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i], w, acc[i], 0, 0, 0);
                }
                af[i] = *reinterpret_cast<const f16x8*>(lds_raw + from + i * 4096);
                // the step's requests one at a time between the MFMAs: a wave whose request finds the address unit busy stands still
                if (g == 3) {
                    constexpr int kEach = (kSlabPieces + RT - 1) / RT;
                    [&]<int... I2>(std::integer_sequence<int, I2...>) {
                        ([&] { if constexpr (I * kEach + I2 < kSlabPieces) request_a(a_from, slot_now, std::integral_constant<int, I * kEach + I2>{}); }(), ...);
                    }(std::make_integer_sequence<int, kEach>{});
                }
            };
            [&]<int... I>(std::integer_sequence<int, I...>) { (row_tile(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, RT>{});
            if (P == 1 && g < 3) {
                constexpr int kEach = (kHead + 2) / 3;
                auto some = [&]<int G>(std::integral_constant<int, G>) {
                    [&]<int... I>(std::integer_sequence<int, I...>) {
                        ([&] { if constexpr (G * kEach + I < kHead) request_w(w_next, sx_next, b + 1, std::integral_constant<int, G * kEach + I>{}); }(), ...);
                    }(std::make_integer_sequence<int, kEach>{});
                };
                if (g == 0) some(std::integral_constant<int, 0>{});
                if (g == 1) some(std::integral_constant<int, 1>{});
                if (g == 2) some(std::integral_constant<int, 2>{});
            }
        }
        const uint32_t freed = slot_now;
        slot_now = slot_next; slot_next = slot_last; slot_last = freed;
        // A wave issues in order: one MFMA, then a few vector instructions and an LDS read, so that the unpacking runs behind the MFMAs
#pragma unroll
        for (int k = 0; k < 4 * RT; ++k) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x002, RT >= 8 ? 2 : RT >= 4 ? (EXACT ? 2 : 4) : 5, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        if constexpr (EXACT && P == 3) {
            // acc += d * blk - dmin * sum_s Sx(hi + lo)[m, s] * mn[n, s]
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const f16x8 sf = *reinterpret_cast<const f16x8*>(lds_raw + sx_at + (b % 2) * kSxBytes + i * 1024);
                const f32x16 zero{};
                const f32x16 low = __builtin_amdgcn_mfma_f32_32x32x16_f16(sf, minima, zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 16; ++v) acc[i][v] = __builtin_fmaf(-fold_dmin, low[v], __builtin_fmaf(fold_d, blk[i][v], acc[i][v]));
            }
        }
    };
    using std::integral_constant;
    {
        const uint8_t* const a0 = a_block(0);
        [&]<int... I>(std::integer_sequence<int, I...>) { (request_w(w_block(0), sx_block(0), 0, integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, kHead>{});
        [&]<int... I>(std::integer_sequence<int, I...>) {
            (request_a(a0, 0, integral_constant<int, I>{}), ...);
            (request_a(a0 + 128, kSlabBytes, integral_constant<int, I>{}), ...);
            (request_a(a0 + 256, 2 * kSlabBytes, integral_constant<int, I>{}), ...);
        }(std::make_integer_sequence<int, kSlabPieces>{});
    }
    lds_barrier_after_loads<2 * kSlabPieces>();  // weights, sums and activations of step 0
    read_header(0);
#pragma unroll
    for (int i = 0; i < RT; ++i) af[i] = *reinterpret_cast<const f16x8*>(lds_raw + a_at[0] + i * 4096);
    for (uint32_t b = 0; b < count; ++b) {
        const uint8_t* const a_now = a_block(b);
        const uint8_t* const a_next = a_block(b + 1);
        const uint8_t* const w_next = w_block(b + 1);
        const uint8_t* const sx_next = EXACT ? sx_block(b + 1) : nullptr;
        step_fn(b, a_now, a_next, w_next, sx_next, integral_constant<int, 0>{});
        step_fn(b, a_now, a_next, w_next, sx_next, integral_constant<int, 1>{});
        step_fn(b, a_now, a_next, w_next, sx_next, integral_constant<int, 2>{});
        step_fn(b, a_now, a_next, w_next, sx_next, integral_constant<int, 3>{});
    }
    wait_all_loads();
    // ---- epilogue. Accumulator v of tile (i, j): row 32 i + 8 (v / 4) + 4 khalf + v % 4 of the wave's rows, weight row col of column tile j
    uint32_t biggest = 0;  // the largest result's bits without the sign: anything not finite shows at the end
    const uint32_t wave_m0 = m0 + wm * (RT * 32) + group * (kOwn * 32), wave_n0 = n0 + wn * 32;
    const bool whole = wave_n0 + 32 <= a.n && reinterpret_cast<uintptr_t>(a.out) % 16 == 0 && a.out_stride % 16 == 0;  // uniform
    __syncthreads();  // every wave has left the rings, and every request into them has landed: the LDS is the epilogue's
    if constexpr (GROUPS > 1) {
        // group g stores row tiles g * kOwn .. of the tile: every group leaves the others' parts in LDS, and the parts of a result
        // are added in the order of the columns, its own among them
        constexpr int kPart = kOwn * 16;  // floats of a lane in one group's share
        static_assert(GROUPS * kShares * kThreadsT * kPart * 4 <= S::kLds);
        float* const parts = reinterpret_cast<float*>(lds_all);  // [group][share][wave][kPart / 4][lane][4]
        auto at = [&](uint32_t from, uint32_t share, int piece) { return parts + (((from * kShares + share) * kGroupWaves + wave) * kPart + piece * 4) * kWave + lane * 4; };
#pragma unroll
        for (int i = 0; i < RT; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q)
                *reinterpret_cast<f32x4*>(at(group, i / kOwn, i % kOwn * 4 + q)) = f32x4{acc[i][4 * q], acc[i][4 * q + 1], acc[i][4 * q + 2], acc[i][4 * q + 3]};
        __syncthreads();
        if (kShares == GROUPS || group < kShares)
#pragma unroll
        for (int i = 0; i < kOwn; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                f32x4 sum = *reinterpret_cast<const f32x4*>(at(0, group, i * 4 + q));
#pragma unroll
                for (int g = 1; g < GROUPS; ++g) sum += *reinterpret_cast<const f32x4*>(at(g, group, i * 4 + q));
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][4 * q + e] = sum[e];
            }
        __syncthreads();
        if (kShares < GROUPS && group >= kShares) return;
    }
    if (whole) {
        // The wave's results go out as whole 16-byte pieces, neighbouring lanes along a row, after a turn through LDS that the
        // wave has to itself (16 or 18 KB: a few row tiles at a time; a row pitch of 16 bytes
        // more than the row keeps the column-wise writes and the row-wise reads off each other's banks). A lane storing
        // its own 2- or 4-byte results one by one, 128 stores, took a fifth of the kernel's time.
        uint8_t* const mine = lds_all + (group * kGroupWaves + wave) * kRegion;
        static_assert(WAVES * kRegion <= S::kLds);
        // four row tiles at a time as bf16, two as f32 (with two column tiles per wave; twice that with four, and four and two with one),
        // or as many as there are
        constexpr int kTilesB = std::min(kOwn, 4), kTilesF = std::min(kOwn, 2);
        auto pass = [&](auto bf16_tag, auto first_tag) {
            constexpr bool BF16 = decltype(bf16_tag)::value;
            constexpr int first_tile = decltype(first_tag)::value;
            constexpr int kTiles = BF16 ? kTilesB : kTilesF, kElem = BF16 ? 2 : 4, kPitch = 32 * kElem + 16;
            static_assert(kTiles * 32 * kPitch <= kRegion && first_tile + kTiles <= kOwn);
#pragma unroll
            for (int t = 0; t < kTiles; ++t) {
                const int i = first_tile + t;
#pragma unroll
                for (int v = 0; v < 16; ++v) {
                    const uint32_t r = t * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
                    const float val = acc[i][v];
                    const uint32_t vb = __float_as_uint(val), magnitude = vb & 0x7fffffffu;
                    biggest = biggest > magnitude ? biggest : magnitude;
                    uint8_t* at = mine + r * kPitch + col * kElem;
                    if constexpr (BF16) *reinterpret_cast<uint16_t*>(at) = uint16_t((vb + 0x7fffu + ((vb >> 16) & 1u)) >> 16);
                    else *reinterpret_cast<float*>(at) = val;
                }
            }
            // written and read back by this wave only: LDS serves a wave's requests in order
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            constexpr int kPieces = 32 * kElem / 16;                    // 16-byte pieces per row
            constexpr int kRounds = kTiles * 32 * kPieces / kWave;      // pieces per lane
#pragma unroll
            for (int q = 0; q < kRounds; ++q) {
                const uint32_t c = q * kWave + lane, r = c / kPieces, piece = c % kPieces;
                const uint4 data = *reinterpret_cast<const uint4*>(mine + r * kPitch + piece * 16);
                const uint32_t row = wave_m0 + first_tile * 32 + r;
                if (row < a.m)
                    *reinterpret_cast<uint4*>(static_cast<uint8_t*>(a.out) + uint64_t(row) * a.out_stride + uint64_t(wave_n0) * kElem + piece * 16) = data;
            }
            __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
        };
        auto passes = [&]<int... I>(auto bf16_tag, std::integer_sequence<int, I...>) {
            (pass(bf16_tag, std::integral_constant<int, I * (decltype(bf16_tag)::value ? kTilesB : kTilesF)>{}), ...);
        };
        if (a.out_bf16) passes(std::true_type{}, std::make_integer_sequence<int, kOwn / kTilesB>{});
        else passes(std::false_type{}, std::make_integer_sequence<int, kOwn / kTilesF>{});
    } else {
        // a ragged column tile or rows that 16 bytes do not align: element by element
#pragma unroll
        for (int i = 0; i < kOwn; ++i) {
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t row = wave_m0 + i * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
                if (row >= a.m) continue;
                uint8_t* orow = static_cast<uint8_t*>(a.out) + uint64_t(row) * a.out_stride;
                const uint32_t n = wave_n0 + col;
                if (n >= a.n) continue;
                const float val = acc[i][v];
                const uint32_t vb = __float_as_uint(val), magnitude = vb & 0x7fffffffu;
                biggest = biggest > magnitude ? biggest : magnitude;
                if (a.out_bf16) reinterpret_cast<uint16_t*>(orow)[n] = uint16_t((vb + 0x7fffu + ((vb >> 16) & 1u)) >> 16);
                else reinterpret_cast<float*>(orow)[n] = val;
            }
        }
    }
    publish_error(biggest >= 0x7f800000u ? uint32_t(TSP_ERRBIT_NONFINITE) : 0u, a.error_word);
}

template <int RT, int WAVES, int TN, int GROUPS, bool EXACT>
int launch(DenseTileArgs a, hipStream_t s) {
    using S = Shape<RT, WAVES, TN, GROUPS, EXACT>;
    if constexpr (S::kAtLaunch) {
        static std::atomic<uint64_t> raised{0};
        int device = 0;
        if (setup_pending(raised, &device)) {
            TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&dense_tile_kernel<RT, WAVES, TN, GROUPS, EXACT>), hipFuncAttributeMaxDynamicSharedMemorySize, S::kLds));
            setup_done(raised, device);
        }
    }
    constexpr uint32_t TM = WAVES / GROUPS / (TN / 32) * RT * 32;
    const uint32_t m_tiles = (a.m + TM - 1) / TM, n_tiles = (a.n + TN - 1) / TN, tiles = m_tiles * n_tiles;
    a.band = dense_band(m_tiles, n_tiles, TM, TN);
    TSP_LAUNCH("gemm_dense_tile", s, (dense_tile_kernel<RT, WAVES, TN, GROUPS, EXACT><<<(tiles + 7) / 8 * 8, WAVES * 64, S::kAtLaunch ? S::kLds : 0, s>>>(a)));
    return launch_status("dense_tile");
}

}  // namespace

namespace tsp {

int launch_dense_tile(const DenseTileArgs& a, hipStream_t s) {
    auto tiles = [&](uint64_t high, uint64_t wide) { return (a.m + high - 1) / high * ((a.n + wide - 1) / wide); };
    if (dense_exact(a.m, a.n)) {
        // Few tiles are dense_fragments.hip's.
        if (a.m <= 32) return launch<1, 4, 64, 2, true>(a, s);
        // 64 x 64 tiles while the chip takes them all at once, two to a compute unit: 13 to 24 us at 2560 columns, 41 for twice as many,
        // where 128 x 128 tiles take 34.
        if (tiles(64, 64) <= 512) return launch<2, 4, 64, 2, true>(a, s);
        return launch<4, 8, 128, 2, true>(a, s);
    }
    // The shape whose rounds over the chip end first, a round of each as measured at 2048 columns, in us: two 64 x 64 tiles per
    // compute unit, or one 128 x 128, 128 x 256 or 256 x 256 tile.
    const uint64_t cost[4] = {(tiles(64, 64) + 511) / 512 * 17, (tiles(128, 128) + 255) / 256 * 25, (tiles(128, 256) + 255) / 256 * 39,
                              (tiles(256, 256) + 255) / 256 * 62};
    switch (std::min_element(cost, cost + 4) - cost) {
        case 0: return launch<2, 4, 64, 2, false>(a, s);
        case 1: return launch<4, 8, 128, 2, false>(a, s);
        case 2: return launch<4, 8, 256, 1, false>(a, s);
        default: return launch<8, 8, 256, 1, false>(a, s);
    }
}

}  // namespace tsp
