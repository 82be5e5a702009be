// Dense Q8_0 GEMM for many token rows (the shared expert of a prefill chunk): out[t, n] = sum_k x[t, k] * d[n, k/32] * q[n, k].
//
// The streaming kernels of q8.hip / q8_mfma.hip read the whole matrix once per 8 or 16 token rows: right for decode,
// hundreds of passes for a 2048-token chunk. Here a weight is the half nearest d * q (11 significant bits, what the engine's own
// kernel stages, include/tokspur/graph.hpp:860 and kernels/grouped_mm.metal:239-243), the token rows are rounded to halves as
// well, and the matrix cores multiply the two with f32 accumulation.
//
// GGUF rows whose tiles go round the chip well are decoded on their way into the MFMAs, together with the token rows (q8_gemm_fused). Else every operand would be
// decoded too often or much of the chip stand idle: one launch decodes both into the workspace and f16_gemm_nt multiplies them.
//
// f16_gemm_nt: a workgroup of four waves owns a 64 x 64 output tile (each wave a 32 x 32 MFMA tile) and walks K in
// steps of 64 halfs. Every byte travels global -> LDS directly (16 bytes per lane, no registers in between) into a ring
// of four stages, three steps ahead of the multiply; chunk c of row r of a slab sits at position r * 8 + (c ^ (r / 2 % 8)),
// which the loads fill linearly by lane and sixteen consecutive lanes of the fragment reads find in all banks. No other vector-memory operation
// exists in the loop, so the wait before a step's barrier is simply "all but the two younger stages have landed". Bound by the way from
// L2 into LDS: 210 MB in 18 us at 2048 tokens, 2560 columns, 640 rows. Tiles of an XCD side by side, its fragments read ahead: a call with its
// conversion 31.0 -> 27.3 us there, 24.6 -> 24.2 at 640 columns x 2560 rows, 20.0 -> 19.2 at 2048 x 512 (128 x 64 tiles 27.1, 26.0 and 21.5,
// 128 x 128 33.7, 26.7 and 27.9: half and a quarter of the compute units without a tile).
#include "mfma_quant.hpp"

using namespace tsp;

namespace {

constexpr int kTile = 64, kStep = 64;                  // output tile edge; halfs of K per step (128 B per row)
constexpr int kSlabBytes = kTile * kStep * 2;          // 8 KB: 64 rows x 128 B
constexpr int kStageBytes = 2 * kSlabBytes;            // token slab, weight slab
constexpr int kRing = 4;

struct F16GemmArgs {
    const _Float16* x;  // [m][k]
    const _Float16* w;  // [n][k]
    float* out;         // rows out_stride bytes apart
    uint64_t out_stride;
    uint32_t m, n, k;
    uint32_t* error_word;
};

struct Q8GemmArgs {
    const float* x;  // rows x_stride bytes apart
    uint64_t x_stride;
    const uint8_t* w;  // [n][k / 32 blocks of 34 B]
    float* out;        // rows out_stride bytes apart
    uint64_t out_stride;
    uint32_t m, n, k;
    uint32_t* error_word;
};

__global__ __launch_bounds__(256, 2) void f16_gemm_nt(F16GemmArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kRing * kStageBytes];  // 64 KB: two workgroups per CU
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const uint32_t col = lane % 32, khalf = lane / 32;
    // an XCD (workgroup id % 8) takes a run of tiles and with it an eighth of the larger operand and all of the smaller one into its L2
    const uint32_t n_tiles = (a.n + kTile - 1) / kTile, m_tiles = (a.m + kTile - 1) / kTile, tiles = n_tiles * m_tiles, per_xcd = (tiles + 7) / 8;
    const uint32_t tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || tile >= tiles) return;
    const bool tall = a.m >= a.n;
    const uint32_t m0 = (tall ? tile / n_tiles : tile % m_tiles) * kTile, n0 = (tall ? tile % n_tiles : tile / m_tiles) * kTile;
    const uint32_t steps = a.k / kStep;

    // piece p = i * 256 + tid of a stage (1024 pieces of 16 bytes): slab p / 512, LDS position q = p % 512 -> row q / 8,
    // chunk (q % 8) ^ (row / 2 % 8). Rows past the matrix re-read its last row (never stored).
    const uint8_t* src[4];
    uint32_t lds_at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t p = i * 256 + tid, slab = p / 512, q = p % 512, r = q / 8, c = (q % 8) ^ (r / 2 % 8);
        uint32_t row = (slab ? n0 : m0) + r;
        const uint32_t limit = slab ? a.n : a.m;
        row = row < limit ? row : limit - 1;
        src[i] = reinterpret_cast<const uint8_t*>(slab ? a.w : a.x) + (uint64_t(row) * a.k + c * 8) * 2;
        lds_at[i] = __builtin_amdgcn_readfirstlane(lds_address(lds) + (i * 256 + wave * kWave) * 16);  // lane 0 of this wave; the hardware adds 16 * lane
    }
    auto request = [&](uint32_t step, uint32_t slot) {  // steps past the end re-read the last one into a slot nobody reads
        const uint32_t s = step < steps ? step : steps - 1;
#pragma unroll
        for (int i = 0; i < 4; ++i) load_to_lds_16(src[i] + uint64_t(s) * kStep * 2, lds_at[i] + slot * kStageBytes);
    };

    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.0f;
    // chunk 2 kc + khalf of the wave's row
    const uint32_t at = col * 128 + ((khalf ^ (col / 2 % 8)) * 16), x_at = (wave / 2) * 4096 + at, w_at = kSlabBytes + (wave % 2) * 4096 + at;
    request(0, 0);
    request(1, 1);
    request(2, 2);
    for (uint32_t s = 0; s < steps; ++s) {
        const uint32_t slot = s % kRing;
        lds_barrier_after_loads<8>();  // stage s has landed (the two younger stages may be on their way); every wave has left slot (s + 3) % 4
        // every fragment is read before the first product: a read right before its product is its latency four times a step
        f16x8 fa[4], fb[4];
        auto read = [&](uint32_t kc) {
            fa[kc] = *reinterpret_cast<const f16x8*>(lds + slot * kStageBytes + (x_at ^ (kc * 32)));
            fb[kc] = *reinterpret_cast<const f16x8*>(lds + slot * kStageBytes + (w_at ^ (kc * 32)));
        };
        read(0);
        read(1);
        request(s + 3, (s + 3) % kRing);
        read(2);
        read(3);
#pragma unroll
        for (int kc = 0; kc < 4; ++kc) acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[kc], fb[kc], acc, 0, 0, 0);
    }
    wait_all_loads();  // the last requests land in slots nobody reads: they must be done before this LDS is given away

    // accumulator v: token row 8 * (v / 4) + 4 * khalf + v % 4 of the wave's tile, weight row `col`
    uint32_t bad = 0;
    const uint32_t n = n0 + (wave % 2) * 32 + col;
#pragma unroll
    for (int v = 0; v < 16; ++v) {
        const uint32_t m = m0 + (wave / 2) * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
        if (m < a.m && n < a.n) {
            if (nonfinite(acc[v])) bad = TSP_ERRBIT_NONFINITE;
            reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.out) + uint64_t(m) * a.out_stride)[n] = acc[v];
        }
    }
    publish_error(bad, a.error_word);
}

using four_floats = f32x4 __attribute__((aligned(4)));
using four_quants = uint32_t __attribute__((aligned(2)));  // rows and blocks are even byte counts

// GGUF rows and a tile to nearly every compute unit: a workgroup of eight waves owns an MT x NT output tile and takes 128 columns a step. A thread reads eight
// columns of each 32nd row as they lie (32 bytes of a token row, eight quants and their scale of a matrix row), rounds them to halves and puts them into
// LDS, DEPTH steps' requests in registers; the waves multiply from there, WM x WN of them side by side and every such group a share of
// the step's columns, whose sums meet in LDS in the groups' order. Chunk c (16 bytes) of row r sits at position c ^ (r % 16) of the
// row's 256 bytes: sixteen consecutive lanes touch every bank once, writing and reading. Fragments are requested from LDS before the next step's
// operands are rounded, and multiplied after that.
// Bound by what a compute unit fetches, some 30 bytes a cycle whether the rest of the chip has work or not (a tile alone takes as long as 256; steps further ahead
// and a step's rounding beside its products gain nothing). Against the 32 x 32 tiles whose waves took 64 columns in turns, or above 600 of them the two launches below, per call, tokens x
// columns -> rows, operands from memory: 203 x 2560 -> 640 11.2 -> 10.3 us, 600 19.6 -> 15.3, 800 20.4 -> 14.8; 1000 x 2048 -> 512 17.3 -> 12.4, 2048 19.5 -> 18.6; 800 x 1024 ->
// 512 10.5 -> 8.1; 203 x 640 -> 2560 8.7 -> 8.1; 2048 x 768 -> 2048 23.9 -> 22.1. Tried: token rows sixteen bytes to a lane and sixteen quants to a load (2048 x 2560 -> 640 27 for
// 23), operands straight into LDS of the wave that multiplies them (24), the matrix in fragment order by a launch before (22, but 32 for 24.9 at 640 x 2560).
template <int MT, int NT, int WM, int WN, int DEPTH, int WAVES_PER_SIMD>
struct FusedShape {
    static constexpr int kM = MT, kN = NT, kDepth = DEPTH, kRowTiles = MT / 32 / WM, kColumnTiles = NT / 32 / WN, kGroups = 8 / (WM * WN), kPasses = kRowTiles * kColumnTiles;
    static constexpr uint32_t kStage = (MT + NT) * 256, kLds = 2 * kStage > (kPasses > 1 ? 65536u : 32768u) ? 2 * kStage : (kPasses > 1 ? 65536u : 32768u);
    static constexpr int kWavesM = WM, kWavesN = WN, kWavesPerSimd = WAVES_PER_SIMD;
    static_assert(kRowTiles * WM * 32 == MT && kColumnTiles * WN * 32 == NT && kGroups * WM * WN == 8);
};

template <class S>
__global__ __launch_bounds__(512, S::kWavesPerSimd) void q8_gemm_fused(Q8GemmArgs a) {
    constexpr uint32_t MT = S::kM, NT = S::kN, XR = MT / 32, WR = NT / 32, TILES = S::kWavesM * S::kWavesN;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid / kWave)));
    // an XCD (workgroup id % 8) takes a run of tiles and with it an eighth of the larger operand and all of the smaller one into its L2
    const uint32_t n_tiles = (a.n + NT - 1) / NT, m_tiles = (a.m + MT - 1) / MT, tiles = n_tiles * m_tiles, per_xcd = (tiles + 7) / 8;
    const uint32_t tile = (blockIdx.x % 8) * per_xcd + blockIdx.x / 8;
    if (blockIdx.x / 8 >= per_xcd || tile >= tiles) return;
    const bool tall = a.m >= a.n;
    const uint32_t m0 = (tall ? tile / n_tiles : tile % m_tiles) * MT, n0 = (tall ? tile % n_tiles : tile / m_tiles) * NT;
    const uint32_t steps = (a.k + 127) / 128, row_bytes = a.k / 32 * 34;

    const uint32_t row = tid / 16, chunk = tid % 16;
    const uint8_t* x_from[XR];
    const uint8_t* w_from[WR];
#pragma unroll
    for (uint32_t i = 0; i < XR; ++i) {  // rows past the matrix re-read its last row (never stored)
        const uint32_t r = m0 + row + 32 * i;
        x_from[i] = reinterpret_cast<const uint8_t*>(a.x) + (r < a.m ? r : a.m - 1) * a.x_stride;
    }
#pragma unroll
    for (uint32_t i = 0; i < WR; ++i) {
        const uint32_t r = n0 + row + 32 * i;
        w_from[i] = a.w + uint64_t(r < a.n ? r : a.n - 1) * row_bytes;
    }
    struct Step { f32x4 x[XR][2]; uint32_t q[WR][2]; uint32_t d[WR]; };
    auto fetch = [&](uint32_t s, Step& t) {
        const uint32_t wanted = s * 128 + chunk * 8, column = wanted < a.k ? wanted : chunk * 8 % 64;  // every request unconditional: past the end some others, unused
        const uint32_t x_at = column * 4, d_at = column / 32 * 34, q_at = d_at + 2 + column % 32;
#pragma unroll
        for (uint32_t i = 0; i < XR; ++i) {
            const four_floats* const from = reinterpret_cast<const four_floats*>(x_from[i] + x_at);
            t.x[i][0] = from[0]; t.x[i][1] = from[1];
        }
#pragma unroll
        for (uint32_t i = 0; i < WR; ++i) {
            const four_quants* const from = reinterpret_cast<const four_quants*>(w_from[i] + q_at);
            t.q[i][0] = from[0]; t.q[i][1] = from[1];
            t.d[i] = *reinterpret_cast<const uint16_t*>(w_from[i] + d_at);
        }
    };
    const uint32_t put_at = row * 256 + ((chunk ^ (row % 16)) * 16);
    auto put = [&](uint32_t s, const Step& t) {
        uint8_t* const to = lds + (s % 2) * S::kStage + put_at;
#pragma unroll
        for (uint32_t i = 0; i < XR; ++i) {
            f16x8 h;
#pragma unroll
            for (int e = 0; e < 8; ++e) h[e] = _Float16(t.x[i][e / 4][e % 4]);
            *reinterpret_cast<f16x8*>(to + i * 8192) = h;
        }
#pragma unroll
        for (uint32_t i = 0; i < WR; ++i) {
            const f16x2 d2 = as_h2(t.d[i] | t.d[i] << 16);
            const f16x8 c = quants8(t.q[i][0], t.q[i][1]);  // exact, as is d: one packed multiply rounds once
            const f16x2 p0 = f16x2{c[0], c[1]} * d2, p1 = f16x2{c[2], c[3]} * d2, p2 = f16x2{c[4], c[5]} * d2, p3 = f16x2{c[6], c[7]} * d2;
            *reinterpret_cast<f16x8*>(to + MT * 256 + i * 8192) = f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
        }
        if (s * 128 + chunk * 8 >= a.k) {  // past the end
#pragma unroll
            for (uint32_t i = 0; i < XR + WR; ++i) *reinterpret_cast<u32x4*>(to + i * 8192) = u32x4{};
        }
    };
    const uint32_t group = wave / TILES, wm = wave % TILES / S::kWavesN, wn = wave % S::kWavesN, col = lane % 32, khalf = lane / 32;
    const uint32_t at = col * 256 + ((khalf ^ (col % 16)) * 16), xs = wm * (S::kRowTiles * 8192) + at, ws = MT * 256 + wn * (S::kColumnTiles * 8192) + at;
    f32x16 acc[S::kRowTiles][S::kColumnTiles] = {};
    constexpr uint32_t kSlices = 8 / S::kGroups;  // of sixteen columns
    struct Fragments { f16x8 x[kSlices][S::kRowTiles], w[kSlices][S::kColumnTiles]; };
    auto read = [&](uint32_t s, Fragments& f) {
        const uint8_t* const from = lds + (s % 2) * S::kStage;
#pragma unroll
        for (uint32_t j = 0; j < kSlices; ++j) {
            const uint32_t k = (group * kSlices + j) * 32;
#pragma unroll
            for (int i = 0; i < S::kRowTiles; ++i) f.x[j][i] = *reinterpret_cast<const f16x8*>(from + (xs ^ k) + i * 8192);
#pragma unroll
            for (int i = 0; i < S::kColumnTiles; ++i) f.w[j][i] = *reinterpret_cast<const f16x8*>(from + (ws ^ k) + i * 8192);
        }
    };
    auto multiply = [&](const Fragments& f) {
#pragma unroll
        for (uint32_t j = 0; j < kSlices; ++j)
#pragma unroll
            for (int i = 0; i < S::kRowTiles; ++i)
#pragma unroll
                for (int c = 0; c < S::kColumnTiles; ++c) acc[i][c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(f.x[j][i], f.w[j][c], acc[i][c], 0, 0, 0);
    };
    Step t[S::kDepth];
#pragma unroll
    for (uint32_t d = 0; d < S::kDepth; ++d) fetch(d, t[d]);
    put(0, t[0]);
    fetch(S::kDepth, t[0]);
    lds_barrier();
    for (uint32_t s0 = 0; s0 < steps; s0 += S::kDepth) {
#pragma unroll
        for (uint32_t d = 0; d < S::kDepth; ++d) {  // steps past the end are zeros
            const uint32_t s = s0 + d;
            Step& next = t[(d + 1) % S::kDepth];
            Fragments f;
            read(s, f);
            __builtin_amdgcn_sched_barrier(0);
            put(s + 1, next);  // while the fragments are on their way
            fetch(s + 1 + S::kDepth, next);
            __builtin_amdgcn_sched_barrier(0);
            multiply(f);
            lds_barrier();
        }
    }
    // the groups' sums, added in their order: a 32 x 32 tile of every wave at a time, the next one's beside it in LDS
    uint32_t bad = 0;  // a token's value that is no finite half makes its whole row so
    f32x4* const sums = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int p = 0; p < S::kPasses; ++p) {
        const f32x16& mine = acc[p / S::kColumnTiles][p % S::kColumnTiles];
        f32x4* const at_pass = sums + (p % 2) * 2048;
#pragma unroll
        for (int b = 0; b < 4; ++b) at_pass[(wave * 4 + b) * 64 + lane] = f32x4{mine[4 * b], mine[4 * b + 1], mine[4 * b + 2], mine[4 * b + 3]};
        lds_barrier();
        // quad b of lane l: token rows 8 b + 4 (l / 32) + 0 .. 3 of the tile, weight row l % 32
#pragma unroll
        for (uint32_t q = tid; q < TILES * 256; q += 512) {
            const uint32_t which = q / 256, b = q / 64 % 4;
            f32x4 value = at_pass[(which * 4 + b) * 64 + lane];
#pragma unroll
            for (uint32_t g = 1; g < S::kGroups; ++g) value += at_pass[((g * TILES + which) * 4 + b) * 64 + lane];
            const uint32_t n = n0 + ((which % S::kWavesN) * S::kColumnTiles + p % S::kColumnTiles) * 32 + col;
            const uint32_t m = m0 + ((which / S::kWavesN) * S::kRowTiles + p / S::kColumnTiles) * 32 + 8 * b + 4 * khalf;
#pragma unroll
            for (uint32_t r = 0; r < 4; ++r)
                if (m + r < a.m && n < a.n) {
                    if (nonfinite(value[r])) bad = TSP_ERRBIT_NONFINITE;
                    reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.out) + (m + r) * a.out_stride)[n] = value[r];
                }
        }
    }
    publish_error(bad, a.error_word);
}

// Both operands to halves in one launch (two small ones cost more than their work): the first `rows` rows of the grid are the matrix's, the others
// the token rows. Workgroup (x, y): rows 4 x .. 4 x + 3, one to a wave, columns 512 y on, eight to a lane, with no division left to the lanes.
// GGUF rows are 34-byte blocks (f16 d, 32 int8); q8_lanes_v1 rows keep the scales first, then runs of 16 blocks with byte = index * width +
// block % 16 (src/expert_lanes.cpp:60-119). A token's value that does not fit a half (or is not finite) raises the non-finite bit.
// Bound by memory from some 1000 rows on, below by a trip there. A flat index divided by the row's length in 64 bits, element-wise loads and sixteen weights
// to a lane before: 2048 x 2560 with 640 matrix rows 9.6 -> 8.2 us, 2048 x 2048 with 512 8.8 -> 7.9, 2048 x 512 with 1024 4.4 -> 4.0.
struct OperandsArgs {
    const uint8_t* matrix;
    const float* x;
    uint64_t x_stride;  // bytes
    _Float16 *w16, *x16;
    uint32_t layout, columns, rows, tokens;
    uint32_t* error_word;
};
__global__ __launch_bounds__(256) void q8_operands_to_f16(OperandsArgs a) {
    const uint32_t lane = threadIdx.x % kWave, row = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), c8 = blockIdx.y * kWave + lane;
    if (row >= a.rows + a.tokens || c8 * 8 >= a.columns) return;
    f16x8 h;
    if (row < a.rows) {
        const uint32_t blocks = a.columns / 32, block = c8 / 4, index = c8 % 4 * 8;
        const uint8_t* const data = a.matrix + uint64_t(row) * blocks * 34;
        float d;
        uint32_t q[2];
        if (a.layout == TSP_LAYOUT_GGUF) {
            const uint8_t* const b = data + block * 34;
            d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(b));
            const four_quants* const from = reinterpret_cast<const four_quants*>(b + 2 + index);
            q[0] = from[0]; q[1] = from[1];
        } else {
            const uint32_t run = block / 16, width = blocks - run * 16 < 16 ? blocks - run * 16 : 16;
            const uint8_t* const from = data + blocks * 2 + run * 512 + block % 16 + index * width;
            d = half_bits_to_float(uint32_t(data[block * 2]) | (uint32_t(data[block * 2 + 1]) << 8));
            q[0] = q[1] = 0;
#pragma unroll
            for (int i = 0; i < 8; ++i) q[i / 4] |= uint32_t(from[i * width]) << (i % 4 * 8);
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = _Float16(d * float(int8_t(q[e / 4] >> (e % 4 * 8))));  // d * q is exact in f32: one rounding
        *reinterpret_cast<f16x8*>(a.w16 + uint64_t(row) * a.columns + c8 * 8) = h;
        return;
    }
    const uint32_t token = row - a.rows;
    const four_floats* const from = reinterpret_cast<const four_floats*>(reinterpret_cast<const uint8_t*>(a.x) + token * a.x_stride + c8 * 32);
    const f32x4 v0 = from[0], v1 = from[1];
    uint32_t bad = 0;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        h[e] = _Float16(e < 4 ? v0[e % 4] : v1[e % 4]);
        if ((__builtin_bit_cast(uint16_t, _Float16(h[e])) & 0x7c00u) == 0x7c00u) bad = TSP_ERRBIT_NONFINITE;
    }
    *reinterpret_cast<f16x8*>(a.x16 + uint64_t(token) * a.columns + c8 * 8) = h;
    publish_error(bad, a.error_word);
}

uint64_t align256(uint64_t v) { return (v + 255) / 256 * 256; }

template <class S>
int launch_fused(const Q8GemmArgs& a, const char* name, hipStream_t s) {
    if constexpr (S::kLds > 65536) {
        static std::atomic<uint64_t> raised{0};
        int device = 0;
        if (setup_pending(raised, &device)) {
            TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_gemm_fused<S>), hipFuncAttributeMaxDynamicSharedMemorySize, int(S::kLds)));
            setup_done(raised, device);
        }
    }
    const uint64_t tiles = uint64_t((a.m + S::kM - 1) / S::kM) * ((a.n + S::kN - 1) / S::kN);
    TSP_LAUNCH(name, s, q8_gemm_fused<S><<<uint32_t((tiles + 7) / 8 * 8), 512, S::kLds, s>>>(a));
    return launch_status("q8_gemm_fused");
}

// Which tile, or none for the two launches: the one whose time, as measured, is shortest. A round of 256 workgroups, one to a compute unit, takes so
// long for each 128 columns and so long to begin and end, between operands that a call before has read and operands from memory (20 steps of 2560 columns,
// us: 32 x 32 8.5 and 11.6, 32 x 64 12.9 and 15.2, 64 x 64 16.4 and 21.5, 64 x 96 23.2 and 27.2, 128 x 128 39 and 48); rounds follow each other, so a tile that just fills
// one is the best. The two launches take 570 ns a step for each round of 64 x 64 tiles, which share the compute units evenly, and the conversion's bytes at
// 5 TB/s; what they read from memory they read once and in long runs, so they keep calls that would gain less than a tenth: 2048 x 2560 -> 640 23.1 and 25.8
// where 64 x 96 takes 22.3 and 27.2, 1000 x 2560 -> 640 18.4 and 19.8 where 64 x 64 takes 17.6 and 21.7, 2048 x 640 -> 2560 24.9 and 26.3 where 128 x 128 takes 31 and 32.9.
struct FusedTile {
    uint32_t m, n, step_ns, ends_ns;
    const char* name;  // in a profile window
    int (*launch)(const Q8GemmArgs&, const char*, hipStream_t);
};
const FusedTile* fused_tile(uint32_t m, uint32_t n, uint32_t k) {
    static constexpr FusedTile choices[] = {{32, 32, 370, 2500, "q8_gemm_fused 32x32", launch_fused<FusedShape<32, 32, 1, 1, 2, 2>>},
                                            {32, 64, 545, 3000, "q8_gemm_fused 32x64", launch_fused<FusedShape<32, 64, 1, 2, 2, 2>>},
                                            {64, 64, 760, 3850, "q8_gemm_fused 64x64", launch_fused<FusedShape<64, 64, 2, 1, 1, 4>>},
                                            {64, 96, 980, 5100, "q8_gemm_fused 64x96", launch_fused<FusedShape<64, 96, 2, 1, 2, 2>>},
                                            {128, 128, 1875, 7500, "q8_gemm_fused 128x128", launch_fused<FusedShape<128, 128, 2, 2, 1, 2>>}};
    const auto tiles = [&](uint32_t tm, uint32_t tn) { return uint64_t((m + tm - 1) / tm) * ((n + tn - 1) / tn); };
    const uint64_t steps = (k + 127) / 128, staged_tiles = tiles(kTile, kTile), staged_rounds = staged_tiles < 220 ? 220 : staged_tiles;  // in 256ths
    uint64_t best = steps * (570 * staged_rounds / 256 + (768ull * m + 392ull * n) / 5000) + 4950 + 550 * staged_rounds / 256;
    best = best * 9 / 10;
    const FusedTile* chosen = nullptr;
    for (const FusedTile& c : choices) {
        const uint64_t ns = (tiles(c.m, c.n) + 255) / 256 * (steps * c.step_ns + c.ends_ns);
        if (ns < best) { best = ns; chosen = &c; }
    }
    return chosen;
}

}  // namespace

// workspace: [decoded matrix, halves][token rows, halves]
extern "C" uint64_t tsp_dense_mm_q8_workspace_bytes(uint32_t tokens, uint32_t columns, uint32_t rows) {
    return align256(uint64_t(rows) * columns * 2) + align256(uint64_t(tokens) * columns * 2);
}

extern "C" int tsp_dense_mm_q8_staged(uint32_t layout, const void* matrix, uint64_t matrix_bytes, const float* input, uint64_t input_stride_bytes,
                                      float* output, uint64_t output_stride_bytes, uint32_t tokens, uint32_t columns, uint32_t rows,
                                      void* workspace, uint64_t workspace_bytes, uint32_t* error_word, void* stream) {
    TSP_REQUIRE(layout == TSP_LAYOUT_GGUF || layout == TSP_LAYOUT_Q8_LANES_V1, "dense Q8_0 GEMM layout");
    TSP_REQUIRE(columns && columns <= 65536 && columns % 64 == 0 && rows && rows <= 1000000 && tokens && tokens <= 65536,
                "staged dense Q8_0 GEMM needs columns in multiples of 64");
    TSP_REQUIRE(uint64_t(columns / 32) * rows * 34 == matrix_bytes, "dense Q8_0 GEMM matrix byte span mismatch");
    TSP_REQUIRE(input_stride_bytes % 4 == 0 && output_stride_bytes % 4 == 0 && input_stride_bytes >= uint64_t(columns) * 4 &&
                    output_stride_bytes >= uint64_t(rows) * 4,
                "dense Q8_0 GEMM row geometry mismatch");
    TSP_REQUIRE(matrix && input && output && workspace && error_word, "null device pointer");
    TSP_REQUIRE(reinterpret_cast<uintptr_t>(workspace) % 16 == 0 && workspace_bytes >= tsp_dense_mm_q8_workspace_bytes(tokens, columns, rows),
                "dense Q8_0 GEMM workspace too small or misaligned");
    const uint64_t in_span = uint64_t(tokens - 1) * input_stride_bytes + uint64_t(columns) * 4;
    const uint64_t out_span = uint64_t(tokens - 1) * output_stride_bytes + uint64_t(rows) * 4;
    TSP_REQUIRE(!ranges_overlap(output, out_span, matrix, matrix_bytes) && !ranges_overlap(output, out_span, input, in_span) &&
                    !ranges_overlap(workspace, workspace_bytes, matrix, matrix_bytes) && !ranges_overlap(workspace, workspace_bytes, input, in_span) &&
                    !ranges_overlap(workspace, workspace_bytes, output, out_span),
                "dense Q8_0 GEMM buffers overlap");
    const auto s = static_cast<hipStream_t>(stream);
    if (layout == TSP_LAYOUT_GGUF) {
        const Q8GemmArgs a{input, input_stride_bytes, static_cast<const uint8_t*>(matrix), output, output_stride_bytes, tokens, rows, columns, error_word};
        if (const FusedTile* tile = fused_tile(tokens, rows, columns)) return tile->launch(a, tile->name, s);
    }
    _Float16* const w16 = static_cast<_Float16*>(workspace);
    _Float16* const x16 = reinterpret_cast<_Float16*>(static_cast<uint8_t*>(workspace) + align256(uint64_t(rows) * columns * 2));
    const OperandsArgs o{static_cast<const uint8_t*>(matrix), input, input_stride_bytes, w16, x16, layout, columns, rows, tokens, error_word};
    TSP_LAUNCH("q8_operands_to_f16", s, q8_operands_to_f16<<<dim3((rows + tokens + 3) / 4, (columns + 511) / 512), 256, 0, s>>>(o));
    const F16GemmArgs a{x16, w16, output, output_stride_bytes, tokens, rows, columns, error_word};
    const uint64_t f16_tiles = uint64_t((rows + kTile - 1) / kTile) * ((tokens + kTile - 1) / kTile);
    TSP_LAUNCH("f16_gemm_nt", s, f16_gemm_nt<<<uint32_t((f16_tiles + 7) / 8 * 8), 256, 0, s>>>(a));
    return launch_status("f16_gemm_nt");
}
