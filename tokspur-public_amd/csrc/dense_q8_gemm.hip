// Dense Q8_0 GEMM for many token rows (the shared expert of a prefill chunk): out[t, n] = sum_k x[t, k] * d[n, k/32] * q[n, k].
//
// The streaming kernels of q8.hip / q8_mfma.hip read the whole matrix once per 8 or 16 token rows: right for decode,
// hundreds of passes for a 2048-token chunk. Here a weight is the half nearest d * q (11 significant bits, what the engine's own
// kernel stages, include/tokspur/graph.hpp:860 and kernels/grouped_mm.metal:239-243), the token rows are rounded to halves as
// well, and the matrix cores multiply the two with f32 accumulation.
//
// GGUF rows whose tiles go round the chip well are decoded on their way into the MFMAs, together with the token rows (q8_gemm_fused; q8_gemm_split for few columns or few
// token rows). Else every operand would be decoded too often or much of the chip stand idle: one launch decodes both into the workspace and f16_gemm_nt multiplies them.
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

// A workgroup is one 32 x 32 output tile and its waves take the columns in turns of 64: a chunk of 64 tokens against 640 rows is 40
// workgroups of eight waves, each wave a chain of five steps. A wave reads a step as it lies (256 bytes of 32 token rows,
// 17 dwords of 32 weight rows), two steps' requests in flight, and puts it into fragment order through LDS of its own: no barrier
// until the waves' sums meet, which are added in wave order.
// For few columns or few token rows, where it has less to begin and to end with than the kernel below: 400 x 64 -> 640 3.2 us, 100 x 3.0, 9 x 5120 -> 1024 15.2 from memory
// (4.4, 3.6 and 16.5 on 32 x 32 or 32 x 64 tiles of that one, 5.2 and more for 64 columns with two launches). f32 rows are read sixteen bytes at a time.
template <int WAVES>
__global__ __launch_bounds__(WAVES * kWave, 4) void q8_gemm_split(Q8GemmArgs a) {
    constexpr uint32_t kEdge = 32, kDwords = 17, kWLoads = (kEdge * kDwords + kWave - 1) / kWave, kPitch = kStep + 8;
    struct WaveLds {
        _Float16 x[kEdge * kPitch];
        uint32_t w[kWLoads * kWave];
    };
    static_assert(sizeof(WaveLds) >= kEdge * kEdge * 4);
    __shared__ __attribute__((aligned(16))) WaveLds lds[WAVES];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = uint32_t(__builtin_amdgcn_readfirstlane(int(tid / kWave)));
    const uint32_t col = lane % 32, khalf = lane / 32;
    const uint32_t m0 = blockIdx.y * kEdge, n0 = blockIdx.x * kEdge, steps = a.k / kStep, row_bytes = a.k / 32 * 34;
    const uint8_t* const w_base = a.w + uint64_t(n0) * row_bytes;
    uint32_t w_at[kWLoads];
#pragma unroll
    for (uint32_t q = 0; q < kWLoads; ++q) {
        const uint32_t id = q * kWave + lane < kEdge * kDwords ? q * kWave + lane : kEdge * kDwords - 1, r = n0 + id / kDwords;
        w_at[q] = ((r < a.n ? r : a.n - 1) - n0) * row_bytes + id % kDwords * 4;
    }
    const uint8_t* x_from[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t r = m0 + i * 4 + lane / 16;
        x_from[i] = reinterpret_cast<const uint8_t*>(a.x) + (r < a.m ? r : a.m - 1) * a.x_stride + lane % 16 * 16;
    }
    struct Step { f32x4 x[8]; uint32_t w[kWLoads]; };
    auto fetch = [&](uint32_t s) {
        Step t;
#pragma unroll
        for (int i = 0; i < 8; ++i) t.x[i] = *reinterpret_cast<const f32x4*>(x_from[i] + uint64_t(s) * (kStep * 4));
#pragma unroll
        for (uint32_t q = 0; q < kWLoads; ++q) t.w[q] = *reinterpret_cast<const uint32_t*>(w_base + uint64_t(s) * (kDwords * 4) + w_at[q]);
        return t;
    };
    _Float16* const xs = lds[wave].x;
    uint32_t* const ws = lds[wave].w;
    uint32_t largest = 0;
    f32x16 acc{};
    Step next = fetch(wave < steps ? wave : steps - 1);
    for (uint32_t s = wave; s < steps; s += WAVES) {
        const Step now = next;
        next = fetch(s + WAVES < steps ? s + WAVES : s);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            f16x4 h;
#pragma unroll
            for (int e = 0; e < 4; ++e) h[e] = _Float16(now.x[i][e]);
            const uint2 bits = __builtin_bit_cast(uint2, h);
            // halves without their signs, two to a word: an exponent of ones carries into the bit above
            largest |= ((bits.x & 0x7fff7fffu) + 0x04000400u) | ((bits.y & 0x7fff7fffu) + 0x04000400u);
            *reinterpret_cast<f16x4*>(xs + (i * 4 + lane / 16) * kPitch + lane % 16 * 4) = h;
        }
#pragma unroll
        for (uint32_t q = 0; q < kWLoads; ++q) ws[q * kWave + lane] = now.w[q];
        __builtin_amdgcn_wave_barrier();
        const uint32_t* const mine = ws + col * kDwords;
        const uint32_t d_even = mine[0] & 0xffffu, d_odd = mine[8] >> 16;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
            // quants 16 (g % 2) + 8 khalf .. + 7 of block g / 2, which starts at byte 34 (g / 2) of the row's 68 with its scale
            const uint32_t* const q = mine + (g < 2 ? 0 : 9) + g % 2 * 4 + khalf * 2;
            uint32_t q0 = q[0], q1 = q[1];
            if (g < 2) {
                q0 = __builtin_amdgcn_alignbyte(q1, q0, 2);
                q1 = __builtin_amdgcn_alignbyte(q[2], q1, 2);
            }
            const uint32_t d = g < 2 ? d_even : d_odd;
            const f16x2 d2 = as_h2(d | d << 16);
            const f16x8 c = quants8(q0, q1);  // exact, as is d: one packed multiply rounds once
            const f16x2 p0 = f16x2{c[0], c[1]} * d2, p1 = f16x2{c[2], c[3]} * d2, p2 = f16x2{c[4], c[5]} * d2, p3 = f16x2{c[6], c[7]} * d2;
            const f16x8 fb{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
            const f16x8 fa = *reinterpret_cast<const f16x8*>(xs + col * kPitch + g * 16 + khalf * 8);
            acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa, fb, acc, 0, 0, 0);
        }
        __builtin_amdgcn_wave_barrier();
    }
    uint32_t bad = largest & 0x80008000u ? uint32_t(TSP_ERRBIT_NONFINITE) : 0u;
    // accumulator v: token row 8 (v / 4) + 4 khalf + v % 4 of the tile, weight row `col`; the sums lie over their wave's operands
    float* const sums = reinterpret_cast<float*>(&lds[wave]);
#pragma unroll
    for (int v = 0; v < 16; ++v) sums[(8 * (v / 4) + 4 * khalf + v % 4) * kEdge + col] = acc[v];
    __syncthreads();
#pragma unroll
    for (uint32_t i = tid; i < kEdge * kEdge; i += WAVES * kWave) {
        float value = 0;
#pragma unroll
        for (int q = 0; q < WAVES; ++q) value += reinterpret_cast<const float*>(&lds[q])[i];
        const uint32_t m = m0 + i / kEdge, n = n0 + i % kEdge;
        if (m < a.m && n < a.n) {
            if (nonfinite(value)) bad = TSP_ERRBIT_NONFINITE;
            reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.out) + m * a.out_stride)[n] = value;
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

template <int WAVES>
int launch_split(const Q8GemmArgs& a, const char* name, hipStream_t s) {
    TSP_LAUNCH(name, s, q8_gemm_split<WAVES><<<dim3((a.n + 31) / 32, (a.m + 31) / 32), WAVES * kWave, 0, s>>>(a));
    return launch_status("q8_gemm_split");
}

struct RawRowsKernel {
    const char* name;  // in a profile window
    int (*launch)(const Q8GemmArgs&, const char*, hipStream_t);
};
constexpr RawRowsKernel kSplit4{"q8_gemm_split", launch_split<4>}, kSplit8{"q8_gemm_split", launch_split<8>}, k32x32{"q8_gemm_fused 32x32", launch_fused<FusedShape<32, 32, 1, 1, 2, 2>>},
    k32x64{"q8_gemm_fused 32x64", launch_fused<FusedShape<32, 64, 1, 2, 2, 2>>}, k64x64{"q8_gemm_fused 64x64", launch_fused<FusedShape<64, 64, 2, 1, 1, 4>>},
    k64x96{"q8_gemm_fused 64x96", launch_fused<FusedShape<64, 96, 2, 1, 2, 2>>}, k128x128{"q8_gemm_fused 128x128", launch_fused<FusedShape<128, 128, 2, 2, 1, 2>>};

// Which kernel decodes GGUF rows on their way, or none for the two launches; `aligned`: rows as q8_gemm_split reads them. All forms were timed at some 2300 calls, 64 to 8192
// columns, 64 to 16 000 matrix rows, 1 to 2048 tokens, with operands at hand, the matrix from memory, and both from memory; times below are the first and the last of these.
//   * Below 384 columns q8_gemm_fused takes longer to begin and end than its products take: q8_gemm_split up to 600 tiles, 1024 of 64 columns (64 -> 640, 700 tokens 3.5
//     us and 4.0, 32 x 64 4.7 and 5.3, two launches 5.4 and 6.1; 64 -> 512, 2048 tokens 4.2 and 4.9, two launches 5.8 and 6.5; 256 and 320 columns are even, at 448 32 x 32 takes
//     0.95 of the time). Beyond that 64 x 64 as below, larger tiles not below 512 columns (1600 tokens, 384 -> 700, 64 x 96 8.8 and 10.8, two launches 8.6 and 10.2).
//   * Up to 16 tokens from 2048 columns on: q8_gemm_split with eight waves, by operands from memory (9 tokens, 4096 -> 4096 11.6 and 13.3, 32 x 32 11.4 and 14.0).
//   * Else the smallest tile that goes round in one round of the compute units, since a second costs as much as the first however few are in it. 32 x 32 and 32 x 64
//     gain whatever they fill (203 tokens, 2560 -> 640 8.6 and 11.5, q8_gemm_split 8.9 and 11.9, two launches 15.5 and 16.3).
//   * 64 x 64 takes as long for one tile as for all (2048 columns 14.5 and 18.5), the two launches less for fewer (16.8 and 17.1 at 152 tiles, 18.1 and 18.8 at 224): seven tenths
//     of a round, half of one up to 1024 columns or 256 tokens. Beyond 2048 columns operands from memory make it the slower one (512 rows, 1800 tokens, 4096 columns: 0.93 and
//     1.09 of the two launches' time) but for so few tokens that they are little (150 tokens, 2560 -> 4096 17.1 and 21.8, two launches 21.6 and 22.6).
//   * 64 x 96 where 64 x 64 would need two rounds: 78 hundredths of one, 75 up to 1024 columns, and within the same columns (1800 tokens, 1024 -> 640 14.0 -> 12.1 and 15.8 -> 14.7).
//   * 128 x 128 for four rounds of the two launches: nine tenths of a round, from 2048 columns on of several, 85 hundredths up to 1024 (2048 tokens, 2560 -> 2048 60.7 -> 43.0
//     and 63.7 -> 51.1; at 75 hundredths even with operands at hand and 1.2 times as long from memory).
// Against the kernels that were chosen by 600 tiles before there was q8_gemm_fused, 512 columns and more: 0.92 of the time on average, 43 of 1716 calls slower by more than 2.5 % in one
// of the three states, two in their mean.
// `units`: the device's compute units; figures are for 256.
const RawRowsKernel* raw_rows_kernel(uint32_t m, uint32_t n, uint32_t k, bool aligned, uint64_t units) {
    const auto tiles = [&](uint32_t tm, uint32_t tn) { return uint64_t((m + tm - 1) / tm) * ((n + tn - 1) / tn); };
    // at most that many rounds, their tiles at least `hundredths` of what they could be
    const auto fill = [&](uint64_t count, uint32_t hundredths, uint64_t rounds = 1) {
        const uint64_t r = (count + units - 1) / units;
        return r <= rounds && count * 100 >= hundredths * r * units;
    };
    const uint64_t smallest = tiles(32, 32);
    const bool split = aligned && smallest <= (k < 128 ? 4 * units : units * 75 / 32), few_columns = k <= 1024, few_tokens = m <= 256;
    if (split && (k < 384 || (m <= 16 && k >= 2048 && smallest <= units))) return k < 2048 ? &kSplit4 : &kSplit8;
    if (k >= 384 && fill(smallest, 0)) return &k32x32;
    if (k >= 384 && fill(tiles(32, 64), 0)) return &k32x64;
    if ((k <= 2048 || few_tokens) && fill(tiles(64, 64), few_columns || (few_tokens && k <= 2048) ? 50 : k <= 2048 ? 70 : 75)) return &k64x64;
    if (k < 512) return nullptr;
    if ((k <= 2048 || m <= 320) && fill(tiles(64, 96), few_columns ? 75 : 78)) return &k64x96;
    if (fill(tiles(128, 128), few_columns ? 85 : 90, k < 2048 ? 1 : ~0ull)) return &k128x128;
    return nullptr;
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
        const bool aligned = reinterpret_cast<uintptr_t>(input) % 16 == 0 && input_stride_bytes % 16 == 0 && reinterpret_cast<uintptr_t>(matrix) % 4 == 0;
        static std::atomic<uint64_t> seen{0};
        static int units_of[64];
        int device = 0;
        if (setup_pending(seen, &device)) {
            TSP_HIP(hipDeviceGetAttribute(&units_of[device], hipDeviceAttributeMultiprocessorCount, device));
            setup_done(seen, device);
        }
        if (const RawRowsKernel* kernel = raw_rows_kernel(tokens, rows, columns, aligned, units_of[device] > 0 ? uint64_t(units_of[device]) : 256)) return kernel->launch(a, kernel->name, s);
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
