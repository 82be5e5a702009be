// Dense Q8_0 GEMM for many token rows (the shared expert of a prefill chunk): out[t, n] = sum_k x[t, k] * d[n, k/32] * q[n, k].
//
// The streaming kernels of q8.hip / q8_mfma.hip read the whole matrix once per 8 or 16 token rows: right for decode,
// hundreds of passes for a 2048-token chunk. Here a weight is the half nearest d * q (11 significant bits, what the engine's own
// kernel stages, include/tokspur/graph.hpp:860 and kernels/grouped_mm.metal:239-243), the token rows are rounded to halves as
// well, and the matrix cores multiply the two with f32 accumulation.
//
// A short chunk goes through one kernel that decodes both operands on their way into the MFMAs (q8_gemm_split, raw rows). With more
// tokens every operand would be decoded again and again, ten to forty times over, so one launch decodes both into the workspace and
// f16_gemm_nt multiplies them.
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
// Bound by latency: 60 tokens, 2560 -> 640 columns 8.8 us, 640 -> 2560 4.9 (two conversions and a GEMM: 18.7 and 14.4).
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
using four_floats = f32x4 __attribute__((aligned(4)));
using four_quants = uint32_t __attribute__((aligned(2)));  // rows and blocks are even byte counts
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
    // Up to 600 tiles of 32 x 32 (two or three rounds over the chip): decoded on the way, else decoded once and multiplied, where a round
    // costs more than the launch saved (2048 columns x 512 rows: 14.8 against 17.2 us at 400 tiles, 20.7 against 18.1 at 656; 640 x
    // 2560 8.4 against 9.5 at 560, 12.5 against 11.5 at 1040). f32 rows are read sixteen bytes at a time.
    const uint64_t tiles = uint64_t((rows + 31) / 32) * ((tokens + 31) / 32);
    if (layout == TSP_LAYOUT_GGUF && tiles <= 600 && reinterpret_cast<uintptr_t>(input) % 16 == 0 && input_stride_bytes % 16 == 0 &&
        reinterpret_cast<uintptr_t>(matrix) % 4 == 0) {
        const Q8GemmArgs a{input, input_stride_bytes, static_cast<const uint8_t*>(matrix), output, output_stride_bytes, tokens, rows, columns, error_word};
        const dim3 grid((rows + 31) / 32, (tokens + 31) / 32);
        if (columns >= 2048 && tiles <= 256) TSP_LAUNCH("q8_gemm_split", s, q8_gemm_split<8><<<grid, 512, 0, s>>>(a));
        else TSP_LAUNCH("q8_gemm_split", s, q8_gemm_split<4><<<grid, 256, 0, s>>>(a));
        return launch_status("q8_gemm_split");
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
