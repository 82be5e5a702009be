// Q8_0 GEMV for up to sixteen token rows on the matrix cores (LM head, verify): y[m, r] = sum_k d[r, k/32] * q[r, k] * x[m, k]. Raw rows of more than 2048 columns
// with up to ten token rows, some of fewer columns with up to eight (rows_by_waves), and q8_lanes_v1 rows; the other raw rows are q8_resident.hip's.
//
// A Q8_0 row is a run of 34-byte blocks (f16 scale + 32 int8). The int8 quants are exact halves and bf16, so a block is one
// 16x16x32 MFMA step per 16 weight rows: the block's 32 columns are the instruction's whole K, a lane (n, kq) supplies the
// eight quants 8 kq .. 8 kq + 7 of weight row n, and the sixteen operand rows on the other side are the token rows (eight
// of them repeated when there are only eight). The block's scale multiplies the f32 result once (4 fused multiply-adds per
// lane and 16 weight rows). Up to 2048 columns the activations are scaled by a power of two per token row and split into hi + lo halves, staged once in
// LDS for all of K, so the result carries 22 significant bits of the row's largest x: this is the f32 GEMV of the engine to within f32
// accumulation error (raw rows: the groups of 256 columns meet in 64 bits, 2048 columns 8.9e-8 of the 2-norm, 1.6e-7 in one f32 chain), at ~1.3 VALU operations per weight byte whatever the number of token rows. Rows of more than 2048
// columns are staged as the floats they are, three bf16 pieces each (mfma_quant.hpp): fifteen operand rows for up to five
// token rows, in the same LDS, or for up to ten where a workgroup takes half of the columns.
//
// Raw rows are only 2-byte aligned inside, so the bytes travel global -> registers -> LDS -> registers: a wave reads
// its 32 weight rows x 8 blocks (272 contiguous bytes per row, 16-byte aligned because 8 blocks = 17 x 16 bytes) with
// whole-chunk loads by consecutive lanes, parks them in a wave-private LDS tile whose row stride (272 bytes: unpadded) spreads
// the rows over all banks, and each lane then picks its 8 quants of a block (for each half of the tile's 32 rows) with
// aligned dword reads and a byte funnel shift. The next group of 8 blocks is in flight while the current one is multiplied.
//
// Workgroups are persistent (one per compute unit, 8 waves): the activations are staged once per workgroup, which owns
// every n-th of the matrix's tiles (n workgroups: at any moment the grid reads one stretch of the matrix, 1 us
// faster at 151 936 x 2048 than a contiguous share per workgroup); its waves take the workgroup's tiles through a counter in LDS. A
// lane asks for its share of the token rows first and for its wave's first weight bytes second, and stages the rows
// while the weights travel. Every address inside the loop is a uniform base plus a lane offset fixed before the loop.
//
// Token rows that do not fit LDS for all of K beside the weight tiles (more than eight, in f32 five) split K in two:
// even workgroups take the first half of the columns, odd ones the second, each over its share of the tiles, and both
// add their f32 partial sums into an output the host cleared before the launch (two addends onto zero: the sum does
// not depend on which arrives first). The matrix is still read once.
#include "q8_mfma.hpp"
#include "q8_resident.hpp"

#include <type_traits>

#include "mfma_quant.hpp"

using namespace tsp;

namespace {

constexpr uint32_t kWaves = 8, kThreads = kWaves * kWave;
constexpr uint32_t kGroupBlocks = 8, kGroupBytes = kGroupBlocks * 34, kGroupChunks = kGroupBytes / 16;  // 272 B = 17 chunks
// Bytes between rows of the LDS weight tile: 68 dwords = 4 mod 64 banks, so the sixteen rows times two column quarters that a
// half-wave reads one dword of land in 32 different banks, and the tile is written as the contiguous run of chunks it is.
constexpr uint32_t kTileStride = kGroupBytes;
constexpr uint32_t kTileBytes = 32 * kTileStride;         // 8 704 B per wave
constexpr uint32_t kStageLoads = (32 * kGroupChunks + kWave - 1) / kWave;  // 9 chunk loads per lane and group (the last half used)

struct Q8MfmaArgs {
    const uint8_t* matrix;
    const float* x;   // token-major [M, columns]
    float* y;         // token-major [M, rows]
    uint32_t columns, rows, m;
    uint32_t* error_word;
};

// Any number of floats at any float's address: whole 16-byte pieces but for the ends. (For numbers of weight rows that four does not
// divide: nine to sixteen token rows took two passes over the matrix there, ten by 151 934 x 2048 145 us where this way takes 86.)
__global__ void clear_rows(float* out, uint64_t count) {
    const uint64_t i = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const uint64_t ahead = (16 - reinterpret_cast<uintptr_t>(out) % 16) % 16 / 4, head = ahead < count ? ahead : count, pieces = (count - head) / 4;
    if (i < pieces) reinterpret_cast<float4*>(out + head)[i] = float4{0, 0, 0, 0};
    if (i < head) out[i] = 0;
    if (i < count - head - 4 * pieces) out[head + 4 * pieces + i] = 0;
}
void clear_output(float* out, uint64_t count, hipStream_t s) {
    TSP_LAUNCH("clear_rows", s, clear_rows<<<uint32_t((count / 4 + 3 + 255) / 256), 256, 0, s>>>(out, count));
}

// The token rows of a workgroup, [kRows, K] from column k0 on, in chunks of eight columns: chunk i = tid + j * kThreads is columns
// 8 (i % (K / 8)) .. + 7 of row i / (K / 8). kRows * K / 8 <= 2048 = kMine * kThreads for K <= 2048 (8 rows) or 1024 (16 rows).
// Five rows in f32: chunk tid of row j (LDS has room for 2560 columns); ten rows, K = 1280 columns: chunk tid % 256 of row j for the first
// four waves, of row 5 + j for the others.
constexpr uint32_t kMine = 4, kHalvesColumns = kMine * kThreads, kMostColumns = 2560;
constexpr int kF32Rows = 5;

template <int kRows>
__device__ __forceinline__ void request_token_rows(const Q8MfmaArgs& a, uint32_t K, uint32_t k0, float4 (&xv)[kMine][2]) {
    const uint32_t chunks = K / 8;
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t i = threadIdx.x + j * kThreads, r = i / chunks, c = i % chunks;
        xv[j][0] = xv[j][1] = float4{0, 0, 0, 0};
        if (i < kRows * chunks && r < a.m) {
            const float4* src = reinterpret_cast<const float4*>(a.x + uint64_t(r) * a.columns + k0 + c * 8);
            xv[j][0] = src[0];
            xv[j][1] = src[1];
        }
    }
}

// Largest magnitude of each row, as bits in `largest` (zeros before), -> power-of-two scale -> hi + lo halves in LDS, the 16-byte chunks of a row swizzled
// by the row's index (chunk c of row r sits at c ^ r). Ends with a barrier.
__device__ __forceinline__ int halves_shift(uint32_t largest) {  // the largest to 2^13; a row that is not finite stays as it is
    const int up = 13 + 127 - int(largest >> 23);
    return largest == 0 || largest >= 0x7f800000u ? 0 : up > 100 ? 100 : up;
}
template <int kRows>
__device__ __forceinline__ void stage_token_rows(const float4 (&xv)[kMine][2], uint32_t K, _Float16* a_hi, _Float16* a_lo, uint32_t* largest, uint32_t& bad) {
    const uint32_t tid = threadIdx.x, chunks = K / 8;
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        uint32_t bits = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            for (const float v : {xv[j][h].x, xv[j][h].y, xv[j][h].z, xv[j][h].w}) bits = max(bits, __float_as_uint(v) & 0x7fffffffu);
        if (bits >= 0x7f800000u) bad = TSP_ERRBIT_NONFINITE;
        bits = row16_largest_bits(bits);  // sixteen lanes are of one row: a row's chunks are a multiple of sixteen
        const uint32_t i = tid + j * kThreads;
        if (tid % 16 == 0 && i < kRows * chunks) atomicMax(&largest[i / chunks], bits);
    }
    __syncthreads();
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t i = tid + j * kThreads, r = i / chunks, c = i % chunks;
        if (i >= kRows * chunks) break;
        const float scale = power_of_two(halves_shift(largest[r]));
        const float v[8] = {xv[j][0].x, xv[j][0].y, xv[j][0].z, xv[j][0].w, xv[j][1].x, xv[j][1].y, xv[j][1].z, xv[j][1].w};
        f16x8 hi, lo;  // zeros for the rows past a.m
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float sv = v[e] * scale;
            hi[e] = _Float16(sv);
            lo[e] = _Float16(sv - float(hi[e]));
        }
        const uint32_t at = (r * chunks + (c ^ r)) * 8;
        *reinterpret_cast<f16x8*>(a_hi + at) = hi;
        *reinterpret_cast<f16x8*>(a_lo + at) = lo;
    }
    __syncthreads();
}
// What undoes the scales of the token rows that a lane's accumulators belong to.
template <int kRows>
__device__ __forceinline__ void halves_back(const uint32_t* largest, uint32_t kq, float (&back)[4]) {
#pragma unroll
    for (uint32_t v = 0; v < 4; ++v) back[v] = power_of_two(-halves_shift(largest[(4 * kq + v) % kRows]));
}

// The same for SETS times five rows in f32: xv[j] is row 5 set + j of the thread's set.
template <int SETS>
__device__ __forceinline__ void request_f32_rows(const Q8MfmaArgs& a, uint32_t K, uint32_t k0, float4 (&xv)[kF32Rows][2]) {
    const uint32_t chunk = threadIdx.x % (kThreads / SETS), set = threadIdx.x / (kThreads / SETS);
#pragma unroll
    for (uint32_t j = 0; j < kF32Rows; ++j) {
        xv[j][0] = xv[j][1] = float4{0, 0, 0, 0};
        if (chunk < K / 8 && set * kF32Rows + j < a.m) {
            const float4* src = reinterpret_cast<const float4*>(a.x + uint64_t(set * kF32Rows + j) * a.columns + k0 + chunk * 8);
            xv[j][0] = src[0];
            xv[j][1] = src[1];
        }
    }
}

// Row s < 4 of a set becomes operand rows s, 4 + s and 12 + s (its pieces from the largest down), row 4 operand rows 8, 9 and 10; a set's
// sixteen operand rows follow the other's. `back` gets what undoes each row's scale. Ends with a barrier.
template <int SETS>
__device__ __forceinline__ void stage_f32_rows(const float4 (&xv)[kF32Rows][2], uint32_t K, __bf16* rows, float (*wave_max)[kWaves], float (&back)[SETS][kF32Rows],
                                               uint32_t& bad) {
    constexpr uint32_t kSetWaves = kWaves / SETS;
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, chunks = K / 8, chunk = tid % (kThreads / SETS), set = tid / (kThreads / SETS);
#pragma unroll
    for (int j = 0; j < kF32Rows; ++j) {
        float biggest = 0;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const float4 v = xv[j][h];
            if (nonfinite(v.x) || nonfinite(v.y) || nonfinite(v.z) || nonfinite(v.w)) bad = TSP_ERRBIT_NONFINITE;
            biggest = fmaxf(biggest, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        }
        biggest = wave_largest(biggest);
        if (lane == 0) wave_max[j][wave] = biggest;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kF32Rows; ++j) {
        float scale = 1.0f;
#pragma unroll
        for (uint32_t q = 0; q < SETS; ++q) {
            float biggest = wave_max[j][q * kSetWaves];
#pragma unroll
            for (uint32_t w = 1; w < kSetWaves; ++w) biggest = fmaxf(biggest, wave_max[j][q * kSetWaves + w]);
            const int shift = row_lift(biggest);
            if (q == set) scale = power_of_two(shift);
            back[q][j] = power_of_two(-shift);
        }
        if (chunk < chunks) {
            const float v[8] = {xv[j][0].x, xv[j][0].y, xv[j][0].z, xv[j][0].w, xv[j][1].x, xv[j][1].y, xv[j][1].z, xv[j][1].w};
            Pieces p[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) p[e] = three_pieces(v[e] * scale);
            auto put = [&](uint32_t row, u32x4 eight) { *reinterpret_cast<u32x4*>(rows + ((set * 16 + row) * chunks + (chunk ^ row)) * 8) = eight; };
            const uint32_t first = j < 4 ? j : 8, second = j < 4 ? 4 + j : 9, third = j < 4 ? 12 + j : 10;
            put(first, u32x4{two_tops(p[0].hi, p[1].hi), two_tops(p[2].hi, p[3].hi), two_tops(p[4].hi, p[5].hi), two_tops(p[6].hi, p[7].hi)});
            put(second, u32x4{two_tops(p[0].mid, p[1].mid), two_tops(p[2].mid, p[3].mid), two_tops(p[4].mid, p[5].mid), two_tops(p[6].mid, p[7].mid)});
            put(third, u32x4{two_tops(p[0].lo, p[1].lo), two_tops(p[2].lo, p[3].lo), two_tops(p[4].lo, p[5].lo), two_tops(p[6].lo, p[7].lo)});
        }
    }
    __syncthreads();
}

// The sums of five rows in f32 out of the accumulators of their fifteen operand rows (row 4 kq + v in acc[v]) for the weight row of
// lane n16: store(token row, sum) in the lanes that hold one. The small pieces first.
template <class Store>
__device__ __forceinline__ void f32_row_sums(const float (&acc)[4], uint32_t kq, const float (&back)[kF32Rows], Store store) {
#pragma unroll
    for (int v = 0; v < 4; ++v) {
        const uint32_t mine = __float_as_uint(kq == 2 ? 0.0f : acc[v]);
        const auto halves = __builtin_amdgcn_permlane32_swap(mine, mine, false, false);  // lanes l and l ^ 32
        const uint32_t outer = __float_as_uint(__uint_as_float(halves[0]) + __uint_as_float(halves[1]));
        const auto quarters = __builtin_amdgcn_permlane16_swap(outer, outer, false, false);  // l and l ^ 16
        const float sum = __uint_as_float(quarters[0]) + __uint_as_float(quarters[1]);
        if (kq == 0) store(uint32_t(v), sum * back[v]);
    }
    if (kq == 2) store(4u, (acc[0] + (acc[1] + acc[2])) * back[4]);
}

// Two workgroups whose halves of a sum meet in an output that starts at zero: the halves may be finite and the sum not, which only the one
// that adds last can see. What an addition found there is kept until the next tile's additions, by when it has long come back.
struct Joined { float mine = 0, found = 0; };
__device__ __forceinline__ Joined join(float* y, uint32_t at, float half) {  // sixteen rows of 1 000 000 at most: 32-bit offsets
    return {half, unsafeAtomicAdd(reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(y) + at * 4), half)};
}
template <int N>
__device__ __forceinline__ void check_joined(Joined (&all)[N], uint32_t& bad) {
#pragma unroll
    for (int i = 0; i < N; ++i) {
        if (nonfinite(all[i].found + all[i].mine)) bad = TSP_ERRBIT_NONFINITE;
        all[i] = Joined{};
    }
}

// DEPTH = (tile, group) items whose bytes are on their way while one is multiplied (1 or 2; it divides the number of groups
// of a workgroup). ROWS = token rows staged: 8, in halves, or in f32 5 (all of K per workgroup) and 10 (half of K per workgroup, sums added into y).
template <int DEPTH, int ROWS>
__global__ __launch_bounds__(kThreads, 1) void q8_mfma_kernel(Q8MfmaArgs a) {
    constexpr bool F32 = ROWS % kF32Rows == 0;
    constexpr int SETS = F32 ? ROWS / kF32Rows : 1;
    constexpr uint32_t KSPLIT = SETS;
    using Operand = std::conditional_t<F32, __bf16, _Float16>;
    using Frag = std::conditional_t<F32, bf16x8, f16x8>;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // [sets of sixteen operand rows, or eight in hi and eight in lo halves][8 weight tiles]
    __shared__ float wave_max[kF32Rows][kWaves];
    __shared__ uint32_t largest[8];
    __shared__ uint32_t next_tile;

    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const uint32_t n16 = lane % 16, kq = lane / 16;  // 16x16x32 MFMA: operand row / column lane % 16, columns 8 kq .. 8 kq + 7 of the block
    // K: the columns this workgroup multiplies, starting at column k0 (group g0 of the rows)
    const uint32_t K = a.columns / KSPLIT, chunks = K / 8, groups = K / 256, row_bytes = a.columns / 32 * 34;
    const uint32_t k0 = (blockIdx.x % KSPLIT) * K, g0 = k0 / 256;
    const uint32_t sharer = blockIdx.x / KSPLIT, sharers = gridDim.x / KSPLIT;  // the host launches a multiple of KSPLIT
    if (tid == 0) next_tile = 0;
    if (!F32 && tid < 8) largest[tid] = 0;
    __syncthreads();  // the tile counter is set before any wave takes from it
    Operand* const operands = reinterpret_cast<Operand*>(lds);
    uint8_t* const tile = lds + SETS * 16 * K * 2 + wave * kTileBytes;

    // ---- the token rows: this lane's 16-byte chunks are requested first (they come from cache and return first), then the
    // wave's first weight bytes, and only then the arithmetic. The weights travel while the rows are staged.
    uint32_t bad = 0;
    float4 xv[F32 ? kF32Rows : kMine][2];
    if constexpr (F32) request_f32_rows<SETS>(a, K, k0, xv);
    else request_token_rows<8>(a, K, k0, xv);
    // chunk `id` of a group tile: row id / 17 of the wave's 32, bytes (id % 17) * 16 of that row's 272. The byte offsets from
    // the tile's first row and the group's first byte never change, so a request is a uniform address plus a lane offset.
    uint32_t chunk_at[kStageLoads];
#pragma unroll
    for (uint32_t t = 0; t < kStageLoads; ++t) {
        uint32_t id = t * kWave + lane;
        id = id < 32 * kGroupChunks ? id : 32 * kGroupChunks - 1;  // the tail lanes repeat the last chunk
        chunk_at[t] = (id / kGroupChunks) * row_bytes + (id % kGroupChunks) * 16;
    }
    uint2 stage[DEPTH][kStageLoads][2];
    auto fetch_group = [&](uint32_t row0, uint32_t group, auto set_tag) {
        constexpr int SET = decltype(set_tag)::value;
        const uint8_t* from = a.matrix + uint64_t(row0) * row_bytes + uint64_t(g0 + group) * kGroupBytes;  // uniform
        const bool whole = row0 + 32 <= a.rows;                                                           // uniform
#pragma unroll
        for (uint32_t t = 0; t < kStageLoads; ++t) {
            uint32_t at = chunk_at[t];
            if (!whole) {  // the matrix's last tile: rows past the end repeat the last row
                uint32_t id = t * kWave + lane;
                id = id < 32 * kGroupChunks ? id : 32 * kGroupChunks - 1;
                const uint32_t row = row0 + id / kGroupChunks < a.rows ? id / kGroupChunks : a.rows - 1 - row0;
                at = row * row_bytes + (id % kGroupChunks) * 16;
            }
            const uint4 v = *reinterpret_cast<const uint4*>(from + at);
            stage[SET][t][0] = uint2{v.x, v.y};
            stage[SET][t][1] = uint2{v.z, v.w};
        }
    };
    // Workgroup b of n owns tiles b, b + n, b + 2 n, ... and its waves take the next free one of them from
    // a counter in LDS (which wave computes a tile does not change the result). The bytes of the next (tile, group) item
    // are requested before the current one is multiplied, so a wave always holds its next tile index one step ahead.
    const uint32_t share_end = (a.rows + 31) / 32;
    auto take_tile = [&]() {
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(&next_tile, 1u);
        return uint32_t(__builtin_amdgcn_readfirstlane(int(t))) * sharers + sharer;
    };
    uint32_t t = take_tile(), t_next = take_tile();
    if (t < share_end) {
        fetch_group(t * 32, 0, std::integral_constant<int, 0>{});
        if constexpr (DEPTH >= 2) fetch_group(t * 32, 1, std::integral_constant<int, 1 % DEPTH>{});
    }
    __builtin_amdgcn_sched_barrier(0);  // every request above is out before the first wait below
    float back[SETS][F32 ? kF32Rows : 4];
    if constexpr (F32) {
        stage_f32_rows<SETS>(xv, K, operands, wave_max, back, bad);
    } else {
        stage_token_rows<8>(xv, K, operands, operands + 8 * K, largest, bad);
        halves_back<8>(largest, kq, back[0]);
    }

    // The activation chunk of block B of group g, columns 8 kq .. 8 kq + 7, is chunk g * 32 + B * 4 + kq of row `arow`, kept at
    // position chunk ^ arow. arow only flips the three or four low bits, which B % kVariants and kq decide: the lane keeps one
    // address per variant and the rest of the chunk index is an offset known when the code is compiled (B) or uniform (g).
    const uint32_t arow = F32 ? n16 : n16 % 8;
    constexpr uint32_t kVariants = F32 ? 4 : 2;
    uint32_t a_at[kVariants];  // in elements, from the start of a set or plane
#pragma unroll
    for (uint32_t v = 0; v < kVariants; ++v) a_at[v] = (arow * chunks + ((v * 4 + kq) ^ arow)) * 8;
    auto store_group = [&](auto set_tag) {
        constexpr int SET = decltype(set_tag)::value;
#pragma unroll
        for (uint32_t t = 0; t < kStageLoads; ++t) {
            uint32_t id = t * kWave + lane;
            id = id < 32 * kGroupChunks ? id : 32 * kGroupChunks - 1;
            uint8_t* at = tile + (id / kGroupChunks) * kTileStride + (id % kGroupChunks) * 16;
            *reinterpret_cast<uint4*>(at) = uint4{stage[SET][t][0].x, stage[SET][t][0].y, stage[SET][t][1].x, stage[SET][t][1].y};
        }
    };

    Joined joined[KSPLIT == 2 ? SETS * 8 : 1];
    for (; t < share_end; t = t_next, t_next = take_tile()) {
        const uint32_t row0 = t * 32;
        std::conditional_t<F32, float, double> acc[SETS][2][4] = {};  // [set][16-row half of the tile][token row 4 kq + v]
        // one item: its bytes go registers -> LDS tile, the item DEPTH ahead is requested into the freed registers, then the
        // tile is multiplied.
        auto item = [&](uint32_t g, auto set_tag) {
            store_group(set_tag);  // the previous item's reads were issued before this point; LDS serves a wave in order
            const uint32_t ahead = g + DEPTH;
            const bool wraps = ahead >= groups;
            // past the workgroup's share: ask again for the group at hand (its lines are in cache), nothing new comes from memory
            const bool more = t_next < share_end;
            const uint32_t following = wraps && more ? t_next : t;
            const uint32_t group = !wraps ? ahead : more ? ahead - groups : g;
            fetch_group(following * 32, group, set_tag);
            const uint8_t* mine = tile + n16 * kTileStride + kq * 8;
            float sums[SETS][2][4] = {};  // a group's blocks are added up by themselves: a tenth as many roundings of the whole sum
            auto block = [&](auto b_tag) {
                constexpr int B = decltype(b_tag)::value;
                // the lane's eight quants of the block, for rows n16 and n16 + 16 of the tile: bytes 34 B + 2 + 8 kq .. + 8 of the
                // row, dword aligned for odd B, 2 bytes past a dword for even B
                constexpr uint32_t Q_AT = 34 * B + 2, ALIGNED = Q_AT & ~3u;
                Frag b_frag[2];
                float scale_d[2];
#pragma unroll
                for (int nt = 0; nt < 2; ++nt) {
                    const uint8_t* row = mine + nt * 16 * kTileStride;
                    uint32_t w[2];
                    if constexpr (Q_AT % 4 == 0) {
                        w[0] = *reinterpret_cast<const uint32_t*>(row + ALIGNED);
                        w[1] = *reinterpret_cast<const uint32_t*>(row + ALIGNED + 4);
                    } else {
                        uint32_t d[3];
#pragma unroll
                        for (int i = 0; i < 3; ++i) d[i] = *reinterpret_cast<const uint32_t*>(row + ALIGNED + 4 * i);
                        w[0] = __builtin_amdgcn_alignbyte(d[1], d[0], 2);
                        w[1] = __builtin_amdgcn_alignbyte(d[2], d[1], 2);
                    }
                    if constexpr (F32) b_frag[nt] = quants8_bf16(w[0], w[1]);
                    else b_frag[nt] = quants8(w[0], w[1]);
                    scale_d[nt] = half_bits_to_float(*reinterpret_cast<const uint16_t*>(tile + (nt * 16 + n16) * kTileStride + 34 * B));
                }
                // columns g * 256 + B * 32 + 8 kq of the lane's token row
                const uint32_t at = a_at[B % kVariants] + (g * 32 + (B / kVariants) * kVariants * 4) * 8;
                const f32x4 zero{};
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int set = SETS - 1; set >= 0; --set) {
                        f32x4 part;
                        if constexpr (F32) {
                            part = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(operands + set * 16 * K + at), b_frag[nt], zero, 0, 0, 0);
                        } else {  // the lo halves of the rows first, the hi halves on top of them: one f32 result per block to scale
                            part = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(operands + 8 * K + at), b_frag[nt], zero, 0, 0, 0);
                            part = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(operands + at), b_frag[nt], part, 0, 0, 0);
                        }
#pragma unroll
                        for (int v = 0; v < 4; ++v) sums[set][nt][v] = __builtin_fmaf(scale_d[nt], part[v], sums[set][nt][v]);
                    }
            };
            block(std::integral_constant<int, 0>{});
            block(std::integral_constant<int, 1>{});
            block(std::integral_constant<int, 2>{});
            block(std::integral_constant<int, 3>{});
            block(std::integral_constant<int, 4>{});
            block(std::integral_constant<int, 5>{});
            block(std::integral_constant<int, 6>{});
            block(std::integral_constant<int, 7>{});
#pragma unroll
            for (int set = 0; set < SETS; ++set)
#pragma unroll
                for (int nt = 0; nt < 2; ++nt)
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[set][nt][v] += sums[set][nt][v];
        };
        uint32_t g = 0;
        do {  // the host picks a DEPTH that divides the number of groups; there is at least one, and the compiler has to know it to count what is in flight
            item(g, std::integral_constant<int, 0>{});
            if constexpr (DEPTH >= 2) item(g + 1, std::integral_constant<int, 1 % DEPTH>{});
        } while ((g += DEPTH) < groups);
        if constexpr (KSPLIT == 2) check_joined(joined, bad);
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) {
            const uint32_t r = row0 + nt * 16 + n16;
            if constexpr (F32) {
#pragma unroll
                for (int set = 0; set < SETS; ++set) {
                    f32_row_sums(acc[set][nt], kq, back[set], [&](uint32_t row, float val) {
                        const uint32_t m = set * kF32Rows + row;
                        if (m >= a.m || r >= a.rows) return;
                        if (nonfinite(val)) bad = TSP_ERRBIT_NONFINITE;
                        if constexpr (KSPLIT == 1) a.y[uint64_t(m) * a.rows + r] = val;
                        else joined[(set * 2 + nt) * 4 + row % 4] = join(a.y, m * a.rows + r, val);  // (row 4 is in other lanes than row 0)
                    });
                }
            } else {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t m = 4 * kq + v;  // lanes with kq >= 2 hold repeats of rows 0 .. 7
                    if (kq >= 2 || m >= a.m || r >= a.rows) continue;
                    const float val = float(acc[0][nt][v]) * back[0][v];
                    if (nonfinite(val)) bad = TSP_ERRBIT_NONFINITE;
                    a.y[uint64_t(m) * a.rows + r] = val;
                }
            }
        }
    }
    if constexpr (KSPLIT == 2) check_joined(joined, bad);
    publish_error(bad, a.error_word);
}

// ---- q8_lanes_v1 rows: [f16 scale x blocks][runs of 16 blocks x 512 B: quant i of the run's sixteen blocks side by side].
// The unit of work is 16 weight rows x one run (512 columns): per row 32 bytes of scales and 512 bytes of quants, both whole
// 16-byte chunks at 16-byte aligned offsets when the row has a multiple of 16 blocks. A wave parks the 34 chunks of each row
// in its LDS tile at a row stride of 560 bytes (140 dwords = 12 mod 64 banks: the sixteen rows that a quarter-wave reads one
// 16-byte chunk of land in 64 different banks). A lane (n, kq) then reads the eight chunks of quants 8 kq .. 8 kq + 7 of row n,
// which hold those quants for all sixteen blocks, and turns each 4 x 4 byte square (4 quants x 4 blocks) into the four dwords
// "4 quants of one block" with two rounds of byte permutes: four permutes per block and lane. From there on a block is what it
// is for raw rows: exact halves, one 16x16x32 MFMA step for the lo and one for the hi halves of the token rows, and the
// block's scale times the f32 result.
constexpr uint32_t kRunBlocks = 16, kRunChunks = 2 + 32;  // 32 B of scales + 512 B of quants per row and run
constexpr uint32_t kLaneRows = 16, kLaneStride = 560, kLaneTileBytes = kLaneRows * kLaneStride;  // 8 960 B per wave
constexpr uint32_t kLaneLoads = (kLaneRows * kRunChunks + kWave - 1) / kWave;  // 9 chunk loads per lane and run (the last half used)

// ROWS = token rows staged: 8 (all of K per workgroup) or 16 (even workgroups the first half of a row's runs, odd ones the second,
// each pair over its share of the tiles, both adding their f32 sums into an output the host cleared: the matrix is read once); 5 and
// 10: the same in f32, ten on rows of five runs only: either workgroup takes two and a half of them, and both read the third, which
// costs less than the second pass over the matrix that five rows at a time take (151 936 rows, six tokens: 168 us of kernels, now 96).
template <int DEPTH, int ROWS>
__global__ __launch_bounds__(kThreads, 1) void q8_lanes_mfma_kernel(Q8MfmaArgs a) {
    constexpr bool F32 = ROWS % kF32Rows == 0;
    constexpr int SETS = F32 ? ROWS / kF32Rows : 1, kRows = F32 ? 8 * SETS : ROWS;  // kRows: of each of two operand planes; as much LDS in f32
    constexpr uint32_t KSPLIT = kRows / 8;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];  // [hi plane][lo plane][8 weight tiles]
    __shared__ float wave_max[kF32Rows][kWaves];
    __shared__ uint32_t largest[16];
    __shared__ uint32_t next_tile;

    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave;
    const uint32_t n16 = lane % 16, kq = lane / 16;
    // K: the columns this workgroup multiplies, runs run0 .. run0 + runs - 1 of every row
    constexpr bool kShared = F32 && KSPLIT == 2;  // the middle run is both workgroups'
    const uint32_t part = blockIdx.x % KSPLIT, all_runs = a.columns / 32 / kRunBlocks;
    const uint32_t K = a.columns / KSPLIT, chunks = K / 8, blocks = a.columns / 32, runs = (all_runs + (kShared ? 1 : 0)) / KSPLIT, row_bytes = blocks * 34;
    const uint32_t run0 = part * (all_runs - runs);
    const uint32_t sharer = blockIdx.x / KSPLIT, sharers = gridDim.x / KSPLIT;  // the host launches a multiple of KSPLIT
    const uint32_t tiles = (a.rows + kLaneRows - 1) / kLaneRows;
    if (tid == 0) next_tile = 0;
    if (!F32 && tid < 16) largest[tid] = 0;
    __syncthreads();
    _Float16* const a_hi = reinterpret_cast<_Float16*>(lds);
    _Float16* const a_lo = a_hi + kRows * K;
    uint8_t* const tile = lds + 2 * kRows * K * 2 + wave * kLaneTileBytes;

    uint32_t bad = 0;
    float4 xv[F32 ? kF32Rows : kMine][2];
    if constexpr (F32) request_f32_rows<SETS>(a, K, part * K, xv);
    else request_token_rows<kRows>(a, K, run0 * (kRunBlocks * 32), xv);

    // chunk `id` of a tile: row id / 34 of the wave's 16, piece id % 34 of that row's run: pieces 0 and 1 are the run's scales
    // (32 bytes per run from the row's start), pieces 2 .. 33 its quants (512 bytes per run after all the scales).
    auto piece_at = [&](uint32_t row, uint32_t piece, uint32_t run) {
        return row * row_bytes + (piece < 2 ? run * 32 + piece * 16 : 2 * blocks + run * 512 + (piece - 2) * 16);
    };
    uint32_t chunk_at[kLaneLoads], chunk_step[kLaneLoads];  // byte offset at run 0 and bytes per run
#pragma unroll
    for (uint32_t t = 0; t < kLaneLoads; ++t) {
        uint32_t id = t * kWave + lane;
        id = id < kLaneRows * kRunChunks ? id : kLaneRows * kRunChunks - 1;  // the tail lanes repeat the last chunk
        chunk_at[t] = piece_at(id / kRunChunks, id % kRunChunks, run0);
        chunk_step[t] = id % kRunChunks < 2 ? 32 : 512;
    }
    uint2 stage[DEPTH][kLaneLoads][2];
    auto fetch_run = [&](uint32_t row0, uint32_t run, auto set_tag) {
        constexpr int SET = decltype(set_tag)::value;
        const uint8_t* from = a.matrix + uint64_t(row0) * row_bytes;  // uniform
        const bool whole = row0 + kLaneRows <= a.rows;               // uniform
#pragma unroll
        for (uint32_t t = 0; t < kLaneLoads; ++t) {
            uint32_t at = chunk_at[t] + run * chunk_step[t];
            if (!whole) {  // the matrix's last tile: rows past the end repeat the last row
                uint32_t id = t * kWave + lane;
                id = id < kLaneRows * kRunChunks ? id : kLaneRows * kRunChunks - 1;
                const uint32_t row = row0 + id / kRunChunks < a.rows ? id / kRunChunks : a.rows - 1 - row0;
                at = piece_at(row, id % kRunChunks, run0 + run);
            }
            const uint4 v = *reinterpret_cast<const uint4*>(from + at);
            stage[SET][t][0] = uint2{v.x, v.y};
            stage[SET][t][1] = uint2{v.z, v.w};
        }
    };
    const uint32_t share_end = tiles;
    auto take_tile = [&]() {
        uint32_t t = 0;
        if (lane == 0) t = atomicAdd(&next_tile, 1u);
        return uint32_t(__builtin_amdgcn_readfirstlane(int(t))) * sharers + sharer;
    };
    uint32_t t = take_tile(), t_next = take_tile();
    if (t < share_end) {
        fetch_run(t * kLaneRows, 0, std::integral_constant<int, 0>{});
        if constexpr (DEPTH >= 2) fetch_run(t * kLaneRows, 1, std::integral_constant<int, 1 % DEPTH>{});
    }
    __builtin_amdgcn_sched_barrier(0);  // every request above is out before the first wait below
    float back[SETS][F32 ? kF32Rows : 4];
    if constexpr (F32) {
        stage_f32_rows<SETS>(xv, K, reinterpret_cast<__bf16*>(lds), wave_max, back, bad);
    } else {
        stage_token_rows<kRows>(xv, K, a_hi, a_lo, largest, bad);
        halves_back<kRows>(largest, kq, back[0]);
    }

    // the activation chunk of block B of run g, columns 8 kq .. 8 kq + 7: chunk g * 64 + B * 4 + kq of row `arow`, kept at
    // chunk ^ arow; arow < kRows flips the three or four low bits, which B % kVariants and kq decide
    constexpr uint32_t kOperandRows = F32 ? 16 : kRows;
    const uint32_t arow = n16 & (kOperandRows - 1);
    constexpr uint32_t kVariants = kOperandRows / 4;
    uint32_t a_at[kVariants];
#pragma unroll
    for (uint32_t v = 0; v < kVariants; ++v) a_at[v] = (arow * chunks + ((v * 4 + kq) ^ arow)) * 8;
    auto store_run = [&](auto set_tag) {
        constexpr int SET = decltype(set_tag)::value;
#pragma unroll
        for (uint32_t t = 0; t < kLaneLoads; ++t) {
            uint32_t id = t * kWave + lane;
            id = id < kLaneRows * kRunChunks ? id : kLaneRows * kRunChunks - 1;
            uint8_t* at = tile + (id / kRunChunks) * kLaneStride + (id % kRunChunks) * 16;
            *reinterpret_cast<uint4*>(at) = uint4{stage[SET][t][0].x, stage[SET][t][0].y, stage[SET][t][1].x, stage[SET][t][1].y};
        }
    };

    Joined joined[KSPLIT == 2 ? SETS * 4 : 1];
    for (; t < share_end; t = t_next, t_next = take_tile()) {
        const uint32_t row0 = t * kLaneRows;
        float acc[SETS][4] = {};  // [set][token row 4 kq + v]
        auto item = [&](uint32_t g, auto set_tag) {
            store_run(set_tag);  // the previous item's reads were issued before this point; LDS serves a wave in order
            const uint32_t ahead = g + DEPTH;
            const bool wraps = ahead >= runs;
            // past the workgroup's share: ask again for the run at hand (its lines are in cache), nothing new comes from memory
            const bool more = t_next < share_end;
            const uint32_t following = wraps && more ? t_next : t;
            const uint32_t run = !wraps ? ahead : more ? ahead - runs : g;
            fetch_run(following * kLaneRows, run, set_tag);
            const uint8_t* mine = tile + n16 * kLaneStride;
            const uint4 s0 = *reinterpret_cast<const uint4*>(mine), s1 = *reinterpret_cast<const uint4*>(mine + 16);
            const uint32_t scales[8] = {s0.x, s0.y, s0.z, s0.w, s1.x, s1.y, s1.z, s1.w};  // two f16 scales per dword
            uint4 q[8];  // q[j]: quant 8 kq + j of the run's sixteen blocks, one byte per block
#pragma unroll
            for (int j = 0; j < 8; ++j) q[j] = *reinterpret_cast<const uint4*>(mine + 32 + (8 * kq + j) * 16);
            float run_sum[SETS][4] = {};  // in f32 a run's blocks are added up by themselves
            const uint32_t columns_at = g * 64 * 8 - (kShared && part ? kRunBlocks / 2 * 4 * 8 : 0);  // of the run, in the staged rows
            auto& sums = F32 ? run_sum : acc;
            auto quad = [&](auto m_tag) {  // blocks 4 M .. 4 M + 3 of the run
                constexpr int M = decltype(m_tag)::value;
                uint32_t d[8];
#pragma unroll
                for (int j = 0; j < 8; ++j) d[j] = M == 0 ? q[j].x : M == 1 ? q[j].y : M == 2 ? q[j].z : q[j].w;
                // byte b of d[j] = quant j of block 4 M + b. First round: pairs of quants interleaved, for blocks 0, 1 (lo) and 2, 3 (hi)
                uint32_t lo[4], hi[4];
#pragma unroll
                for (int p = 0; p < 4; ++p) {
                    lo[p] = __builtin_amdgcn_perm(d[2 * p + 1], d[2 * p], 0x05010400u);
                    hi[p] = __builtin_amdgcn_perm(d[2 * p + 1], d[2 * p], 0x07030602u);
                }
                // second round: w[b][0] = quants 0 .. 3 and w[b][1] = quants 4 .. 7 of block 4 M + b
                uint32_t w[4][2];
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    w[0][half] = __builtin_amdgcn_perm(lo[2 * half + 1], lo[2 * half], 0x05040100u);
                    w[1][half] = __builtin_amdgcn_perm(lo[2 * half + 1], lo[2 * half], 0x07060302u);
                    w[2][half] = __builtin_amdgcn_perm(hi[2 * half + 1], hi[2 * half], 0x05040100u);
                    w[3][half] = __builtin_amdgcn_perm(hi[2 * half + 1], hi[2 * half], 0x07060302u);
                }
#pragma unroll
                for (int b = 0; b < 4; ++b) {
                    constexpr int kBase = 4 * M;
                    const int B = kBase + b;
                    const float scale_d = half_bits_to_float((scales[B / 2] >> (16 * (B % 2))) & 0xffffu);
                    const uint32_t at = a_at[B % kVariants] + columns_at + (B / kVariants) * kVariants * 4 * 8;  // columns g * 512 + B * 32 + 8 kq of the lane's token row
                    const f32x4 zero{};
                    f32x4 product;
                    if constexpr (F32) {
                        const bf16x8 b_frag = quants8_bf16(w[b][0], w[b][1]);
#pragma unroll
                        for (int set = 0; set < SETS; ++set) {
                            product = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(a_hi + set * 16 * K + at), b_frag, zero, 0, 0, 0);
#pragma unroll
                            for (int v = 0; v < 4; ++v) sums[set][v] = __builtin_fmaf(scale_d, product[v], sums[set][v]);
                        }
                    } else {
                        const f16x8 b_frag = quants8(w[b][0], w[b][1]);
                        product = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(a_lo + at), b_frag, zero, 0, 0, 0);
                        product = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(a_hi + at), b_frag, product, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 4; ++v) sums[0][v] = __builtin_fmaf(scale_d, product[v], sums[0][v]);
                    }
                }
            };
            // of the middle run the first workgroup takes the first half, the second the second: uniform
            if (!kShared || part == 0 || g != 0) {
                quad(std::integral_constant<int, 0>{});
                quad(std::integral_constant<int, 1>{});
            }
            if (!kShared || part != 0 || g + 1 != runs) {
                quad(std::integral_constant<int, 2>{});
                quad(std::integral_constant<int, 3>{});
            }
            if constexpr (F32) {
#pragma unroll
                for (int set = 0; set < SETS; ++set)
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[set][v] += run_sum[set][v];
            }
        };
        uint32_t g = 0;
        do {  // the host picks a DEPTH that divides the number of runs; there is at least one
            item(g, std::integral_constant<int, 0>{});
            if constexpr (DEPTH >= 2) item(g + 1, std::integral_constant<int, 1 % DEPTH>{});
        } while ((g += DEPTH) < runs);
        const uint32_t r = row0 + n16;
        if constexpr (KSPLIT == 2) check_joined(joined, bad);
        if constexpr (F32) {
#pragma unroll
            for (int set = 0; set < SETS; ++set) {
                f32_row_sums(acc[set], kq, back[set], [&](uint32_t row, float val) {
                    const uint32_t m = set * kF32Rows + row;
                    if (m >= a.m || r >= a.rows) return;
                    if (nonfinite(val)) bad = TSP_ERRBIT_NONFINITE;
                    if constexpr (KSPLIT == 1) a.y[uint64_t(m) * a.rows + r] = val;
                    else joined[set * 4 + row % 4] = join(a.y, m * a.rows + r, val);
                });
            }
            continue;
        }
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const uint32_t m = 4 * kq + v;  // with eight token rows the lanes with kq >= 2 hold repeats of rows 0 .. 7
            if (m < kRows && m < a.m && r < a.rows) {
                const float val = acc[0][v] * back[0][v];
                if (nonfinite(val)) bad = TSP_ERRBIT_NONFINITE;
                if constexpr (KSPLIT == 1) a.y[uint64_t(m) * a.rows + r] = val;
                else joined[v] = join(a.y, m * a.rows + r, val);
            }
        }
    }
    if constexpr (KSPLIT == 2) check_joined(joined, bad);
    publish_error(bad, a.error_word);
}

}  // namespace

namespace tsp {

// Up to eight token rows in halves against a large matrix, where a wave with whole matrix rows is through before q8_resident.hip's workgroups (the bits are the
// same). `tiles`: of 32 rows, for each of 256 compute units; eight are as many as its waves here. us a call, there and here:
//   1536 and 2048 columns: where the tiles nearly fill a round of these waves, or fall short of half of the next one, and those of the second round and half of the third, where
//   there is little between them: eight by 48 100 x 2048 27.1 and 28.6, 58 000 32.6 and 29.8, 71 200 37.5 and 34.7, 97 600 46.6 and 46.1, 100 900 49.4 and 53.2, 124 000 58.9 and
//   57.6, 151 936 70.0 and 69.3, 168 000 76.2 and 80.7; four by 84 400 42.3 and 40.7, 151 936 66.6 and 67.1; with five only from ten tiles on (67 900 36.3 and 39.1, 84 400 42.4 and
//   41.6), with one and three in one stretch (three by 58 000 31.2 and 30.5), with two nowhere (58 000 31.1 and 32.2); by 1536 columns eight by 51 400 25.6 and 24.2, 97 600
//   38.7 and 38.4; five by 67 900 30.6 and 28.7, three by 84 400 34.8 and 34.4. (Matrices in rotation. Called with one matrix over and over, a good part of which the last-level
//   cache then keeps, this kernel is the faster one from 143 900 rows on: one by 151 936 62.3 and 60.1.)
//   1280 and 1792: five and seven waves there, one such workgroup a compute unit, are too few bytes on their way: eight by 58 000 x 1792 31.5 and 29.7, 71 200 36.5
//   and 32.8, 153 700 67.7 and 61.6, x 1280 49.9 and 46.3; with few token rows there is less to do beside them: two by 67 900 x 1792 34.4 and 34.6, 84 400 40.1 and 37.7; one by
//   54 700 (fewer are gemv.hip's) 28.3 and 26.1, 67 900 34.1 and 37.1, 91 000 41.4 and 39.1.
//   256: a workgroup of one wave there: eight by 31 600 6.7 and 6.9, 34 900 8.3 and 7.1, 150 400 14.7 and 13.6; one by 367 650 24.9 and 23.7.
//   512 to 1024: with eight, half a microsecond in a stretch each (77 800 x 512 16.3 and 15.7, 58 000 x 1024 19.4 and 18.8), else never (100 900 x 1024 27.1 and 31.8).
static bool rows_by_waves(uint32_t columns, uint32_t rows, uint32_t width) {
    const uint32_t tiles = rows / 8192;
    if (width > 8) return false;
    switch (columns / 256) {
    case 1: return tiles >= 4;
    case 2: return width == 8 && tiles >= 8 && tiles < 11;
    case 4: return width == 8 && tiles == 7;
    case 5: return tiles >= (width > 5 ? 7 : width > 2 ? 8 : width == 2 ? 10 : 12);
    case 6: return width >= 5 ? (tiles >= (width == 8 ? 6 : 8) && tiles < 12) || (tiles >= 14 && tiles < 20) : width == 3 && tiles == 10;
    case 7: return (width == 1 && tiles < 8) || tiles >= (width > 6 ? 7 : width > 3 ? 8 : 10);
    case 8: return width >= 4 && tiles < 12 ? tiles >= (width == 5 ? 10 : 6) : width >= 5 ? tiles >= 14 && tiles < 20 : width != 2 && width != 4 && tiles == 7;
    default: return false;
    }
}

bool q8_mfma_supported(const void* matrix, const float* x, uint32_t columns, uint32_t rows) {
    return columns % 256 == 0 && columns <= kMostColumns && rows >= 32 && reinterpret_cast<uintptr_t>(matrix) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(x) % 16 == 0;
}

int q8_mfma(const void* matrix, const float* x, float* y, uint32_t columns, uint32_t rows, uint32_t width, uint32_t* error_word, hipStream_t s) {
    // Up to ten token rows of 2560 columns (five where the columns are no two halves) are one pass here, with fewer matrix instructions than pieces by themselves
    // take: 2560 columns, eight token rows by 64 001 55.7 us with the top-64 behind, 63.3 the other way; sixteen, two passes, 109.7 against 71.7.
    const uint32_t at_once = columns % 512 == 0 ? 2 * kF32Rows : kF32Rows;
    // Up to 2048 columns a small matrix is multiplied by floats in three pieces, at no cost there; two halves, which the large ones take, are 2 to 3 % faster
    // (eight token rows by 151 936 x 2048 82.9 us with the top-64 behind, 85.3 in three pieces). Large: 24 576 rows, 14 000 with nine token rows or more of whole
    // 512 columns. What is below has never had fewer bits than the floats it is given.
    const bool floats = rows < (width > 8 && columns % 512 == 0 ? 14000u : 24576u);
    const bool whole_rows = columns <= kHalvesColumns && !floats && rows_by_waves(columns, rows, width);
    if (!whole_rows && (columns <= kHalvesColumns || width > at_once)) return q8_resident(false, floats, matrix, x, y, columns, rows, width, error_word, s);
    const Q8MfmaArgs a{static_cast<const uint8_t*>(matrix), x, y, columns, rows, width, error_word};
    // five rows x all columns and ten rows x half the columns stage the same number of bytes
    const uint32_t lds_bytes = 2 * 8 * columns * 2 + kWaves * kTileBytes;
    static std::atomic<uint64_t> raised{0};
    static int units_of[64] = {};
    int device = 0;
    if (setup_pending(raised, &device)) {
        const int most = int(2 * 8 * kMostColumns * 2 + kWaves * kTileBytes);
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_mfma_kernel<1, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_mfma_kernel<2, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_mfma_kernel<1, kF32Rows>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_mfma_kernel<2, kF32Rows>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_mfma_kernel<1, 2 * kF32Rows>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipDeviceGetAttribute(&units_of[device], hipDeviceAttributeMultiprocessorCount, device));
        setup_done(raised, device);
    }
    const int compute_units = units_of[device];
    const uint32_t tiles = (rows + 31) / 32;
    uint32_t grid = uint32_t(compute_units > 0 ? compute_units : 256);
    if (width > kF32Rows && !whole_rows) {  // two workgroups (one per half of the columns) share each run of tiles; the output starts at zero
        uint32_t pairs = grid / 2 ? grid / 2 : 1;
        if (pairs * kWaves > tiles) pairs = (tiles + kWaves - 1) / kWaves;
        clear_output(y, uint64_t(width) * rows, s);
        TSP_LAUNCH("q8_mfma", s, q8_mfma_kernel<1, 2 * kF32Rows><<<2 * pairs, kThreads, lds_bytes, s>>>(a));
        return launch_status("q8_mfma");
    }
    if (grid * kWaves > tiles) grid = (tiles + kWaves - 1) / kWaves;
    if (whole_rows) {
        // two items in flight measured best on MI355X (one: 72 us, two: 69 us, four: 75 us at 151 936 x 2048)
        if ((columns / 256) % 2 == 0) TSP_LAUNCH("q8_mfma", s, q8_mfma_kernel<2, 8><<<grid, kThreads, lds_bytes, s>>>(a));
        else TSP_LAUNCH("q8_mfma", s, q8_mfma_kernel<1, 8><<<grid, kThreads, lds_bytes, s>>>(a));
        return launch_status("q8_mfma");
    }
    if ((columns / 256) % 2 == 0) TSP_LAUNCH("q8_mfma", s, q8_mfma_kernel<2, kF32Rows><<<grid, kThreads, lds_bytes, s>>>(a));
    else TSP_LAUNCH("q8_mfma", s, q8_mfma_kernel<1, kF32Rows><<<grid, kThreads, lds_bytes, s>>>(a));
    return launch_status("q8_mfma");
}

bool q8_lanes_mfma_supported(const void* matrix, const float* x, uint32_t columns, uint32_t rows) {
    return columns % 512 == 0 && columns <= kMostColumns && rows >= 16 && reinterpret_cast<uintptr_t>(matrix) % 16 == 0 &&
           reinterpret_cast<uintptr_t>(x) % 16 == 0;
}

bool q8_lanes_mfma_supported_16(const void* matrix, const float* x, uint32_t columns, uint32_t rows) {
    if (columns > kHalvesColumns) return q8_lanes_mfma_supported(matrix, x, columns, rows);
    return q8_lanes_mfma_supported(matrix, x, columns, rows) && columns % 1024 == 0 && rows >= 32;
}

int q8_lanes_mfma(const void* matrix, const float* x, float* y, uint32_t columns, uint32_t rows, uint32_t width, uint32_t* error_word,
                  hipStream_t s) {
    // In one pass instead of two, though a wave's 256 columns are half a run there: 2560 columns, 16 token rows by 151 936 215 -> 157 us with the top-64 behind,
    // twelve by 33 000 71 -> 52. Where one pass is enough here it is the faster one (2048 columns, four token rows by 151 936 79 against 88).
    if (columns > kHalvesColumns && width > 2 * kF32Rows) return q8_resident(true, true, matrix, x, y, columns, rows, width, error_word, s);
    const Q8MfmaArgs a{static_cast<const uint8_t*>(matrix), x, y, columns, rows, width, error_word};
    const uint32_t lds_bytes = 2 * 8 * columns * 2 + kWaves * kLaneTileBytes;
    static std::atomic<uint64_t> raised{0};
    static int units_of[64] = {};
    int device = 0;
    if (setup_pending(raised, &device)) {
        const int most = int(2 * 8 * kMostColumns * 2 + kWaves * kLaneTileBytes);
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_lanes_mfma_kernel<1, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_lanes_mfma_kernel<2, 8>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_lanes_mfma_kernel<1, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_lanes_mfma_kernel<2, 16>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_lanes_mfma_kernel<1, kF32Rows>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&q8_lanes_mfma_kernel<1, 2 * kF32Rows>), hipFuncAttributeMaxDynamicSharedMemorySize, most));
        TSP_HIP(hipDeviceGetAttribute(&units_of[device], hipDeviceAttributeMultiprocessorCount, device));
        setup_done(raised, device);
    }
    const int compute_units = units_of[device];
    const uint32_t tiles = (rows + kLaneRows - 1) / kLaneRows;
    uint32_t grid = uint32_t(compute_units > 0 ? compute_units : 256);
    // two workgroups (one per half of a row's runs) share each stretch of tiles; the output starts at zero
    uint32_t pairs = grid / 2 ? grid / 2 : 1;
    if (pairs * kWaves > tiles) pairs = (tiles + kWaves - 1) / kWaves;
    if (columns > kHalvesColumns && width > kF32Rows) {
        // 2560 columns: one pass for up to ten token rows, where five at a time take two (151 936 rows, six token rows with the top-64 behind: 183 -> 111 us)
        clear_output(y, uint64_t(width) * rows, s);
        TSP_LAUNCH("q8_lanes_mfma", s, q8_lanes_mfma_kernel<1, 2 * kF32Rows><<<2 * pairs, kThreads, lds_bytes, s>>>(a));
        return launch_status("q8_lanes_mfma");
    }
    if (width > 8 && columns <= kHalvesColumns) {
        clear_output(y, uint64_t(width) * rows, s);
        if ((columns / 1024) % 2 == 0) TSP_LAUNCH("q8_lanes_mfma", s, q8_lanes_mfma_kernel<2, 16><<<2 * pairs, kThreads, lds_bytes, s>>>(a));
        else TSP_LAUNCH("q8_lanes_mfma", s, q8_lanes_mfma_kernel<1, 16><<<2 * pairs, kThreads, lds_bytes, s>>>(a));
        return launch_status("q8_lanes_mfma");
    }
    if (grid * kWaves > tiles) grid = (tiles + kWaves - 1) / kWaves;
    if (columns > kHalvesColumns) {  // 2560: five runs
        TSP_LAUNCH("q8_lanes_mfma", s, q8_lanes_mfma_kernel<1, kF32Rows><<<grid, kThreads, lds_bytes, s>>>(a));
        return launch_status("q8_lanes_mfma");
    }
    if ((columns / 512) % 2 == 0) TSP_LAUNCH("q8_lanes_mfma", s, q8_lanes_mfma_kernel<2, 8><<<grid, kThreads, lds_bytes, s>>>(a));
    else TSP_LAUNCH("q8_lanes_mfma", s, q8_lanes_mfma_kernel<1, 8><<<grid, kThreads, lds_bytes, s>>>(a));
    return launch_status("q8_lanes_mfma");
}

}  // namespace tsp
