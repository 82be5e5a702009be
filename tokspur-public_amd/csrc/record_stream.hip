// The two products of the T <= 8 routed MoE as streams over the union records' weights, for experts of any width:
//   gate/up + SwiGLU   h[route] = silu(Wg x_token) * (Wu x_token)   Q4_K planes
//   down               y[route] = Wd h[route]                       Q8_0, Q5_1 or Q6_K planes
//
// A step of a few tokens meets some fifty experts with one or two rows each: the launch is a stream of about a megabyte of
// weights per expert and product, and what it costs is how early that stream starts, how evenly it is cut and how many
// instructions a weight takes. Hence:
//
//   * One workgroup of eight waves per compute unit takes an equal contiguous share of the (record, 16 weight rows) tiles.
//     Inside the workgroup the share is cut once more, in pieces of two steps (512 columns; 256 for the 32-weight blocks), evenly
//     over the waves whatever tile they fall in; every piece leaves its sums in LDS, and after one barrier the pieces of a row
//     are added up in column order. No wave waits for another in between, neither an odd number of super-blocks per row nor
//     one of records leaves waves idle, and a result does not depend on how the launch was cut.
//   * The rows of the share's records go to LDS once, as an operand of sixteen rows for the 16x16x32 matrix instructions, which
//     meet 512 weights at a time; the block scales are applied to the f32 sums. Two forms:
//     f32 rows (Q8_0, Q5_1, and Q4_K above 2048 columns): at most five rows, each as three bf16 pieces that are the float
//     exactly (mfma_quant.hpp), against the integer codes q; a record of more rows is passed twice.
//     Rows of 22 bits (Q4_K and Q6_K up to 2048 columns, as the kernels for their other widths have them, skinny.hip): at most eight,
//     under a power of two per row that brings the largest magnitude near 2^14, as high halves (operand rows 0..7) and low halves
//     (rows 8..15), against the integers sc * q, resp. sc * (q - 32) (above 2048 without their lowest bit), which have too many
//     bits for bf16. Half as many scalings, and eight rows at once: at 1024 x 512, 8 tokens, a sublayer takes 34 us so and 41 in
//     the other form.
//   * A step's weight bytes are requested three steps ahead, whole 128-byte pieces of rows by neighbouring lanes, into
//     registers; they turn into fragment order through 2 to 3.5 KB of LDS of the wave's own. (A lane that requests the pieces
//     of its own row makes the address unit take ~50 cycles per request, more than the memory needs for the bytes.)
//
// Measured (kernel trace, 2560 channels x 640 hidden units, 8 tokens, 69 distinct experts: 131 MB of gate/up, 120 MB of Q8_0 or
// 85 MB of Q5_1 down): 45 us, 36 and 41, where the per-element kernels took 194 and 142. (With rows of 22 bits 43 and 34: the
// f32 form costs a scaling per 32 columns in Q4_K, and a Q5_1 block its nearest code.) Some 7 us are the launch's serial
// beginning (ids, records, table, first bytes; a microsecond more with divisions in the table's planning, 5 tokens 30.0 -> 28.6 us), the rest is a stream at 5 TB/s beside an instruction stream of equal length.
// Two tiles per step against one read of the operand (a tenth fewer instructions), and the LDS round trip of a step overlapped
// with the products of the one before, were each built and made no difference. For rows of 1, 2, 4 or 8 super-blocks the
// kernels that keep a wave's columns in registers (record_resident.hip, skinny.hip) stay the faster ones where they apply: no
// operand is read from LDS there.
//
// Error against sums in 64 bits (2-norm, per row of 16 experts, normal rows): gate/up at 2560 x 640 1.35e-7 of h (per element in f32
// 2.1e-7, rows of 22 bits 2.0e-7), Q8_0 down 8.0e-8 (8.8e-8, 9.2e-8), Q5_1 down 7.6e-8 (6.6e-8, 9.7e-8).
#include "record_stream.hpp"

#include <type_traits>

#include "grouping_device.hpp"
#include "mfma_quant.hpp"

using namespace tsp;

namespace {

constexpr uint32_t kWaves = 8, kThreads = kWaves * kWave;
constexpr uint32_t kTile = 16;        // weight rows per tile
constexpr uint32_t kMostRows = 8;     // rows of a record
constexpr uint32_t kMaxTiles = 64;    // tiles per pass over the waves, if their pieces' sums fit
constexpr uint32_t kPiece = 2;        // steps per piece
constexpr uint32_t kMaxColumns = 2560;
constexpr uint32_t kBlockWords = 2320;  // the union block
constexpr uint32_t kDepth = 3;          // steps requested ahead of the one being multiplied
constexpr uint32_t kPartialBytes = 20480;
static_assert(kUnionScratchWords * 4 <= kPartialBytes, "the union build borrows the partial results' space");
typedef uint32_t u32x4_any __attribute__((ext_vector_type(4), aligned(2)));  // 16 bytes at any even address

enum Kind : int { K_Q4K = 0, K_Q6K = 1, K_Q8 = 2, K_Q51 = 3, K_Q4K_F32 = 4 };
constexpr bool is_q4(int kind) { return kind == K_Q4K || kind == K_Q4K_F32; }

// slots: activation rows held at a time. Of f32 rows slot s < 4 has its three pieces in operand rows s, 4 + s and 12 + s, slot 4 in
// rows 8, 9 and 10: the sums of a row's pieces meet across the lane quarters, resp. in the third quarter's own registers, the two
// small ones first (sum_bytes: a slot's sums of a super-block, eight of each half, resp. of each piece). The minima are added up with the second pieces: apart from the largest sums, so that a block costs those one rounding.
template <int KIND> struct Traits;
template <> struct Traits<K_Q4K> { static constexpr uint32_t step = 256, block = 256, bytes = 128, stage = 2048 + 512, slots = 8, sum_bytes = 32; };
template <> struct Traits<K_Q4K_F32> { static constexpr uint32_t step = 256, block = 256, bytes = 128, stage = 2048 + 512, slots = 5, sum_bytes = 48; };
template <> struct Traits<K_Q6K> { static constexpr uint32_t step = 256, block = 256, bytes = 128, stage = 2048 + 1024 + 512, slots = 8; };
template <> struct Traits<K_Q8> { static constexpr uint32_t step = 128, block = 32, bytes = 32, stage = 2048 + 256, slots = 5; };
template <> struct Traits<K_Q51> { static constexpr uint32_t step = 128, block = 32, bytes = 16, stage = 1024 + 256 + 768, slots = 5; };
constexpr uint32_t kQ51SumBytes = 32;  // the slots' sums of a block: slots 0..3, zero, slot 4, two zeros

template <int KIND> constexpr uint32_t q4_sum_bytes() { if constexpr (is_q4(KIND)) return Traits<KIND>::sum_bytes; else return 0; }

// n / d as one multiplication: magic = 2^32 / d rounded up is off by less than d / 2^32 per unit, so the quotient is exact for n * d < 2^32.
struct Divisor { uint32_t d, magic; };
__device__ __forceinline__ uint32_t operator/(uint32_t n, const Divisor& v) { return v.d == 1 ? n : __umulhi(n, v.magic); }
Divisor divisor(uint32_t d) { return Divisor{d, d == 1 ? 0 : uint32_t((1ull << 32) / d + ((1ull << 32) % d != 0))}; }

struct StreamArgs {
    const float* x;            // rows of the product: tokens (gate/up) or routes (down), x_stride bytes apart
    uint64_t x_stride;
    const uint8_t* w0;         // pair_lo | down
    const uint8_t* w1;         // pair_hi
    const uint8_t* shared_w0;  // the always-on expert: gate | down
    const uint8_t* shared_w1;  // up
    const float* shared_x;     // its rows, by token
    uint64_t shared_x_stride;
    tsp_planar_spec spec;
    const uint32_t* ids;       // the routes' expert ids
    uint32_t* meta;            // the union block: written by the gate/up launch, read by the down launch; null for one token
    float* out;                // rows by route
    uint64_t out_stride;
    float* shared_out;         // rows by token
    uint64_t shared_out_stride;
    uint32_t experts, tokens, selected, n, k;  // n: weight rows (hidden units | channels); k: columns
    Divisor units, ppt;                        // tiles of a record, pieces of a tile
    uint32_t per_group;                        // 2^32 / workgroups, rounded down
    uint32_t* error_word;
};

// What a pass works on, worked out by the first wave and read by all.
struct PassTable {
    uint32_t item1, rows, tiles, next_row;  // next_row: where the pass after this one goes on in the same record, 0: with the next items
    uint64_t src[kMostRows], dst[kMostRows];  // a row's operand and result rows
    float back[kMostRows];                    // the power of two that takes a row's scaling off again
    u32x4 tile[kMaxTiles];              // expert's base (two words), first block, first slot | rows << 8 | tile within the expert << 16
};

// LDS: [16 operand rows][sub-block sums][128 zero bytes][union block][pass table][partial results][wave stages]. The operand rows
// are 16 bytes longer than their columns: sixteen lanes reading 16 bytes of sixteen rows touch all banks once.
struct Layout { uint32_t row_bytes, sums, zero, block, table, partial, stages, total; };
template <int KIND>
__host__ __device__ Layout layout_of(uint32_t columns) {
    const uint32_t padded = (columns + 255) / 256 * 256;
    Layout l;
    l.row_bytes = padded * 2 + 16;
    l.sums = 16 * l.row_bytes;
    l.zero = l.sums + (is_q4(KIND) ? Traits<KIND>::slots * (padded / 256) * q4_sum_bytes<KIND>() : KIND == K_Q51 ? padded / 32 * kQ51SumBytes : 0);
    l.block = l.zero + 128;
    l.table = l.block + kBlockWords * 4;
    l.partial = l.table + sizeof(PassTable);
    l.stages = l.partial + kPartialBytes;
    l.total = l.stages + kWaves * Traits<KIND>::stage;
    return l;
}

// PIECES: 256-column pieces of a row a lane holds while it is staged, at least k / 256 rounded up.
template <int KIND, bool SWIGLU, uint32_t PIECES>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void record_stream(StreamArgs a) {
    using T = Traits<KIND>;
    constexpr bool F32 = KIND != K_Q6K && KIND != K_Q4K, Q4 = is_q4(KIND);
    constexpr uint32_t kSlots = T::slots;
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const Layout at = layout_of<KIND>(a.k);
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t n16 = lane % 16, kq = lane / 16;
    uint32_t* const block = reinterpret_cast<uint32_t*>(lds + at.block);
    PassTable& pass = *reinterpret_cast<PassTable*>(lds + at.table);
    float* const partial = reinterpret_cast<float*>(lds + at.partial);
    uint8_t* const stage_lds = lds + at.stages + wave * T::stage;
    uint32_t bad = 0;

    // ---- the records
    if (tid < 32) reinterpret_cast<uint32_t*>(lds + at.zero)[tid] = 0;
    if (a.meta == nullptr) {  // one token: a record per route
        if (tid < a.selected) {
            block[8 + tid] = a.ids[tid]; block[136 + tid] = 1; block[264 + tid * 8] = 0; block[1288 + tid * 8] = tid;
        }
        if (tid == 0) block[6] = a.selected;
    } else if constexpr (SWIGLU) {
        const uint32_t mine = tid < a.tokens * a.selected ? a.ids[tid] : 0xffffffffu;
        const bool writer = blockIdx.x == 0;
        if (!union_block(mine, tid, kThreads, a.experts, a.selected, a.tokens, a.n, a.k, reinterpret_cast<uint32_t*>(partial),
                         [&](uint32_t word, uint32_t value) { block[word] = value; if (writer) a.meta[word] = value; },
                         [&]() { if (writer) atomicOr(a.error_word, TSP_ERRBIT_INDEX); }))
            return;
    } else {
        for (uint32_t i = tid; i < kBlockWords; i += kThreads) block[i] = a.meta[i];
    }
    __syncthreads();

    // ---- this workgroup's items: (record, 16 rows), in record order; n is a multiple of 16
    constexpr uint32_t kMats = SWIGLU ? 2 : 1;
    const uint32_t limit = a.tokens * a.selected < 128 ? a.tokens * a.selected : 128;
    const uint32_t listed = __builtin_amdgcn_readfirstlane(block[6]), live = listed < limit ? listed : limit;
    const uint32_t units = a.n / kTile, records = live + (a.shared_w0 ? 1 : 0), items = records * units;  // at most 129 x 4096
    // Where share b begins: any monotone cut will do, and this one is a multiplication (a division is some thirty dependent instructions of a
    // wave that is alone, and they all stand before the first byte is requested).
    auto share_at = [&](uint32_t b) { return b == gridDim.x ? items : __umulhi(items * b, a.per_group); };
    const uint32_t share1 = share_at(blockIdx.x + 1);
    const uint32_t bpr = a.k / T::block, last_block = a.n * bpr - 1;
    const uint32_t spt = (a.k + T::step - 1) / T::step, ppt = a.ppt.d;  // steps and pieces per tile
    if (listed > limit) bad |= TSP_ERRBIT_INDEX;

    // Lane l of the first wave looks after record k0 + l, then row slot l, then tile l. A record that does not check out has no
    // rows and reads expert 0: the batch is refused.
    // A record of more rows than slots makes passes of its own, over the same items with the rows from row0 on.
    auto plan_pass = [&](uint32_t item0, uint32_t row0) {
        const uint32_t k0 = item0 / a.units, k = k0 + lane, index = k < 128 ? k : 0;
        const bool shared = a.shared_w0 != nullptr && k == live;
        uint32_t expert = shared ? 0 : block[8 + index], count = shared ? a.tokens : block[136 + index];
        if (k >= records) count = 0;
        else if (count > kMostRows || expert >= a.experts) { count = 0; expert = 0; bad |= TSP_ERRBIT_INDEX; }
        const uint32_t first = __builtin_amdgcn_readlane(count, 0);
        const bool split = first > kSlots;
        uint32_t upto = count;
        // sums over the first sixteen lanes: more records than slots are never taken
        auto add_shifted = [&](auto control) { upto += uint32_t(__builtin_amdgcn_update_dpp(0, int(upto), decltype(control)::value, 0xf, 0xf, true)); };
        add_shifted(std::integral_constant<int, 0x111>{});
        add_shifted(std::integral_constant<int, 0x112>{});
        add_shifted(std::integral_constant<int, 0x114>{});
        add_shifted(std::integral_constant<int, 0x118>{});
        uint32_t item1 = share1 - item0 > kMaxTiles / kMats ? item0 + kMaxTiles / kMats : share1;
        const uint64_t fits = __builtin_amdgcn_ballot_w64(lane < 16 && k * units < item1 && (lane == 0 || upto <= kSlots));
        const uint32_t taken = __builtin_ctzll(~fits);  // records of this pass: nearly always all of the share's
        if ((k0 + taken) * units < item1) item1 = (k0 + taken) * units;
        const uint32_t whole = __builtin_amdgcn_readlane(upto, taken - 1), rows = !split ? whole : first - row0 < kSlots ? first - row0 : kSlots;
        // kPartialBytes / 4 / (rows * kTile * ppt * kMats), the same for a record's passes; quotients of small numbers, at least 1 / 128 apart from a whole one
        const uint32_t room = uint32_t(float(kPartialBytes / 4 / (kTile * kMats)) * __builtin_amdgcn_rcpf(float((split ? kSlots : rows ? rows : 1) * ppt)) + 0.001f);
        if (item1 - item0 > room) item1 = item0 + room;
        const uint32_t tiles = (item1 - item0) * kMats;
        if (lane == 0) { pass.item1 = item1; pass.rows = rows; pass.tiles = tiles; pass.next_row = split && row0 + rows < first ? row0 + rows : 0; }
        // slot `lane` is row `in` of record k0 + q
        uint32_t q = 0;
        for (uint32_t i = 0; i < taken; ++i) q += uint32_t(__builtin_amdgcn_readlane(upto, i)) <= lane ? 1 : 0;
        const uint32_t in = lane - (__shfl(upto, q, kWave) - __shfl(count, q, kWave)) + row0;
        if (lane < kSlots && lane >= rows) pass.src[lane] = reinterpret_cast<uint64_t>(a.x);  // read and not used
        if (lane < rows) {
            const uint32_t rk = k0 + q, ri = rk < 128 ? rk : 0;
            const bool rs = a.shared_w0 != nullptr && rk == live;
            uint32_t token = rs ? in : block[264 + ri * 8 + in], route = rs ? in : block[1288 + ri * 8 + in];
            if (!rs && (token >= a.tokens || route >= a.tokens * a.selected)) { token = route = 0; bad |= TSP_ERRBIT_INDEX; }
            pass.src[lane] = reinterpret_cast<uint64_t>(rs ? a.shared_x : a.x) + uint64_t(SWIGLU ? token : route) * (rs ? a.shared_x_stride : a.x_stride);
            pass.dst[lane] = reinterpret_cast<uint64_t>(rs ? a.shared_out : a.out) + uint64_t(route) * (rs ? a.shared_out_stride : a.out_stride);
        }
        const uint32_t tile = lane < tiles ? lane : 0, item = item0 + tile / kMats, mat = tile % kMats, tk = item / a.units - k0;
        const uint32_t te = __shfl(expert, tk, kWave), tc = __shfl(count, tk, kWave), tu = __shfl(upto, tk, kWave), unit = item - (tk + k0) * units;
        const uint8_t* base;
        if (a.shared_w0 != nullptr && tk + k0 == live) base = mat ? a.shared_w1 : a.shared_w0;
        else if constexpr (SWIGLU) {
            const uint32_t half_e = a.experts / 2;
            base = (te < half_e ? a.w0 : a.w1) + (uint64_t(te < half_e ? te : te - half_e) * 2 + mat) * a.spec.planar_expert_bytes;
        } else base = a.w0 + uint64_t(te) * a.spec.planar_expert_bytes;
        const uint64_t bits = reinterpret_cast<uint64_t>(base);
        if (lane < tiles) pass.tile[lane] = u32x4{uint32_t(bits), uint32_t(bits >> 32), unit * kTile * bpr, (tu - tc) | (split ? rows : tc) << 8 | unit << 16};
    };

    // ---- request addresses: a uniform base per step plus these lane parts.
    // Quants: 16-byte pieces, eight (four) lanes side by side on a row; piece c of row r goes to position c ^ (r / 2 % 8)
    // (c ^ (r / 4 % 4) where a row has four) of the stage. Where a row does not fill its last step, the lanes go on into the
    // row behind it, and at the end of the plane into the plane behind it: those weights meet zeros.
    struct Stage { u32x4 q[KIND == K_Q6K ? 3 : KIND == K_Q51 ? 1 : 2]; u32x4 hdr; };
    uint32_t q_lane[3] = {}, hdr_lane, hdr_step = 0;
    if constexpr (KIND == K_Q51) {
        q_lane[0] = lane / 4 * bpr * 16 + ((lane % 4) ^ (lane / 16)) * 16;
    } else {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t r = q * 8 + lane / 8;
            q_lane[q] = r * bpr * T::bytes + ((lane % 8) ^ (r / 2 % 8)) * 16;
        }
        if constexpr (KIND == K_Q6K) q_lane[2] = uint32_t(a.spec.qh_offset) + lane / 4 * bpr * 64 + ((lane % 4) ^ (lane / 16)) * 16;
    }
    if constexpr (Q4 || KIND == K_Q6K) {
        // lanes 0..15 (and 32..47) a row's scales, 16 bytes; the others the 16 bytes that END with its d (so that the last one
        // stays inside the expert)
        constexpr uint32_t d_bytes = Q4 ? 4 : 2;
        hdr_lane = lane & 16 ? uint32_t(a.spec.dm_offset) + (n16 * bpr + 1) * d_bytes - 16 : uint32_t(a.spec.sm_offset) + n16 * bpr * 16;
        hdr_step = lane & 16 ? d_bytes : 16;
    } else {
        hdr_lane = n16 * bpr + kq;
    }
    // ---- fragment addresses (LDS): the lane's columns of operand row n16, and of the sums
    const uint32_t a_lane = n16 * at.row_bytes + (KIND == K_Q4K ? kq * 128 : KIND == K_Q6K ? kq / 2 * 256 + kq % 2 * 32 : kq * 16);
    uint32_t s_lane = at.zero, s_step = 0;
    if constexpr (KIND == K_Q4K) {  // the high-half rows; the others get zeros
        if (n16 < 8 && kq < 2) { s_lane = at.sums + n16 * ((at.row_bytes - 16) / 512) * T::sum_bytes + kq * 16; s_step = T::sum_bytes; }
    } else if constexpr (KIND == K_Q4K_F32) {  // the rows of the second pieces
        if (kq < 3 && ((n16 >= 4 && n16 < 8) || n16 == 9)) {
            s_lane = at.sums + (n16 < 8 ? n16 - 4 : 4) * ((at.row_bytes - 16) / 512) * T::sum_bytes + kq * 16;
            s_step = T::sum_bytes;
        }
    } else if constexpr (KIND == K_Q51) {
        if (kq == 1 || kq == 2) { s_lane = at.sums + (kq - 1) * 16; s_step = 4 * kQ51SumBytes; }
    }

    const Q4Consts q4c = q4_consts();
    Q4ScaleConsts q4s = q4_scale_consts();
    const uint32_t q4_sel = kq & 1 ? 0x04030402u : 0x04010400u;

    uint32_t row0 = 0;
    for (uint32_t item0 = share_at(blockIdx.x); item0 < share1;) {
        if (wave == 0) plan_pass(item0, row0);
        lds_barrier();
        const uint32_t item1 = __builtin_amdgcn_readfirstlane(pass.item1), rows = __builtin_amdgcn_readfirstlane(pass.rows), tiles = __builtin_amdgcn_readfirstlane(pass.tiles);
        row0 = __builtin_amdgcn_readfirstlane(pass.next_row);  // of the next pass
        const uint32_t stride = rows * kTile, pieces = tiles * ppt, each = (pieces + kWaves - 1) / kWaves;
        const uint32_t p0 = wave * each < pieces ? wave * each : pieces, p1 = p0 + each < pieces ? p0 + each : pieces;
        const uint32_t tile0 = p0 / a.ppt, tile1 = p1 / a.ppt;
        const uint32_t s0 = tile0 * spt + (p0 - tile0 * ppt) * kPiece, s1 = tile1 * spt + (p1 - tile1 * ppt) * kPiece;

        // ---- this wave's row, requested first: loads come back in the order they were asked for
        // (Every wave asks, also where there are fewer rows than waves: a load under a branch makes the compiler drain all loads later.)
        f32x4 row[PIECES];
        const uint32_t my_slot = wave < rows ? wave : 0;
        const GlobalBytes src = uniform_address(uint32_t(pass.src[my_slot]), uint32_t(pass.src[my_slot] >> 32));
#pragma unroll
        for (uint32_t j = 0; j < PIECES; ++j) {
            const uint32_t c = j * 256 + lane * 4;
            row[j] = global_at<f32x4>(src, (c < a.k ? c : a.k - 4) * 4);
        }

        // ---- the request cursor: step -> (tile, column step); the tile's expert and first block come from the table
        uint32_t f_tile = tile0, f_step = tile0 < tiles ? s0 - tile0 * spt : 0, f_block = 0, f_left = s1 > s0 ? s1 - s0 - 1 : 0;
        GlobalBytes f_base = nullptr;
        auto enter_tile = [&](uint32_t tile) {
            const u32x4 t = pass.tile[tile];
            f_base = uniform_address(t[0], t[1]);
            f_block = __builtin_amdgcn_readfirstlane(t[2]);
        };
        auto fetch = [&](Stage& st) {  // 32-bit offsets inside one expert (the host refuses larger ones)
            const uint32_t b = f_block + f_step * (T::step / T::block);
            GlobalBytes q = f_base + uint64_t(b) * T::bytes;
            st.q[0] = global_at<u32x4>(q, q_lane[0]);
            if constexpr (KIND != K_Q51) st.q[1] = global_at<u32x4>(q, q_lane[1]);
            if constexpr (KIND == K_Q6K) st.q[2] = global_at<u32x4>(f_base + uint64_t(b) * 64, q_lane[2]);
            if constexpr (Q4 || KIND == K_Q6K) {
                st.hdr = global_at<u32x4_any>(f_base, hdr_lane + b * hdr_step);
            } else {
                uint32_t e = hdr_lane + b;
                e = e < last_block ? e : last_block;
                if constexpr (KIND == K_Q8) {
                    st.hdr[0] = global_at<uint16_t>(f_base + a.spec.dm_offset, e * 2);
                } else {
                    st.hdr[0] = global_at<uint32_t>(f_base + a.spec.qh_offset, e * 4);
                    st.hdr[1] = global_at<uint32_t>(f_base + a.spec.dm_offset, e * 4);
                }
            }
            if (f_left != 0) {  // past the wave's last step the last one is requested again (unused)
                --f_left;
                if (++f_step == spt) { f_step = 0; enter_tile(++f_tile); }
            }
        };
        Stage st[kDepth];
        if (tile0 >= tiles) f_tile = tiles - 1;  // a wave without steps asks for bytes nobody uses
        enter_tile(f_tile);
#pragma unroll
        for (uint32_t i = 0; i < kDepth; ++i) fetch(st[i]);
        __builtin_amdgcn_sched_barrier(0);  // everything is requested before the first wait

        // ---- the row becomes its operand rows
        if (wave < rows) {
            float biggest = 0;
#pragma unroll
            for (uint32_t j = 0; j < PIECES; ++j) {
                if (j * 256 + lane * 4 >= a.k) row[j] = f32x4{};
                if (nonfinite(row[j].x) || nonfinite(row[j].y) || nonfinite(row[j].z) || nonfinite(row[j].w)) bad |= TSP_ERRBIT_NONFINITE;
                biggest = fmaxf(biggest, fmaxf(fmaxf(fabsf(row[j].x), fabsf(row[j].y)), fmaxf(fabsf(row[j].z), fabsf(row[j].w))));
            }
            biggest = wave_largest(biggest);
            int shift = 0;
            if constexpr (F32) {
                shift = row_lift(biggest);
            } else if (biggest > 0 && !nonfinite(biggest)) {  // the largest |x * scale| comes to just below 2^14
                shift = 13 - (int((__float_as_uint(biggest) >> 23) & 0xffu) - 127);
                shift = shift > 100 ? 100 : shift < -100 ? -100 : shift;
            }
            const float scale = power_of_two(shift);
            if (lane == 0) pass.back[wave] = power_of_two(-shift);
            uint8_t* const at0 = lds + (!F32 || wave < 4 ? wave : 8) * at.row_bytes + lane * 8;  // of the first piece; the others follow at
            const uint32_t second = (!F32 ? 8 : wave < 4 ? 4 : 1) * at.row_bytes, third = (wave < 4 ? 12 : 2) * at.row_bytes;
#pragma unroll
            for (uint32_t j = 0; j < PIECES; ++j) {
                if (j * 256 >= a.k) break;
                const float s4[4] = {row[j].x * scale, row[j].y * scale, row[j].z * scale, row[j].w * scale};
                uint8_t* const here = at0 + j * 512;
                if constexpr (F32) {
                    const Pieces p[4] = {three_pieces(s4[0]), three_pieces(s4[1]), three_pieces(s4[2]), three_pieces(s4[3])};
                    *reinterpret_cast<uint2*>(here) = uint2{two_tops(p[0].hi, p[1].hi), two_tops(p[2].hi, p[3].hi)};
                    *reinterpret_cast<uint2*>(here + second) = uint2{two_tops(p[0].mid, p[1].mid), two_tops(p[2].mid, p[3].mid)};
                    *reinterpret_cast<uint2*>(here + third) = uint2{two_tops(p[0].lo, p[1].lo), two_tops(p[2].lo, p[3].lo)};
                } else {
                    _Float16 hi[4], lo[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) { hi[e] = _Float16(s4[e]); lo[e] = _Float16(s4[e] - float(hi[e])); }
                    constexpr int I1 = KIND == K_Q4K ? 2 : 1, I2 = 3 - I1;  // Q4_K: the order in which a dword of nibbles unpacks
                    *reinterpret_cast<f16x4*>(here) = f16x4{hi[0], hi[I1], hi[I2], hi[3]};
                    *reinterpret_cast<f16x4*>(here + second) = f16x4{lo[0], lo[I1], lo[I2], lo[3]};
                }
                if constexpr (Q4 || KIND == K_Q51) {
                    const float sum = octet_sum((s4[0] + s4[1]) + (s4[2] + s4[3]));  // eight lanes hold 32 columns
                    if (lane % 8 == 0) {
                        if constexpr (Q4) {
                            uint16_t* o = reinterpret_cast<uint16_t*>(lds + at.sums + (wave * ((at.row_bytes - 16) / 512) + j) * T::sum_bytes) + lane / 8;
                            if constexpr (F32) {
                                const Pieces p = three_pieces(sum);
                                o[0] = uint16_t(__float_as_uint(p.hi) >> 16);
                                o[8] = uint16_t(__float_as_uint(p.mid) >> 16);
                                o[16] = uint16_t(__float_as_uint(p.lo) >> 16);
                            } else {
                                const float s32 = sum * 0.03125f;
                                const _Float16 high = _Float16(s32);
                                o[0] = __builtin_bit_cast(uint16_t, high);
                                o[8] = __builtin_bit_cast(uint16_t, _Float16(s32 - float(high)));
                            }
                        } else {
                            *reinterpret_cast<float*>(lds + at.sums + (j * 8 + lane / 8) * kQ51SumBytes + (wave < 4 ? wave : 5) * 4) = sum;
                        }
                    }
                }
            }
        } else if (KIND == K_Q51 && wave >= kSlots) {  // the first and third piece of slot 4 and the row after them
            const uint32_t none = wave == kSlots ? 4 : wave;
            for (uint32_t i = lane; i < (at.zero - at.sums) / kQ51SumBytes; i += kWave) *reinterpret_cast<float*>(lds + at.sums + i * kQ51SumBytes + none * 4) = 0;
        }
        lds_barrier();

        // ---- the steps
        uint32_t c_step = s0 - tile0 * spt;
        uint32_t a_at = a_lane + c_step * (T::step * 2), s_at = s_lane + c_step * s_step;
        f32x4 acc{};
        float* out = partial + p0 * stride + (F32 ? 0 : kq * 4 * kTile) + n16;
        auto leave_piece = [&]() {
            auto halves_sum = [](float v) {  // over lanes l and l ^ 32
                const auto both = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
                return __uint_as_float(both[0]) + __uint_as_float(both[1]);
            };
            if constexpr (F32) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {  // slot v: lanes 0..15 get first + (second + third)
                    const float outer = halves_sum(kq == 2 ? 0.0f : acc[v]);
                    const auto quarters = __builtin_amdgcn_permlane16_swap(__float_as_uint(outer), __float_as_uint(outer), false, false);
                    const float all = __uint_as_float(quarters[0]) + __uint_as_float(quarters[1]);
                    if (kq == 0 && v < rows) out[v * kTile] = all;
                }
                if (kq == 2 && rows > 4) out[4 * kTile] = acc[0] + (acc[1] + acc[2]);  // in the same order
            } else {  // low-half rows 8..15 (lanes 32..63) join the high-half rows; then lanes 0..31 hold rows 4 kq + v of column n16
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const float both = halves_sum(acc[v]);
                    if (lane < 32 && kq * 4 + v < rows) out[v * kTile] = both;
                }
            }
            acc = f32x4{};
            out += stride;
        };
        auto operand = [&](uint32_t bytes) { return *reinterpret_cast<const f16x8*>(lds + a_at + bytes); };
        auto exact_operand = [&](uint32_t bytes) { return *reinterpret_cast<const bf16x8*>(lds + a_at + bytes); };
        auto body = [&](Stage& cur) {
            // registers -> LDS, and the stage is free for the step kDepth ahead (past the row's end the scales are another row's, and stay out)
            if constexpr (Q4 || KIND == K_Q6K) {
                *reinterpret_cast<u32x4*>(stage_lds + lane * 16) = cur.q[0];
                *reinterpret_cast<u32x4*>(stage_lds + 1024 + lane * 16) = cur.q[1];
                if constexpr (KIND == K_Q6K) *reinterpret_cast<u32x4*>(stage_lds + 2048 + lane * 16) = cur.q[2];
                *reinterpret_cast<u32x4*>(stage_lds + T::stage - 512 + lane % 32 * 16) = cur.hdr;
            } else if constexpr (KIND == K_Q8) {
                *reinterpret_cast<u32x4*>(stage_lds + lane * 16) = cur.q[0];
                *reinterpret_cast<u32x4*>(stage_lds + 1024 + lane * 16) = cur.q[1];
                *reinterpret_cast<float*>(stage_lds + 2048 + (n16 * 4 + kq) * 4) = c_step * 4 + kq < bpr ? half_bits_to_float(cur.hdr[0]) : 0.0f;
            } else {
                *reinterpret_cast<u32x4*>(stage_lds + lane * 16) = cur.q[0];
                *reinterpret_cast<uint32_t*>(stage_lds + 1024 + (n16 * 4 + kq) * 4) = cur.hdr[0];
                // d q + m = d (q - c) + (m + c d) with the code c that comes nearest to zero: neither part is larger than the weight by
                // more than d / 2, so the two sums lose no more than the weights' own would
                const float d = half_bits_to_float(cur.hdr[1] & 0xffffu), least = half_bits_to_float(cur.hdr[1] >> 16);
                const float c = fminf(fmaxf(__builtin_rintf(-least * __builtin_amdgcn_rcpf(d)), 0.0f), 31.0f);
                const bool inside = c_step * 4 + kq < bpr;
                *reinterpret_cast<float*>(stage_lds + 1280 + (n16 * 4 + kq) * 4) = inside ? d : 0.0f;
                *reinterpret_cast<float*>(stage_lds + 1536 + (n16 * 4 + kq) * 4) = inside ? __builtin_fmaf(c, d, least) : 0.0f;
                *reinterpret_cast<uint32_t*>(stage_lds + 1792 + (n16 * 4 + kq) * 4) = uint32_t(c) * 0x01010101u;
            }
            fetch(cur);
            const f32x4 zero{};
            if constexpr (KIND == K_Q4K) {
                // lane (row n16, kq): the 32 bytes of pair kq of the row's super-block, sub-blocks 2 kq (low nibbles) and 2 kq + 1
                const uint32_t swz = n16 / 2;
                const u32x4 raw0 = *reinterpret_cast<const u32x4*>(stage_lds + n16 * 128 + ((2 * kq) ^ swz) * 16);
                const u32x4 raw1 = *reinterpret_cast<const u32x4*>(stage_lds + n16 * 128 + ((2 * kq + 1) ^ swz) * 16);
                const u32x4 sm = *reinterpret_cast<const u32x4*>(stage_lds + 2048 + n16 * 16);
                const uint32_t dm = *reinterpret_cast<const uint32_t*>(stage_lds + 2048 + 256 + n16 * 16 + 12);
                const f16x2 sc = as_h2(__builtin_amdgcn_perm(q4s.k64, kq & 2 ? sm[1] : sm[0], q4_sel)) + q4s.off;
                const Q4PairScale ps{sc * q4s.mul, sc * q4s.bias};
                f32x4 blk;
                f16x8 f[2];
                frags_q4k_pair(raw0, ps, 0, q4c, f);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(0), f[0], zero, 0, 0, 0);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(16), f[1], blk, 0, 0, 0);
                frags_q4k_pair(raw1, ps, 0, q4c, f);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(32), f[0], blk, 0, 0, 0);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(48), f[1], blk, 0, 0, 0);
                frags_q4k_pair(raw0, ps, 1, q4c, f);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(64), f[0], blk, 0, 0, 0);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(80), f[1], blk, 0, 0, 0);
                frags_q4k_pair(raw1, ps, 1, q4c, f);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(96), f[0], blk, 0, 0, 0);
                blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(112), f[1], blk, 0, 0, 0);
                // minima: operand columns 0..7 are the high halves of the sums / 32, 8..15 their residuals, the rest and the low-half rows zero
                HdrQ4 h;
                h.mn[0] = sm[2]; h.mn[1] = sm[3];
                const f32x4 mins = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const f16x8*>(lds + s_at), minima_frag(h), zero, 0, 0, 0);
                const float d = half_bits_to_float(dm & 0xffffu), dmin = -32.0f * half_bits_to_float(dm >> 16);
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(dmin, mins[v], __builtin_fmaf(d, blk[v], acc[v]));
            } else if constexpr (KIND == K_Q4K_F32) {
                const uint32_t swz = n16 / 2;
                const u32x4 sm = *reinterpret_cast<const u32x4*>(stage_lds + 2048 + n16 * 16);
                const uint32_t dm = *reinterpret_cast<const uint32_t*>(stage_lds + 2048 + 256 + n16 * 16 + 12);
                const float d = half_bits_to_float(dm & 0xffffu), dmin = -half_bits_to_float(dm >> 16);
#pragma unroll
                for (int p = 0; p < 4; ++p) {  // sub-blocks 2 p (low nibbles) and 2 p + 1: lane kq has weights 8 kq .. 8 kq + 7 of each
                    const uint2 q = *reinterpret_cast<const uint2*>(stage_lds + n16 * 128 + ((2 * p + kq / 2) ^ swz) * 16 + kq % 2 * 8);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const bf16x8 f = nibbles8_bf16((q.x >> (4 * h)) & 0x0f0f0f0fu, (q.y >> (4 * h)) & 0x0f0f0f0fu);
                        const f32x4 sub = __builtin_amdgcn_mfma_f32_16x16x32_bf16(exact_operand((2 * p + h) * 64), f, zero, 0, 0, 0);
                        const float scale = d * float((sm[p / 2] >> (p % 2 * 16 + h * 8)) & 0xffu);
#pragma unroll
                        for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(scale, sub[v], acc[v]);
                    }
                }
                // minima: operand columns 8 i .. 8 i + 7 are the i-th pieces of the sums, the last eight and all other rows zero
                const f32x4 mins = __builtin_amdgcn_mfma_f32_16x16x32_bf16(*reinterpret_cast<const bf16x8*>(lds + s_at), codes8_bf16(sm[2], sm[3]), zero, 0, 0, 0);
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(dmin, mins[v], acc[v]);
            } else if constexpr (KIND == K_Q6K) {
                const uint32_t sec = kq / 2, half = kq % 2, swz = n16 / 2;
                RawQ6 raw;
                raw.la = *reinterpret_cast<const u32x4*>(stage_lds + n16 * 128 + ((sec * 4 + half) ^ swz) * 16);
                raw.lb = *reinterpret_cast<const u32x4*>(stage_lds + n16 * 128 + ((sec * 4 + 2 + half) ^ swz) * 16);
                raw.qh = *reinterpret_cast<const u32x4*>(stage_lds + 2048 + n16 * 64 + (kq ^ (n16 / 4)) * 16);
                const uint2 sc = *reinterpret_cast<const uint2*>(stage_lds + 3072 + n16 * 16 + sec * 8);
                raw.sc[0] = sc.x; raw.sc[1] = sc.y;
                const float d = half_bits_to_float(*reinterpret_cast<const uint16_t*>(stage_lds + 3072 + 256 + n16 * 16 + 14));
                f32x4 blk{};
                auto quarter = [&](auto q_tag) {
                    constexpr int Q = decltype(q_tag)::value;
                    f16x8 f[2];
                    frags_q6k<Q>(raw, half, f);
                    blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(Q * 64), f[0], blk, 0, 0, 0);
                    blk = __builtin_amdgcn_mfma_f32_16x16x32_f16(operand(Q * 64 + 16), f[1], blk, 0, 0, 0);
                };
                quarter(std::integral_constant<int, 0>{});
                quarter(std::integral_constant<int, 1>{});
                quarter(std::integral_constant<int, 2>{});
                quarter(std::integral_constant<int, 3>{});
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(d, blk[v], acc[v]);
            } else if constexpr (KIND == K_Q8) {
                const f32x4 d = *reinterpret_cast<const f32x4*>(stage_lds + 2048 + n16 * 16);
                const uint32_t swz = n16 / 2;
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // a block is one instruction: lane kq has quants 8 kq .. 8 kq + 7
                    const uint2 q = *reinterpret_cast<const uint2*>(stage_lds + n16 * 128 + ((2 * j + kq / 2) ^ swz) * 16 + kq % 2 * 8);
                    const f32x4 blk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(exact_operand(j * 64), quants8_bf16(q.x, q.y), zero, 0, 0, 0);
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(d[j], blk[v], acc[v]);
                }
            } else {
                const u32x4 qh = *reinterpret_cast<const u32x4*>(stage_lds + 1024 + n16 * 16);
                const f32x4 d = *reinterpret_cast<const f32x4*>(stage_lds + 1280 + n16 * 16), m = *reinterpret_cast<const f32x4*>(stage_lds + 1536 + n16 * 16);
                const u32x4 nearest = *reinterpret_cast<const u32x4*>(stage_lds + 1792 + n16 * 16);
                const uint32_t swz = n16 / 4;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    // lane kq has weights 8 kq .. 8 kq + 7: low nibbles of the first or second eight bytes for kq < 2, then the high ones
                    const uint2 q = *reinterpret_cast<const uint2*>(stage_lds + n16 * 64 + (j ^ swz) * 16 + kq % 2 * 8);
                    const uint32_t fifth = qh[j] >> (8 * kq);
                    // bit i of the eight goes to bit 4 of byte i % 4; a byte's code is then 128 more until c is off it
                    const uint32_t f0 = ((fifth & 15u) * 0x00204081u & 0x01010101u) << 4, f1 = ((fifth >> 4 & 15u) * 0x00204081u & 0x01010101u) << 4;
                    const uint32_t w0 = (((q.x >> (kq / 2 * 4) & 0x0f0f0f0fu) | f0 | 0x80808080u) - nearest[j]) ^ 0x80808080u;
                    const uint32_t w1 = (((q.y >> (kq / 2 * 4) & 0x0f0f0f0fu) | f1 | 0x80808080u) - nearest[j]) ^ 0x80808080u;
                    const f32x4 blk = __builtin_amdgcn_mfma_f32_16x16x32_bf16(exact_operand(j * 64), quants8_bf16(w0, w1), zero, 0, 0, 0);
                    // the block's minimum times its rows' sums: once per row (the operand rows of the other pieces read zeros)
                    const f32x4 s = *reinterpret_cast<const f32x4*>(lds + s_at + j * kQ51SumBytes);
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[v] = __builtin_fmaf(m[j], s[v], __builtin_fmaf(d[j], blk[v], acc[v]));
                }
            }
            ++c_step;
            a_at += T::step * 2;
            s_at += s_step;
            if (c_step % kPiece == 0 || c_step == spt) leave_piece();
            if (c_step == spt) { c_step = 0; a_at = a_lane; s_at = s_lane; }
        };
        uint32_t s = s0;
        for (; s + kDepth <= s1; s += kDepth)
#pragma unroll
            for (uint32_t i = 0; i < kDepth; ++i) body(st[i]);
#pragma unroll
        for (uint32_t i = 0; i < kDepth - 1; ++i)
            if (s + i < s1) body(st[i]);
        lds_barrier();

        // ---- a row's pieces meet, in column order; a thread finishes one value of a row
        for (uint32_t i = tid / 128; i < item1 - item0; i += kThreads / 128) {
            const uint32_t info = pass.tile[i * kMats][3], r = tid / 16 % 8, slot = (info & 255u) + r, n = (info >> 16) * kTile + n16;
            if (r >= (info >> 8 & 255u)) continue;
            auto total = [&](uint32_t tile) {
                const float* piece = partial + tile * ppt * stride + slot * kTile + n16;
                float sum = piece[0];
                for (uint32_t q = 1; q < ppt; ++q) sum += piece[q * stride];
                return sum * pass.back[slot];
            };
            float value;
            if constexpr (SWIGLU) {
                const float g = total(i * 2), u = total(i * 2 + 1);
                value = (g * sigmoid_stable(g)) * u;
                if (nonfinite(g) || nonfinite(u) || nonfinite(value)) bad |= TSP_ERRBIT_NONFINITE;
            } else {
                value = total(i);
                if (nonfinite(value)) bad |= TSP_ERRBIT_NONFINITE;
            }
            reinterpret_cast<float __attribute__((address_space(1)))*>(pass.dst[slot])[n] = value;
        }
        if (row0 == 0) item0 = item1;
        if (item0 < share1) __syncthreads();  // the table, the rows and the partial results are taken over by the next pass
    }
    publish_error(bad, a.error_word);
}

int compute_units(int* out) {
    static std::atomic<uint64_t> seen{0};
    static int cus[64];
    int device = 0;
    if (setup_pending(seen, &device)) {
        int n = 0;
        TSP_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device));
        cus[device] = n >= 1 ? n : 1;
        setup_done(seen, device);
    }
    *out = cus[device];
    return TSP_OK;
}

template <int KIND, bool SWIGLU, uint32_t PIECES>
int launch_pieces(const char* name, const StreamArgs& a, hipStream_t s) {
    static std::atomic<uint64_t> raised{0};
    int device = 0, cus = 0;
    if (setup_pending(raised, &device)) {
        TSP_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(&record_stream<KIND, SWIGLU, PIECES>), hipFuncAttributeMaxDynamicSharedMemorySize,
                                    int(layout_of<KIND>(PIECES * 256).total)));
        setup_done(raised, device);
    }
    const int rc = compute_units(&cus);
    if (rc != TSP_OK) return rc;
    StreamArgs g = a;
    const uint32_t spt = (a.k + Traits<KIND>::step - 1) / Traits<KIND>::step;
    g.units = divisor(a.n / kTile);
    g.ppt = divisor((spt + kPiece - 1) / kPiece);
    g.per_group = uint32_t((1ull << 32) / (cus > 1 ? cus : 2));
    TSP_LAUNCH(name, s, record_stream<KIND, SWIGLU, PIECES><<<cus > 1 ? cus : 2, kThreads, layout_of<KIND>(a.k).total, s>>>(g));
    return launch_status(name);
}

template <int KIND, bool SWIGLU>
int launch(const char* name, const StreamArgs& a, hipStream_t s) {
    constexpr bool narrow = KIND != K_Q4K_F32, wide = KIND != K_Q4K && KIND != K_Q6K;  // up to 2048 columns, beyond
    if constexpr (narrow) {
        if (a.k <= 4 * 256) return launch_pieces<KIND, SWIGLU, 4>(name, a, s);
        if (!wide || a.k <= 8 * 256) return launch_pieces<KIND, SWIGLU, 8>(name, a, s);
    }
    if constexpr (wide) return launch_pieces<KIND, SWIGLU, kMaxColumns / 256>(name, a, s);
}

bool aligned16(const void* p, uint64_t stride) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 16 == 0; }

}  // namespace

namespace tsp {

bool record_stream_gate_up_takes(const SkinnyMoe& m) {
    return m.gu.source_type == 12 && m.channels <= kMaxColumns && m.gu.planar_expert_bytes < (1ull << 32) && aligned16(m.x, m.x_stride) && m.tokens <= kMostRows && m.hidden % kTile == 0;
}

int launch_record_stream_gate_up(const SkinnyMoe& m, hipStream_t s) {
    StreamArgs a{};
    a.x = m.x; a.x_stride = m.x_stride; a.w0 = m.pair_lo; a.w1 = m.pair_hi; a.spec = m.gu; a.ids = m.ids; a.meta = m.tokens > 1 ? m.meta : nullptr;
    a.out = m.h; a.out_stride = m.h_stride; a.experts = m.experts; a.tokens = m.tokens; a.selected = m.selected; a.n = m.hidden; a.k = m.channels;
    a.error_word = m.error_word;
    if (m.shared_gate) {
        a.shared_w0 = m.shared_gate; a.shared_w1 = m.shared_up; a.shared_x = m.x; a.shared_x_stride = m.x_stride;
        a.shared_out = m.shared_h; a.shared_out_stride = m.shared_h_stride;
    }
    // Q4_K rows of more columns than the kernels in halves take keep f32 rows
    return m.channels > 2048 ? launch<K_Q4K_F32, true>("record_gate_up_swiglu", a, s) : launch<K_Q4K, true>("record_gate_up_swiglu", a, s);
}

bool record_stream_down_takes(const SkinnyMoe& m) {
    // Q6_K in halves only as far as its other widths are (skinny.hip): beyond, the per-element kernel keeps the rows in f32
    return (m.dn.source_type == 8 || m.dn.source_type == 7 || (m.dn.source_type == 14 && m.hidden <= 2048)) && m.hidden <= kMaxColumns && m.dn.planar_expert_bytes < (1ull << 32) &&
           aligned16(m.h, m.h_stride) && m.tokens <= kMostRows && m.channels % kTile == 0;
}

int launch_record_stream_down(const SkinnyMoe& m, hipStream_t s) {
    StreamArgs a{};
    a.x = m.h; a.x_stride = m.h_stride; a.w0 = m.down; a.spec = m.dn; a.ids = m.ids; a.meta = m.tokens > 1 ? m.meta : nullptr;
    a.out = m.y; a.out_stride = m.y_stride; a.experts = m.experts; a.tokens = m.tokens; a.selected = m.selected; a.n = m.channels; a.k = m.hidden;
    a.error_word = m.error_word;
    if (m.shared_down) {
        a.shared_w0 = m.shared_down; a.shared_x = m.shared_h; a.shared_x_stride = m.shared_h_stride;
        a.shared_out = m.shared_y; a.shared_out_stride = m.shared_y_stride;
    }
    if (m.dn.source_type == 8) return launch<K_Q8, false>("record_down", a, s);
    if (m.dn.source_type == 7) return launch<K_Q51, false>("record_down", a, s);
    return launch<K_Q6K, false>("record_down", a, s);
}

}  // namespace tsp
