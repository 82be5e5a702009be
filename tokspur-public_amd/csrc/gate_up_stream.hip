// Grouped gate/up GEMM with fused SwiGLU for Q4_K experts of any width: weights and activations both stream through LDS.
//
// A workgroup of four waves owns one task (at most 64 activation rows of one expert) x 128 hidden units; a wave the gate and the up rows of 32
// units. Two workgroups share a compute unit. Products are v_mfma_f32_32x32x16_f16 on the exact integers sc * q, a super-block of 256
// columns at a time; d multiplies its f32 sum and the minima are one more product with the rows' sub-block sums (hi + lo halves).
//
// What the loop is built around: a matrix instruction leaves half of its 32 cycles to the vector ALUs, and only to instructions that
// stand between it and the next one, so unpacking must run beside multiplying all the time, with everything it needs in registers one
// group of sixteen columns ahead. 128 registers hold sums (64 rows x 64 weight rows, twice), so nothing may wait in
// registers for its turn:
//   * Every byte goes global -> LDS directly, whole lines by eight neighbouring lanes (half lines cost the address unit twice as much).
//     Activations: 64 rows x 128 bytes per step of 64 columns, into a ring of three slabs, three steps ahead. Weights: a wave's
//     own, no barrier: 32 rows' lines of the gate and of the up matrix, a super-block each, go to registers whole as its
//     first products begin, and the places are free for the next ones, three and two steps ahead. Headers (16 + 4 bytes a row) four super-blocks
//     at a time: once per super-block, 64 lanes on as many lines, they are 2.2 M more line fetches (285 -> 270 us below).
//   * Each group's fragments are read from LDS, and its codes unpacked, among the products of the group before. The one
//     barrier per step stands before the step's last group: by then every wave has the whole slab in registers, so the
//     barrier frees it and publishes the next.
//   * Every request is unconditional (past the end the last one again), so each wave waits with an exact count.
//   * A workgroup finds its task in one word pair at a place that its id names, and asks for the routes ahead of everything else: two trips
//     stand before the rows' request where there were five. The places are filled so that the XCDs' runs are alike and end on light tasks (task_order_block).
// 2048 tokens, 512 experts of 2560 x 640: 340 -> 278 us a launch (half lines through registers, a fragment read from LDS right before its product
// before; 8 us of it are the sigmoid); 2048 x 512: 224 -> 196 (the resident kernel; 4 us are sums by super-block). With places and routes first, measured
// in turn on another box: 203 -> 191 (2048 x 512), 290 -> 281. Bound by what it fetches and by its instructions at once (2048 x 512 and 2560 x 640): 0.91 and 1.36 GB,
// the planes once per task, the headers' lines twice, 0.1 GB of rows, in 167 and 250 us without any arithmetic (5.4 TB/s); the arithmetic alone
// takes 158 and 215 with nothing to wait for, 40 and 46 of it where a super-block's sums are scaled and added. Barriers and reads of rows from LDS are free.
// Rows past a task's end are zeros: in a run of launches the clock goes by the power, 189 us after a pause and 213 in a row, and there rows of
// zeros are cheap products (a first row repeated: 213 -> 209, 295 -> 292 at 2560 x 640).
// Tried: the minima's products a group ahead of their use (the other workgroup's wave fills that time already), persistent workgroups that request the next item's bytes during the last steps of this
// one (298 for 270), tasks of more than 32 rows first (280), nibbles' lines as non-temporal (285), an expert's tasks on one column tile side by side (they do not
// meet in L2 either: as many bytes).
#include "gate_up_resident.hpp"
#include "mfma_quant.hpp"
#include "resident_tasks.hpp"

#include <type_traits>

using namespace tsp;

namespace {

constexpr uint32_t kTaskRows = 64, kUnits = 128;  // rows and hidden units of a workgroup
constexpr uint32_t kSlab = kTaskRows * 128, kLines = 32 * 128;
constexpr uint32_t kLinesAt = 3 * kSlab, kHeadersAt = kLinesAt + 4 * 2 * kLines, kHeaderBytes = 64 * 64 + 64 * 16, kSumsAt = kHeadersAt + 4 * kHeaderBytes;
constexpr uint32_t kLdsBytes = kSumsAt + kTaskRows * 32;
static_assert(kLdsBytes <= 80 * 1024, "two workgroups per compute unit");

__device__ __forceinline__ void load_to_lds_4(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(lds_base), "v"(lane_offset), "s"(uniform_base) : "memory", "m0");
}

// The same from a buffer: a lane whose offset lies past its end brings zeros, and costs no fetch.
__device__ __forceinline__ void buffer_to_lds_16(u32x4 buffer, uint32_t lane_offset, uint32_t offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(lds_base), "v"(lane_offset), "s"(buffer), "s"(offset) : "memory", "m0");
}

// BY_BLOCKS: super-blocks are summed by themselves and then added up, in order, as the resident kernel's waves do, and with its roundings: a row's
// bits may not tell which of the two has had it, since that goes by the rows of the whole call. Else the two products of a super-block go
// straight to the sum, an instruction less for each.
template <bool BY_BLOCKS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void gate_up_stream_kernel(ResidentGateUpArgs a) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[kLdsBytes];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t col = lane % 32, khalf = lane / 32;
    const uint32_t bpr = a.channels / 256, steps = 4 * bpr, col_tiles = (a.hidden + kUnits - 1) / kUnits;

    // ---- (task, units) from the workgroup id: ids go to the eight XCDs in turn, and the units of a task meet in one L2
    const uint32_t place = blockIdx.x / 8;
    const OrderedTask mine = a.order[(blockIdx.x % 8) * order_pitch(a.task_slots) + place / col_tiles];
    if (!(mine.what >> 31)) return;
    ResidentTask t;
    t.task = mine.task; t.expert = mine.what & 1023u; t.start = (mine.what >> 10 & 63u) * kTaskRows; t.nrows = mine.what >> 16 & 127u;
    t.shared = t.expert == a.experts;
    const uint32_t unit0 = (place % col_tiles) * kUnits + wave * 32;
    const uint32_t half_e = a.experts / 2;
    const uint8_t* const pair = (t.expert < half_e ? a.pair_lo : a.pair_hi) + uint64_t(t.expert < half_e ? t.expert : t.expert - half_e) * 2 * a.spec.planar_expert_bytes;
    const uint8_t* const gate = t.shared ? a.shared_gate : pair;
    const uint8_t* const up = t.shared ? a.shared_up : pair + a.spec.planar_expert_bytes;

    // ---- requests
    const uint32_t lds_at = __builtin_amdgcn_readfirstlane(lds_address(lds)), my_lines = kLinesAt + wave * (2 * kLines), my_headers = kHeadersAt + wave * kHeaderBytes;
    // weights: instruction q covers rows 8 q .. 8 q + 7 of the wave's 32, eight lanes per line; position p of row n holds chunk p ^ (n / 2) % 8.
    // Hidden units come in 32s: a wave past the last one works on that and stores nothing.
    const uint32_t unit = min(unit0, a.hidden - 32);
    uint32_t w_lane[2];
#pragma unroll
    for (uint32_t q = 0; q < 2; ++q) w_lane[q] = (lane / 8) * (bpr * 128) + (((lane % 8) ^ (4 * q + lane / 16)) * 16);
    auto request_lines = [&](const uint8_t* matrix, uint32_t b, uint32_t place) {
        const uint8_t* base = matrix + a.spec.qs_offset + (uint64_t(unit) * bpr + min(b, bpr - 1)) * 128;
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) load_to_lds_16(base + q * (8 * bpr * 128), w_lane[q % 2], lds_at + place + q * 1024);
    };
    // headers, four super-blocks at a time: instruction q covers sixteen of the 32 gate and 32 up rows, four lanes per row's 64 bytes of scales and
    // minima (piece c of row n sits at position c ^ (n / 4) % 4) and its four words of d and dmin. A request past the plane's end stays on its last piece.
    const uint32_t last_block = a.hidden * bpr - 1;
    auto request_headers = [&](uint32_t b) {
#pragma unroll
        for (uint32_t q = 0; q < 4; ++q) {
            const uint8_t* const matrix = q / 2 ? up : gate;
            const uint32_t block = (unit + (q % 2) * 16 + lane / 4) * bpr + b, c = (lane % 4) ^ (lane / 16);
            load_to_lds_16(matrix + a.spec.sm_offset, min(block + c, last_block) * 16, lds_at + my_headers + q * 1024);
            load_to_lds_4(matrix + a.spec.dm_offset, min(block + lane % 4, last_block) * 4, lds_at + my_headers + 4096 + q * 256);
        }
    };
    const uint32_t gate_at = my_lines, up_at = gate_at + kLines;
    // The task's routes first, each wave its own copy: their answer alone has to be there before the rows can be asked for (a table of the
    // workgroup's behind the weights, with the expert's id of each route looked up before its row is, was three more trips one after the other).
    const uint32_t my_routes = kSumsAt + wave * 512;
    if (!t.shared) load_to_lds_4(a.token_map + uint64_t(t.expert) * a.tokens + t.start, (lane < t.nrows ? lane : 0) * 4, lds_at + my_routes);
    request_lines(gate, 0, gate_at);
    request_lines(up, 0, up_at);
    request_headers(0);

    // ---- the task's rows: a row past the end is zeros and not stored (its sums are the first row's); a route that is not the expert's shows behind the first wait,
    // and the batch is refused. Activations: instruction i covers rows 8 wave + 32 i .. + 7, eight lanes per row; sums: 16 bytes each of 64 rows x 32, sixteen rows per wave.
    uint32_t bad = 0;
    const uint32_t my_rows[3] = {wave * 8 + lane / 8, wave * 8 + lane / 8 + 32, wave * 16 + col / 2};
    uint32_t token[3], named[2] = {t.expert, t.expert};  // the experts that the first two rows' routes name
    if (t.shared) {
#pragma unroll
        for (int i = 0; i < 3; ++i) token[i] = t.start + (my_rows[i] < t.nrows ? my_rows[i] : 0);
    } else {
        wait_after_loads<16>();  // all but the requests for weights
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            uint32_t rid = *reinterpret_cast<const uint32_t*>(lds + my_routes + my_rows[i] * 4);
            if (rid >= a.tokens * a.selected) { bad = TSP_ERRBIT_INDEX; rid = 0; }
            token[i] = rid / a.selected;
            if (i < 2) named[i] = a.ids[rid];
        }
    }
    // chunk c of row n sits at position c ^ (n / 2) % 8
    const uint32_t a_chunk = ((lane % 8) ^ ((4 * wave + lane / 16) % 8)) * 16;
    uint32_t a_lane[2];  // byte offsets: 2048 tokens of 65536 channels at most
#pragma unroll
    for (uint32_t i = 0; i < 2; ++i) a_lane[i] = my_rows[i] < t.nrows ? token[i] * (a.channels * 2) + a_chunk : 0x80000000u;
    const uint64_t x_at = reinterpret_cast<uint64_t>(a.xh);
    const u32x4 x_rows{uint32_t(x_at), uint32_t(x_at >> 32) & 0xffffu, a.tokens * a.channels * 2, 0x00020000u};
    const uint32_t s_lane = token[2] * (bpr * 32) + (col % 2) * 16;
    auto request_sums = [&](uint32_t b) { if (lane < 32) load_to_lds_16(reinterpret_cast<const uint8_t*>(a.sx) + b * 32, s_lane, lds_at + kSumsAt + wave * 512); };

    // ---- fragment addresses: chunk 4 (q / 2) + 2 khalf + q % 2 of row col in a slab, chunk 2 P + khalf of row col in a wave's lines
    const uint32_t a_at = col * 128 + (((2 * khalf) ^ (col / 2 % 8)) * 16), w_at = col * 128 + ((khalf ^ (col / 2 % 8)) * 16);
    const Q4Masks masks = q4_masks();
    const Q4ScaleConsts q4s = q4_scale_consts();
    uint32_t biggest = 0;  // the largest carried half's bits without the sign: anything not finite shows at the end

    // One loop per number of 32-row tiles.
    auto run = [&](auto tiles_tag) {
        constexpr int MT = decltype(tiles_tag)::value;
        auto request_rows = [&](uint32_t step, uint32_t slab) {
            const uint32_t at = min(step, steps - 1) * 128;
#pragma unroll
            for (int i = 0; i < MT; ++i) buffer_to_lds_16(x_rows, a_lane[i], at, lds_at + slab + i * 4096 + wave * 1024);
        };
        uint32_t slab = 0, slab1 = kSlab, slab2 = 2 * kSlab;  // this step's, the next, the one after
        request_rows(0, slab);
        request_rows(1, slab1);
        request_rows(2, slab2);
        wait_all_loads();
        asm volatile("" : "+v"(named[0]), "+v"(named[1]));  // looked at from here on: sooner would be a wait for everything older
        if (named[0] != t.expert || named[1] != t.expert) bad = TSP_ERRBIT_INDEX;
        __syncthreads();

        f32x16 acc[MT][2] = {}, blk[MT][2];
        f16x8 rows[MT], w[2];    // the present group's fragments
        u32x4 raw[4][2];  // the present super-block's nibbles by step
        f16x2 scale[2];
        uint4 sm[2], sm_next[2];
        uint32_t dm[2], dm_next[2];
        auto read_rows = [&](uint32_t from, int q, f16x8 (&into)[MT]) {
            const uint32_t at = (a_at ^ uint32_t((q / 2) * 64 + (q % 2) * 16)) + from;
#pragma unroll
            for (int i = 0; i < MT; ++i) into[i] = *reinterpret_cast<const f16x8*>(lds + at + i * 4096);
        };
        auto read_raw = [&]() {
#pragma unroll
            for (uint32_t p = 0; p < 4; ++p) {
                raw[p][0] = *reinterpret_cast<const u32x4*>(lds + gate_at + (w_at ^ (p * 32)));
                raw[p][1] = *reinterpret_cast<const u32x4*>(lds + up_at + (w_at ^ (p * 32)));
            }
        };
        auto read_headers = [&](uint32_t b, uint4 (&s)[2], uint32_t (&d)[2]) {
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j) {
                s[j] = *reinterpret_cast<const uint4*>(lds + my_headers + (j * 32 + col) * 64 + (((b % 4) ^ (col / 4 % 4)) * 16));
                d[j] = *reinterpret_cast<const uint32_t*>(lds + my_headers + 4096 + (j * 32 + col) * 16 + b % 4 * 4);
            }
        };
        auto unpack = [&](auto p_tag, auto g_tag, const uint4 (&s)[2], f16x8 (&into)[2]) {
            constexpr int P = decltype(p_tag)::value, G = decltype(g_tag)::value;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (G == 0) scale[j] = q4_pair_scale<P>(s[j].x, s[j].y, q4s);
                into[j] = scaled8_q4_swapped<G / 2>(raw[P][j][2 * (G % 2)], raw[P][j][2 * (G % 2) + 1], f16x2{scale[j][G / 2], scale[j][G / 2]}, masks);
            }
        };
        // Group G (sixteen columns) of step P of super-block b
        auto group = [&](uint32_t b, auto p_tag, auto g_tag) {
            constexpr int P = decltype(p_tag)::value, G = decltype(g_tag)::value, NP = G < 3 ? P : (P + 1) % 4, NG = (G + 1) % 4;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (G == 3) {
                // What has to be there now: the next step's slab, the first request of two barriers ago; at P == 3 also the next
                // super-block's lines, requested after it and before. Younger than that are (and now and then headers, which make the wait stricter):
                constexpr int W[4] = {MT, MT + 5, MT + 9, MT};
                lds_barrier_after_loads<W[P]>();
                request_rows(b * 4 + P + 3, slab);
                if (P == 0) {
                    if (b % 4 == 3) request_headers(b + 1);  // the last of the four is in registers
                    request_sums(b);
                    request_lines(gate, b + 1, gate_at);
                }
                if (P == 1) request_lines(up, b + 1, up_at);
                const uint32_t freed = slab;
                slab = slab1; slab1 = slab2; slab2 = freed;
            }
            f16x8 rows_next[MT], w_next[2];
            read_rows(slab, NG, rows_next);
            if constexpr (G == 3 && P == 3) { read_headers(b + 1, sm_next, dm_next); read_raw(); }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const f32x16 zero{};
                    blk[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(rows[i], w[j], P == 0 && G == 0 ? zero : blk[i][j], 0, 0, 0);
                }
            unpack(std::integral_constant<int, NP>{}, std::integral_constant<int, NG>{}, P == 3 && G == 3 ? sm_next : sm, w_next);
            if constexpr (P == 3 && G == 3) {
                // acc += d * blk - dmin * sum_s Sx(hi + lo)[m, s] * mn[n, s]
                f16x8 mn[2];
                float d[2], dmin[2];
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    HdrQ4 h;
                    h.mn[0] = sm[j].z; h.mn[1] = sm[j].w;
                    mn[j] = minima_frag(h);
                    d[j] = half_bits_to_float(dm[j] & 0xffffu) * kQ4Lift; dmin[j] = half_bits_to_float(dm[j] >> 16);
                    asm volatile("" : "+v"(d[j]), "+v"(dmin[j]));  // as floats in registers: as halves they make every multiply-add a mixed-precision one
                }
#pragma unroll
                for (int i = 0; i < MT; ++i) {
                    const f16x8 sums = *reinterpret_cast<const f16x8*>(lds + kSumsAt + (i * 32 + col) * 32 + khalf * 16);
#pragma unroll
                    for (int j = 0; j < 2; ++j) {
                        const f32x16 zero{};
                        const f32x16 m = __builtin_amdgcn_mfma_f32_32x32x16_f16(sums, mn[j], zero, 0, 0, 0);
#pragma unroll
                        for (int v = 0; v < 16; ++v) {
                            if constexpr (BY_BLOCKS) acc[i][j][v] += __builtin_fmaf(-dmin[j], m[v], d[j] * blk[i][j][v]);
                            else acc[i][j][v] = __builtin_fmaf(-dmin[j], m[v], __builtin_fmaf(d[j], blk[i][j][v], acc[i][j][v]));
                        }
                    }
                }
                sm[0] = sm_next[0]; sm[1] = sm_next[1]; dm[0] = dm_next[0]; dm[1] = dm_next[1];
            } else {
#pragma unroll
                for (int m = 0; m < 2 * MT; ++m) {
                    __builtin_amdgcn_sched_group_barrier(0x8, 1, 0);             // a matrix instruction,
                    __builtin_amdgcn_sched_group_barrier(0x2, 12 / MT, 0);       // vector instructions in turn
                }
            }
#pragma unroll
            for (int i = 0; i < MT; ++i) rows[i] = rows_next[i];
            w[0] = w_next[0]; w[1] = w_next[1];
        };
        read_headers(0, sm, dm);
        read_raw();
        read_rows(slab, 0, rows);
        unpack(std::integral_constant<int, 0>{}, std::integral_constant<int, 0>{}, sm, w);
        for (uint32_t b = 0; b < bpr; ++b) {
            auto step = [&](auto p) {
                group(b, p, std::integral_constant<int, 0>{});
                group(b, p, std::integral_constant<int, 1>{});
                group(b, p, std::integral_constant<int, 2>{});
                group(b, p, std::integral_constant<int, 3>{});
            };
            step(std::integral_constant<int, 0>{});
            step(std::integral_constant<int, 1>{});
            step(std::integral_constant<int, 2>{});
            step(std::integral_constant<int, 3>{});
        }
        wait_all_loads();  // the last requests fetched what nobody reads: they must have landed before the LDS is given away

        // accumulator v of tile (i, j): row i*32 + 8*(v/4) + 4*khalf + v%4, hidden unit col. h travels to the down product as the half
        // nearest to h * 2^-8; a sum that is not finite, or a product too large for a half, leaves an infinity or a NaN there. The sigmoid is
        // the resident kernel's short one only where rows share that kernel's bits; at other widths it is good to its last places (2560 x 640,
        // 2048 tokens: 740 us a sublayer with the short one, 749).
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int v = 0; v < 16; ++v) {
                const uint32_t r = i * 32 + 8 * (v / 4) + 4 * khalf + (v % 4);
                const float g = acc[i][0][v], h = (g * (BY_BLOCKS ? sigmoid_fast(g) : sigmoid_stable(g))) * acc[i][1][v];
                const _Float16 carried = _Float16(h * 0.00390625f);
                if (r < t.nrows && unit0 < a.hidden) {
                    const uint32_t magnitude = __builtin_bit_cast(uint16_t, carried) & 0x7fffu;
                    biggest = biggest > magnitude ? biggest : magnitude;
                    a.hbuf[(uint64_t(t.task) * kTaskRows + r) * a.hidden + unit + col] = carried;
                }
            }
    };
    if (t.nrows <= 32) run(std::integral_constant<int, 1>{});
    else run(std::integral_constant<int, 2>{});
    if (biggest >= 0x7c00u) bad |= TSP_ERRBIT_NONFINITE;
    publish_error(bad, a.error_word);
}

}  // namespace

namespace tsp {

// Half a round of an XCD's 64 workgroups (one, one and a half and two: the same to 0.3 % of a sublayer, 2048 tokens).
uint32_t stream_gate_up_tail(uint32_t hidden) { return 32 / ((hidden + kUnits - 1) / kUnits); }

int launch_stream_gate_up(const ResidentGateUpArgs& a, hipStream_t s) {
    const uint32_t groups = 8 * order_pitch(a.task_slots) * ((a.hidden + kUnits - 1) / kUnits);
    if (resident_gate_up_takes(a.channels, a.hidden)) TSP_LAUNCH("gemm_gate_up_swiglu", s, gate_up_stream_kernel<true><<<groups, 256, 0, s>>>(a));
    else TSP_LAUNCH("gemm_gate_up_swiglu", s, gate_up_stream_kernel<false><<<groups, 256, 0, s>>>(a));
    return launch_status("gate_up_stream");
}

}  // namespace tsp
