// Grouped down GEMM for experts in Q8_0 planes (quants / d) or Q5_1 planes (nibbles / fifth bits / d, m) of 128 to 768 hidden units
// in multiples of 128 (512: small layers with a route an expert and more, gemm.hip), the task's h rows in LDS: y[route, channel] = 256 * sum_k h[slot, k] / 256 * w[channel, k].
//
// The launch is a stream of expert weights from HBM and of f32 results back to it; what it costs is how many requests are on
// their way. Hence:
//   * One persistent workgroup of eight waves per compute unit takes a contiguous share of the (task, 256 channels) items, as long as everyone's
//     (share_begin); consecutive shares go to one XCD. The task's <= 64 rows of h sit in LDS (80 KB at 640 hidden units), whole, so a wave sums a
//     32-channel tile over all columns by itself: no partial results, and no barrier except where the task changes.
//   * Weights are requested a whole tile ahead into registers (half a tile where all six steps would not fit them), a step of 128 columns
//     as the step at hand frees them: 5 x 4 KB per wave in flight at 640 hidden units, whole 128-byte pieces of rows by neighbouring
//     lanes. They turn into fragment order through 4 KB (2 KB) of LDS of the wave's own.
//   * A tile's results are stored at the beginning of the next one: then the requests outstanding at the head of the loop are the same
//     from wherever it is entered, and each wait counts exactly. In a task's first round there are none: the buffer they go to
//     has no bytes, and the hardware drops them. Rows a task does not have go past its end likewise; they come from past the end of the
//     h rows' buffer, as zeros, which take the least power to multiply (a first row repeated: 742.9 us a sublayer as below, now 740.7).
//   * A weight is the half nearest to d * q (d * q + m), the engine's arithmetic for these kinds: one packed half operation, one
//     rounding.
//   * Where the task changes, the next one's rows are on their way before the last results of the old one are stored.
//
// Measured (2048 tokens, 512 experts of 2560 x 640, ten selected, 615 tasks; 891 MB of Q8_0 weights and 210 MB of results): 250 us,
// where the staged kernel's short-lived workgroups took 495 (planar_staged.hip, which stays for other widths). Bound by the
// stream: 4.9 TB/s counting the rows of heavy experts that are read once per task.
#include "down_resident.hpp"
#include "mfma_quant.hpp"
#include "resident_tasks.hpp"

#include <type_traits>
#include <utility>

using namespace tsp;

namespace {

constexpr int kWaves = 8, kThreads = kWaves * kWave, kTaskRows = 64;
constexpr int kQ8 = 8, kQ51 = 7;  // the planes' source types
constexpr uint32_t kInfoSlots = kResidentInfoSlots;
constexpr uint32_t kNoRow = 0xffff0000u;  // an offset past the end of any output taken here; the 128 bytes of a tile behind it don't wrap

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
template <int KIND> struct Stage;
template <> struct Stage<kQ8> { u32x4 q[4]; u32x2 d; };
template <> struct Stage<kQ51> { u32x4 q[2], fifth, dm; };

template <int KIND, int STEPS>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void down_wide_kernel(ResidentDownArgs a) {
    constexpr uint32_t kColumns = STEPS * 128, bpr = STEPS * 4;
    constexpr uint32_t kPitch = kColumns * 2 + 16;  // sixteen lanes reading 16 bytes of sixteen rows touch all banks once
    constexpr uint32_t kStageBytes = KIND == kQ8 ? 4096 : 2048;
    constexpr int kDepth = STEPS == 6 ? 3 : STEPS;  // steps requested ahead
    constexpr bool kHalves = STEPS == 4;  // two sums of 256 columns, added: the bits of down_resident.hip, which takes the same calls with fewer routes
    constexpr uint32_t kRowAt = kTaskRows * kPitch, kInfoAt = kRowAt + kTaskRows * 4, kStagesAt = kInfoAt + 2 * kInfoSlots * 16;
    __shared__ __attribute__((aligned(16))) uint8_t lds_raw[kStagesAt + kWaves * kStageBytes];
    static_assert(sizeof(lds_raw) <= 160 * 1024, "one workgroup per compute unit");
    uint32_t* const row_at = reinterpret_cast<uint32_t*>(lds_raw + kRowAt);

    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = __builtin_amdgcn_readfirstlane(tid / kWave);
    const uint32_t n = lane % 32, khalf = lane / 32;
    const uint32_t units = a.channels / 256;
    uint8_t* const stage = lds_raw + kStagesAt + wave * kStageBytes;

    const uint32_t bound = a.task_slots, listed = a.tasks[0];
    if (listed > bound || a.tasks[1] != a.tokens * a.selected || a.classes[0] + a.classes[1] != listed) {
        if (tid == 0 && blockIdx.x == 0) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
        return;
    }
    const uint32_t groups = gridDim.x, share = (blockIdx.x % 8) * (groups / 8) + blockIdx.x / 8;

    // ---- per-lane parts of the request addresses. Q8_0: request i covers rows 8i .. 8i+7 of the tile, eight lanes per row; position
    // lane % 8 of row r holds piece (lane % 8) ^ (r / 2 % 8). Q5_1: rows 16i .. 16i+15, four lanes per row, piece (lane % 4) ^ (r / 4 % 4).
    uint32_t q_lane[2];
    if constexpr (KIND == kQ8) {
        q_lane[0] = lane / 8 * kColumns + ((lane % 8) ^ (lane / 16)) * 16;
        q_lane[1] = q_lane[0] ^ 64;  // r / 2 % 8 has its bit 2 set for odd i; a row is a multiple of 128 bytes
    } else {
        q_lane[0] = q_lane[1] = lane / 4 * (bpr * 16) + ((lane % 4) ^ (lane / 16)) * 16;
    }
    const uint32_t d_lane = n * bpr * (KIND == kQ8 ? 2 : 4);
    const uint32_t a_lane = n * kPitch + khalf * 32;
    const uint32_t w_lane = KIND == kQ8 ? n * 128 : n * 64, w_swz = KIND == kQ8 ? n / 2 % 8 : n / 4 % 4;

    uint32_t bad = 0, biggest = 0;  // biggest: the largest result's bits without the sign; anything not finite shows at the end

    auto pass = [&](auto mt_tag) {
        constexpr int MT = decltype(mt_tag)::value;
        const uint32_t* list = a.classes + 2 + (MT - 1) * bound;
        constexpr ItemLengths kLengths = KIND == kQ8 ? ItemLengths{19, 4, 2} : ItemLengths{17, 3, 2};
        const uint32_t it0 = share_begin<MT>(a.classes, units, share, groups, kLengths), it1 = share_begin<MT>(a.classes, units, share + 1, groups, kLengths);
        if (it0 >= it1) return;
        const uint32_t k0 = it0 / units, k1 = (it1 - 1) / units;  // first and last position in the kind's list
        auto first_unit = [&](uint32_t k) { return k == k0 ? it0 % units : 0; };
        auto end_unit = [&](uint32_t k) { return k == k1 ? (it1 - 1) % units + 1 : units; };
        // the share's tasks, looked up once; every wave writes the whole table for itself (the same words), one table per pass
        uint4* const info = reinterpret_cast<uint4*>(lds_raw + kInfoAt) + (MT - 1) * kInfoSlots;
        auto resolve = [&](uint32_t k) { return resolve_resident_task(a.tasks, a.counts, list[k], listed, a.experts, a.tokens, false); };
        if (lane < kInfoSlots && k0 + lane <= k1) {
            const ResidentTask t = resolve(k0 + lane);
            if (!t.ok) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
            info[lane] = pack_resident_task(t);
        }
        auto info_at = [&](uint32_t k) { return unpack_resident_task(k - k0 < kInfoSlots ? info[k - k0] : pack_resident_task(resolve(k))); };

        // ---- the request cursor, kDepth steps ahead of the arithmetic; past the end of the share the last tile is requested again (unused)
        uint32_t rk = k0, runit = first_unit(k0);
        GlobalBytes rbase, rq, rfifth, rd;
        auto point = [&]() {
            const uint32_t tile = runit * 8 + wave;
            rq = rbase + a.spec.qs_offset + uint64_t(tile) * (32 * bpr * (KIND == kQ8 ? 32 : 16));
            if constexpr (KIND == kQ51) rfifth = rbase + a.spec.qh_offset + uint64_t(tile) * (32 * bpr * 4);
            rd = rbase + a.spec.dm_offset + uint64_t(tile) * (32 * bpr * (KIND == kQ8 ? 2 : 4));
        };
        auto enter = [&]() {
            const uint64_t bits = reinterpret_cast<uint64_t>(a.down) + uint64_t(info_at(rk).expert) * a.spec.planar_expert_bytes;
            rbase = uniform_address(uint32_t(bits), uint32_t(bits >> 32));
        };
        auto advance = [&]() {
            if (runit + 1 < end_unit(rk)) ++runit;
            else if (rk != k1) { ++rk; runit = 0; enter(); }
            point();
        };
        Stage<KIND> st[kDepth];
        auto fetch = [&](Stage<KIND>& s, int step) {
#pragma unroll
            for (int i = 0; i < int(kStageBytes / 1024); ++i) s.q[i] = global_at<u32x4>(rq, q_lane[i % 2] + (KIND == kQ8 ? i * 8 * kColumns + step * 128 : i * 16 * bpr * 16 + step * 64));
            if constexpr (KIND == kQ8) {
                s.d = global_at<u32x2>(rd, d_lane + step * 8);
            } else {
                s.fifth = global_at<u32x4>(rfifth, d_lane + step * 16);
                s.dm = global_at<u32x4>(rd, d_lane + step * 16);
            }
        };
        enter();
        point();
#pragma unroll
        for (int s = 0; s < kDepth; ++s) fetch(st[s], s);
        __builtin_amdgcn_sched_barrier(0);

        f32x16 blk[MT], first[kHalves ? MT : 1];
#pragma unroll
        for (int i = 0; i < MT; ++i) blk[i] = f32x16{};
        auto store_tile = [&](uint32_t tile, bool live) {
            const uint32_t from = tile * 128;
            __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<uint8_t*>(a.y) + from, 0, live ? int(a.out_bytes - from) : 0, 0x00020000);
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    // accumulator 4 c + e of row tile i is task row 32 i + 8 c + 4 khalf + e, channel n of the tile
                    const u32x4 to = *reinterpret_cast<const u32x4*>(&row_at[i * 32 + 8 * c + 4 * khalf]);
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float val = blk[i][4 * c + e] * a.out_scale;
                        const uint32_t magnitude = __float_as_uint(val) & 0x7fffffffu;
                        biggest = biggest > magnitude ? biggest : magnitude;
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(val), out, to[e] + n * 4, 0, 0);
                    }
                }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto step = [&](auto s_tag) {
            constexpr int S = decltype(s_tag)::value;
            Stage<KIND>& cur = st[S % kDepth];
            constexpr bool kFresh = S == 0 || (kHalves && S == STEPS / 2);  // sums begin here
            if constexpr (kFresh && S > 0)
#pragma unroll
                for (int i = 0; i < MT; ++i) first[i] = blk[i];
#pragma unroll
            for (int i = 0; i < int(kStageBytes / 1024); ++i) *reinterpret_cast<u32x4*>(stage + i * 1024 + lane * 16) = cur.q[i];
            // everything a stage holds is used up before it is requested again: a value carried over would be moved at the end of
            // the loop, and the move waits for the request
            f16x2 d2[4], m2[4];
            uint32_t fifth[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                if constexpr (KIND == kQ8) {
                    const uint32_t pair = b < 2 ? cur.d.x : cur.d.y;
                    d2[b] = as_h2(__builtin_amdgcn_perm(pair, pair, b % 2 ? 0x07060706u : 0x05040504u));
                } else {
                    d2[b] = as_h2(__builtin_amdgcn_perm(cur.dm[b], cur.dm[b], 0x05040504u));
                    m2[b] = as_h2(__builtin_amdgcn_perm(cur.dm[b], cur.dm[b], 0x07060706u));
                    fifth[b] = cur.fifth[b] >> (16 * khalf);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            if (S == STEPS - kDepth) advance();
            fetch(cur, (S + kDepth) % STEPS);
            __builtin_amdgcn_sched_barrier(0);  // the tile ahead is on its way before this one is worked on
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                f16x8 f[2];
                if constexpr (KIND == kQ8) {
                    const u32x4 q = *reinterpret_cast<const u32x4*>(stage + w_lane + ((2 * b + khalf) ^ w_swz) * 16);
#pragma unroll
                    for (int ff = 0; ff < 2; ++ff) {
                        const f16x8 whole = quants8(q[2 * ff], q[2 * ff + 1]);
                        const f16x2 p0 = f16x2{whole[0], whole[1]} * d2[b], p1 = f16x2{whole[2], whole[3]} * d2[b];
                        const f16x2 p2 = f16x2{whole[4], whole[5]} * d2[b], p3 = f16x2{whole[6], whole[7]} * d2[b];
                        f[ff] = f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
                    }
                } else {
                    const u32x4 q = *reinterpret_cast<const u32x4*>(stage + w_lane + (b ^ w_swz) * 16);
                    q51_frags(q, fifth[b], d2[b], m2[b], khalf, f);
                }
#pragma unroll
                for (int ff = 0; ff < 2; ++ff)
#pragma unroll
                    for (int i = 0; i < MT; ++i) {
                        const f16x8 rows = *reinterpret_cast<const f16x8*>(lds_raw + a_lane + i * 32 * kPitch + S * 256 + b * 64 + ff * 16);
                        const f32x16 zero{};
                        blk[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(rows, f[ff], kFresh && b == 0 && ff == 0 ? zero : blk[i], 0, 0, 0);
                    }
            }
            if constexpr (kHalves && S == STEPS - 1)
#pragma unroll
                for (int i = 0; i < MT; ++i) blk[i] = first[i] + blk[i];
        };

        // ---- a task's rows: requested before the last results of the task before go out, put down when every wave has left that task
        constexpr int kPieces = MT * STEPS, kBatch = kPieces <= 8 ? kPieces : STEPS == 5 ? 8 : 6;  // as many at a time as registers are left
        u32x4 piece[kBatch];
        uint32_t route = 0;
        auto request_rows = [&](const ResidentTask& t, int from) {
            __amdgpu_buffer_rsrc_t src = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(reinterpret_cast<const uint8_t*>(a.hbuf)) + uint64_t(t.task) * (kTaskRows * kColumns * 2), 0, int(t.nrows * (kColumns * 2)), 0x00020000);
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {  // a row past the end lies past the buffer's and is zeros
                const uint32_t c = tid + (from + j) * kThreads, r = c / (STEPS * 16);
                if (from + j < kPieces) piece[j] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(src, r * (kColumns * 2) + c % (STEPS * 16) * 16, 0, 0));
            }
        };
        auto put_rows = [&](int from) {
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const uint32_t c = tid + (from + j) * kThreads, r = c / (STEPS * 16);
                if (from + j < kPieces) *reinterpret_cast<u32x4*>(lds_raw + r * kPitch + c % (STEPS * 16) * 16) = piece[j];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
        auto request_task = [&](const ResidentTask& t) {
            route = a.token_map[uint64_t(t.expert) * a.tokens + t.start + (lane < t.nrows ? lane : 0)];
            request_rows(t, 0);
            __builtin_amdgcn_sched_barrier(0);
        };
        ResidentTask cur = info_at(k0);
        request_task(cur);
        for (uint32_t k = k0; k <= k1; ++k) {
            const uint32_t u0 = first_unit(k), u1 = end_unit(k);
            lds_barrier();  // every wave has left the rows of the task before
            put_rows(0);
            if constexpr (kBatch < kPieces) {
                request_rows(cur, kBatch);
                put_rows(kBatch);
            }
            // Where task row `lane` goes. The gate/up product of the same call has checked every route against the expert; here the
            // index only has to stay inside the output.
            uint32_t at = kNoRow;
            if (lane < cur.nrows) {
                if (route < a.tokens * a.selected) at = route * uint32_t(a.y_stride);
                else bad |= TSP_ERRBIT_INDEX;
            }
            if (wave == 0) row_at[lane] = at;
            lds_barrier();
            for (uint32_t unit = u0; unit < u1; ++unit) {
                store_tile((unit != u0 ? unit - 1 : unit) * 8 + wave, unit != u0);
                [&]<int... S>(std::integer_sequence<int, S...>) { (step(std::integral_constant<int, S>{}), ...); }(std::make_integer_sequence<int, STEPS>{});
            }
            if (k < k1) cur = info_at(k + 1);
            request_task(cur);  // the last task's once more, unused
            store_tile((u1 - 1) * 8 + wave, true);
        }
    };
    pass(std::integral_constant<int, 2>{});
    pass(std::integral_constant<int, 1>{});
    if (biggest >= 0x7f800000u) bad |= TSP_ERRBIT_NONFINITE;
    publish_error(bad, a.error_word);
}

template <int KIND, int STEPS>
int launch_steps(const ResidentDownArgs& a, int groups, hipStream_t s) {
    TSP_LAUNCH("gemm_down", s, (down_wide_kernel<KIND, STEPS><<<groups, kThreads, 0, s>>>(a)));
    return launch_status("down_wide");
}
template <int KIND>
int launch_kind(const ResidentDownArgs& a, uint32_t hidden, int groups, hipStream_t s) {
    switch (hidden / 128) {
        case 1: return launch_steps<KIND, 1>(a, groups, s);
        case 2: return launch_steps<KIND, 2>(a, groups, s);
        case 3: return launch_steps<KIND, 3>(a, groups, s);
        case 4: return launch_steps<KIND, 4>(a, groups, s);
        case 5: return launch_steps<KIND, 5>(a, groups, s);
        default: return launch_steps<KIND, 6>(a, groups, s);
    }
}

}  // namespace

namespace tsp {

// The rows of 1024 hidden units (132 KB) would leave no LDS for the waves' stages; 896 are not built.
bool wide_down_takes(uint32_t source_type, uint32_t channels, uint32_t hidden) {
    return (source_type == kQ8 || source_type == kQ51) && hidden >= 128 && hidden <= 768 && hidden % 128 == 0 && channels >= 256 && channels % 256 == 0;
}

int launch_wide_down(const ResidentDownArgs& a, uint32_t hidden, hipStream_t s) {
    static std::atomic<uint64_t> seen{0};
    static int cus[64];
    int device = 0;
    if (setup_pending(seen, &device)) {
        int n = 0;
        TSP_HIP(hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, device));
        cus[device] = n >= 8 ? n / 8 * 8 : 8;
        setup_done(seen, device);
    }
    return a.spec.source_type == kQ8 ? launch_kind<kQ8>(a, hidden, cus[device], s) : launch_kind<kQ51>(a, hidden, cus[device], s);
}

}  // namespace tsp
