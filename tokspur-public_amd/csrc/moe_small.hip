// Routed MoE for 1..8 token rows (decode and speculative verify) on Pack v3 planar experts:
//   h[rid, r] = silu(Wg[e] x_t . r) * (Wu[e] x_t . r)      gate + up + SwiGLU, one kernel
//   y[rid, c] = Wd[e] h[rid] . c                            down projection
// with rid = t*selected + slot and e = ids[rid]. HBM-bound. Rows, sums and weights are f32 or more, but for the integer part of a
// Q6_K weight of up to 2048 columns against h rows that 16 bytes align: sc * (q - 32) is a half there (above 2048 in size it loses its lowest bit).
//
// This file holds the entry points, the choice of a kernel and the per-element arm, which takes any planar encoding, width and
// alignment on the union records (one per distinct expert, up to 8 tokens each). The kernels for Q4_K gate/up and for down rows
// that fit in LDS are in moe_few.hip.
#include "decode.hpp"
#include "moe_few.hpp"

using namespace tsp;

namespace {

struct SmallMoeArgs {
    const uint8_t* pair_lo;   // experts 0..E/2-1 as [gate_e, up_e]
    const uint8_t* pair_hi;   // experts E/2..E-1
    const uint8_t* down;      // [experts] planar
    const uint32_t* ids;      // [tokens*selected]
    uint32_t* meta;           // union block, or nullptr for tokens == 1
    const float* x;           // [tokens] rows, x_stride bytes apart
    float* h;                 // [tokens*selected] rows, h_stride bytes apart
    float* y;                 // [tokens*selected] rows, y_stride bytes apart
    uint64_t x_stride, h_stride, y_stride;
    uint32_t channels, hidden, experts, selected, tokens;
    tsp_planar_spec gu, dn;
    uint32_t* error_word;
};

struct Record { uint32_t expert, count; uint32_t token[8], route[8]; };

// Record `index` of the launch: a union record, or a single route when there is no union block.
__device__ __forceinline__ bool load_record(const SmallMoeArgs& a, uint32_t index, Record& r) {
    if (a.meta) {
        if (index >= a.meta[6]) return false;
        r.expert = a.meta[8 + index];
        r.count = a.meta[136 + index];
#pragma unroll
        for (int k = 0; k < 8; ++k) { r.token[k] = a.meta[264 + index * 8 + k]; r.route[k] = a.meta[1288 + index * 8 + k]; }
    } else {
        if (index >= a.tokens * a.selected) return false;
        r.expert = a.ids[index];
        r.count = 1;
#pragma unroll
        for (int k = 0; k < 8; ++k) { r.token[k] = index / a.selected; r.route[k] = index; }
    }
    return true;
}

__device__ __forceinline__ float silu_mul(float g, float u) {
    const float s = sigmoid_stable(g);
    return (g * s) * u;
}

// ------------------------------------------------------------------------------------ planar element decode (generic arm)
template <uint32_t T>
__device__ __forceinline__ float planar_element(const uint8_t* base, const tsp_planar_spec& s, uint64_t blk, uint32_t e) {
    if constexpr (T == 12 || T == 13) {
        const uint32_t grp = e / 32, l = e % 32;
        uint32_t q = (uint32_t(base[s.qs_offset + blk * 128 + (grp >> 1) * 32 + l]) >> ((grp & 1u) * 4u)) & 15u;
        if constexpr (T == 13) q |= ((uint32_t(base[s.qh_offset + blk * 32 + l]) >> grp) & 1u) << 4;
        const uint8_t* sm = base + s.sm_offset + blk * 16;
        const uint8_t* dm = base + s.dm_offset + blk * 4;
        return (half_bits_to_float(ld16(dm)) * float(sm[grp])) * float(q) - half_bits_to_float(ld16(dm + 2)) * float(sm[8 + grp]);
    } else if constexpr (T == 14) {
        const uint32_t sec = e / 128, t = e % 128;
        const uint32_t low = (uint32_t(base[s.qs_offset + blk * 128 + sec * 64 + t % 64]) >> (4 * (t / 64))) & 15u;
        const uint32_t high = (uint32_t(base[s.qh_offset + blk * 64 + sec * 32 + t % 32]) >> (2 * (t / 32))) & 3u;
        return (half_bits_to_float(ld16(base + s.dm_offset + blk * 2)) * float(int(int8_t(base[s.sm_offset + blk * 16 + e / 16])))) *
               float(int(low | (high << 4)) - 32);
    } else if constexpr (T == 7) {
        const uint32_t low = (uint32_t(base[s.qs_offset + blk * 16 + e % 16]) >> (4 * (e / 16))) & 15u;
        const uint32_t q = low | (((ld32(base + s.qh_offset + blk * 4) >> e) & 1u) << 4);
        const uint8_t* dm = base + s.dm_offset + blk * 4;
        return half_bits_to_float(ld16(dm)) * float(q) + half_bits_to_float(ld16(dm + 2));
    } else {
        static_assert(T == 8);
        return half_bits_to_float(ld16(base + s.dm_offset + blk * 2)) * float(int(int8_t(base[s.qs_offset + blk * 32 + e])));
    }
}

template <uint32_t T> constexpr uint32_t planar_block_elements() { return (T == 7 || T == 8) ? 32u : 256u; }

__device__ __forceinline__ const uint8_t* pair_base(const SmallMoeArgs& a, uint32_t expert) {
    const uint32_t half = a.experts / 2;
    const uint8_t* base = expert < half ? a.pair_lo : a.pair_hi;
    return base + uint64_t(expert < half ? expert : expert - half) * 2 * a.gu.planar_expert_bytes;
}

// grid (ceil(hidden/4), records): one wave per hidden unit, all tokens of the record.
template <uint32_t T>
__global__ __launch_bounds__(256) void gate_up_generic(SmallMoeArgs a) {
    Record rec;
    if (!load_record(a, blockIdx.y, rec)) return;
    uint32_t bad = 0;
    if (rec.expert >= a.experts) {
        if (threadIdx.x == 0 && blockIdx.x == 0) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
        return;
    }
    constexpr uint32_t E = planar_block_elements<T>();
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t r = blockIdx.x * 4 + wave;
    if (r >= a.hidden) return;
    const uint8_t* gate = pair_base(a, rec.expert);
    const uint8_t* up = gate + a.gu.planar_expert_bytes;
    const uint32_t bpr = a.channels / E;
    for (uint32_t k = 0; k < rec.count; ++k) {
        const float* x = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.x) + rec.token[k] * a.x_stride);
        float g = 0, u = 0;
        for (uint32_t c = lane; c < a.channels; c += kWave) {
            const uint64_t blk = uint64_t(r) * bpr + c / E;
            const float xv = x[c];
            g = __builtin_fmaf(planar_element<T>(gate, a.gu, blk, c % E), xv, g);
            u = __builtin_fmaf(planar_element<T>(up, a.gu, blk, c % E), xv, u);
        }
        g = wave_sum(g);
        u = wave_sum(u);
        if (lane == 0) {
            const float act = silu_mul(g, u);
            if (nonfinite(g) || nonfinite(u) || nonfinite(act)) bad = TSP_ERRBIT_NONFINITE;
            reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.h) + rec.route[k] * a.h_stride)[r] = act;
        }
    }
    publish_error(bad, a.error_word);
}

// grid (ceil(channels/4), records)
template <uint32_t T>
__global__ __launch_bounds__(256) void down_generic(SmallMoeArgs a) {
    Record rec;
    if (!load_record(a, blockIdx.y, rec)) return;
    if (rec.expert >= a.experts) return;  // flagged by the gate/up kernel of the same batch
    constexpr uint32_t E = planar_block_elements<T>();
    const uint32_t lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
    const uint32_t r = blockIdx.x * 4 + wave;
    if (r >= a.channels) return;
    const uint8_t* w = a.down + uint64_t(rec.expert) * a.dn.planar_expert_bytes;
    const uint32_t bpr = a.hidden / E;
    uint32_t bad = 0;
    for (uint32_t k = 0; k < rec.count; ++k) {
        const float* hrow = reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.h) + rec.route[k] * a.h_stride);
        float acc = 0;
        for (uint32_t c = lane; c < a.hidden; c += kWave)
            acc = __builtin_fmaf(planar_element<T>(w, a.dn, uint64_t(r) * bpr + c / E, c % E), hrow[c], acc);
        acc = wave_sum(acc);
        if (lane == 0) {
            if (nonfinite(acc)) bad = TSP_ERRBIT_NONFINITE;
            reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.y) + rec.route[k] * a.y_stride)[r] = acc;
        }
    }
    publish_error(bad, a.error_word);
}

// ------------------------------------------------------------------------------------ host side
bool coloc_pair_kinds(uint32_t gate_kind, uint32_t up_kind, uint32_t* type) {
    if (gate_kind == TSP_KIND_Q4K_COLOC_GATE && up_kind == TSP_KIND_Q4K_COLOC_UP) { *type = 12; return true; }
    if (gate_kind == TSP_KIND_Q5K_COLOC_GATE && up_kind == TSP_KIND_Q5K_COLOC_UP) { *type = 13; return true; }
    if (gate_kind == TSP_KIND_Q8_COLOC_GATE && up_kind == TSP_KIND_Q8_COLOC_UP) { *type = 8; return true; }
    return false;
}

int fill_common(const tsp_small_moe* m, SmallMoeArgs* a, bool need_down) {
    TSP_REQUIRE(m, "null small MoE description");
    uint32_t gu_type = 0;
    TSP_REQUIRE(coloc_pair_kinds(m->gate_kind, m->up_kind, &gu_type), "planar v3 co-located gate/up registration mismatch");
    TSP_REQUIRE(m->experts >= 2 && m->experts <= 512 && m->experts % 2 == 0, "co-located planar v3 requires even experts >= 2");
    TSP_REQUIRE(m->tokens >= 1 && m->tokens <= 8 && m->selected >= 1 && m->selected <= 16 && m->selected <= m->experts,
                "planar v3 gate/up row or stride geometry mismatch");
    TSP_REQUIRE(m->x_stride_bytes >= uint64_t(m->channels) * 4 && m->x_stride_bytes % 4 == 0 &&
                    m->h_stride_bytes >= uint64_t(m->hidden) * 4 && m->h_stride_bytes % 4 == 0,
                "planar v3 gate/up row or stride geometry mismatch");
    int rc = tsp_make_expert_spec(gu_type, m->channels, m->hidden, &a->gu);
    if (rc != TSP_OK) return rc;
    TSP_REQUIRE(m->pair_lo && m->pair_hi && m->ids && m->x && m->h && m->error_word, "null device pointer");
    TSP_REQUIRE(m->tokens == 1 || m->union_meta, "planar v3 small MoE requires the union block for more than one token");
    TSP_REQUIRE(reinterpret_cast<uintptr_t>(m->pair_lo) % 16 == 0 && reinterpret_cast<uintptr_t>(m->pair_hi) % 16 == 0,
                "planar v3 matrices require 16-byte alignment");
    const uint32_t routes = m->tokens * m->selected;
    const uint64_t pair_bytes = uint64_t(m->experts / 2) * 2 * a->gu.planar_expert_bytes;
    const uint64_t x_span = uint64_t(m->tokens - 1) * m->x_stride_bytes + uint64_t(m->channels) * 4;
    const uint64_t h_span = uint64_t(routes - 1) * m->h_stride_bytes + uint64_t(m->hidden) * 4;
    TSP_REQUIRE(!ranges_overlap(m->h, h_span, m->pair_lo, pair_bytes) && !ranges_overlap(m->h, h_span, m->pair_hi, pair_bytes) &&
                    !ranges_overlap(m->h, h_span, m->x, x_span) && !ranges_overlap(m->h, h_span, m->ids, uint64_t(routes) * 4) &&
                    !ranges_overlap(m->h, h_span, m->union_meta, m->union_meta ? 9280 : 0),
                "planar v3 small MoE outputs overlap inputs");
    a->pair_lo = static_cast<const uint8_t*>(m->pair_lo); a->pair_hi = static_cast<const uint8_t*>(m->pair_hi);
    a->ids = m->ids; a->meta = m->tokens > 1 ? m->union_meta : nullptr; a->x = m->x; a->h = m->h;
    a->x_stride = m->x_stride_bytes; a->h_stride = m->h_stride_bytes;
    a->channels = m->channels; a->hidden = m->hidden; a->experts = m->experts; a->selected = m->selected; a->tokens = m->tokens;
    a->error_word = m->error_word;
    if (need_down) {
        const uint32_t dn_type = m->down_kind == TSP_KIND_Q51_PLANAR ? 7u : m->down_kind == TSP_KIND_Q8_PLANAR ? 8u :
                                 m->down_kind == TSP_KIND_Q6K_PLANAR_X ? 14u : 0u;
        TSP_REQUIRE(dn_type, "planar v3 down registration mismatch");
        rc = tsp_make_expert_spec(dn_type, m->hidden, m->channels, &a->dn);
        if (rc != TSP_OK) return rc;
        TSP_REQUIRE(m->down && m->y && reinterpret_cast<uintptr_t>(m->down) % 16 == 0, "planar v3 down pointer/alignment");
        TSP_REQUIRE(m->y_stride_bytes >= uint64_t(m->channels) * 4 && m->y_stride_bytes % 4 == 0, "planar v3 down output geometry mismatch");
        const uint64_t y_span = uint64_t(routes - 1) * m->y_stride_bytes + uint64_t(m->channels) * 4;
        const uint64_t dn_bytes = uint64_t(m->experts) * a->dn.planar_expert_bytes;
        TSP_REQUIRE(!ranges_overlap(m->y, y_span, m->down, dn_bytes) && !ranges_overlap(m->y, y_span, m->h, h_span) &&
                        !ranges_overlap(m->y, y_span, m->x, x_span) && !ranges_overlap(m->y, y_span, m->ids, uint64_t(routes) * 4) &&
                        !ranges_overlap(m->y, y_span, m->pair_lo, pair_bytes) && !ranges_overlap(m->y, y_span, m->pair_hi, pair_bytes) &&
                        !ranges_overlap(m->y, y_span, m->union_meta, m->union_meta ? 9280 : 0) &&
                        !ranges_overlap(m->h, h_span, m->down, dn_bytes),
                    "planar v3 small MoE outputs overlap inputs");
        a->down = static_cast<const uint8_t*>(m->down); a->y = m->y; a->y_stride = m->y_stride_bytes;
    }
    return TSP_OK;
}

uint32_t record_slots(const SmallMoeArgs& a) {
    const uint32_t routes = a.tokens * a.selected;
    return routes < 128 ? routes : 128;
}

FewMoe few_view(const SmallMoeArgs& a, const tsp_shared_rows* shared = nullptr) {
    FewMoe v{a.pair_lo, a.pair_hi, a.down, a.ids, a.meta, a.x, a.h, a.y, a.x_stride, a.h_stride, a.y_stride,
             a.channels, a.hidden, a.experts, a.selected, a.tokens, a.gu, a.dn, a.error_word};
    if (shared) {
        v.shared_gate = static_cast<const uint8_t*>(shared->gate); v.shared_up = static_cast<const uint8_t*>(shared->up);
        v.shared_down = static_cast<const uint8_t*>(shared->down);
        v.shared_h = shared->h; v.shared_h_stride = shared->h_stride_bytes; v.shared_y = shared->y; v.shared_y_stride = shared->y_stride_bytes;
    }
    return v;
}

// The shapes the always-on expert may ride with: Q4_K co-located gate/up and Q6_K planes down, columns a multiple of 256 up to 2048,
// 16-byte aligned rows.
bool shared_may_ride(const SmallMoeArgs& a) {
    auto aligned16 = [](const void* p, uint64_t stride) { return reinterpret_cast<uintptr_t>(p) % 16 == 0 && stride % 16 == 0; };
    return a.gu.source_type == 12 && a.dn.source_type == 14 && a.channels % 256 == 0 && a.channels <= 2048 && a.hidden % 256 == 0 && a.hidden <= 2048 &&
           aligned16(a.x, a.x_stride) && aligned16(a.h, a.h_stride);
}

// Q4_K experts take the kernels of moe_few.hip, which build the union records themselves (and leave them in `meta` for the down launch
// and the caller): no launch of the union kernel goes before them. Other encodings, rows so wide that two of them don't fit in LDS, and
// Q6_K down rows whose weights are to stay floats, go weight by weight.
bool gate_up_builds_union(const SmallMoeArgs& a) { return few_gate_up_takes(few_view(a)); }

int launch_gate_up(const SmallMoeArgs& a, hipStream_t s, const tsp_shared_rows* shared = nullptr) {
    const FewMoe v = few_view(a, shared);
    if (few_gate_up_takes(v)) return launch_few_gate_up(v, s);
    TSP_REQUIRE(!shared, "the always-on expert rides only on the kernels for few tokens");
    const dim3 grid((a.hidden + 3) / 4, record_slots(a));
    switch (a.gu.source_type) {
    case 12: TSP_LAUNCH("gate_up_generic", s, gate_up_generic<12><<<grid, 256, 0, s>>>(a)); break;
    case 13: TSP_LAUNCH("gate_up_generic", s, gate_up_generic<13><<<grid, 256, 0, s>>>(a)); break;
    default: TSP_LAUNCH("gate_up_generic", s, gate_up_generic<8><<<grid, 256, 0, s>>>(a)); break;
    }
    return launch_status("gate_up_generic");
}

int launch_down(const SmallMoeArgs& a, hipStream_t s, const tsp_shared_rows* shared = nullptr) {
    const FewMoe v = few_view(a, shared);
    if (few_down_takes(v)) return launch_few_down(v, s);
    TSP_REQUIRE(!shared, "the always-on expert rides only on the kernels for few tokens");
    const dim3 grid((a.channels + 3) / 4, record_slots(a));
    switch (a.dn.source_type) {
    case 7: TSP_LAUNCH("down_generic", s, down_generic<7><<<grid, 256, 0, s>>>(a)); break;
    case 8: TSP_LAUNCH("down_generic", s, down_generic<8><<<grid, 256, 0, s>>>(a)); break;
    default: TSP_LAUNCH("down_generic", s, down_generic<14><<<grid, 256, 0, s>>>(a)); break;
    }
    return launch_status("down_generic");
}

}  // namespace

extern "C" int tsp_planar_moe_gate_up_swiglu_m8(const tsp_small_moe* m, void* stream) {
    SmallMoeArgs a{};
    int rc = fill_common(m, &a, false);
    if (rc != TSP_OK) return rc;
    const auto s = static_cast<hipStream_t>(stream);
    if (m->tokens > 1 && !gate_up_builds_union(a)) {
        rc = tsp_planar_union_build(m->ids, m->union_meta, m->experts, m->selected, m->tokens, m->hidden, m->channels, m->error_word, stream);
        if (rc != TSP_OK) return rc;
    }
    return launch_gate_up(a, s);
}

extern "C" int tsp_planar_moe_routed_m8(const tsp_small_moe* m, void* stream) {
    SmallMoeArgs a{};
    int rc = fill_common(m, &a, true);
    if (rc != TSP_OK) return rc;
    const auto s = static_cast<hipStream_t>(stream);
    if (m->tokens > 1 && !gate_up_builds_union(a)) {
        rc = tsp_planar_union_build(m->ids, m->union_meta, m->experts, m->selected, m->tokens, m->hidden, m->channels, m->error_word, stream);
        if (rc != TSP_OK) return rc;
    }
    rc = launch_gate_up(a, s);
    if (rc != TSP_OK) return rc;
    return launch_down(a, s);
}

extern "C" int tsp_planar_moe_routed_m8_shared(const tsp_small_moe* m, const tsp_shared_rows* shared, void* stream) {
    TSP_REQUIRE(shared, "null shared expert description");
    SmallMoeArgs a{};
    int rc = fill_common(m, &a, true);
    if (rc != TSP_OK) return rc;
    TSP_REQUIRE(shared->gate && shared->up && shared->down && shared->h && shared->y, "null device pointer");
    TSP_REQUIRE(shared_may_ride(a),
                "the always-on expert rides only with Q4_K co-located gate/up and Q6_K planes down, 16-byte aligned rows");
    TSP_REQUIRE(reinterpret_cast<uintptr_t>(shared->gate) % 16 == 0 && reinterpret_cast<uintptr_t>(shared->up) % 16 == 0 &&
                    reinterpret_cast<uintptr_t>(shared->down) % 16 == 0 && reinterpret_cast<uintptr_t>(shared->h) % 16 == 0 &&
                    shared->h_stride_bytes % 16 == 0 && shared->h_stride_bytes >= uint64_t(m->hidden) * 4 && shared->y_stride_bytes % 4 == 0 &&
                    shared->y_stride_bytes >= uint64_t(m->channels) * 4,
                "planar v3 small MoE shape or stride mismatch");
    const uint64_t h_span = uint64_t(m->tokens - 1) * shared->h_stride_bytes + uint64_t(m->hidden) * 4;
    const uint64_t y_span = uint64_t(m->tokens - 1) * shared->y_stride_bytes + uint64_t(m->channels) * 4;
    const uint32_t routes = m->tokens * m->selected;
    const void* others[] = {m->x, m->ids, m->h, m->y, shared->gate, shared->up, shared->down, m->union_meta};
    const uint64_t spans[] = {uint64_t(m->tokens - 1) * m->x_stride_bytes + uint64_t(m->channels) * 4, uint64_t(routes) * 4,
                              uint64_t(routes - 1) * m->h_stride_bytes + uint64_t(m->hidden) * 4, uint64_t(routes - 1) * m->y_stride_bytes + uint64_t(m->channels) * 4,
                              a.gu.planar_expert_bytes, a.gu.planar_expert_bytes, a.dn.planar_expert_bytes, m->union_meta ? 9280u : 0u};
    for (int i = 0; i < 8; ++i)
        TSP_REQUIRE(!ranges_overlap(shared->h, h_span, others[i], spans[i]) && !ranges_overlap(shared->y, y_span, others[i], spans[i]),
                    "planar v3 small MoE outputs overlap inputs");
    TSP_REQUIRE(!ranges_overlap(shared->h, h_span, shared->y, y_span), "planar v3 small MoE outputs overlap inputs");
    const auto s = static_cast<hipStream_t>(stream);
    if (m->tokens > 1 && !gate_up_builds_union(a)) {
        rc = tsp_planar_union_build(m->ids, m->union_meta, m->experts, m->selected, m->tokens, m->hidden, m->channels, m->error_word, stream);
        if (rc != TSP_OK) return rc;
    }
    rc = launch_gate_up(a, s, shared);
    if (rc != TSP_OK) return rc;
    return launch_down(a, s, shared);
}
