// The two products of the routed MoE for ONE token: each route's expert meets a single activation row, so the launch is a set of
// matrix-vector products over the routes' planes (ten experts, 13 MB of gate/up and 9 MB of Q6_K down at 2048 x 512).
//
// Every weight is multiplied as the float it stands for, up to its block's scale (a Q6_K weight sc * (q - 32) as the half that the
// kernels for more tokens have): codes become floats and meet the activations in fused multiply-adds, four chains to a block, and
// scales, minima and the sum over the blocks are 64 bits wide. No value shares an exponent with its neighbours. Against 64 bits
// throughout: 1.4e-7 of h's size and 5.5e-8 of y's (2560 x 640, Q8_0 down), where the kernels for more tokens have 1.8e-7 and 6.9e-8.
//
// Bound by one trip to memory, the launch and the issue of two instructions per weight, in about equal parts, not by the stream. So
// a wave asks for everything it will ever need before it waits: L lanes share a weight row, a lane owns every L-th unit of 64 (32)
// weights of TWO rows, the gate and up rows of a hidden unit or two rows of down, so that an activation read from LDS serves two
// weights; R units per row and lane are all in flight at once. Neighbouring lanes read neighbouring pieces, where the operand order
// of the matrix cores gathers 16 bytes from 64 places per request.
// Kernel times, ten of 512 experts (with the kernels for up to eight tokens before): gate/up 2048 x 512 9.5 -> 6.3 us, 2560 x 640
// 14.6 -> 9.2; down 512 -> 2048 Q6_K 6.6 -> 5.2, 640 -> 2560 Q8_0 9.2 -> 5.6, 768 -> 2048 Q5_1 of eight 10.1 -> 5.2.
// Lanes per row: 2048 columns at L = 32, 16, 8 take 6.3, 7.2, 7.7 us; 2560 columns at L = 32, 16, 8
// 9.8, 9.2, 10.1 (24 of 64, 8 of 48 and no lanes idle, against fewer and longer waves). Workgroups of 128 threads: 10.3 there.
#include "moe_one.hpp"

#include <type_traits>

#include "mfma_quant.hpp"

using namespace tsp;

namespace {

struct OneArgs {
    const uint8_t* w0;      // pair_lo | down experts
    const uint8_t* w1;      // pair_hi
    tsp_planar_spec spec;
    const uint32_t* ids;    // the token's routes
    const float* x;         // gate/up: the token row (stride 0); down: a row per route
    uint64_t x_stride;
    float* out;             // a row per route
    uint64_t out_stride;
    uint32_t experts, routes, n, k;
    uint32_t* error_word;
    // the always-on expert, task `routes` of the launch
    const uint8_t* shared_w0;
    const uint8_t* shared_w1;
    const float* shared_x;
    float* shared_out;
};

constexpr uint32_t unit_weights(uint32_t type) { return type == 12 || type == 14 ? 64 : 32; }
// A unit's activations lie together in LDS in the order its codes unpack; behind them the sums of its sub-blocks and padding, so
// that neighbouring lanes' 16-byte reads fall in different banks.
constexpr uint32_t unit_floats(uint32_t type) { return unit_weights(type) + 4; }

// A unit's bytes as they come from memory.
template <uint32_t T> struct Piece;
template <> struct Piece<12> { u32x4 q0, q1; uint16_t sc, mn; uint32_t dm; };
template <> struct Piece<14> { u32x4 la, lb, qh; uint2 sc; uint16_t d; };
template <> struct Piece<8> { u32x4 q0, q1; uint16_t d; };
template <> struct Piece<7> { u32x4 q; uint32_t qh, dm; };

template <uint32_t T>
__device__ __forceinline__ Piece<T> fetch(const uint8_t* w, const tsp_planar_spec& spec, uint64_t row, uint32_t units, uint32_t u) {
    const uint64_t at = row * units + u;  // the unit's place in the plane
    Piece<T> p;
    if constexpr (T == 12) {  // sub-blocks 2 (u % 4) and 2 (u % 4) + 1 of super-block u / 4
        const uint8_t* q = w + spec.qs_offset + at * 32;
        p.q0 = *reinterpret_cast<const u32x4*>(q);
        p.q1 = *reinterpret_cast<const u32x4*>(q + 16);
        const uint8_t* sm = w + spec.sm_offset + at / 4 * 16 + at % 4 * 2;
        p.sc = *reinterpret_cast<const uint16_t*>(sm);
        p.mn = *reinterpret_cast<const uint16_t*>(sm + 8);
        p.dm = *reinterpret_cast<const uint32_t*>(w + spec.dm_offset + at / 4 * 4);
    } else if constexpr (T == 14) {  // section u / 2 % 2, the 16-byte half u % 2 of each of its pieces
        const uint64_t blk = at / 4;
        const uint32_t sec = uint32_t(at) / 2 % 2, half = uint32_t(at) % 2;
        const uint8_t* ql = w + spec.qs_offset + blk * 128 + sec * 64 + half * 16;
        p.la = *reinterpret_cast<const u32x4*>(ql);
        p.lb = *reinterpret_cast<const u32x4*>(ql + 32);
        p.qh = *reinterpret_cast<const u32x4*>(w + spec.qh_offset + blk * 64 + sec * 32 + half * 16);
        p.sc = *reinterpret_cast<const uint2*>(w + spec.sm_offset + blk * 16 + sec * 8);
        p.d = *reinterpret_cast<const uint16_t*>(w + spec.dm_offset + blk * 2);
    } else if constexpr (T == 8) {
        const uint8_t* q = w + spec.qs_offset + at * 32;
        p.q0 = *reinterpret_cast<const u32x4*>(q);
        p.q1 = *reinterpret_cast<const u32x4*>(q + 16);
        p.d = *reinterpret_cast<const uint16_t*>(w + spec.dm_offset + at * 2);
    } else {
        p.q = *reinterpret_cast<const u32x4*>(w + spec.qs_offset + at * 16);
        p.qh = *reinterpret_cast<const uint32_t*>(w + spec.qh_offset + at * 4);
        p.dm = *reinterpret_cast<const uint32_t*>(w + spec.dm_offset + at * 4);
    }
    return p;
}

// Four unsigned (signed) byte codes against four activations, a chain each.
__device__ __forceinline__ void four(uint32_t codes, const float4& x, float (&sum)[4]) {
    asm("" : "+v"(codes));  // one v_cvt_f32_ubyteN per code: seen through, a masked word becomes a shift or bit field and a conversion
    sum[0] = __builtin_fmaf(float(codes & 0xffu), x.x, sum[0]);
    sum[1] = __builtin_fmaf(float((codes >> 8) & 0xffu), x.y, sum[1]);
    sum[2] = __builtin_fmaf(float((codes >> 16) & 0xffu), x.z, sum[2]);
    sum[3] = __builtin_fmaf(float(codes >> 24), x.w, sum[3]);
}
__device__ __forceinline__ void four_signed(uint32_t codes, const float4& x, float (&sum)[4]) {
    sum[0] = __builtin_fmaf(float(int8_t(codes)), x.x, sum[0]);
    sum[1] = __builtin_fmaf(float(int8_t(codes >> 8)), x.y, sum[1]);
    sum[2] = __builtin_fmaf(float(int8_t(codes >> 16)), x.z, sum[2]);
    sum[3] = __builtin_fmaf(float(int8_t(codes >> 24)), x.w, sum[3]);
}

__device__ __forceinline__ float all(const float (&sum)[4]) { return (sum[0] + sum[1]) + (sum[2] + sum[3]); }

// Two rows' units against the same activations: total[n] += the unit's share of row n.
template <uint32_t T>
__device__ __forceinline__ void multiply(const Piece<T> (&p)[2], uint32_t u, const float* xs, double (&total)[2]) {
    auto quad = [&](int i) { return *reinterpret_cast<const float4*>(xs + 4 * i); };
    if constexpr (T == 12) {
        float sum[2][2][4] = {};
#pragma unroll
        for (int i = 0; i < 8; ++i) {  // the low nibbles are the first sub-block's codes, the high ones the second's (times 16)
            const float4 a = quad(i), b = quad(8 + i);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const uint32_t word = i < 4 ? p[n].q0[i % 4] : p[n].q1[i % 4];
                four(word & 0x0f0f0f0fu, a, sum[n][0]);
                four(word & 0xf0f0f0f0u, b, sum[n][1]);
            }
        }
        const float2 sx = *reinterpret_cast<const float2*>(xs + 64);
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            const float d = half_bits_to_float(p[n].dm & 0xffffu), dmin = half_bits_to_float(p[n].dm >> 16);
            // a scale times its code is exact in 32 bits
            total[n] = __builtin_fma(double(d * float(p[n].sc & 0xffu)), double(all(sum[n][0])), total[n]);
            total[n] = __builtin_fma(double(d * (0.0625f * float(p[n].sc >> 8))), double(all(sum[n][1])), total[n]);
            total[n] = __builtin_fma(-double(dmin * float(p[n].mn & 0xffu)), double(sx.x), total[n]);
            total[n] = __builtin_fma(-double(dmin * float(p[n].mn >> 8)), double(sx.y), total[n]);
        }
    } else if constexpr (T == 14) {
        RawQ6 raw[2];
        float sum[2][4] = {};
#pragma unroll
        for (int n = 0; n < 2; ++n) { raw[n].la = p[n].la; raw[n].lb = p[n].lb; raw[n].qh = p[n].qh; raw[n].sc[0] = p[n].sc.x; raw[n].sc[1] = p[n].sc.y; }
        auto quarter = [&](auto q_tag) {  // 16 weights of one sub-scale, sc * (q - 32) as halves
            constexpr int Q = decltype(q_tag)::value;
            f16x8 f[2][2];
#pragma unroll
            for (int n = 0; n < 2; ++n) frags_q6k<Q>(raw[n], u % 2, f[n]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 x = quad(4 * Q + i);
#pragma unroll
                for (int n = 0; n < 2; ++n) {
                    const f16x8& h = f[n][i / 2];
                    sum[n][0] = __builtin_fmaf(float(h[i % 2 * 4]), x.x, sum[n][0]);
                    sum[n][1] = __builtin_fmaf(float(h[i % 2 * 4 + 1]), x.y, sum[n][1]);
                    sum[n][2] = __builtin_fmaf(float(h[i % 2 * 4 + 2]), x.z, sum[n][2]);
                    sum[n][3] = __builtin_fmaf(float(h[i % 2 * 4 + 3]), x.w, sum[n][3]);
                }
            }
        };
        quarter(std::integral_constant<int, 0>{});
        quarter(std::integral_constant<int, 1>{});
        quarter(std::integral_constant<int, 2>{});
        quarter(std::integral_constant<int, 3>{});
#pragma unroll
        for (int n = 0; n < 2; ++n) total[n] = __builtin_fma(double(half_bits_to_float(p[n].d)), double(all(sum[n])), total[n]);
    } else if constexpr (T == 8) {
        float sum[2][4] = {};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 a = quad(i);
#pragma unroll
            for (int n = 0; n < 2; ++n) four_signed(i < 4 ? p[n].q0[i % 4] : p[n].q1[i % 4], a, sum[n]);
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) total[n] = __builtin_fma(double(half_bits_to_float(p[n].d)), double(all(sum[n])), total[n]);
    } else {
        float sum[2][4] = {};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float4 a = quad(i);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const uint32_t nib = (i < 4 ? p[n].q[i % 4] : p[n].q[i % 4] >> 4) & 0x0f0f0f0fu;
                // the fifth bits of codes 4 i .. 4 i + 3, one to a byte
                const uint32_t fifth = (__umul24((p[n].qh >> (4 * i)) & 15u, 0x204081u) & 0x01010101u) << 4;
                four(nib | fifth, a, sum[n]);
            }
        }
        const float sx = xs[32];
#pragma unroll
        for (int n = 0; n < 2; ++n) {
            total[n] = __builtin_fma(double(half_bits_to_float(p[n].dm & 0xffffu)), double(all(sum[n])), total[n]);
            total[n] = __builtin_fma(double(half_bits_to_float(p[n].dm >> 16)), double(sx), total[n]);
        }
    }
}

template <int Ctrl>
__device__ __forceinline__ double dpp_add_f64(double v) {
    const uint64_t bits = uint64_t(__double_as_longlong(v));
    const uint32_t low = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(bits)), Ctrl, 0xf, 0xf, true));
    const uint32_t high = uint32_t(__builtin_amdgcn_update_dpp(0, int(uint32_t(bits >> 32)), Ctrl, 0xf, 0xf, true));
    return v + __longlong_as_double((long long)(uint64_t(high) << 32 | low));
}
// Sum over aligned groups of L lanes (8, 16, 32); every lane of a group gets it.
template <int L>
__device__ __forceinline__ double lanes_sum(double v) {
    v = dpp_add_f64<0xB1>(v);
    v = dpp_add_f64<0x4E>(v);
    v = dpp_add_f64<0x141>(v);
    if constexpr (L >= 16) v = dpp_add_f64<0x140>(v);
    if constexpr (L >= 32) v += __shfl_xor(v, 16, kWave);
    return v;
}

constexpr uint32_t kThreads = 256;

// grid (ceil(n / rows of a workgroup), routes (+ 1)). PAIR: gate and up of a hidden unit, SwiGLU at the end; else two rows of down.
template <uint32_t T, bool PAIR, int L, int R>
__global__ __launch_bounds__(kThreads) void one_row(OneArgs a) {
    constexpr uint32_t kUnit = unit_weights(T), kFloats = unit_floats(T);
    constexpr uint32_t kGroups = kWave / L;                       // lane groups of a wave, each two rows
    constexpr uint32_t kRows = kGroups * (PAIR ? 1 : 2);          // output values of a wave
    constexpr uint32_t kMine = (L * R * kUnit / 4 + kThreads - 1) / kThreads;  // float4 of activations per thread
    __shared__ __attribute__((aligned(16))) float staged[L * R * kFloats];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, in_row = lane % L, group = lane / L;
    const bool shared = a.shared_w0 != nullptr && blockIdx.y == a.routes;
    const uint32_t units = a.k / kUnit, quads = a.k / 4;

    // ---- the activations first: a few cached kilobytes, they come back first
    const float* x = shared ? a.shared_x : reinterpret_cast<const float*>(reinterpret_cast<const uint8_t*>(a.x) + blockIdx.y * a.x_stride);
    float4 xv[kMine];
    const bool x_quads = reinterpret_cast<uintptr_t>(x) % 16 == 0;  // else a row that only floats align
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t quad = tid + j * kThreads;
        xv[j] = make_float4(0, 0, 0, 0);
        if (quad < quads) {
            if (x_quads) xv[j] = reinterpret_cast<const float4*>(x)[quad];
            else xv[j] = make_float4(x[4 * quad], x[4 * quad + 1], x[4 * quad + 2], x[4 * quad + 3]);
        }
    }
    const uint32_t expert = shared ? 0 : a.ids[blockIdx.y];
    if (expert >= a.experts) {
        if (tid == 0 && blockIdx.x == 0) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
        return;
    }

    // ---- all of the wave's weights behind them (rows past the end repeat the last one, units past the row its last one)
    const uint32_t first = (blockIdx.x * (kThreads / kWave) + wave) * kRows + group;
    const uint8_t* w[2];
    uint32_t row[2];
    if constexpr (PAIR) {
        const uint32_t half = a.experts / 2;
        const uint8_t* pair = (expert < half ? a.w0 : a.w1) + uint64_t(expert < half ? expert : expert - half) * 2 * a.spec.planar_expert_bytes;
        w[0] = shared ? a.shared_w0 : pair;
        w[1] = shared ? a.shared_w1 : pair + a.spec.planar_expert_bytes;
        row[0] = row[1] = first;
    } else {
        w[0] = w[1] = shared ? a.shared_w0 : a.w0 + uint64_t(expert) * a.spec.planar_expert_bytes;
        row[0] = first;
        row[1] = first + kGroups;
    }
    Piece<T> cur[R][2];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t u0 = r * L + in_row, u = u0 < units ? u0 : units - 1;
#pragma unroll
        for (int n = 0; n < 2; ++n) cur[r][n] = fetch<T>(w[n], a.spec, row[n] < a.n ? row[n] : a.n - 1, units, u);
    }
    __builtin_amdgcn_sched_barrier(0);  // every request is out before the first wait

    // ---- the activations to LDS while the weights travel
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t quad = tid + j * kThreads;
        if constexpr (T == 12 || T == 7) {  // the sum of a sub-block of 32: eight neighbouring threads
            const float sum = octet_sum((xv[j].x + xv[j].y) + (xv[j].z + xv[j].w));
            if (quad % 8 == 0 && quad < quads) staged[quad / (kUnit / 4) * kFloats + kUnit + quad / 8 % (kUnit / 32)] = sum;
        }
        uint32_t at;
        if constexpr (T == 14) at = (quad / 64 * 4 + quad / 32 % 2 * 2 + quad / 4 % 2) * kFloats + quad / 8 % 4 * 16 + quad % 4 * 4;  // section, half | quarter
        else at = quad / (kUnit / 4) * kFloats + quad % (kUnit / 4) * 4;
        if (quad < quads) *reinterpret_cast<float4*>(staged + at) = xv[j];
    }
    __syncthreads();

    double sums[2] = {0, 0};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t u = r * L + in_row;
        if (u < units) multiply<T>(cur[r], u, staged + u * kFloats, sums);
    }
    float total[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) total[n] = float(lanes_sum<L>(sums[n]));

    uint32_t bad = 0;
    float* const out = shared ? a.shared_out : reinterpret_cast<float*>(reinterpret_cast<uint8_t*>(a.out) + blockIdx.y * a.out_stride);
    if (in_row == 0) {
        if constexpr (PAIR) {
            if (row[0] < a.n) {
                const float g = total[0], up = total[1], h = (g * sigmoid_stable(g)) * up;
                if (nonfinite(g) || nonfinite(up) || nonfinite(h)) bad = TSP_ERRBIT_NONFINITE;
                out[row[0]] = h;
            }
        } else {
#pragma unroll
            for (int n = 0; n < 2; ++n)
                if (row[n] < a.n) {
                    if (nonfinite(total[n])) bad = TSP_ERRBIT_NONFINITE;
                    out[row[n]] = total[n];
                }
        }
    }
    publish_error(bad, a.error_word);
}

template <uint32_t T, bool PAIR, int L, int R>
int launch(const char* name, const OneArgs& a, hipStream_t s) {
    constexpr uint32_t per_group = kThreads / L * (PAIR ? 1 : 2);
    const dim3 grid((a.n + per_group - 1) / per_group, a.routes + (a.shared_w0 ? 1 : 0));
    TSP_LAUNCH(name, s, one_row<T, PAIR, L, R><<<grid, kThreads, 0, s>>>(a));
    return launch_status(name);
}

// Lanes per row, and units per lane of the widest instantiation: rows of up to 3072 columns for gate/up, 1024 for down. Wider ones
// would need more registers in flight than two waves per SIMD have, or a loop; they keep the kernels for up to eight tokens.
constexpr uint32_t kGateUpLanes = 16, kGateUpMost = 3, kDownLanes = 8, kDownMost = 4;

}  // namespace

namespace tsp {

bool one_gate_up_takes(const SkinnyMoe& m) { return m.tokens == 1 && m.gu.source_type == 12 && m.channels / 64 <= kGateUpLanes * kGateUpMost; }
bool one_down_takes(const SkinnyMoe& m) {
    if (m.tokens != 1) return false;
    if (m.dn.source_type == 14) return m.hidden / 64 <= kDownLanes * 2;
    return (m.dn.source_type == 8 || m.dn.source_type == 7) && m.hidden / 32 <= kDownLanes * kDownMost;
}

int launch_one_gate_up(const SkinnyMoe& m, hipStream_t s) {
    const OneArgs a{m.pair_lo, m.pair_hi, m.gu, m.ids, m.x, 0, m.h, m.h_stride, m.experts, m.selected, m.hidden, m.channels, m.error_word,
                    m.shared_gate, m.shared_up, m.x, m.shared_h};
    const uint32_t units = m.channels / 64;
    if (units <= 16) return launch<12, true, 16, 1>("one_gate_up", a, s);
    if (units <= 32) return launch<12, true, 32, 1>("one_gate_up", a, s);
    return launch<12, true, kGateUpLanes, kGateUpMost>("one_gate_up", a, s);
}

template <uint32_t T>
static int launch_one_down_blocks(const OneArgs& a, hipStream_t s) {
    const uint32_t rounds = (a.k / 32 + kDownLanes - 1) / kDownLanes;
    if (rounds <= 2) return launch<T, false, kDownLanes, 2>("one_down", a, s);
    return rounds == 3 ? launch<T, false, kDownLanes, 3>("one_down", a, s) : launch<T, false, kDownLanes, kDownMost>("one_down", a, s);
}

int launch_one_down(const SkinnyMoe& m, hipStream_t s) {
    const OneArgs a{m.down, nullptr, m.dn, m.ids, m.h, m.h_stride, m.y, m.y_stride, m.experts, m.selected, m.channels, m.hidden, m.error_word,
                    m.shared_down, nullptr, m.shared_h, m.shared_y};
    switch (m.dn.source_type) {
    case 7: return launch_one_down_blocks<7>(a, s);
    case 8: return launch_one_down_blocks<8>(a, s);
    default: return m.hidden / 64 <= kDownLanes ? launch<14, false, kDownLanes, 1>("one_down", a, s) : launch<14, false, kDownLanes, 2>("one_down", a, s);
    }
}

}  // namespace tsp
