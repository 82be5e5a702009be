// The two products of the routed MoE for one to eight tokens: an expert meets one activation row, seldom two (eight tokens and ten
// of 512 experts: 75 experts, five of them twice), so a launch is a set of matrix-vector products over the routes' planes.
//
// Every weight is multiplied as the float it stands for, up to its block's scale (a Q6_K weight sc * (q - 32) as a half): codes
// become floats and meet the activations in fused multiply-adds, four chains to a block, and scales, minima and the sum over the
// blocks are 64 bits wide. No value shares an exponent with its neighbours. Against 64 bits throughout: 1.4e-7 to 1.6e-7 of h's size
// and 5.0e-8 to 5.7e-8 of y's (Q8_0, Q5_1). (Rows as two halves or three bf16 pieces on the matrix cores: 1.8e-7 to 3.2e-7, 6.7e-8
// to 7.3e-8.)
//
// Matrix cores are not needed for it: two and a half instructions per weight and row are in the end a quarter of the time where experts meet one
// row each, while their operand order gathers 16 bytes from 64 places per request, or takes a plan over the step's records first, and both cost more.
// L lanes share a weight row and read neighbouring pieces of it; a lane owns every L-th unit of 64 (32) weights of TWO rows, the
// gate and up rows of a hidden unit or two rows of down, so that an activation read from LDS serves two weights.
//
//  one_row   one token. Bound by one trip to memory, the launch and the issue of its instructions, in about equal parts: a wave
//            asks for everything it will ever need before it waits, R units of each row.
//  few_rows  more tokens, and one token's rows that are too wide for that. Bound by memory with a head of one trip and a tail of one
//            unit's arithmetic: the next unit's bytes travel while one is multiplied, three or four waves per SIMD. Both activation rows are
//            asked for whole, ahead of the first weights: piece by piece as they are staged they were three more trips (eight tokens, gate/up
//            2048 x 512, 24.4 -> 23.3 us).
//
// Kernel times, before -> now (ten of 512 experts; the kernels before were one super-block per wave, rows kept in registers, or a
// stream over the records, each on the matrix cores):
//   one token     gate/up 2048 x 512 9.5 -> 6.3 us, 2560 x 640 14.6 -> 9.0; down 512 -> 2048 Q6_K 6.6 -> 5.2, 640 -> 2560 Q8_0 9.2 -> 5.6
//   three tokens  gate/up 2048 x 512 15.7 -> 11.6, down 512 -> 2048 Q8_0 13.4 -> 7.4
//   five tokens   gate/up 2560 x 640 30.8 -> 22.8 (88 MB: 18 us at the rate of a copy), down Q8_0 26.0 -> 17.6
//   eight tokens  gate/up 2048 x 512 27.1 -> 23.1, down Q6_K 19.6 -> 17.1; eight of 128, down 768 -> 2048 Q5_1 31.4 -> 17.2
// Tokens that agree, a whole call of eight at 2048 x 512 with Q6_K, against the kernels with records on the matrix cores before (us): eight sets of
// experts 45.6 -> 39.9, four 34.5 -> 29.5, two 27.5 -> 27.4, all on the same ten 21.0 -> 27.3; five on the same ten 20.7 -> 21.3, four 20.4, both, three
// 18.6 -> 17.2. Wider and larger layers gain throughout (eight on the same eight of 4096 x 1536, Q8_0: 539 -> 90). What the last of the eight lose is
// arithmetic, 2.75 waves a SIMD of it: rows that come for nothing on the matrix cores. v_mfma_f32_4x4x1 gives the bits of these multiply-adds, but
// not beside vector instructions (10 cycles, and 20 with one conversion between); up to four rows to a task share a conversion more, in 244
// registers where three waves a SIMD have 168 (gate/up 16 -> 50 us with what that spills).
#include "moe_few.hpp"

#include <type_traits>

#include "grouping_device.hpp"
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

__device__ __forceinline__ void opaque(Piece<12> (&p)[2]) { asm volatile("" : "+v"(p[0].q0), "+v"(p[0].q1), "+v"(p[1].q0), "+v"(p[1].q1)); }
__device__ __forceinline__ void opaque(Piece<14> (&p)[2]) {
    asm volatile("" : "+v"(p[0].la), "+v"(p[0].lb), "+v"(p[0].qh), "+v"(p[1].la), "+v"(p[1].lb), "+v"(p[1].qh));
}
__device__ __forceinline__ void opaque(Piece<8> (&p)[2]) { asm volatile("" : "+v"(p[0].q0), "+v"(p[0].q1), "+v"(p[1].q0), "+v"(p[1].q1)); }
__device__ __forceinline__ void opaque(Piece<7> (&p)[2]) { asm volatile("" : "+v"(p[0].q), "+v"(p[1].q), "+v"(p[0].qh), "+v"(p[1].qh)); }

// The planes of an expert; a unit's bytes lie `at` units into them (row * units of a row + unit: 32 bits reach every expert below 4 GiB,
// and one offset from a uniform base is one register where a pointer each is two and two instructions a step).
struct Planes { const uint8_t *q, *qh, *sm, *dm; };
__device__ __forceinline__ Planes planes_of(const uint8_t* w, const tsp_planar_spec& s) { return {w + s.qs_offset, w + s.qh_offset, w + s.sm_offset, w + s.dm_offset}; }

template <uint32_t T>
__device__ __forceinline__ Piece<T> fetch(const Planes& w, uint32_t at) {
    Piece<T> p;
    if constexpr (T == 12) {  // sub-blocks 2 (u % 4) and 2 (u % 4) + 1 of super-block u / 4
        p.q0 = *reinterpret_cast<const u32x4*>(w.q + at * 32);
        p.q1 = *reinterpret_cast<const u32x4*>(w.q + (at * 32 + 16));
        const uint32_t sm = at / 4 * 16 + at % 4 * 2;
        p.sc = *reinterpret_cast<const uint16_t*>(w.sm + sm);
        p.mn = *reinterpret_cast<const uint16_t*>(w.sm + (sm + 8));
        p.dm = *reinterpret_cast<const uint32_t*>(w.dm + at / 4 * 4);
    } else if constexpr (T == 14) {  // section u / 2 % 2, the 16-byte half u % 2 of each of its pieces
        const uint32_t ql = at / 2 * 64 + at % 2 * 16;
        p.la = *reinterpret_cast<const u32x4*>(w.q + ql);
        p.lb = *reinterpret_cast<const u32x4*>(w.q + (ql + 32));
        p.qh = *reinterpret_cast<const u32x4*>(w.qh + at * 16);
        p.sc = *reinterpret_cast<const uint2*>(w.sm + at / 2 * 8);
        p.d = *reinterpret_cast<const uint16_t*>(w.dm + at / 4 * 2);
    } else if constexpr (T == 8) {
        p.q0 = *reinterpret_cast<const u32x4*>(w.q + at * 32);
        p.q1 = *reinterpret_cast<const u32x4*>(w.q + (at * 32 + 16));
        p.d = *reinterpret_cast<const uint16_t*>(w.dm + at * 2);
    } else {
        p.q = *reinterpret_cast<const u32x4*>(w.q + at * 16);
        p.qh = *reinterpret_cast<const uint32_t*>(w.qh + at * 4);
        p.dm = *reinterpret_cast<const uint32_t*>(w.dm + at * 4);
    }
    return p;
}

// Four unsigned (signed) byte codes against four activations of each of X rows, a chain each.
template <int X>
__device__ __forceinline__ void four(uint32_t codes, const float4 (&x)[X], float (&sum)[X][4]) {
    asm("" : "+v"(codes));  // one v_cvt_f32_ubyteN per code: seen through, a masked word becomes a shift or bit field and a conversion
    const float c[4] = {float(codes & 0xffu), float((codes >> 8) & 0xffu), float((codes >> 16) & 0xffu), float(codes >> 24)};
#pragma unroll
    for (int j = 0; j < X; ++j) {
        sum[j][0] = __builtin_fmaf(c[0], x[j].x, sum[j][0]);
        sum[j][1] = __builtin_fmaf(c[1], x[j].y, sum[j][1]);
        sum[j][2] = __builtin_fmaf(c[2], x[j].z, sum[j][2]);
        sum[j][3] = __builtin_fmaf(c[3], x[j].w, sum[j][3]);
    }
}
template <int X>
__device__ __forceinline__ void four_signed(uint32_t codes, const float4 (&x)[X], float (&sum)[X][4]) {
    const float c[4] = {float(int8_t(codes)), float(int8_t(codes >> 8)), float(int8_t(codes >> 16)), float(int8_t(codes >> 24))};
#pragma unroll
    for (int j = 0; j < X; ++j) {
        sum[j][0] = __builtin_fmaf(c[0], x[j].x, sum[j][0]);
        sum[j][1] = __builtin_fmaf(c[1], x[j].y, sum[j][1]);
        sum[j][2] = __builtin_fmaf(c[2], x[j].z, sum[j][2]);
        sum[j][3] = __builtin_fmaf(c[3], x[j].w, sum[j][3]);
    }
}

__device__ __forceinline__ float all(const float (&sum)[4]) { return (sum[0] + sum[1]) + (sum[2] + sum[3]); }

// Two weight rows' units against the same activations, of X rows that lie `stride` floats apart: total[j][n] += weight row n's
// unit with activation row j. What happens to a row does not depend on X.
template <uint32_t T, int X>
__device__ __forceinline__ void multiply(const Piece<T> (&p)[2], uint32_t u, const float* xs, uint32_t stride, double (&total)[X][2]) {
    struct Quads { float4 v[X]; };
    auto quad = [&](int i) {
        Quads q;
#pragma unroll
        for (int j = 0; j < X; ++j) q.v[j] = *reinterpret_cast<const float4*>(xs + j * stride + 4 * i);
        return q;
    };
    if constexpr (T == 12) {
#pragma unroll
        for (int b = 0; b < 2; ++b) {  // the low nibbles are the first sub-block's codes, the high ones the second's (times 16)
            float sum[2][X][4] = {};
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const Quads a = quad(8 * b + i);
#pragma unroll
                for (int n = 0; n < 2; ++n) four<X>((i < 4 ? p[n].q0[i % 4] : p[n].q1[i % 4]) & (b ? 0xf0f0f0f0u : 0x0f0f0f0fu), a.v, sum[n]);
            }
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const float d = half_bits_to_float(p[n].dm & 0xffffu), dmin = half_bits_to_float(p[n].dm >> 16);
                // a scale times its code is exact in 32 bits
                const double scale = b ? d * (0.0625f * float(p[n].sc >> 8)) : d * float(p[n].sc & 0xffu);
                const double least = -(dmin * float(b ? p[n].mn >> 8 : p[n].mn & 0xff));
#pragma unroll
                for (int j = 0; j < X; ++j) {
                    total[j][n] = __builtin_fma(scale, double(all(sum[n][j])), total[j][n]);
                    total[j][n] = __builtin_fma(least, double(xs[j * stride + 64 + b]), total[j][n]);
                }
            }
        }
    } else if constexpr (T == 14) {
        RawQ6 raw[2];
        float sum[2][X][4] = {};
#pragma unroll
        for (int n = 0; n < 2; ++n) { raw[n].la = p[n].la; raw[n].lb = p[n].lb; raw[n].qh = p[n].qh; raw[n].sc[0] = p[n].sc.x; raw[n].sc[1] = p[n].sc.y; }
        auto quarter = [&](auto q_tag) {  // 16 weights of one sub-scale, sc * (q - 32) as halves
            constexpr int Q = decltype(q_tag)::value;
            f16x8 f[2][2];
#pragma unroll
            for (int n = 0; n < 2; ++n) frags_q6k<Q>(raw[n], u % 2, f[n]);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const Quads x = quad(4 * Q + i);
#pragma unroll
                for (int n = 0; n < 2; ++n)
#pragma unroll
                    for (int j = 0; j < X; ++j) {
                        const f16x8& h = f[n][i / 2];
                        float (&s)[4] = sum[n][j];
                        s[0] = __builtin_fmaf(float(h[i % 2 * 4]), x.v[j].x, s[0]);
                        s[1] = __builtin_fmaf(float(h[i % 2 * 4 + 1]), x.v[j].y, s[1]);
                        s[2] = __builtin_fmaf(float(h[i % 2 * 4 + 2]), x.v[j].z, s[2]);
                        s[3] = __builtin_fmaf(float(h[i % 2 * 4 + 3]), x.v[j].w, s[3]);
                    }
            }
        };
        quarter(std::integral_constant<int, 0>{});
        quarter(std::integral_constant<int, 2>{});
        quarter(std::integral_constant<int, 1>{});
        quarter(std::integral_constant<int, 3>{});
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int j = 0; j < X; ++j) total[j][n] = __builtin_fma(double(half_bits_to_float(p[n].d)), double(all(sum[n][j])), total[j][n]);
    } else if constexpr (T == 8) {
        float sum[2][X][4] = {};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const Quads a = quad(i);
#pragma unroll
            for (int n = 0; n < 2; ++n) four_signed<X>(i < 4 ? p[n].q0[i % 4] : p[n].q1[i % 4], a.v, sum[n]);
        }
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int j = 0; j < X; ++j) total[j][n] = __builtin_fma(double(half_bits_to_float(p[n].d)), double(all(sum[n][j])), total[j][n]);
    } else {
        float sum[2][X][4] = {};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const Quads a = quad(i);
#pragma unroll
            for (int n = 0; n < 2; ++n) {
                const uint32_t nib = (i < 4 ? p[n].q[i % 4] : p[n].q[i % 4] >> 4) & 0x0f0f0f0fu;
                // the fifth bits of codes 4 i .. 4 i + 3, one to a byte
                const uint32_t fifth = (__umul24((p[n].qh >> (4 * i)) & 15u, 0x204081u) & 0x01010101u) << 4;
                four<X>(nib | fifth, a.v, sum[n]);
            }
        }
#pragma unroll
        for (int n = 0; n < 2; ++n)
#pragma unroll
            for (int j = 0; j < X; ++j) {
                total[j][n] = __builtin_fma(double(half_bits_to_float(p[n].dm & 0xffffu)), double(all(sum[n][j])), total[j][n]);
                total[j][n] = __builtin_fma(double(half_bits_to_float(p[n].dm >> 16)), double(xs[j * stride + 32]), total[j][n]);
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
// Sum over aligned groups of L lanes (4 to 32); every lane of a group gets it.
template <int L>
__device__ __forceinline__ double lanes_sum(double v) {
    v = dpp_add_f64<0xB1>(v);
    v = dpp_add_f64<0x4E>(v);
    if constexpr (L >= 8) v = dpp_add_f64<0x141>(v);
    if constexpr (L >= 16) v = dpp_add_f64<0x140>(v);
    if constexpr (L >= 32) v += __shfl_xor(v, 16, kWave);
    return v;
}

// A float4 of a row of activations to its place in LDS.
template <uint32_t T>
__device__ __forceinline__ void stage(float* staged, uint32_t quad, const float4& v, bool live) {
    constexpr uint32_t kUnit = unit_weights(T), kFloats = unit_floats(T);
    if constexpr (T == 12 || T == 7) {  // the sum of a sub-block of 32: eight neighbouring threads
        const float sum = octet_sum((v.x + v.y) + (v.z + v.w));
        if (quad % 8 == 0 && live) staged[quad / (kUnit / 4) * kFloats + kUnit + quad / 8 % (kUnit / 32)] = sum;
    }
    uint32_t at;
    if constexpr (T == 14) at = (quad / 64 * 4 + quad / 32 % 2 * 2 + quad / 4 % 2) * kFloats + quad / 8 % 4 * 16 + quad % 4 * 4;  // section, half | quarter
    else at = quad / (kUnit / 4) * kFloats + quad % (kUnit / 4) * 4;
    if (live) *reinterpret_cast<float4*>(staged + at) = v;
}

// Sums of codes times activations have yet to meet the blocks' scales, so an activation row with something at or above 2^100 in it
// (2^18 below the largest float, which is what codes and block length can add) goes through LDS 2^-64 of its size; its totals, 64
// bits wide, come back up. Every wave leaves a flag per row before the barrier that follows the staging.
constexpr uint32_t kHuge = (127u + 100u) << 23;
constexpr float kDown64 = 0x1p-64f;
constexpr double kUp64 = 0x1p64;
__device__ __forceinline__ uint32_t largest_bits(const float4& v) {
    const uint32_t a = __float_as_uint(v.x) & 0x7fffffffu, b = __float_as_uint(v.y) & 0x7fffffffu, c = __float_as_uint(v.z) & 0x7fffffffu, d = __float_as_uint(v.w) & 0x7fffffffu;
    return max(max(a, b), max(c, d));
}
constexpr uint32_t kThreads = 256;  // (one token, 2560 columns, workgroups of 128: 10.3 us, 256: 9.2)

// grid (ceil(n / rows of a workgroup), routes (+ 1)). PAIR: gate and up of a hidden unit, SwiGLU at the end; else two rows of down.
template <uint32_t T, bool PAIR, int L, int R>
__global__ __launch_bounds__(kThreads) void one_row(OneArgs a) {
    constexpr uint32_t kUnit = unit_weights(T), kFloats = unit_floats(T);
    constexpr uint32_t kGroups = kWave / L;                       // lane groups of a wave, each two rows
    constexpr uint32_t kRows = kGroups * (PAIR ? 1 : 2);          // output values of a wave
    constexpr uint32_t kMine = (L * R * kUnit / 4 + kThreads - 1) / kThreads;  // float4 of activations per thread
    __shared__ __attribute__((aligned(16))) float staged[L * R * kFloats];
    __shared__ __attribute__((aligned(16))) uint32_t huge[kThreads / kWave];
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
    const Planes planes[2] = {planes_of(w[0], a.spec), planes_of(w[1], a.spec)};
    Piece<T> cur[R][2];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t u0 = r * L + in_row, u = u0 < units ? u0 : units - 1;
#pragma unroll
        for (int n = 0; n < 2; ++n) cur[r][n] = fetch<T>(planes[n], (row[n] < a.n ? row[n] : a.n - 1) * units + u);
    }
    __builtin_amdgcn_sched_barrier(0);  // every request is out before the first wait

    // ---- the activations to LDS while the weights travel
    uint32_t largest = 0;
#pragma unroll
    for (uint32_t j = 0; j < kMine; ++j) {
        const uint32_t quad = tid + j * kThreads;
        largest = max(largest, largest_bits(xv[j]));
        stage<T>(staged, quad, xv[j], quad < quads);
    }
    const bool over = __builtin_amdgcn_ballot_w64(largest >= kHuge) != 0;
    if (lane == 0) huge[wave] = over;
    __syncthreads();
    const uint4 flags = *reinterpret_cast<const uint4*>(huge);
    const bool down = (flags.x | flags.y | flags.z | flags.w) != 0;  // the same in every wave
    if (down) {
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < kMine; ++j) {
            const uint32_t quad = tid + j * kThreads;
            stage<T>(staged, quad, make_float4(xv[j].x * kDown64, xv[j].y * kDown64, xv[j].z * kDown64, xv[j].w * kDown64), quad < quads);
        }
        __syncthreads();
    }

    double sums[1][2] = {};
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const uint32_t u = r * L + in_row;
        if (u < units) multiply<T, 1>(cur[r], u, staged + u * kFloats, 0, sums);
    }
    float total[2];
#pragma unroll
    for (int n = 0; n < 2; ++n) total[n] = float(lanes_sum<L>(sums[0][n]) * (down ? kUp64 : 1.0));

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

// ---------------------------------------------------------------- two to eight tokens
// A task is an expert and one or two of its routes: every workgroup reads the step's ids, finds the routes of its own route's
// expert with two ballots and leaves if its own is in their second half. Nothing is planned or written first; one workgroup of the
// gate/up launch writes the union block that the call promises. The always-on expert's tasks are its tokens by twos.
// JOINT: a second row uses the first one's converted codes, at the price of registers (165 against 122 at Q4_K, a wave per SIMD
// less); else the codes are converted again. Up to 2048 columns joint: 23.8 against 24.6 us for eight tokens on even experts,
// 27.6 against 30.0 for the call where all take the same. 2560 columns: 25.0 and 23.2 us for five tokens; Q8_0 down 21.0 and 17.7.
struct FewArgs {
    OneArgs one;              // x_stride: between the token rows (gate/up) or route rows (down)
    uint32_t tokens, selected, shared_tasks;
    uint64_t shared_x_stride, shared_out_stride;
    uint32_t* meta;           // gate/up: the union block, which one workgroup writes for the caller
    uint32_t hidden, channels;
};

template <uint32_t T, bool PAIR, int L, int Q, bool JOINT>
__global__ __launch_bounds__(kThreads) void few_rows(FewArgs f) {
    const OneArgs& a = f.one;
    constexpr uint32_t kUnit = unit_weights(T), kFloats = unit_floats(T), kGroups = kWave / L, kRows = kGroups * (PAIR ? 1 : 2);
    extern __shared__ __attribute__((aligned(16))) float staged[];
    __shared__ __attribute__((aligned(16))) uint32_t huge[2][kThreads / kWave];
    const uint32_t tid = threadIdx.x, lane = tid % kWave, wave = tid / kWave, in_row = lane % L, group = lane / L;
    const uint32_t units = a.k / kUnit, quads = a.k / 4, row_floats = units * kFloats, rounds = (units + L - 1) / L;
    // every id of the step, and whether any of them is none
    const uint32_t id_low = lane < a.routes ? a.ids[lane] : 0u, id_high = kWave + lane < a.routes ? a.ids[kWave + lane] : 0u;
    const bool refused = __builtin_amdgcn_ballot_w64(id_low >= a.experts || id_high >= a.experts) != 0;
    if (PAIR && blockIdx.y == f.shared_tasks + a.routes) {  // the union block
        if (blockIdx.x == 0)
            union_block(tid < a.routes ? a.ids[tid] : 0u, tid, kThreads, a.experts, f.selected, f.tokens, f.hidden, f.channels,
                        reinterpret_cast<uint32_t*>(staged), [&](uint32_t i, uint32_t v) { f.meta[i] = v; },
                        [&] { atomicOr(a.error_word, TSP_ERRBIT_INDEX); });
        return;
    }
    if (refused && f.tokens > 1) {  // no record of the batch stands
        if (tid == 0 && blockIdx.x == 0 && blockIdx.y == 0) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
        return;
    }
    const bool shared = blockIdx.y < f.shared_tasks;
    uint32_t expert = 0, row_in[2], row_out[2], count = 1;
    if (shared) {
        row_in[0] = row_out[0] = 2 * blockIdx.y;
        row_in[1] = row_out[1] = 2 * blockIdx.y + 1;
        count = row_in[1] < f.tokens ? 2 : 1;
    } else {
        const uint32_t route = blockIdx.y - f.shared_tasks;
        expert = uint32_t(__builtin_amdgcn_readlane(int(route < kWave ? id_low : id_high), int(route % kWave)));
        // the routes of this expert: each of the first half of them takes one of the second half along, so that workgroups with nothing to do come
        // behind those that have something (with neighbours in pairs, eight tokens on the same ten experts: 16.9 us of gate/up, 16.2 so)
        const uint64_t low = __builtin_amdgcn_ballot_w64(lane < a.routes && id_low == expert);
        const uint64_t high = __builtin_amdgcn_ballot_w64(kWave + lane < a.routes && id_high == expert);
        if (expert >= a.experts) {  // one token: the other routes do
            if (tid == 0 && blockIdx.x == 0) atomicOr(a.error_word, TSP_ERRBIT_INDEX);
            return;
        }
        const uint32_t in_low = __builtin_popcountll(low), all = in_low + __builtin_popcountll(high), half = (all + 1) / 2;
        const uint64_t below = (1ull << (route % kWave)) - 1;
        const uint32_t before = route < kWave ? __builtin_popcountll(low & below) : in_low + __builtin_popcountll(high & below);
        if (before >= half) return;
        uint32_t next = route;
        if (before + half < all) {
            uint32_t n = before + half;
            uint64_t left = n < in_low ? low : high;
            for (n = n < in_low ? n : n - in_low; n; --n) left &= left - 1;
            next = (before + half < in_low ? 0 : kWave) + __builtin_ctzll(left);
            count = 2;
        }
        row_out[0] = route; row_out[1] = next;
        row_in[0] = PAIR ? route / f.selected : route;
        row_in[1] = PAIR ? next / f.selected : next;
    }
    const uint8_t* const x_base = reinterpret_cast<const uint8_t*>(shared ? a.shared_x : a.x);
    const uint64_t x_stride = shared ? f.shared_x_stride : a.x_stride;
    const float* x[2] = {reinterpret_cast<const float*>(x_base + row_in[0] * x_stride), reinterpret_cast<const float*>(x_base + row_in[1] * x_stride)};
    auto load = [&](const float* from, uint32_t quad) {
        if (quad >= quads) return make_float4(0, 0, 0, 0);
        if (reinterpret_cast<uintptr_t>(from) % 16 == 0) return reinterpret_cast<const float4*>(from)[quad];
        return make_float4(from[4 * quad], from[4 * quad + 1], from[4 * quad + 2], from[4 * quad + 3]);
    };
    float4 held[2][Q];
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (uint32_t(j) < count) held[j][q] = load(x[j], tid + q * kThreads);

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
    const Planes planes[2] = {planes_of(w[0], a.spec), planes_of(w[1], a.spec)};
    const uint32_t begin[2] = {(row[0] < a.n ? row[0] : a.n - 1) * units, (row[1] < a.n ? row[1] : a.n - 1) * units};
    auto ask = [&](uint32_t round, Piece<T> (&p)[2]) {
        const uint32_t u0 = round * L + in_row, u = u0 < units ? u0 : units - 1;
#pragma unroll
        for (int n = 0; n < 2; ++n) p[n] = fetch<T>(planes[n], begin[n] + u);
    };
    Piece<T> next[2], now[2];
    ask(0, next);
    __builtin_amdgcn_sched_barrier(0);
    const uint32_t rounded = (quads + kThreads - 1) / kThreads * kThreads;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (uint32_t(j) >= count) break;
        uint32_t largest = 0;
        auto take = [&](const float4& here, uint32_t quad) {
            largest = max(largest, largest_bits(here));
            stage<T>(staged + j * row_floats, quad, here, quad < quads);
        };
#pragma unroll
        for (int q = 0; q < Q; ++q)
            if (q * kThreads < quads) take(held[j][q], tid + q * kThreads);
        for (uint32_t quad = tid + Q * kThreads; quad < rounded; quad += kThreads) take(load(x[j], quad), quad);
        const bool over = __builtin_amdgcn_ballot_w64(largest >= kHuge) != 0;
        if (lane == 0) huge[j][wave] = over;
    }
    __syncthreads();
    bool down[2] = {false, false};  // the same in every wave
    for (uint32_t j = 0; j < count; ++j) {
        const uint4 flags = *reinterpret_cast<const uint4*>(huge[j]);
        const bool over = (flags.x | flags.y | flags.z | flags.w) != 0;
        if (j) down[1] = over;
        else down[0] = over;
        if (!over) continue;
        __syncthreads();
        for (uint32_t quad = tid; quad < rounded; quad += kThreads) {
            const float4 v = load(x[j], quad);
            stage<T>(staged + j * row_floats, quad, make_float4(v.x * kDown64, v.y * kDown64, v.z * kDown64, v.w * kDown64), quad < quads);
        }
        __syncthreads();
    }

    double one[1][2] = {}, other[1][2] = {};  // of the first and the second activation row
    for (uint32_t round = 0; round < rounds; ++round) {
        now[0] = next[0]; now[1] = next[1];
        if (round + 1 < rounds) ask(round + 1, next);
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t u = round * L + in_row;
        if (u < units) {
            const float* const xs = staged + u * kFloats;
            if constexpr (!JOINT) {
#pragma unroll 1
                for (uint32_t j = 0; j < count; ++j) {
                    opaque(now);
                    double mine[1][2] = {{j ? other[0][0] : one[0][0], j ? other[0][1] : one[0][1]}};
                    multiply<T, 1>(now, u, xs + j * row_floats, 0, mine);
#pragma unroll
                    for (int n = 0; n < 2; ++n) {
                        one[0][n] = j ? one[0][n] : mine[0][n];
                        other[0][n] = j ? mine[0][n] : other[0][n];
                    }
                }
            } else if (count == 1) {
                multiply<T, 1>(now, u, xs, 0, one);
            } else {
                opaque(now);
                double both[2][2] = {{one[0][0], one[0][1]}, {other[0][0], other[0][1]}};
                multiply<T, 2>(now, u, xs, row_floats, both);
                one[0][0] = both[0][0]; one[0][1] = both[0][1]; other[0][0] = both[1][0]; other[0][1] = both[1][1];
            }
        }
    }

    uint32_t bad = 0;
    uint8_t* const out_base = reinterpret_cast<uint8_t*>(shared ? a.shared_out : a.out);
    const uint64_t out_stride = shared ? f.shared_out_stride : a.out_stride;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        if (uint32_t(j) >= count) break;
        float total[2];
#pragma unroll
        for (int n = 0; n < 2; ++n) total[n] = float(lanes_sum<L>(j ? other[0][n] : one[0][n]) * ((j ? down[1] : down[0]) ? kUp64 : 1.0));
        float* const out = reinterpret_cast<float*>(out_base + row_out[j] * out_stride);
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
    }
    publish_error(bad, a.error_word);
}

template <uint32_t T, bool PAIR, int L, int Q, bool JOINT>
int launch_few(const char* name, const FewArgs& f, hipStream_t s) {
    constexpr uint32_t per_group = kThreads / L * (PAIR ? 1 : 2);
    const dim3 grid((f.one.n + per_group - 1) / per_group, f.shared_tasks + f.one.routes + (PAIR && f.meta ? 1 : 0));
    uint32_t lds = 2 * (f.one.k / unit_weights(T)) * unit_floats(T) * 4;
    if (PAIR && lds < kUnionScratchWords * 4) lds = kUnionScratchWords * 4;
    TSP_LAUNCH(name, s, few_rows<T, PAIR, L, Q, JOINT><<<grid, kThreads, lds, s>>>(f));
    return launch_status(name);
}

template <uint32_t T, bool PAIR, int L, int R>
int launch(const char* name, const OneArgs& a, hipStream_t s) {
    constexpr uint32_t per_group = kThreads / L * (PAIR ? 1 : 2);
    const dim3 grid((a.n + per_group - 1) / per_group, a.routes + (a.shared_w0 ? 1 : 0));
    TSP_LAUNCH(name, s, one_row<T, PAIR, L, R><<<grid, kThreads, 0, s>>>(a));
    return launch_status(name);
}

// Q6_K rows up to here, and aligned to 16 bytes, have sc * (q - 32) as a half; wider and other ones the weight as it decodes: the
// per-element kernel, since nobody has asked for fewer bits there.
constexpr uint32_t kMostHalves = 2048;
// What few_rows stages of two activation rows at most, and the widest row whose loads one_row keeps all in flight.
constexpr uint32_t kMostLds = 64 * 1024, kOneGateUp = 3072, kOneDown = 1024;

}  // namespace

namespace tsp {

static bool few_fits(uint32_t type, uint32_t columns, uint64_t expert_bytes) {
    return expert_bytes < (1ull << 32) && 2 * (columns / unit_weights(type)) * unit_floats(type) * 4 <= kMostLds;
}
bool few_gate_up_takes(const FewMoe& m) { return m.gu.source_type == 12 && few_fits(12, m.channels, m.gu.planar_expert_bytes); }
bool few_down_takes(const FewMoe& m) {
    const uint32_t type = m.dn.source_type;
    const bool aligned = reinterpret_cast<uintptr_t>(m.h) % 16 == 0 && m.h_stride % 16 == 0;
    return (type == 7 || type == 8 || (type == 14 && m.hidden <= kMostHalves && aligned)) && few_fits(type, m.hidden, m.dn.planar_expert_bytes);
}

static FewArgs few_args(const FewMoe& m, const OneArgs& a) {
    return {a, m.tokens, m.selected, m.shared_gate ? (m.tokens + 1) / 2 : 0, 0, 0, m.meta, m.hidden, m.channels};
}

int launch_few_gate_up(const FewMoe& m, hipStream_t s) {
    const OneArgs a{m.pair_lo, m.pair_hi, m.gu, m.ids, m.x, 0, m.h, m.h_stride, m.experts, m.selected, m.hidden, m.channels, m.error_word,
                    m.shared_gate, m.shared_up, m.x, m.shared_h};
    if (m.tokens > 1 || m.channels > kOneGateUp) {
        FewArgs f = few_args(m, a);
        f.one.x_stride = f.shared_x_stride = m.x_stride; f.shared_out_stride = m.shared_h_stride; f.one.routes = m.tokens * m.selected;
        return m.channels <= 2048 ? launch_few<12, true, 8, 2, true>("few_gate_up", f, s) : launch_few<12, true, 8, 3, false>("few_gate_up", f, s);
    }
    // 2048 columns with 32, 16 and 8 lanes to a row: 6.3, 7.2, 7.7 us; 2560 columns 9.8, 9.2, 10.1 (24 of 64, 8 of 48 and no lanes
    // idle, against fewer and longer waves)
    const uint32_t units = m.channels / 64;
    if (units <= 16) return launch<12, true, 16, 1>("one_gate_up", a, s);
    if (units <= 32) return launch<12, true, 32, 1>("one_gate_up", a, s);
    return launch<12, true, 16, 3>("one_gate_up", a, s);
}

template <uint32_t T>
static int launch_one_down_blocks(const OneArgs& a, hipStream_t s) {
    const uint32_t units = a.k / 32;
    if (units <= 16) return launch<T, false, 8, 2>("one_down", a, s);
    return units <= 24 ? launch<T, false, 8, 3>("one_down", a, s) : launch<T, false, 8, 4>("one_down", a, s);
}

int launch_few_down(const FewMoe& m, hipStream_t s) {
    const OneArgs a{m.down, nullptr, m.dn, m.ids, m.h, m.h_stride, m.y, m.y_stride, m.experts, m.selected, m.channels, m.hidden, m.error_word,
                    m.shared_down, nullptr, m.shared_h, m.shared_y};
    if (m.tokens > 1 || m.hidden > kOneDown) {
        FewArgs f = few_args(m, a);
        f.shared_x_stride = m.shared_h_stride; f.shared_out_stride = m.shared_y_stride; f.one.routes = m.tokens * m.selected;
        // Wide rows are few rows, and with four lanes to one a wave has eight rounds or more: 2048 -> 1024 Q6_K, two tokens, 25.0
        // us a call with four lanes, 19.6 with eight; 2560 -> 1024 Q8_0 29.5 with four, 19.9 with sixteen. Short rows the other way
        // round (640 -> 2560 Q8_0, five tokens: 18.2 and, with eight lanes, 18.8).
        const bool wide = m.hidden > kOneDown;
        switch (m.dn.source_type) {
        case 7: return wide ? launch_few<7, false, 16, 2, true>("few_down", f, s) : launch_few<7, false, 8, 1, true>("few_down", f, s);
        case 8: return wide ? launch_few<8, false, 16, 2, false>("few_down", f, s) : launch_few<8, false, 4, 1, false>("few_down", f, s);
        default: return wide ? launch_few<14, false, 8, 2, true>("few_down", f, s) : launch_few<14, false, 4, 1, true>("few_down", f, s);
        }
    }
    switch (m.dn.source_type) {
    case 7: return launch_one_down_blocks<7>(a, s);
    case 8: return launch_one_down_blocks<8>(a, s);
    default: return m.hidden <= 512 ? launch<14, false, 8, 1>("one_down", a, s) : launch<14, false, 8, 2>("one_down", a, s);
    }
}

}  // namespace tsp
