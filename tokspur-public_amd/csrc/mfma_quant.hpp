// Shared pieces of the matrix-core kernels: vector types, the LDS-only barrier, and the unpacking of K-quant blocks
// into MFMA B fragments of exact integer products (sc * q for Q4_K, sc * (q - 32) for Q6_K) as packed halves.
#pragma once
#include "decode.hpp"

namespace tsp {

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

enum BKind : int { B_Q4K_RAW = 0, B_Q4K_PLANAR = 1, B_Q6K_PLANAR = 2 };

// Workgroup barrier that waits for this wave's LDS traffic only. __syncthreads() also drains every outstanding
// global load, which would serialise the prefetch of the next K step behind the barrier.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// The same, after all but the YOUNGEST vector-memory operations of this wave have completed (they complete in issue
// order): for data that a direct global -> LDS load is bringing in, which no register dependency waits for.
template <int YOUNGEST>
__device__ __forceinline__ void lds_barrier_after_loads() {
    static_assert(YOUNGEST >= 0 && YOUNGEST < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(YOUNGEST) : "memory");
}
// The wait alone, for this wave.
template <int YOUNGEST>
__device__ __forceinline__ void wait_after_loads() {
    static_assert(YOUNGEST >= 0 && YOUNGEST < 64, "vmcnt is a 6-bit counter");
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(YOUNGEST) : "memory");
}
// 16 bytes per lane from global memory straight into LDS at lds_base + 16 * lane (lds_base uniform over the wave).
// The compiler does not know this load: it counts in vmcnt like any other, so waits the compiler places for its own
// loads are only ever longer than needed, and whoever reads the bytes waits for them with lds_barrier_after_loads.
__device__ __forceinline__ void load_to_lds_16(const void* src, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(lds_base), "v"(src) : "memory", "m0");
}
// The same with the global address as a uniform base (scalar registers) plus a 32-bit byte offset per lane.
__device__ __forceinline__ void load_to_lds_16(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_base), "v"(lane_offset), "s"(uniform_base) : "memory", "m0");
}
// The same for whole lines that hardly anyone will want again: they don't take the place of others in the caches.
__device__ __forceinline__ void load_once_to_lds_16(const void* uniform_base, uint32_t lane_offset, uint32_t lds_base) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_base), "v"(lane_offset), "s"(uniform_base) : "memory", "m0");
}
__device__ __forceinline__ uint32_t lds_address(const void* p) {
    return uint32_t(reinterpret_cast<uintptr_t>((__attribute__((address_space(3))) const void*)p));
}
__device__ __forceinline__ void wait_all_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// An address that came through LDS says so itself: the compiler would take the generic path, which counts every load among the
// LDS accesses as well and drains all of them at each wait.
typedef const uint8_t __attribute__((address_space(1)))* GlobalBytes;
template <class V> __device__ __forceinline__ V global_at(GlobalBytes base, uint32_t offset) {
    asm volatile("" : "+v"(offset));  // a scalar base and a lane offset, not a 64-bit address per lane
    return *reinterpret_cast<const V __attribute__((address_space(1)))*>(base + offset);
}
__device__ __forceinline__ GlobalBytes uniform_address(uint32_t lo, uint32_t hi) {
    return reinterpret_cast<GlobalBytes>(uint64_t(uint32_t(__builtin_amdgcn_readfirstlane(hi))) << 32 | uint32_t(__builtin_amdgcn_readfirstlane(lo)));
}

__device__ __forceinline__ f16x2 as_h2(uint32_t bits) { return __builtin_bit_cast(f16x2, bits); }
__device__ __forceinline__ uint32_t as_u32(f16x2 v) { return __builtin_bit_cast(uint32_t, v); }
__device__ __forceinline__ f16x2 splat(float v) { const _Float16 h = _Float16(v); return f16x2{h, h}; }
// one rounding per lane: the products below are only exact as fused multiply-adds
__device__ __forceinline__ f16x2 fma2(f16x2 a, f16x2 b, f16x2 c) { return __builtin_elementwise_fma(a, b, c); }

// Bytes (b0, b1) resp. (b2, b3) of `codes` into the low bytes of two f16 lanes whose high bytes are `hi`.
__device__ __forceinline__ uint32_t spread01(uint32_t codes, uint32_t hi) { return __builtin_amdgcn_perm(hi, codes, 0x04010400u); }
__device__ __forceinline__ uint32_t spread23(uint32_t codes, uint32_t hi) { return __builtin_amdgcn_perm(hi, codes, 0x04030402u); }

// Eight int8 quants (two dwords) as exact halves: q ^ 0x80 = q + 128 in 0..255, 0x6400 | u = 1024 + u, minus 1152.
__device__ __forceinline__ f16x8 quants8(uint32_t w0, uint32_t w1) {
    constexpr uint32_t K = 0x64646464u;
    const uint32_t u0 = w0 ^ 0x80808080u, u1 = w1 ^ 0x80808080u;
    const f16x2 off = splat(-1152.0f);
    const f16x2 p0 = as_h2(spread01(u0, K)) + off, p1 = as_h2(spread23(u0, K)) + off;
    const f16x2 p2 = as_h2(spread01(u1, K)) + off, p3 = as_h2(spread23(u1, K)) + off;
    return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// ---------------------------------------------------------------- f32 operands
// A float is three bf16 values, its top eight significant bits, the next eight and the last eight: cut off the top, subtract, again.
// Every step is exact and the pieces have a float's own exponent range, so three products with the same integer weights, summed
// in f32, are the f32 product whatever else is in the row. (Two halves under a power of two per row carry 22 bits, and fewer for
// what is far below the row's largest value.) Pieces below 2^-133 are cut off: `row_lift` is the power of two that brings a row's largest
// magnitude to 2^80 (by 120 binades at most, which is enough for subnormals), so that only what is 2^-189 of it loses bits, and
// sums that the blocks' scales, up to 2^22, have yet to meet stay finite.
__device__ __forceinline__ float top_bits(float v) { return __uint_as_float(__float_as_uint(v) & 0xffff0000u); }
struct Pieces { float hi, mid, lo; };  // the upper 16 bits of each
__device__ __forceinline__ Pieces three_pieces(float v) {
    const float rest = v - top_bits(v);
    return Pieces{v, rest, rest - top_bits(rest)};
}
__device__ __forceinline__ uint32_t two_tops(float a, float b) { return __builtin_amdgcn_perm(__float_as_uint(b), __float_as_uint(a), 0x07060302u); }
__device__ __forceinline__ int row_lift(float biggest) {
    const int up = 80 + 127 - int((__float_as_uint(biggest) >> 23) & 0xffu);
    return up > 120 ? 120 : up;
}
__device__ __forceinline__ float power_of_two(int e) { return __uint_as_float(uint32_t(127 + e) << 23); }

// Integers of at most eight bits as exact bf16: eight int8 quants, or eight codes 0 .. 255 (one per byte of w0, w1).
__device__ __forceinline__ bf16x8 quants8_bf16(uint32_t w0, uint32_t w1) {
    auto f = [](uint32_t w, int i) { return float(int(int8_t(w >> (8 * i)))); };
    return __builtin_bit_cast(bf16x8, u32x4{two_tops(f(w0, 0), f(w0, 1)), two_tops(f(w0, 2), f(w0, 3)), two_tops(f(w1, 0), f(w1, 1)), two_tops(f(w1, 2), f(w1, 3))});
}
// Sixteen weights of a Q5_1 block as two fragments. Element e is nibble e % 16 (low for e < 16, high above) of byte e % 16 with bit e
// of the block's fifth-bit word on top; the lane's k-half takes elements 16 khalf .. 16 khalf + 15. A weight is the half nearest to
// d * q + m (bits: the k-half's sixteen fifth bits): q exact as a half, one packed fused multiply-add, one rounding (the f32 evaluation rounds the sum to f32 first,
// which can move the half only when that sum sits on a tie).
__device__ __forceinline__ void q51_frags(const u32x4& nibble_bytes, uint32_t bits, f16x2 d2, f16x2 m2, uint32_t khalf, f16x8 frag[2]) {
    const f16x2 off = splat(-1024.0f);
#pragma unroll
    for (int ff = 0; ff < 2; ++ff) {
        f16x2 p[4];
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            const int w = 2 * ff + j;  // bytes 4 w .. 4 w + 3 of the block: elements 16 khalf + 4 w .. + 3
            const uint32_t nibbles = (nibble_bytes[w] >> (4 * khalf)) & 0x0f0f0f0fu;
            // bits 4 w .. 4 w + 3 of the fifth-bit half-word to bit 0 of four bytes: no two partial products share a bit
            const uint32_t four = ((bits >> (4 * w)) & 15u) * 0x00204081u & 0x01010101u;
            const uint32_t codes = nibbles | (four << 4);
            p[2 * j] = fma2(as_h2(spread01(codes, 0x64646464u)) + off, d2, m2);
            p[2 * j + 1] = fma2(as_h2(spread23(codes, 0x64646464u)) + off, d2, m2);
        }
        frag[ff] = f16x8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
    }
}

// ---------------------------------------------------------------- Q4_K operands
struct HdrQ4 { uint32_t sc[2], mn[2]; float d, dmin; };  // eight 6-bit scales and minima, one per byte

// The header of super-block b of a row, as loaded: for planes the 16 bytes of scales and minima and the word holding d and dmin,
// for GGUF rows the block's first 16 bytes (d, dmin, the 12 packed bytes). Kept apart from its decoding so that a kernel
// can request a header a step ahead and touch the bytes only when it needs them: any arithmetic on a loaded register makes
// the compiler wait for the load on the spot, and with it for every request issued before it.
struct RawHdrQ4 { uint4 words; uint32_t dm; };

template <int BKIND>
__device__ __forceinline__ RawHdrQ4 fetch_hdr_q4k(const uint8_t* base, const tsp_planar_spec& s, uint64_t row, uint32_t bpr, uint32_t b) {
    const uint64_t blk = row * bpr + b;
    RawHdrQ4 r;
    if constexpr (BKIND == B_Q4K_PLANAR) {
        r.words = *reinterpret_cast<const uint4*>(base + s.sm_offset + blk * 16);
        r.dm = *reinterpret_cast<const uint32_t*>(base + s.dm_offset + blk * 4);
    } else {
        r.words = *reinterpret_cast<const uint4*>(base + blk * 144);
        r.dm = 0;
    }
    return r;
}

template <int BKIND>
__device__ __forceinline__ HdrQ4 decode_hdr_q4k(const RawHdrQ4& r) {
    HdrQ4 h;
    if constexpr (BKIND == B_Q4K_PLANAR) {
        h.sc[0] = r.words.x; h.sc[1] = r.words.y; h.mn[0] = r.words.z; h.mn[1] = r.words.w;
        h.d = half_bits_to_float(r.dm & 0xffffu); h.dmin = half_bits_to_float(r.dm >> 16);
    } else {
        const uint4 g = r.words;
        h.d = half_bits_to_float(g.x & 0xffffu); h.dmin = half_bits_to_float(g.x >> 16);
        // 12 packed bytes -> one byte per value: sub-blocks 0..3 are the low six bits of bytes 0..7, sub-blocks
        // 4..7 take four bits from bytes 8..11 and two from the top of bytes 0..7
        h.sc[0] = g.y & 0x3f3f3f3fu;
        h.mn[0] = g.z & 0x3f3f3f3fu;
        h.sc[1] = (g.w & 0x0f0f0f0fu) | ((g.y >> 2) & 0x30303030u);
        h.mn[1] = ((g.w >> 4) & 0x0f0f0f0fu) | ((g.z >> 2) & 0x30303030u);
    }
    return h;
}

// Fragments of pair P: bytes 16h..16h+15 of the 32-byte pair; low nibbles (HI = 0) are sub-block 2P, high nibbles
// sub-block 2P+1. Fragment f of a half covers activation columns HI*32 + 16h + f*8 .. +8 of the 64-column slab.
// The columns of every eight come in the order (0, 2, 1, 3, 4, 6, 5, 7), for activations stored in that order: one mask per pair of weights
// instead of a mask and two byte permutes per four. A masked pair of nibbles is two subnormal halves, q * 2^-24 or, where the high ones sit, 16 q * 2^-24;
// times 2^8 sc or 2^4 sc that is sc * q * 2^-16, as exact as sc * q itself (a scale byte of 255 still fits), in two instructions for two
// weights, and the block's d makes up for the power of two (kQ4Lift). An and of two vector registers issues at twice the rate of an and-or, or of an and
// with a scalar register, when two waves share a SIMD (1.0 against 1.9 ns an instruction): hence no bits to be or'ed in, and the masks in vector registers. (Where what
// follows an and is two mixed-precision multiply-adds a pair, weights8_q4_swapped, it is not the ands that are waited for: dense_tile.hip keeps its masks for those in scalar registers.)
struct Q4Masks { uint32_t lo, hi; };
__device__ __forceinline__ Q4Masks q4_masks() {
    Q4Masks m{0x000f000fu, 0x00f000f0u};
    asm volatile("" : "+v"(m.lo), "+v"(m.hi));
    return m;
}
template <int HI>
__device__ __forceinline__ f16x8 scaled8_q4_swapped(uint32_t w0, uint32_t w1, f16x2 sc, const Q4Masks& masks) {
    const uint32_t m = HI ? masks.hi : masks.lo;
    const f16x2 p0 = as_h2(w0 & m) * sc, p1 = as_h2((w0 >> 8) & m) * sc;
    const f16x2 p2 = as_h2(w1 & m) * sc, p3 = as_h2((w1 >> 8) & m) * sc;
    return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}
constexpr float kQ4Lift = 65536.0f;
// Byte N of a word as a float: one v_cvt_f32_ubyteN.
template <int N>
__device__ __forceinline__ float byte_as_float(uint32_t word) { return float((word >> (8 * N)) & 0xffu); }

// Two weights from two codes sitting in the mantissas of two halves (q or q << 4 per half, everything else zero): each is scale *
// code + offset evaluated as one f32 fused multiply-add whose result is rounded to half (v_fma_mix widens the half operand
// inside the instruction, subnormals included). With scale = d * sc * 2^24 (2^20) and offset = -dmin * mn this is the f32 value
// d * sc * q - dmin * mn exactly, then rounded once.
__device__ __forceinline__ uint32_t two_weights(uint32_t codes, float scale, float offset) {
    const f16x2 c = as_h2(codes);
    const _Float16 lo = _Float16(__builtin_fmaf(float(c[0]), scale, offset)), hi = _Float16(__builtin_fmaf(float(c[1]), scale, offset));
    return as_u32(f16x2{lo, hi});
}
// Eight weights from two words of nibbles, in the swapped order; mask: where the codes sit.
__device__ __forceinline__ f16x8 weights8_q4_swapped(uint32_t w0, uint32_t w1, uint32_t mask, float scale, float offset) {
    return __builtin_bit_cast(f16x8, u32x4{two_weights(w0 & mask, scale, offset), two_weights((w0 >> 8) & mask, scale, offset), two_weights(w1 & mask, scale, offset),
                                           two_weights((w1 >> 8) & mask, scale, offset)});
}
// The scale set-up is shared by a pair of sub-blocks: the six-bit scales of sub-blocks 2P and 2P + 1 sit in neighbouring bytes of the
// header; one byte permute puts them under 0x64 (1024 + sc as halves, side by side), one packed add takes the 1024 off, and one
// packed multiply makes (2^8 sc, 2^4 sc): the factors of the low-nibble and of the high-nibble codes. Three instructions per pair.
struct Q4ScaleConsts { uint32_t sel[2]; uint32_t k64; f16x2 off, mul; };
__device__ __forceinline__ Q4ScaleConsts q4_scale_consts() {
    // selector bytes: 0..3 pick a byte of the header word, 4..7 a byte of the constant 0x64646464
    Q4ScaleConsts c{{0x04010400u, 0x04030402u}, 0x64646464u, f16x2{_Float16(-1024.0f), _Float16(-1024.0f)}, f16x2{_Float16(256.0f), _Float16(16.0f)}};
    asm volatile("" : "+s"(c.sel[0]), "+s"(c.sel[1]), "+v"(c.k64));
    return c;
}
template <int P>
__device__ __forceinline__ f16x2 q4_pair_scale(uint32_t sc_lo4, uint32_t sc_hi4, const Q4ScaleConsts& c) {
    const uint32_t word = P < 2 ? sc_lo4 : sc_hi4;  // scales 0..3 | 4..7, one per byte
    return (as_h2(__builtin_amdgcn_perm(c.k64, word, c.sel[P & 1])) + c.off) * c.mul;
}
__device__ __forceinline__ void frags_q4k_pair(const u32x4& raw, f16x2 scale, int hi, const Q4Masks& masks, f16x8 frag[2]) {
    const f16x2 s2 = hi ? f16x2{scale[1], scale[1]} : f16x2{scale[0], scale[0]};
    if (hi) {
        frag[0] = scaled8_q4_swapped<1>(raw[0], raw[1], s2, masks);
        frag[1] = scaled8_q4_swapped<1>(raw[2], raw[3], s2, masks);
    } else {
        frag[0] = scaled8_q4_swapped<0>(raw[0], raw[1], s2, masks);
        frag[1] = scaled8_q4_swapped<0>(raw[2], raw[3], s2, masks);
    }
}

// B operand of the minima term: the eight integer minima, the same in both k-halves (hi and lo sums).
__device__ __forceinline__ f16x8 minima_frag(const HdrQ4& h) {
    constexpr uint32_t K = 0x64646464u;
    const f16x2 one = splat(1.0f), off = splat(-1024.0f);
    const f16x2 p0 = fma2(as_h2(spread01(h.mn[0], K)), one, off), p1 = fma2(as_h2(spread23(h.mn[0], K)), one, off);
    const f16x2 p2 = fma2(as_h2(spread01(h.mn[1], K)), one, off), p3 = fma2(as_h2(spread23(h.mn[1], K)), one, off);
    return f16x8{p0[0], p0[1], p1[0], p1[1], p2[0], p2[1], p3[0], p3[1]};
}

// ---------------------------------------------------------------- Q6_K operands (planes ql / qh / sc / d)
struct RawQ6 { u32x4 la, lb, qh; uint32_t sc[2]; };  // one section: low nibbles of quarters 0/2 and 1/3, high bit pairs, 8 sub-scales

// Quarter Q of the section (elements Q*32 .. Q*32+31): this lane's 16 bytes are elements Q*32 + 16h + 0..15, all in
// the 16-weight group 2Q + h. Fragment f covers activation columns Q*32 + 16h + f*8 .. +8 of the section.
template <int Q>
__device__ __forceinline__ void frags_q6k(const RawQ6& r, uint32_t khalf, f16x8 frag[2]) {
    // A code c = low nibble | two high bits << 4 becomes the half 0x5400 | c << 4 = 64 + c, and (64 + c) * sc - 96 * sc =
    // (c - 32) * sc in one fused multiply-add. The half is put together from its two bytes, four weights at a time: the low
    // byte is the nibble << 4, the high byte 0x54 | the two high bits, and a byte permute pairs them up; the six-bit code
    // itself is never formed (that took a shift and an or per pair of weights more).
    constexpr uint32_t MH = 0xf0f0f0f0u, M2 = 0x03030303u;
    uint32_t K = 0x54545454u;
    asm("" : "+v"(K));  // in a vector register: with two scalar constants (x & M2) | K is two instructions, not one v_and_or_b32
    const u32x4& l = (Q & 1) ? r.lb : r.la;
    const uint32_t g = 2 * Q + khalf;
    const int sc = int(int8_t((r.sc[g >> 2] >> ((g & 3) * 8)) & 0xffu));
    const f16x2 s2 = splat(float(sc)), bias = s2 * splat(-96.0f);
    f16x2 p[8];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t low = Q < 2 ? (l[i] << 4) & MH : l[i] & MH;
        const uint32_t high = ((Q == 0 ? r.qh[i] : r.qh[i] >> (2 * Q)) & M2) | K;  // bits 2Q..2Q+1 of every byte of qh
        p[2 * i] = fma2(as_h2(__builtin_amdgcn_perm(high, low, 0x05010400u)), s2, bias);      // weights 0, 1 of the four
        p[2 * i + 1] = fma2(as_h2(__builtin_amdgcn_perm(high, low, 0x07030602u)), s2, bias);  // weights 2, 3
    }
    frag[0] = f16x8{p[0][0], p[0][1], p[1][0], p[1][1], p[2][0], p[2][1], p[3][0], p[3][1]};
    frag[1] = f16x8{p[4][0], p[4][1], p[5][0], p[5][1], p[6][0], p[6][1], p[7][0], p[7][1]};
}


}  // namespace tsp
