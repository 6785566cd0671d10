// Sign planes -> fp16 weights in matrix-core operand registers, for gfx950 (wave64).
//
// With several activation rows a BCQ product is a GEMM, and its weights are worth forming once per
// row tile instead of once per bit plane: W = sum_b +-alpha_b takes 2^nb values per alpha group, so a
// lane keeps those values as a byte-wise table in registers and picks four weights at a time with
// v_perm_b32 by the nb sign bits of each:
//   * 13 shift / bit-field-insert instructions merge the nb sign words of 32 inputs into nibbles, four byte
//     permutes (eight for one operand at a time) put the nibbles of four inputs into the bytes of one register;
//   * per four weights: mask, one v_perm_b32 for the high bytes, one for the low bytes, two that
//     interleave them into two packed fp16 pairs.
// About two vector instructions per weight at three planes, where expanding every plane to +-alpha
// takes one per weight AND PLANE plus a matrix instruction per plane.
//
// Precision: the table entries are formed in fp32 (scaled by a power of two that keeps them in the
// middle of fp16's range) and rounded to fp16 once; what the rounding leaves over is a second table,
// whose product is added as well wherever an entry is not exact.  Power-of-two alphas, which is what
// the reference's quantiser emits (quantizers/bcq_quant/bcq_shift.py:15-24), are exact and skip it.
// The power of two (the unit) belongs to ONE output, or to one alpha row group of a block format, and
// follows that output's weights along K: it is chosen anew wherever an inexact step has left the window
// [64, 32768] (outputs of one wave may be any number of binades apart, and so may the groups of an output).
// Two pieces then hold a weight to 2^-23 of itself or 2^-31 of the largest weight of the same output in
// the same K-step (64 or 128 inputs), whichever is larger.  (One unit for all 64 outputs of a wave, as these
// kernels had at first, lost a bit per binade beyond the tenth and every bit beyond the thirty-third.)
#ifndef LUT_DEQUANT_DEVICE_H
#define LUT_DEQUANT_DEVICE_H

#include <type_traits>

#include "lutgemm_common.h"

namespace lutgemm {

// how alphas are laid out, as far as forming weights goes
enum WeightFormat : int {
    kWeightRow = 0,      // one alpha per (group of inputs, plane, output)
    kWeightUniform = 1,  // alpha and q_bias per (group of inputs, output)
    kWeightBlock = 2,    // one alpha per (8 inputs, plane, row group)
};

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

// Entries of a table as bytes: entry i's high byte is byte i & 3 of hi[i >> 2], its low byte the same of
// lo[i >> 2].  Four planes: 8 entries for the three planes relative to plane 3, whose sign is applied
// afterwards; uniform mode (whose q_bias breaks that symmetry): 16 entries.
template <int NB, bool UNI>
struct WeightTable {
    static constexpr int kRegs = NB <= 2 ? 1 : (NB == 4 && UNI) ? 4 : 2;
    uint32_t hi[kRegs], lo[kRegs];
};

// bytes of four packed halves: high bytes / low bytes in entry order, or in reverse
__device__ __forceinline__ uint32_t high_bytes(uint32_t p01, uint32_t p23) { return __builtin_amdgcn_perm(p23, p01, 0x07050301u); }
__device__ __forceinline__ uint32_t low_bytes(uint32_t p01, uint32_t p23) { return __builtin_amdgcn_perm(p23, p01, 0x06040200u); }
__device__ __forceinline__ uint32_t high_bytes_rev(uint32_t p01, uint32_t p23) { return __builtin_amdgcn_perm(p23, p01, 0x01030507u); }
__device__ __forceinline__ uint32_t low_bytes_rev(uint32_t p01, uint32_t p23) { return __builtin_amdgcn_perm(p23, p01, 0x00020406u); }

// The distinct fp32 entries of a table, from which the others follow by symmetry.
//   a[b]: the planes' multipliers; UNI: a[b] = alpha / 2^(b+1) and q = q_bias.
template <int NB, bool UNI>
struct TableEntries {
    static constexpr int kCount = UNI ? (NB == 1 ? 2 : 1 << NB) : NB == 4 ? 8 : NB == 3 ? 4 : NB == 2 ? 2 : 1;
    float e[kCount];
};

template <int NB, bool UNI>
__device__ __forceinline__ TableEntries<NB, UNI> table_entries(const float (&a)[NB], float q)
{
    TableEntries<NB, UNI> t;
    if constexpr (UNI) {
#pragma unroll
        for (int i = 0; i < t.kCount; ++i) {
            float v = q;
#pragma unroll
            for (int b = 0; b < NB; ++b) v += ((i >> b) & 1) ? a[b] : -a[b];
            t.e[i] = v;
        }
    } else if constexpr (NB == 1) {
        t.e[0] = a[0];                          // entry 1
    } else if constexpr (NB == 2) {
        t.e[0] = a[1] - a[0];                   // entries 2, 3
        t.e[1] = a[1] + a[0];
    } else if constexpr (NB == 3) {
        const float s = a[0] + a[1], d = a[0] - a[1];
        t.e[0] = a[2] - s;                      // entries 4..7
        t.e[1] = a[2] + d;
        t.e[2] = a[2] - d;
        t.e[3] = a[2] + s;
    } else {
        // entry i: plane 3 negative, plane b of the sign of plane 3 where bit b of i is set
        const float s = a[0] + a[1], d = a[0] - a[1], u = -a[3] - a[2], v = a[2] - a[3];
        t.e[0] = v + s;                         // -(a3 - a2 - a1 - a0)
        t.e[1] = v - d;
        t.e[2] = v + d;
        t.e[3] = v - s;
        t.e[4] = u + s;
        t.e[5] = u - d;
        t.e[6] = u + d;
        t.e[7] = u - s;
    }
    return t;
}

// Entries -> byte table.
template <int NB, bool UNI>
__device__ __forceinline__ void pack_table(const TableEntries<NB, UNI> &t, WeightTable<NB, UNI> &w)
{
    if constexpr (UNI) {
        if constexpr (NB == 1) {
            const uint32_t p = pack_halves(t.e[0], t.e[1]);
            w.hi[0] = high_bytes(p, p);
            w.lo[0] = low_bytes(p, p);
        } else {
#pragma unroll
            for (int r = 0; r < w.kRegs; ++r) {
                const uint32_t p01 = pack_halves(t.e[4 * r], t.e[4 * r + 1]), p23 = pack_halves(t.e[4 * r + 2], t.e[4 * r + 3]);
                w.hi[r] = high_bytes(p01, p23);
                w.lo[r] = low_bytes(p01, p23);
            }
        }
    } else if constexpr (NB == 1) {
        const uint32_t p = pack_halves(t.e[0], t.e[0]);
        w.hi[0] = high_bytes(p, p) ^ 0x00800080u;      // entry 0 (bytes 0 and 2) negative
        w.lo[0] = low_bytes(p, p);
    } else if constexpr (NB == 2) {
        const uint32_t p = pack_halves(t.e[0], t.e[1]);   // entries 2, 3; 1 = -2, 0 = -3
        w.hi[0] = __builtin_amdgcn_perm(p, p, 0x03010103u) ^ 0x00008080u;
        w.lo[0] = __builtin_amdgcn_perm(p, p, 0x02000002u);
    } else if constexpr (NB == 3) {
        const uint32_t p45 = pack_halves(t.e[0], t.e[1]), p67 = pack_halves(t.e[2], t.e[3]);
        w.hi[1] = high_bytes(p45, p67);
        w.lo[1] = low_bytes(p45, p67);
        w.hi[0] = high_bytes_rev(p45, p67) ^ 0x80808080u;
        w.lo[0] = low_bytes_rev(p45, p67);
    } else {
#pragma unroll
        for (int r = 0; r < 2; ++r) {
            const uint32_t p01 = pack_halves(t.e[4 * r], t.e[4 * r + 1]), p23 = pack_halves(t.e[4 * r + 2], t.e[4 * r + 3]);
            w.hi[r] = high_bytes(p01, p23);
            w.lo[r] = low_bytes(p01, p23);
        }
    }
}

// What rounding the entries to fp16 leaves over (zero where they are exact).
template <int NB, bool UNI>
__device__ __forceinline__ TableEntries<NB, UNI> table_residual(const TableEntries<NB, UNI> &t)
{
    TableEntries<NB, UNI> r;
#pragma unroll
    for (int i = 0; i < t.kCount; ++i) r.e[i] = __builtin_fmaf(__half2float(__float2half_rn(t.e[i])), -1.0f, t.e[i]);   // one mixed-precision instruction
    return r;
}

// Whether some entry may be no fp16 number.  The entries of up to three planes are looked at themselves.
// More of them are bounded by the multipliers, a third of the instructions: all are sums of these, so they are fp16 numbers where
// every multiplier is a multiple of u, their sum of magnitudes at most 2048 u (eleven bits) and u no less than 2^-24 (the
// smallest fp16 number).  NaN and infinity are inexact.  LOWEST: u is the smallest of the multipliers' lowest set bits.  (bits & bits
// - 1 clears the lowest mantissa bit; on a power of two it clears an exponent bit instead, which halves u at worst.  A zero
// multiplier counts for nothing.)  Otherwise u follows from the sum, and adding and taking away 1.5 * 2^23 u rounds a multiplier to
// a multiple of it: half the instructions (outputs x inputs x planes: 11008x4096x4 at 1024 rows 142 -> 136 us, 4096x4096x4 57.3 -> 54.4, 432x18016x4 at
// 407 35.3 -> 32.6, 8192x28672x4 at 32 44.1 -> 43.4), but 16-row tiles, which have no registers for it, lose (8192x8192x4 in groups of 32 at 8 rows 21.9 -> 28.8).
template <int NB, bool UNI, bool LOWEST>
__device__ __forceinline__ bool may_round(const TableEntries<NB, UNI> &t, const float (&a)[NB], float q)
{
    if constexpr (TableEntries<NB, UNI>::kCount <= 4) {
        const TableEntries<NB, UNI> r = table_residual(t);
        uint32_t bits = 0;
#pragma unroll
        for (int i = 0; i < t.kCount; ++i) bits |= __builtin_bit_cast(uint32_t, r.e[i]);
        return (bits << 1) != 0u;
    }
    if constexpr (!LOWEST) {
        float sum = UNI ? fabsf(q) : 0.0f;
#pragma unroll
        for (int b = 0; b < NB; ++b) sum += fabsf(a[b]);
        const float below = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, sum) & 0x7f800000u);   // 2^10 u
        const float magic = fmaxf(below, 0x1p-14f) * 0x1.8p13f;
        auto off = [&](float v) { return !((v + magic) - magic == v); };
        bool rounds = !(sum <= 32768.0f);
#pragma unroll
        for (int b = 0; b < NB; ++b) rounds = off(a[b]) || rounds;
        if constexpr (UNI) rounds = off(q) || rounds;
        return rounds;
    }
    float sum = 0.0f, least = 3.0e38f;
    auto take = [&](float v) {
        const uint32_t bits = __builtin_bit_cast(uint32_t, v) & 0x7fffffffu;
        const float mag = __builtin_bit_cast(float, bits);
        const float u = mag - __builtin_bit_cast(float, bits & (bits - 1u));
        sum += mag;
        least = fminf(least, u > 0.0f ? u : 3.0e38f);
    };
#pragma unroll
    for (int b = 0; b < NB; ++b) take(a[b]);
    if constexpr (UNI) take(q);
    return !(sum <= least * 2048.0f) || sum > 32768.0f || least < 0x1p-24f;
}

// The sign words of 32 inputs of one output, one per plane -> z: bytes 0, 1 of z[2 h + p] hold the table indices of
// inputs 16 h + 2 p, 16 h + 2 p + 1 (low nibbles) and of the inputs 4 further on (high nibbles), bytes 2, 3 those of the
// inputs 8 further on.  Bits above the index are garbage, except bit 3 at four planes (plane 3 itself).
template <int NB, bool UNI>
__device__ __forceinline__ void sign_pairs(const uint32_t (&w)[NB], uint32_t (&z)[4])
{
    // (as one three-input bit operation, truth table (m & a) | (~m & b): the compiler takes a chain of them apart)
    auto bfi = [](uint32_t m, uint32_t a, uint32_t b) { return __builtin_amdgcn_bitop3_b32(m, a, b, 0xca); };
    uint32_t n[4];
    if constexpr (NB == 1) {
#pragma unroll
        for (int t = 0; t < 4; ++t) n[t] = w[0] >> t;
    } else {
        uint32_t w0 = w[0], w1 = w[1], w2 = NB > 2 ? w[NB > 2 ? 2 : 0] : 0u;
        [[maybe_unused]] const uint32_t w3 = NB > 3 ? w[NB > 3 ? 3 : 0] : 0u;
        if constexpr (NB == 4 && !UNI) {
            w0 = ~(w0 ^ w3);
            w1 = ~(w1 ^ w3);
            w2 = ~(w2 ^ w3);
        }
        // pairs of planes as two-bit fields of the even and of the odd inputs, then nibbles
        const uint32_t even = bfi(0x55555555u, w0, w1 << 1), odd = bfi(0x55555555u, w0 >> 1, w1);
        n[0] = even;
        n[1] = odd;
        n[2] = even >> 2;
        n[3] = odd >> 2;
        if constexpr (NB == 3) {
            n[0] = bfi(0x33333333u, n[0], w2 << 2);
            n[1] = bfi(0x33333333u, n[1], w2 << 1);
            n[2] = bfi(0x33333333u, n[2], w2);
            n[3] = bfi(0x33333333u, n[3], w2 >> 1);
        } else if constexpr (NB == 4) {
            const uint32_t even2 = bfi(0x55555555u, w2, w3 << 1), odd2 = bfi(0x55555555u, w2 >> 1, w3);
            n[0] = bfi(0x33333333u, n[0], even2 << 2);
            n[1] = bfi(0x33333333u, n[1], odd2 << 2);
            n[2] = bfi(0x33333333u, n[2], even2);
            n[3] = bfi(0x33333333u, n[3], odd2);
        }
    }
    z[0] = __builtin_amdgcn_perm(n[1], n[0], 0x05010400u);
    z[1] = __builtin_amdgcn_perm(n[3], n[2], 0x05010400u);
    z[2] = __builtin_amdgcn_perm(n[1], n[0], 0x07030602u);
    z[3] = __builtin_amdgcn_perm(n[3], n[2], 0x07030602u);
}

// The same in the order of one operand at a time (tables that change every 8 inputs) -> y[c]: byte i of it holds the
// indices of inputs 8 c + i (low nibble) and 8 c + 4 + i (high nibble).
template <int NB, bool UNI>
__device__ __forceinline__ void sign_indices(const uint32_t (&w)[NB], uint32_t (&y)[4])
{
    uint32_t z[4];
    sign_pairs<NB, UNI>(w, z);
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        y[2 * h] = __builtin_amdgcn_perm(z[2 * h + 1], z[2 * h], 0x05040100u);
        y[2 * h + 1] = __builtin_amdgcn_perm(z[2 * h + 1], z[2 * h], 0x07060302u);
    }
}

// The four weights of the bytes' low (HALF 0) or high nibbles: the first two and the last two, packed.
template <int NB, bool UNI, int HALF>
__device__ __forceinline__ u32x2 pick_four(uint32_t y, const WeightTable<NB, UNI> &t)
{
    constexpr uint32_t kMask = NB == 1 ? 0x01010101u : NB == 2 ? 0x03030303u : 0x07070707u;
    constexpr bool half = HALF != 0;
    const uint32_t sel = (half ? y >> 4 : y) & kMask;
    uint32_t h, l;
    if constexpr (NB <= 2) {
        h = __builtin_amdgcn_perm(t.hi[0], t.hi[0], sel);
        l = __builtin_amdgcn_perm(t.lo[0], t.lo[0], sel);
    } else {
        h = __builtin_amdgcn_perm(t.hi[1], t.hi[0], sel);
        l = __builtin_amdgcn_perm(t.lo[1], t.lo[0], sel);
        if constexpr (NB == 4 && !UNI) {
            // plane 3 positive: the other sign (h ^ (bits & mask))
            h = __builtin_amdgcn_bitop3_b32(half ? y : y << 4, 0x80808080u, h, 0x6a);
        } else if constexpr (NB == 4) {
            const uint32_t top = ((half ? y >> 7 : y >> 3) & 0x01010101u);
            const uint32_t mask = (top << 8) - top;       // bytes of 0xff where plane 3 is positive
            const uint32_t h1 = __builtin_amdgcn_perm(t.hi[3], t.hi[2], sel), l1 = __builtin_amdgcn_perm(t.lo[3], t.lo[2], sel);
            h = (h & ~mask) | (h1 & mask);
            l = (l & ~mask) | (l1 & mask);
        }
    }
    return (u32x2){__builtin_amdgcn_perm(h, l, 0x05010400u), __builtin_amdgcn_perm(h, l, 0x07030602u)};
}

// Eight weights (inputs 8 c .. 8 c + 7, in order) as a matrix operand, from sign_indices' y[c].
template <int NB, bool UNI>
__device__ __forceinline__ u32x4 pick_weights(uint32_t y, const WeightTable<NB, UNI> &t)
{
    const u32x2 a = pick_four<NB, UNI, 0>(y, t), b = pick_four<NB, UNI, 1>(y, t);
    return (u32x4){a.x, a.y, b.x, b.y};
}

// Sixteen weights of one table as two operands, from sign_pairs' z[2 h], z[2 h + 1]: four instructions fewer per
// output and sign word than through sign_indices.
template <int NB, bool UNI>
__device__ __forceinline__ void pick_pair(uint32_t z0, uint32_t z1, const WeightTable<NB, UNI> &t, u32x4 (&out)[2])
{
    const u32x2 a = pick_four<NB, UNI, 0>(z0, t), b = pick_four<NB, UNI, 0>(z1, t);
    const u32x2 c = pick_four<NB, UNI, 1>(z0, t), d = pick_four<NB, UNI, 1>(z1, t);
    out[0] = (u32x4){a.x, b.x, c.x, d.x};
    out[1] = (u32x4){a.y, b.y, c.y, d.y};
}

// ---- block formats: one multiplier, as it lies in memory and decoded --------------------------------------
// `at`: its index, below `count`, the multipliers of the tensor (at least four).
__device__ __forceinline__ uint32_t raw_multiplier(const void *alpha, int mode, uint32_t at, uint32_t count)
{
    if (mode == kBlockApotI8) {   // three bytes, as part of four that lie inside the tensor
        const uint32_t from = min(3u * at, 3u * count - 4u);
        uint32_t v;
        __builtin_memcpy(&v, (const char *)alpha + from, 4);
        return v >> (8u * (3u * at - from));
    }
    return (uint32_t) * (const uint16_t *)((const char *)alpha + 2u * at);
}

__device__ __forceinline__ float decode_multiplier(uint32_t u, int mode)
{
    if (mode == kBlockF16) return half_bits_to_float(u & 0xffffu);
    if (mode == kBlockShiftU16) return (float)((1u << (u & 7u)) + (1u << ((u >> 3) & 7u)) + (1u << ((u >> 6) & 7u)));
    float v = 0.0f;
#pragma unroll
    for (int e = 0; e < 3; ++e) {
        const int x = (int)(int8_t)(u >> (8 * e));
        v += x == -128 ? 0.0f : ldexpf(1.0f, x);
    }
    return v;
}

// ---- the power of two that keeps an output's weights in the middle of fp16's range -------------------------
// (`from`: opaque, so that a loop does not keep the many sums of it and constants in registers of their own)
__device__ __forceinline__ int opaque(int from)
{
    asm volatile("" : "+v"(from));
    return from;
}

__device__ __forceinline__ float lane_value(float v, int src)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_ds_bpermute(4 * src, __builtin_bit_cast(int, v)));
}

// Maximum over the 64 lanes, as a scalar (v is not negative).
__device__ __forceinline__ float wave_max(float v)
{
    v = fmaxf(v, dpp_move<0xb1>(v));    // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_move<0x4e>(v));    // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_move<0x141>(v));   // row_half_mirror
    v = fmaxf(v, dpp_move<0x140>(v));   // row_mirror
    const int vi = __builtin_bit_cast(int, v);
    auto row = [&](int l) { return (uint32_t)__builtin_amdgcn_readlane(vi, l); };
    return __builtin_bit_cast(float, max(max(row(0), row(16)), max(row(32), row(48))));
}

// Upper bound of |W| from the multipliers; NaN and infinity count as 0 (no unit helps them).
template <int NB>
__device__ __forceinline__ float finite_magnitude(const float (&a)[NB], float q)
{
    float s = fabsf(q);
#pragma unroll
    for (int b = 0; b < NB; ++b) s += fabsf(a[b]);
    return s < __builtin_inff() ? s : 0.0f;
}

// The unit that brings `most` to 2^12 .. 2^13: room to grow by eight and to shrink by 64 before another one is
// needed.  At most 2^60, where a weight is held to 2^-85, which no sum of 2^17 products with fp16 activations
// shows in units of 2^-31; sums on the scale of the unit stay finite in fp32.
__device__ __forceinline__ float unit_for(float most)
{
    const int e = most > 0.0f ? (int)(__builtin_bit_cast(uint32_t, most) >> 23) - 127 : 12;
    return __builtin_bit_cast(float, (uint32_t)(127 + min(max(12 - e, -115), 60)) << 23);
}

__device__ __forceinline__ float inverse_unit(float unit)   // exact: a unit is a power of two
{
    return __builtin_bit_cast(float, 0x7f000000u - __builtin_bit_cast(uint32_t, unit));
}

// Whether two pieces of weights of magnitude `most` (0: none) call for another unit: beyond 32768 fp16
// overflows, below 64 the second piece loses bits under 2^-24.
__device__ __forceinline__ bool outside_window(float most, float unit)
{
    const float m = most * unit;
    return m > 32768.0f || (m < 64.0f && m > 0.0f && unit < 0x1p60f);
}

}  // namespace lutgemm

#endif
