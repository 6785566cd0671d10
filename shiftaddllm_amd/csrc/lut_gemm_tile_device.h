// GEMM kernel templates for BCQ linear layers with many activation rows (prompts, large batches) on
// MI355X (gfx950, wave64), every alpha format.
//
//   out[m][n] = init[m][n] + sum_k x[m][k] * W[n][k],  W formed from the sign planes on the fly.
//
// A workgroup of 4 waves (or of two such teams, each on half of the inputs) owns 256 outputs x 32 * MF activation rows.  Each wave forms the weights of its
// own 64 outputs in registers (lut_dequant_device.h), directly in the layout of the matrix
// instruction's A operand (v_mfma_f32_32x32x16_f16: lane l holds output l % 32 and eight inputs), so a
// weight is formed once per workgroup and never stored; the activations, the B operand, go through LDS
// and are read by all four waves.  64 outputs per wave is what keeps the LDS reads at half a
// 16-byte read per matrix instruction.
//
// A K-step is 64 inputs = two sign words: lanes 0..31 take the first word, lanes 32..63 the second, and
// matrix instruction j multiplies byte j of either.  While the matrix cores work on step t the vector
// ALU forms the weights of step t + 1 from sign words that were requested in step t - 1, and the
// activations of step t + 2 travel from memory to registers (they enter LDS in step t + 1).
#ifndef LUT_GEMM_TILE_DEVICE_H
#define LUT_GEMM_TILE_DEVICE_H

#include <utility>

#include "lut_dequant_device.h"

namespace lutgemm {

constexpr int kTileThreads = 256;
constexpr int kTileN = 256;            // outputs per workgroup
constexpr int kTileWaveN = 64;         // outputs per wave
constexpr int kTileStepK = 64;
constexpr int kTileMaxRowGroups = 66;  // alpha row groups a tile of 256 outputs can touch (4 outputs each at least)

enum TileFormat : int {
    kTileRow = kWeightRow,
    kTileUniform = kWeightUniform,
    kTileBlock = kWeightBlock,
    kTileBlockWide = 3,  // block format where 64 outputs never straddle a row group
};

template <int MF>
constexpr int kTileXBytes = 32 * MF * kTileStepK * 2;
template <int FMT>   // scales of one step
constexpr int kTileStageBytes = FMT == kTileRow ? 2 * kTileN * 8 : FMT == kTileUniform ? 2 * kTileN * 4 : 8 * kTileMaxRowGroups * 16;
template <int FMT, int MF>
constexpr int kTileLdsBytes = 2 * kTileXBytes<MF> + 4 * kTileStageBytes<FMT>;

template <int... Is, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, Is...>, F &&f)
{
    (f(std::integral_constant<int, Is>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

// How a workgroup goes about its tile:
enum TileKind : int {
    kTileAlone = 0,   // four waves, one K-slice
    // Eight waves: two teams of four take half of the slice's steps each, in LDS of their own, and add up at the end.
    // For calls whose workgroups have a CU to themselves: two waves per SIMD instead of one, whose vector and matrix work
    // overlap, without more slices, whose sums cost memory traffic (5120x13824x2 int8 exponents at 512 rows, 3 slices 105.7 -> 88.3
    // us; 6 slices of four waves, which fill the chip as well, 92.1).
    kTilePair = 1,
    // Four waves take all K-slices in turn and add them up as tile_sum_kernel does: the bits are those of slices
    // that run side by side, and no memory is needed.  The second form: slices of teams, half by half.
    kTileSerial = 2,
    kTileSerialPair = 3,
};

// tid: the thread among the team's 256;  lds: the workgroup's, of which team `team` takes part `team`
template <int NB, int FMT, int MF, int KIND>
__device__ __forceinline__ void gemm_tile(const TileProblem &p, int n_tile, int m_tile, int slice, int tid, int team, char *lds_all)
{
    char *const lds = lds_all + team * kTileLdsBytes<FMT, MF>;
    constexpr bool UNI = FMT == kTileUniform;
    constexpr bool BLOCK = FMT >= kTileBlock;
    constexpr int kTabs = BLOCK ? 4 : 1;                       // tables per 32-output fragment and step
    constexpr int kFragTabs = FMT == kTileBlockWide ? 1 : 2;   // fragments with tables of their own
    const int lane = tid & 63, wave = tid >> 6, l32 = lane & 31, kh = lane >> 5;
    const int n0 = __builtin_amdgcn_readfirstlane(n_tile * kTileN + wave * kTileWaveN);
    const int m0 = m_tile * 32 * MF;
    int nn[2];
#pragma unroll
    for (int f = 0; f < 2; ++f) nn[f] = min(n0 + 32 * f + l32, p.N - 1);

    // ---- activations: global -> registers -> LDS ------------------------------------------------
    // Thread t carries 16-byte chunk t % 8 of rows t / 8 + 32 i; chunk c of row r sits in slot c ^ (r / 2 % 8) of
    // the row's 128 bytes, which spreads the 16 rows that one LDS cycle serves over all banks.  (With r % 8, rows r and
    // r + 8 fell on the same ones: 8 cycles per 16-byte read of a wave instead of 4, 11008x4096x3 at 2048 rows 205 us
    // instead of 203.)
    const int xr = tid >> 3, xc = tid & 7;
    uint32_t xoff[MF];
#pragma unroll
    for (int i = 0; i < MF; ++i) xoff[i] = (uint32_t)min(m0 + xr + 32 * i, p.M - 1) * (uint32_t)p.K * 2u;
    const uint32_t xslot = (uint32_t)(xr * 128 + ((xc ^ ((xr >> 1) & 7)) * 16));
    u32x4 xreg[MF];
    auto load_x = [&](int t) {
        const uint32_t k = (uint32_t)min(t * kTileStepK + xc * 8, p.K - 8) * 2u;
#pragma unroll
        for (int i = 0; i < MF; ++i) xreg[i] = *(const u32x4 *)((const char *)p.x + (xoff[i] + k));
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < MF; ++i) *(u32x4 *)(lds + buf * kTileXBytes<MF> + xslot + i * 4096) = xreg[i];
    };
    // matrix instruction j reads chunk 4 * kh + j of the lane's row, i.e. slot (4 * kh ^ l32 / 2 % 8) ^ j
    const uint32_t bslot = (uint32_t)(l32 * 128 + ((4 * kh ^ ((l32 >> 1) & 7)) * 16));

    // ---- signs and scales --------------------------------------------------------------------------
    uint32_t words[2][NB];
    auto load_fragment = [&](int t, int f, uint32_t (&w)[NB]) {
        const int wd = min(2 * t + kh, p.kwords - 1);
        const uint32_t row = (uint32_t)wd * NB * (uint32_t)p.N;
#pragma unroll
        for (int b = 0; b < NB; ++b)
            w[b] = *(const uint32_t *)((const char *)p.W + (row + (uint32_t)b * (uint32_t)p.N + (uint32_t)nn[f]) * 4u);
    };
    auto load_words = [&](int t, uint32_t (&w)[2][NB]) {
#pragma unroll
        for (int f = 0; f < 2; ++f) load_fragment(t, f, w[f]);
    };
    // The scales of a step go through LDS as well (four steps' worth: while step t runs, those of steps t
    // and t + 1 are read and those of step t + 2 written), fetched at the start of a step and written at
    // its end:
    //   row-wise: [word 0, 1][output 0..255][plane 0..3] fp16;  uniform: [word][output][alpha, q_bias] fp16;
    //   block formats: the decoded multipliers, [chunk 0..7][row group of the tile][plane 0..3] fp32.
    char *stage = lds + 2 * kTileXBytes<MF>;
    auto stage_at = [&](int t) { return stage + (t & 3) * kTileStageBytes<FMT>; };
    [[maybe_unused]] int rg0 = 0, n_rg = 1;
    [[maybe_unused]] uint32_t rgl[2] = {0u, 0u};
    if constexpr (BLOCK) {
        const int first = n_tile * kTileN;
        rg0 = first / p.rows_per_group;
        n_rg = min(first + kTileN - 1, p.N - 1) / p.rows_per_group - rg0 + 1;
#pragma unroll
        for (int f = 0; f < 2; ++f) rgl[f] = (uint32_t)(nn[f] / p.rows_per_group - rg0);
    }
    constexpr int kFetched = BLOCK ? 1 : UNI ? 2 : NB;
    uint32_t fetched[kFetched];
    // block formats: multiplier i of a step = row group i % n_rg of the tile, (chunk, plane) number i / n_rg
    struct ScaleSlot {
        int cb, r, dst;
    };
    [[maybe_unused]] auto scale_slot = [&](int i) {
        ScaleSlot z;
        z.cb = i / n_rg;
        z.r = i - z.cb * n_rg;
        const int c = z.cb / NB;
        z.dst = (c * kTileMaxRowGroups + z.r) * 4 + (z.cb - c * NB);
        return z;
    };
    [[maybe_unused]] ScaleSlot own{};
    if constexpr (BLOCK) own = scale_slot(min(tid, 8 * NB * n_rg - 1));
    [[maybe_unused]] auto raw_scale = [&](int t, const ScaleSlot &z) {
        const int rows = p.K / 8 * NB;
        const uint32_t at = (uint32_t)min(8 * NB * t + z.cb, rows - 1) * (uint32_t)p.R + (uint32_t)(rg0 + z.r);
        return raw_multiplier(p.alpha, p.mode, at, (uint32_t)rows * (uint32_t)p.R);
    };
    [[maybe_unused]] auto put_scale = [&](int t, const ScaleSlot &z, uint32_t u) {
        ((float *)stage_at(t))[z.dst] = decode_multiplier(u, p.mode);
    };
    auto fetch_scales = [&](int t, uint32_t (&to)[kFetched]) {
        if constexpr (BLOCK) {
            to[0] = raw_scale(t, own);
        } else {
            // threads 0..127: two outputs each for the step's first word, the others for its second
            const uint32_t n = (uint32_t)min(n_tile * kTileN + 2 * (tid & 127), p.N - 2);
            const uint32_t g = (uint32_t)fast_div(min(2 * t + (tid >> 7), p.kwords - 1), p.by_group_words);
            if constexpr (UNI) {
                const uint32_t at = (g * (uint32_t)p.N + n) * 2u;
                to[0] = *(const uint32_t *)((const char *)p.alpha + at);
                to[1] = *(const uint32_t *)((const char *)p.qbias + at);
            } else {
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    to[b] = *(const uint32_t *)((const char *)p.alpha + ((g * NB + (uint32_t)b) * (uint32_t)p.N + n) * 2u);
            }
        }
    };
    auto store_scales = [&](int t, const uint32_t (&from)[kFetched]) {
        if constexpr (BLOCK) {
            const int all = 8 * NB * n_rg;
            if (tid < all) put_scale(t, own, from[0]);
            for (int i = tid + kTileThreads; i < all; i += kTileThreads) {   // (row groups of a few outputs)
                const ScaleSlot z = scale_slot(i);
                put_scale(t, z, raw_scale(t, z));
            }
        } else {
            constexpr int kEach = UNI ? 2 : 4;   // halves per output
            unsigned short *dst = (unsigned short *)stage_at(t) + 2 * tid * kEach;
#pragma unroll
            for (int b = 0; b < kFetched; ++b) {
                dst[b] = (unsigned short)from[b];
                dst[kEach + b] = (unsigned short)(from[b] >> 16);
            }
        }
    };
    // multipliers of fragment f (and, block formats, chunk c of the lane's word) in step t, unscaled
    auto multipliers = [&](int t, int f, int c, float (&a)[NB], float &q) {
        q = 0.0f;
        if constexpr (BLOCK) {
            const f32x4 v = *(const f32x4 *)(stage_at(t) + ((4 * kh + c) * kTileMaxRowGroups + rgl[f]) * 16);
#pragma unroll
            for (int b = 0; b < NB; ++b) a[b] = v[b];
        } else {
            const int at = kh * kTileN + wave * kTileWaveN + 32 * f + l32;
            if constexpr (UNI) {
                const uint32_t v = ((const uint32_t *)stage_at(t))[at];
                const float alpha = half_bits_to_float(v & 0xffffu);
#pragma unroll
                for (int b = 0; b < NB; ++b) a[b] = alpha * (1.0f / (float)(2 << b));
                q = half_bits_to_float(v >> 16);
            } else {
                const u32x2 v = ((const u32x2 *)stage_at(t))[at];
                const uint32_t v2[2] = {v.x, v.y};
#pragma unroll
                for (int b = 0; b < NB; ++b) a[b] = half_bits_to_float((v2[b >> 1] >> (16 * (b & 1))) & 0xffffu);
            }
        }
    };

    // ---- the step's weights -----------------------------------------------------------------------
    u32x4 A[2][4][2];            // [step parity][matrix instruction][fragment]
    bool lo_cur = false;         // rounding the current step's weights to fp16 left something over (uniform over the wave)
    WeightTable<NB, UNI> tab[kFragTabs][kTabs];
    // weights are formed as W * unit, a power of two per output (block formats: per row group)
    float unit[kFragTabs];       // (of this lane's outputs)
    auto magnitude = [&](int t, int f) {   // upper bound of |W| in this lane's tables of fragment f
        float most = 0.0f;
#pragma unroll
        for (int c = 0; c < kTabs; ++c) {
            float a[NB], q;
            multipliers(t, f, c, a, q);
            most = fmaxf(most, finite_magnitude(a, q));
        }
        return most;
    };
    auto largest = [&](int t, int f) {   // of the step's two words
        const float m = magnitude(t, f);
        return fmaxf(m, lane_value(m, opaque(lane) ^ 32));
    };
    // One table of step t, or of what its rounding leaves over; true when some entry may not
    // be an fp16 number.
    auto make_table = [&](int t, bool lo, int f, int c) {
        const float u = 2 * t + kh < p.kwords ? unit[f] : 0.0f;   // a word beyond K has no weight
        float a[NB], q;
        multipliers(t, f, c, a, q);
#pragma unroll
        for (int b = 0; b < NB; ++b) a[b] *= u;
        const TableEntries<NB, UNI> e = table_entries<NB, UNI>(a, q * u);
        if (lo) {
            pack_table(table_residual(e), tab[f][c]);
            return false;
        }
        pack_table(e, tab[f][c]);
        return may_round<NB, UNI, FMT == kTileBlock>(e, a, q * u);
    };
    auto make_tables = [&](int t, bool lo) {
        bool inexact = false;
#pragma unroll
        for (int f = 0; f < kFragTabs; ++f)
#pragma unroll
            for (int c = 0; c < kTabs; ++c) inexact = make_table(t, lo, f, c) || inexact;
        return inexact;
    };
    auto pick = [&](int f, int c, const uint32_t (&y)[4]) {
        return pick_weights<NB, UNI>(y[c], tab[FMT == kTileBlockWide ? 0 : f][BLOCK ? c : 0]);
    };

    f32x16 acc[2][MF];
    auto activations = [&](int buf, int j, int i) {
        return __builtin_bit_cast(f16x8, *(const u32x4 *)(lds + buf * kTileXBytes<MF> + i * 4096 + (bslot ^ (uint32_t)(16 * j))));
    };
    auto multiply = [&](int buf, int j, const u32x4 (&a)[2]) {
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            const f16x8 b = activations(buf, j, i);
#pragma unroll
            for (int f = 0; f < 2; ++f)
                acc[f][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a[f]), b, acc[f][i], 0, 0, 0);
        }
    };

    // Sums times a factor per unit: register 4 g + r of a fragment is its output 8 g + 4 kh + r.  (In the main loop
    // the factors are fetched a few at a time: registers are short there.)
    auto scale_sums = [&](const float (&by)[kFragTabs], auto in_loop) {
        const int first = opaque(4 * kh);
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const float v = by[f % kFragTabs];
                const float x = FMT == kTileBlockWide ? v : lane_value(v, first + 8 * (r >> 2) + (r & 3));
#pragma unroll
                for (int i = 0; i < MF; ++i) acc[f][i][r] *= x;
                if constexpr (decltype(in_loop)::value)
                    if (r % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
    };

    uint32_t words_lo[2][NB];
    // Some weight of step t (in A[set]) is no fp16 number: a second piece is due in that step, after a change
    // of the units that do not suit it.
    auto second_piece = [&](int t, int set) {
        load_words(t, words_lo);
        bool outside = false;
#pragma unroll
        for (int f = 0; f < kFragTabs; ++f) outside = outside_window(magnitude(t, f), unit[f]) || outside;
        if (__builtin_amdgcn_ballot_w64(outside) != 0ull) {
            float by[kFragTabs];
#pragma unroll
            for (int f = 0; f < kFragTabs; ++f) {
                const float most = largest(t, f), fresh = outside_window(most, unit[f]) ? unit_for(most) : unit[f];
                by[f] = fresh * inverse_unit(unit[f]);
                unit[f] = fresh;
            }
            scale_sums(by, std::true_type());
#pragma unroll
            for (int f = 0; f < 2; ++f) {
                uint32_t y[4];
                sign_indices<NB, UNI>(words_lo[f], y);
#pragma unroll
                for (int c = 0; c < 4; ++c) {
                    if (c < kTabs) (void)make_table(t, false, f % kFragTabs, c);
                    A[set][c][f] = pick(f, c, y);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
        }
    };

    // step t with parity P: buffer P of LDS holds its activations, A[P] its weights; `words` belong to step t + 1,
    // words_lo, where a second piece is due, to step t.
    auto step = [&](int t, auto parity) {
        constexpr int P = decltype(parity)::value;
        store_x(P ^ 1);
        fetch_scales(t + 2, fetched);
        load_x(t + 2);
        if (lo_cur) {
            uint32_t y[2][4];
#pragma unroll
            for (int f = 0; f < 2; ++f) sign_indices<NB, UNI>(words_lo[f], y[f]);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (j < kTabs)
#pragma unroll
                    for (int f = 0; f < kFragTabs; ++f) (void)make_table(t, true, f, j);
                const u32x4 a[2] = {pick(0, j, y[0]), pick(1, j, y[1])};
                multiply(P, j, a);
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        // The matrix instructions of step t, two at a time (one activation fragment against both weight
        // fragments), each pair with its share of the vector work on step t + 1 and the request for the
        // next activation fragment.  (Left to itself the compiler puts all vector work in front of all
        // matrix work and waits for every fragment right behind its request.)
        bool inexact = false;
        uint32_t y[2][4];
        // (One fragment after the other, and block formats a chunk's table, then its weights, so that few tables and
        // indices are live at a time; where both fragments share their tables, chunk after chunk.  The loop needs every
        // register there is: with both fragments' at once it reloaded spilled values behind all loads in flight,
        // 8192x8192x4 at 128 rows 51 us instead of 41.5, 11008x4096x4 at 2048 rows 294 instead of 242.)
        // Items, in order, and about how many vector instructions each takes; an item goes to the slot in which its share
        // of all of them lies, so that the matrix instructions have as even a load beside them as may be.  Against items of whole
        // operands, as many in each slot, it is worth 1 % (outputs x inputs x planes: 4096x4096x4 at 1024 rows 53.0 -> 52.5 us,
        // 11008x4096x4 134.8 -> 133.6, 11008x4096x3 at 2048 204.8 -> 203.7; 5376x640x3 at 759 and two planes level, 432x18016x4 at
        // 407 rows 32.4 -> 32.6).
        constexpr bool WIDE = FMT == kTileBlockWide;
        constexpr int kSigns = NB == 4 ? 23 : 5 + 4 * NB, kLoad = 2 * NB, kTable = 8 << (NB - 1), kQuarter = NB == 4 ? 7 : 6;
        constexpr int kFragment = BLOCK ? 2 + 4 * 2 : 3 + 8, kItems = WIDE ? 3 + 4 * 5 : 2 * kFragment, kSlots = 4 * MF;
        auto weight = [](int k) constexpr {
            if (WIDE) return k < 2 ? kSigns + 4 : k == 2 ? 2 * kLoad : (k - 3) % 5 == 0 ? kTable : kQuarter;
            const int r = k % kFragment - 2;
            return r == -2 ? +kSigns : r == -1 ? +kLoad : r == 0 ? +kTable : +kQuarter;
        };
        auto first_item = [weight](int slot) constexpr {
            if (BLOCK && !WIDE) return slot * kItems / kSlots;   // (finer items cost registers it does not have: 4160x4096x4 at 700 rows 68 -> 78 us)
            int all = 0, before = 0, k = 0;
            for (int i = 0; i < kItems; ++i) all += weight(i);
            while (k < kItems && (2 * before + weight(k)) * kSlots < 2 * all * slot) before += weight(k++);
            return k;
        };
        auto item = [&](auto k_c) {
            constexpr int k = decltype(k_c)::value;
            if constexpr (WIDE) {
                constexpr int r = k - 3, c = r / 5, q = r % 5 - 1;
                if constexpr (k < 2)
                    sign_indices<NB, UNI>(words[k], y[k]);
                else if constexpr (k == 2)
                    load_words(t + 2, words);
                else if constexpr (q < 0)
                    inexact = make_table(t + 1, false, 0, c) || inexact;
                else {   // half of an operand
                    constexpr int f = q / 2, half = q % 2;
                    const u32x2 v = pick_four<NB, UNI, half>(y[f][c], tab[0][c]);
                    A[P ^ 1][c][f][2 * half] = v.x;
                    A[P ^ 1][c][f][2 * half + 1] = v.y;
                }
            } else {
                constexpr int f = k / kFragment, r = k % kFragment - 2;
                if constexpr (r == -2 && BLOCK)
                    sign_indices<NB, UNI>(words[f], y[f]);
                else if constexpr (r == -2)
                    sign_pairs<NB, UNI>(words[f], y[f]);
                else if constexpr (r == -1)
                    load_fragment(t + 2, f, words[f]);
                else if constexpr (BLOCK) {
                    constexpr int c = r / 2;
                    if constexpr (r % 2 == 0)
                        inexact = make_table(t + 1, false, f, c) || inexact;
                    else
                        A[P ^ 1][c][f] = pick(f, c, y[f]);
                } else if constexpr (r == 0) {
                    inexact = make_table(t + 1, false, f, 0) || inexact;
                } else {   // a quarter of a pair of operands
                    constexpr int q = r - 1, h = q / 4, z = q % 2, half = q / 2 % 2;
                    const u32x2 v = pick_four<NB, UNI, half>(y[f][2 * h + z], tab[f][0]);
                    A[P ^ 1][2 * h][f][z + 2 * half] = v.x;
                    A[P ^ 1][2 * h + 1][f][z + 2 * half] = v.y;
                }
            }
        };
        f16x8 b = activations(P, 0, 0);
        static_for<kSlots>([&](auto s_c) {
            constexpr int s = decltype(s_c)::value, j = s / MF, i = s % MF;
            f16x8 next = b;
            if constexpr (s + 1 < kSlots) next = activations(P, (s + 1) / MF, (s + 1) % MF);
#pragma unroll
            for (int f = 0; f < 2; ++f)
                acc[f][i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, A[P][j][f]), b, acc[f][i], 0, 0, 0);
            constexpr int first = first_item(s), count = (s + 1 < kSlots ? first_item(s + 1) : kItems) - first;
            static_for<count>([&](auto c_c) { item(std::integral_constant<int, first + decltype(c_c)::value>()); });
            b = next;
            __builtin_amdgcn_sched_barrier(0);
        });
        lo_cur = __builtin_amdgcn_ballot_w64(inexact) != 0ull;
        if (lo_cur) second_piece(t + 1, P ^ 1);
        store_scales(t + 2, fetched);
        __syncthreads();
    };

    auto take_steps = [&](int t0, int t1) {   // (even numbers)
#pragma unroll
        for (int f = 0; f < 2; ++f)
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[f][i][r] = 0.0f;
        // ---- prologue: step 0's activations in LDS, its weights in A[0] --------------------------------------
        load_x(t0);
        load_words(t0, words);
        uint32_t of_first[kFetched];
        fetch_scales(t0, of_first);
        fetch_scales(t0 + 1, fetched);
        __builtin_amdgcn_sched_barrier(0);
        store_scales(t0, of_first);
        store_scales(t0 + 1, fetched);
        store_x(0);
        load_x(t0 + 1);
        __syncthreads();
#pragma unroll
        for (int f = 0; f < kFragTabs; ++f) unit[f] = unit_for(largest(t0, f));
        lo_cur = __builtin_amdgcn_ballot_w64(make_tables(t0, false)) != 0ull;
        if (lo_cur) load_words(t0, words_lo);
#pragma unroll
        for (int f = 0; f < 2; ++f) {
            uint32_t y[4];
            sign_indices<NB, UNI>(words[f], y);
#pragma unroll
            for (int c = 0; c < 4; ++c) A[0][c][f] = pick(f, c, y);
        }
        load_words(t0 + 1, words);
#pragma clang loop unroll(disable)
        for (int t = t0; t < t1; t += 2) {
            step(t, std::integral_constant<int, 0>());
            step(t + 1, std::integral_constant<int, 1>());
        }

        float back[kFragTabs];
#pragma unroll
        for (int f = 0; f < kFragTabs; ++f) back[f] = inverse_unit(unit[f]);
        scale_sums(back, std::false_type());
    };
    auto each_sum = [&](auto &&f) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int r = 0; r < 16; ++r) f(h, i, r);
    };
    // the steps of a slice, and where its second half begins
    auto first_step = [&](int sl) { return sl * p.slice_steps; };
    auto last_step = [&](int sl) { return min((sl + 1) * p.slice_steps, p.steps); };
    auto second_half = [&](int sl) { return first_step(sl) + (((last_step(sl) - first_step(sl)) / 2 + 1) & ~1); };
    constexpr bool SERIAL = KIND == kTileSerial || KIND == kTileSerialPair;
    if constexpr (SERIAL) {
        f32x16 total[2][MF];
        each_sum([&](int h, int i, int r) { total[h][i][r] = 0.0f; });
#pragma clang loop unroll(disable)
        for (int sl = 0; sl < p.ksplit; ++sl) {   // (every wave has left the LDS of a slice behind the barrier of its last step)
            if constexpr (KIND == kTileSerialPair) {
                f32x16 half[2][MF];
                each_sum([&](int h, int i, int r) { half[h][i][r] = 0.0f; });
#pragma clang loop unroll(disable)
                for (int part = 0; part < 2; ++part) {
                    take_steps(part ? second_half(sl) : first_step(sl), part ? last_step(sl) : second_half(sl));
                    each_sum([&](int h, int i, int r) { half[h][i][r] += acc[h][i][r]; });
                }
                each_sum([&](int h, int i, int r) { total[h][i][r] += half[h][i][r]; });
            } else {
                take_steps(first_step(sl), last_step(sl));
                each_sum([&](int h, int i, int r) { total[h][i][r] += acc[h][i][r]; });
            }
        }
        each_sum([&](int h, int i, int r) { acc[h][i][r] = total[h][i][r]; });
    } else if constexpr (KIND == kTilePair) {
        const int from = first_step(slice), middle = second_half(slice), to = last_step(slice);
        take_steps(team ? middle : from, team ? to : middle);
        // (a barrier per step: the team with fewer of them joins the others')
        for (int t = team ? to - middle : middle - from; t < middle - from; ++t) __syncthreads();
    } else {
        take_steps(first_step(slice), last_step(slice));
    }

    // ---- write-out: lane l holds row l % 32 of a 32-row fragment and outputs 8 g + 4 (l / 32) + 0..3 ------
    // (K cut into slices: the sums of this slice, for tile_sum_kernel to add up)
    // (Sizes below: outputs x inputs x planes.)  What the sums are added to is requested a 32-row fragment ahead of its use (piece by piece
    // where it is added 15360x256x3 at 330 rows with a bias 16.7 us, so 15.0; 2176x1024x3 int8 exponents at 1230 31.8 and 30.6).
    // `turn`: Stored from the accumulators, an instruction touches 32 rows' lines.  Teams, whose sums pass through LDS anyway, turn
    // them round there (16-byte chunk c of row r in slot c ^ r), so that an instruction stores 32 outputs of eight rows: 4096x4096x4 at
    // 512 rows, two slices, 38.5 -> 37.0 us, 2176x1024x3 int8 exponents at 1230 rows with a bias 32.7 -> 30.6.  A lone team's two more
    // passes through LDS cost more than it gives: 5376x640x3 at 759 rows 19.1 -> 20.3.
    float *sums = !SERIAL && p.ksplit > 1 ? p.partial + (size_t)slice * tile_slice_stride(p.M, p.N) : nullptr;
    const bool add = !sums && !p.overwrite;
    auto write_out = [&](auto f_c, auto &&turn) {
        constexpr int f = decltype(f_c)::value;
        constexpr bool TURN = KIND == kTilePair;
        const int here = opaque(lane);   // (nothing formed from it is worth a register of the main loop)
        // piece u of a fragment: the lane's row and output in it
        auto row = [&](int u) { return TURN ? here / 8 + 8 * u : here & 31; };
        auto output = [&](int u) { return n0 + 32 * f + (TURN ? 4 * (here & 7) : 8 * u + 4 * (here / 32)); };
        u32x2 init[2][4];
        auto request = [&](int i) {
            if (add)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    init[i & 1][u] = *(const u32x2_of_halves *)(p.init + (size_t)min(m0 + 32 * i + row(u), p.M - 1) * p.init_stride + min(output(u), p.N - 4));
        };
        request(0);
#pragma unroll
        for (int i = 0; i < MF; ++i) {
            if (i + 1 < MF) request(i + 1);
            f32x4 v4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
#pragma unroll
                for (int r = 0; r < 4; ++r) v4[u][r] = acc[f][i][4 * u + r];
            if constexpr (TURN) {
                char *const at = turn(i);
#pragma unroll
                for (int u = 0; u < 4; ++u) *(f32x4 *)(at + (here & 31) * 128 + (((2 * u + here / 32) ^ (here & 7)) * 16)) = v4[u];
                wave_handover();
#pragma unroll
                for (int u = 0; u < 4; ++u) v4[u] = *(const f32x4 *)(at + row(u) * 128 + (((here & 7) ^ (row(u) & 7)) * 16));
            }
            auto store_all = [&](auto &&store) {
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int m = m0 + 32 * i + row(u), n = output(u);
                    if (m < p.M && n < p.N) store((size_t)m * p.N + n, v4[u]);
                }
            };
            if (sums) {
                store_all([&](size_t at, const f32x4 &v) { *(f32x4 *)(sums + at) = v; });
                continue;
            }
            if (add)
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    asm volatile("" : "+v"(init[i & 1][u]));   // (as new values: or they are converted, and waited for, where they were requested)
                    float v[4] = {v4[u][0], v4[u][1], v4[u][2], v4[u][3]};
                    add_halves(v, init[i & 1][u]);
                    v4[u] = (f32x4){v[0], v[1], v[2], v[3]};
                }
            auto results = [&](int type) {
                store_all([&](size_t at, const f32x4 &v4) {
                    const float v[4] = {v4[0], v4[1], v4[2], v4[3]};
                    store_results(p.out, at, v, type);
                });
            };
            if (p.out_type == kIoF32) results(kIoF32);
            else if (p.out_type == kIoBF16) results(kIoBF16);
            else results(kIoF16);
        }
    };
    if constexpr (KIND == kTilePair) {
        // team 0 finishes the waves' first 32 outputs, team 1 the others: each leaves what the other finishes in LDS
        auto at = [&](int of, int i, int g) { return (f32x4 *)(lds_all + (((of * 4 + wave) * MF + i) * 4 + g) * 1024 + lane * 16); };
        auto finish = [&](auto mine_c) {
            constexpr int mine = decltype(mine_c)::value;
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    f32x4 v;
#pragma unroll
                    for (int r = 0; r < 4; ++r) v[r] = acc[1 - mine][i][4 * g + r];
                    *at(mine, i, g) = v;
                }
            __syncthreads();
#pragma unroll
            for (int i = 0; i < MF; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x4 v = *at(1 - mine, i, g);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[mine][i][4 * g + r] += v[r];
                }
            wave_handover();   // (the lanes' pieces have been read: the wave turns its sums round where they lay)
            write_out(mine_c, [&](int i) { return lds_all + ((1 - mine) * 4 + wave) * MF * 4096 + i * 4096; });
        };
        __syncthreads();   // (the LDS of both teams changes hands)
        if (team == 0)
            finish(std::integral_constant<int, 0>());
        else
            finish(std::integral_constant<int, 1>());
    } else {
        write_out(std::integral_constant<int, 0>(), nullptr);
        write_out(std::integral_constant<int, 1>(), nullptr);
    }
}

// Flat workgroup index -> (output tile, row tile, K-slice).  Workgroups go to the 8 XCDs in turn: the row
// tiles of an output tile, which stream the same sign words, sit on one XCD, behind one L2.
__device__ __forceinline__ void decode_tile(const TileProblem &p, int b, int &n_tile, int &m_tile, int &slice)
{
    const int q = b >> 3;
    m_tile = q % p.m_tiles;
    const int strip = (q / p.m_tiles) * 8 + (b & 7);   // output tile and slice
    n_tile = strip % p.n_tiles;
    slice = strip / p.n_tiles;
}

// Four outputs per thread: the slices' sums, in slice order, and what they are added to.  One launch behind
// the tiles rather than the last slice's workgroup of each tile: that one alone reads at 60 GB/s
// (4096 x 4096, 128 rows, 16 slices: 32 us, most of them this tail).
static __global__ void __launch_bounds__(256) tile_sum_kernel(const TileProblem p)
{
    const uint32_t quads = (uint32_t)p.N / 4u;
    const uint32_t at = blockIdx.x * 256u + threadIdx.x;
    if (at >= quads * (uint32_t)p.M) return;
    const size_t stride = tile_slice_stride(p.M, p.N);
    const float *src = p.partial + (size_t)at * 4u;
    f32x4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
    int sl = 0;
    for (; sl + 4 <= p.ksplit; sl += 4) {
        f32x4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = *(const f32x4 *)(src + (size_t)(sl + u) * stride);
#pragma unroll
        for (int u = 0; u < 4; ++u) sum += q[u];
    }
    for (; sl < p.ksplit; ++sl) sum += *(const f32x4 *)(src + (size_t)sl * stride);
    float v[4] = {sum[0], sum[1], sum[2], sum[3]};
    const uint32_t m = at / quads, n = 4u * (at - m * quads);
    if (!p.overwrite) add_halves(v, p.init + (size_t)m * p.init_stride + n);
    store_results(p.out, (size_t)m * p.N + n, v, p.out_type);
}

template <int NB, int FMT, int MF, int KIND>
__device__ __forceinline__ void gemm_workgroup(const TileProblem &p, char *lds)
{
    int n_tile, m_tile, slice;
    decode_tile(p, (int)blockIdx.x, n_tile, m_tile, slice);
    if (slice >= (KIND == kTileSerial || KIND == kTileSerialPair ? 1 : p.ksplit)) return;
    const int tid = (int)threadIdx.x & (kTileThreads - 1);
    const int team = KIND == kTilePair ? __builtin_amdgcn_readfirstlane((int)threadIdx.x / kTileThreads) : 0;
    if constexpr (FMT == kTileBlock) {
        // most tiles have no wave whose outputs lie in two row groups, and need half the tables
        bool straddles = false;
#pragma unroll
        for (int w = 0; w < kTileN / kTileWaveN; ++w) {
            const int first = n_tile * kTileN + w * kTileWaveN, last = min(first + kTileWaveN, p.N) - 1;
            straddles = straddles || (first < p.N && first / p.rows_per_group != last / p.rows_per_group);
        }
        if (!straddles) {
            gemm_tile<NB, kTileBlockWide, MF, KIND>(p, n_tile, m_tile, slice, tid, team, lds);
            return;
        }
    }
    gemm_tile<NB, FMT, MF, KIND>(p, n_tile, m_tile, slice, tid, team, lds);
}

template <int NB, int FMT, int MF>
__global__ void __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
lut_gemm_tile_kernel(const TileProblem p)
{
    __shared__ __attribute__((aligned(16))) char lds[kTileLdsBytes<FMT, MF>];
    gemm_workgroup<NB, FMT, MF, kTileAlone>(p, lds);
}

template <int NB, int FMT, int MF>
__global__ void __launch_bounds__(2 * kTileThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
lut_gemm_tile_pair_kernel(const TileProblem p)
{
    // (what the teams hand over at the end: 32 outputs x 32 MF rows of every wave)
    constexpr int kHandOver = 2 * 4 * 32 * 32 * MF * 4, kTeams = 2 * kTileLdsBytes<FMT, MF>;
    __shared__ __attribute__((aligned(16))) char lds[kTeams > kHandOver ? kTeams : kHandOver];
    gemm_workgroup<NB, FMT, MF, kTilePair>(p, lds);
}

// One workgroup per tile and per CU (a call that is cut has at most 256 tiles): two sets of accumulators fit, or three
// of 64 rows.
template <int NB, int FMT, int MF, int KIND>
__global__ void __launch_bounds__(kTileThreads) __attribute__((amdgpu_waves_per_eu(1, 1)))
lut_gemm_tile_serial_kernel(const TileProblem p)
{
    __shared__ __attribute__((aligned(16))) char lds[kTileLdsBytes<FMT, MF>];
    gemm_workgroup<NB, FMT, MF, KIND>(p, lds);
}

}  // namespace lutgemm

#endif
