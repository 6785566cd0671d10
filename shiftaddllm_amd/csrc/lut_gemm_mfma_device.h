// Matrix-core kernel templates for BCQ linear layers with a few activation rows (2 to about 128) on MI355X
// (gfx950, wave64), every alpha format: the semantics of lut_gemm/mv_fp16_bias.hpp:8-579 in the ShiftAddLLM
// checkout extended to M rows.
#ifndef LUT_GEMM_MFMA_DEVICE_H
#define LUT_GEMM_MFMA_DEVICE_H

#include "lut_dequant_device.h"

namespace lutgemm {

// ---------------------------------------------------------------------------
// A table look-up costs one LDS read and two VALU operations per sign byte PER ROW, so beyond a row or
// two the look-up kernel is VALU/LDS bound.  Here every weight is formed once as fp16
// (lut_dequant_device.h) and multiplied with 16 activation rows at a time by v_mfma_f32_16x16x32_f16.
// Forming it costs about two to three vector instructions per weight, whatever the row count, which is
// what bounds the kernel up to 32 rows; expanding each plane to +-alpha, as this kernel did before, cost
// one per weight and plane and a matrix instruction per plane instead of one per weight.
//
// Work split: a workgroup of 8 waves owns 64 outputs; its waves take different K-steps (128 inputs = 4
// sign words) and their accumulators meet in LDS at the end, so that the number of cross-workgroup
// atomics does not grow with the K parallelism.  Lane l (li = l&15, kb = l>>4) loads the sign words of
// outputs n = base + 4*li .. +3 for word kb of its step (256-byte runs per row).  Matrix instruction
// (e, c) takes from every lane the eight weights of byte c of its word of output e: its A rows are
// outputs base + 4*i + e and its K block kb is byte c of word kb.
//
// Tables.  Where the step lies in one alpha group, or the alphas are per block, a step needs 64 tables for
// a wave (one per output) or 16 (one per 8 inputs and row group): lane (li, kb) forms the one of output
// base + 4*li + kb, or of chunk li and row group kb, and the lanes hand them round by ds_bpermute.
// Shorter groups (OWN) leave every lane with four tables of its own.
//
// Activations: a lane's B operands of a step are the 32 activations of row li under its word kb, 64 contiguous
// bytes.  With 16 rows a lane loads them itself.  A request's 64 lanes then touch 32 cache lines, 32 bytes of each, and
// every line is asked for four times; at 32 rows that bounded the kernel (8192x28672x4 46.4 us, 36.3 with the activations
// left out, 45.0 with the weights left unformed).  So with 32 rows a request takes four rows' 256 contiguous bytes and the
// wave turns them round in LDS of its own: 42.4 us; 28672x8192x4 54.9 -> 49.4, 11008x4096x3 15.4 -> 14.2.  (With 16 rows
// the detour costs more than it gives, registers above all: 8192x8192x4 at 4 rows 12.0 -> 16.2; nor does it where weights come in two pieces and forming
// them bounds the kernel: uniform 8192x8192x4 at 17 rows 30.3 -> 31.3.)
//
// There is no barrier in the main loop: each wave runs its own two-deep pipeline of (signs, scales, activations) and
// the waves of a workgroup drift freely until the final reduction.
// ---------------------------------------------------------------------------
constexpr int kMfmaThreads = 512;
constexpr int kMfmaWaves = kMfmaThreads / 64;
constexpr int kMfmaTileCols = 64;     // outputs per workgroup
constexpr int kMfmaStepK = 128;
constexpr int kMfmaMaxRowGroups = 4;  // alpha row groups 64 outputs may touch (block formats)
constexpr int kRedRow = 65;           // the final reduction's LDS rows, padded against bank conflicts
template <int MT>
constexpr int kMfmaRedBytes = kMfmaWaves * 16 * MT * kRedRow * 4;
// a wave's activations on their way to operands: 16 rows of 128 inputs, 16 bytes apart, so that the 16 rows of a
// read spread over all banks
constexpr int kTurnRow = 256 + 16;
template <int MT>
constexpr int kMfmaTurnBytes = MT > 1 ? kMfmaWaves * MT * 16 * kTurnRow : 0;
// the rows' reciprocal RMS sit behind both
template <int MT>
constexpr int kMfmaScaleAt = kMfmaTurnBytes<MT> > kMfmaRedBytes<MT> ? kMfmaTurnBytes<MT> : kMfmaRedBytes<MT>;
template <int MT>
constexpr int kMfmaLdsBytes = kMfmaScaleAt<MT> + 16 * MT * 4;

// Operands of one K-step of a wave: per bit plane word kb of 4 outputs; per 16-row tile the lane's 32 activations (to
// be turned round: chunk li of rows kb, kb + 4, ...); the scales of the lane's table(s), as they lie in memory.
template <int NB, int MT, int FMT, bool OWN>
struct MfmaOperands {
    static constexpr int kScales = FMT == kWeightUniform ? (OWN ? 4 : 2) : (OWN ? 2 * NB : NB);
    u32x4 w[NB];
    u32x4 x[MT][4];
    uint32_t s[kScales];
};

// xs: kMfmaLdsBytes<MT> bytes of LDS for the final reduction (and, behind them, the reciprocal RMS of the
// tile's rows).
// OWN: every lane forms its own four tables (per-column alphas with groups that are no multiple of 128
//      inputs, or K no multiple of 128).
// EXTRA: the launch honours the split-RMSNorm fields of the problem (next_in, sumsq_*).
// ONE: every K-slice of the launch is a single round, i.e. a wave takes at most one step (the
//      host's choice): nothing is requested beyond that step.
// GATE: the launch's two problems are a gate and an up projection (`side` 0 and 1) whose product goes to gated.act:
//      whoever completes the second of an output's two sums finds the first in the output's word and forms it.
template <int NB, int MT, int FMT = kWeightRow, bool OWN = false, bool EXTRA = false, bool ONE = false, bool GATE = false>
__device__ __forceinline__ void mfma_tile(const Problem &p, int local_block, char *xs, const GatedPair &gated = GatedPair(), int side = 0)
{
    constexpr bool UNI = FMT == kWeightUniform;
    static_assert(!OWN || FMT != kWeightBlock, "block formats share their tables");
    typedef MfmaOperands<NB, MT, FMT, OWN> Operands;
    typedef WeightTable<NB, UNI> Table;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int li = lane & 15;
    const int kb = lane >> 4;
    // flat workgroup index (relative to the problem) -> (tile, K-slice, row chunk)
    const int slice = quotient(local_block, p.n_tiles, p.tiles_reciprocal);
    const int tile = local_block - slice * p.n_tiles;
    const int mchunk = quotient(slice, p.ksplit, p.ksplit_reciprocal);
    const int kslice = slice - mchunk * p.ksplit;
    const int m0 = mchunk * 16 * MT;
    const int n_base = tile * kMfmaTileCols;

    const uint32_t wcol4 = (uint32_t)min(n_base + 4 * li, p.N - 4) * 4u;

    const int step_begin = kslice * p.sets_per_split;
    const int step_end = min(step_begin + p.sets_per_split, p.nsets);

    // the lane's activations: row li of each 16-row tile, or rows kb + 4 c (rows beyond M are clamped to the last one:
    // computed twice, written once; byte offsets: the host keeps M * K * 2 below 2^32, and what wraps beyond it belongs
    // to no row)
    constexpr bool TURN = MT > 1 && !UNI;
    const uint32_t row_bytes_x = (uint32_t)p.K * 2u, xlast = (uint32_t)(p.M - 1) * row_bytes_x;
    uint32_t xfirst[TURN ? 1 : MT];
#pragma unroll
    for (int mt = 0; mt < (TURN ? 1 : MT); ++mt)
        xfirst[mt] = (uint32_t)(TURN ? m0 + kb : min(m0 + 16 * mt + li, p.M - 1)) * row_bytes_x;
    [[maybe_unused]] char *const turn_in = xs + wave * (MT * 16 * kTurnRow) + kb * kTurnRow + li * 16;
    [[maybe_unused]] const char *const turn_out = xs + wave * (MT * 16 * kTurnRow) + li * kTurnRow + kb * 64;

    // block formats: the tile's row groups; this lane forms tables of group rg and looks its own outputs up
    // among those of lane group rg_of
    [[maybe_unused]] int rg = 0, rg_of = 0;
    if constexpr (FMT == kWeightBlock) {
        const int rg0 = n_base / p.rows_per_group, n_rg = min(n_base + kMfmaTileCols - 1, p.N - 1) / p.rows_per_group - rg0 + 1;
        rg = rg0 + min(kb, n_rg - 1);
        rg_of = (int)(wcol4 >> 2) / p.rows_per_group - rg0;
    }

    auto load = [&](Operands &r, int step) {
        // (a word beyond K, in the last step only: clamped; its weights are zero)
        const int kbc = OWN || FMT == kWeightBlock ? min(kb, p.kwords - 1 - 4 * step) : kb;
        const uint32_t row_bytes = (uint32_t)p.N * 4u;
        const char *wbase = (const char *)p.W + (size_t)step * 4 * NB * row_bytes;
        const uint32_t wrow = (uint32_t)kbc * (NB * row_bytes);
#pragma unroll
        for (int b = 0; b < NB; ++b)
            r.w[b] = __builtin_nontemporal_load((const u32x4 *)(wbase + (size_t)b * row_bytes + (wrow + wcol4)));
        if constexpr (FMT == kWeightBlock) {
            const int rows = p.K / 8 * NB;
#pragma unroll
            for (int b = 0; b < NB; ++b)
                r.s[b] = raw_multiplier(p.alpha, p.alpha_mode, (uint32_t)(min(16 * step + li, p.K / 8 - 1) * NB + b) * (uint32_t)p.R + (uint32_t)rg,
                                        (uint32_t)rows * (uint32_t)p.R);
        } else if constexpr (OWN) {
            const uint32_t g = (uint32_t)fast_div(4 * step + kbc, p.by_group_words);
            if constexpr (UNI) {
                const uint32_t at = g * (p.N * 2u) + (wcol4 >> 1);
                const u32x2 a = *(const u32x2 *)((const char *)p.alpha + at), q = *(const u32x2 *)((const char *)p.qbias + at);
                r.s[0] = a.x;
                r.s[1] = a.y;
                r.s[2] = q.x;
                r.s[3] = q.y;
            } else {
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    const u32x2 a = *(const u32x2 *)((const char *)p.alpha + ((g * NB + (uint32_t)b) * (p.N * 2u) + (wcol4 >> 1)));
                    r.s[2 * b] = a.x;
                    r.s[2 * b + 1] = a.y;
                }
            }
        } else {
            const int g = fast_div(step * 4, p.by_group_words);
            const uint32_t col2 = (wcol4 >> 1) + 2u * (uint32_t)kb;
            if constexpr (UNI) {
                r.s[0] = *(const unsigned short *)((const char *)p.alpha + (size_t)g * (p.N * 2u) + col2);
                r.s[1] = *(const unsigned short *)((const char *)p.qbias + (size_t)g * (p.N * 2u) + col2);
            } else {
#pragma unroll
                for (int b = 0; b < NB; ++b)
                    r.s[b] = *(const unsigned short *)((const char *)p.alpha + (size_t)(g * NB + b) * (p.N * 2u) + col2);
            }
        }
        // (beyond K: the last chunk, for weights of zero)
        [[maybe_unused]] const uint32_t xchunk = (uint32_t)min(16 * step + li, p.K / 8 - 1) * 16u;
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int c = 0; c < 4; ++c)
                r.x[mt][c] = TURN ? *(const u32x4 *)((const char *)p.x + (min(xfirst[0] + (uint32_t)(16 * mt + 4 * c) * row_bytes_x, xlast) + xchunk))
                                  : *(const u32x4 *)((const char *)p.x + (xfirst[TURN ? 0 : mt] + (uint32_t)(4 * step + kbc) * 64u) + 16 * c);
    };

    // split RMSNorm, consuming side: wave w sums the slots of rows w, w + 8, ... and leaves
    // their reciprocal RMS in LDS for the hand-over
    // The slots are requested here, ahead of everything else, and summed once the first
    // step's operands have been requested behind them (see the main loop): loads return in
    // order, so that wait is for the slots alone.
    float *row_scale = (float *)(xs + kMfmaScaleAt<MT>);
    constexpr int kScaleRows = 2 * MT;  // rows per wave
    bool scaled = false;
    [[maybe_unused]] f32x4 slot4[kScaleRows];
    // (the wave index as a scalar, so that the rows' addresses are a scalar base plus one lane offset)
    const int wave_s = __builtin_amdgcn_readfirstlane(wave);
    if constexpr (EXTRA) {
        scaled = p.sumsq_in != nullptr;
        if (scaled) {
            // one 16-byte request per row and lane: 256 slots, inputs up to 8192 (slots = K / 32
            // and K % 128 == 0 on this path)
            const int quads = p.sumsq_slots >> 2;
#pragma unroll
            for (int i = 0; i < kScaleRows; ++i) {
                const float *slots = p.sumsq_in + (size_t)min(m0 + wave_s + kMfmaWaves * i, p.M - 1) * p.sumsq_slots;
                slot4[i] = *((const f32x4 *)slots + min(lane, quads - 1));
            }
        }
    }
    auto row_scales = [&]() {
        const int quads = p.sumsq_slots >> 2;
#pragma unroll
        for (int i = 0; i < kScaleRows; ++i) {
            const int row = wave_s + kMfmaWaves * i;
            const float *slots = p.sumsq_in + (size_t)min(m0 + row, p.M - 1) * p.sumsq_slots;
            float t = lane < quads ? (slot4[i].x + slot4[i].y) + (slot4[i].z + slot4[i].w) : 0.0f;
            for (int c = 4 * 64 + lane; c < p.sumsq_slots; c += 64) t += slots[c];  // inputs beyond 8192
            t = wave_sum(t);
            if (lane == 0) row_scale[row] = rsqrtf(t / (float)p.K + p.norm_eps);
        }
    };

    f32x4 acc[4][MT];
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) acc[e][mt] = (f32x4){0.0f, 0.0f, 0.0f, 0.0f};

    // ---- one K-step ---------------------------------------------------------------------------------
    constexpr int kTables = OWN ? 4 : 1;   // tables this lane forms
    // Weights are formed as W * unit, a power of two per output (block formats: per row group), held by the lane
    // whose table it scales.  OWN: by the four lanes whose tables they are, the biased exponents of a lane's four as the
    // bytes of one register (8192x8192x4 in groups of 32, 8 rows 38 us with four registers, 29 with one; 34 when one
    // unit served the whole wave); all begin with the unit that suits the wave's largest output, which is what
    // ordinary layers stay with: their sums are scaled back by one number.  A single step (ONE) has the units it
    // chose and needs no check.
    typename std::conditional<OWN, uint32_t, float>::type units = OWN ? 0 : 1;
    bool chosen = false;
    bool same = OWN;                       // all units of the wave are one
    auto unit = [&](int i) {
        if constexpr (OWN) return __builtin_bit_cast(float, ((units >> (8 * i)) & 0xffu) << 23);
        else return units;
    };
    // multipliers of this lane's table i
    auto multipliers = [&](const Operands &ops, int i, float (&a)[NB], float &q) {
        q = 0.0f;
        auto half_of = [&](int r) { return half_bits_to_float((ops.s[r + (i >> 1)] >> (16 * (i & 1))) & 0xffffu); };   // (OWN)
        if constexpr (FMT == kWeightBlock) {
#pragma unroll
            for (int b = 0; b < NB; ++b) a[b] = decode_multiplier(ops.s[b], p.alpha_mode);
        } else if constexpr (UNI) {
            const float alpha = OWN ? half_of(0) : half_bits_to_float(ops.s[0]);
#pragma unroll
            for (int b = 0; b < NB; ++b) a[b] = alpha * (1.0f / (float)(2 << b));
            q = OWN ? half_of(2) : half_bits_to_float(ops.s[1]);
        } else {
#pragma unroll
            for (int b = 0; b < NB; ++b) a[b] = OWN ? half_of(2 * b) : half_bits_to_float(ops.s[b]);
        }
    };
    auto magnitude = [&](const Operands &ops, int i) {   // upper bound of |W| in the lane's table i
        float a[NB], q;
        multipliers(ops, i, a, q);
        return finite_magnitude(a, q);
    };
    // its maximum over the tables that share a unit
    auto largest = [&](const Operands &ops, int i) {
        float m = magnitude(ops, i);
        if constexpr (OWN) {   // the step's four words
            m = fmaxf(m, lane_value(m, opaque(lane) ^ 16));
            m = fmaxf(m, lane_value(m, opaque(lane) ^ 32));
        } else if constexpr (FMT == kWeightBlock) {   // the step's sixteen chunks: a row of 16 lanes
            m = fmaxf(m, dpp_move<0xb1>(m));
            m = fmaxf(m, dpp_move<0x4e>(m));
            m = fmaxf(m, dpp_move<0x141>(m));
            m = fmaxf(m, dpp_move<0x140>(m));
        }
        return m;
    };
    // Accumulators times a factor per unit: register r of acc[e] is output 4 * (4 * kb + r) + e of the tile.
    // In the main loop the factors are fetched a few at a time (all sixteen in flight are registers that the
    // operands of the steps need).
    auto scale_sums = [&](const float (&by)[kTables], auto in_loop) {
        [[maybe_unused]] const float of_quad = FMT == kWeightBlock ? lane_value(by[0], 16 * rg_of) : 0.0f;
        const int quad = opaque(4 * kb);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            [[maybe_unused]] const float of_group = FMT == kWeightBlock ? lane_value(of_quad, quad + r) : 0.0f;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float f = FMT == kWeightBlock ? of_group : OWN ? lane_value(by[e % kTables], quad + r) : lane_value(by[0], 16 * e + quad + r);
#pragma unroll
                for (int mt = 0; mt < MT; ++mt) acc[e][mt][r] *= f;
            }
            if constexpr (decltype(in_loop)::value) __builtin_amdgcn_sched_barrier(0);
        }
    };
    auto refit = [&](const Operands &ops) {   // units that suit this step
        float by[kTables];
        decltype(units) now = 0;
#pragma unroll
        for (int i = 0; i < kTables; ++i) {
            const float most = largest(ops, i), old = unit(i), fresh = outside_window(most, old) ? unit_for(most) : old;
            by[i] = fresh * inverse_unit(old);
            if constexpr (OWN) now |= (__builtin_bit_cast(uint32_t, fresh) >> 23) << (8 * i);
            else now = fresh;
        }
        units = now;
        same = false;
        if constexpr (!ONE) scale_sums(by, std::true_type());
    };
    auto any_outside = [&](const Operands &ops) {
        bool outside = false;
#pragma unroll
        for (int i = 0; i < kTables; ++i) outside = outside_window(magnitude(ops, i), unit(i)) || outside;
        return __builtin_amdgcn_ballot_w64(outside) != 0ull;
    };
    // The lane's tables of a step, or of what rounding their entries leaves over; true when some entry may
    // not be an fp16 number.
    auto make_tables = [&](const Operands &ops, int step, bool lo, Table (&tab)[kTables]) {
        bool inexact = false;
#pragma unroll
        for (int i = 0; i < kTables; ++i) {
            float u = unit(i);
            if constexpr (FMT == kWeightBlock) u = 16 * step + li < p.K / 8 ? u : 0.0f;
            if constexpr (OWN) u = 4 * step + kb < p.kwords ? u : 0.0f;
            float a[NB], q;
            multipliers(ops, i, a, q);
#pragma unroll
            for (int b = 0; b < NB; ++b) a[b] *= u;
            const TableEntries<NB, UNI> e = table_entries<NB, UNI>(a, q * u);
            if (lo) {
                pack_table(table_residual(e), tab[i]);
            } else {
                inexact = may_round<NB, UNI, MT == 1>(e, a, q * u) || inexact;
                pack_table(e, tab[i]);
            }
        }
        return inexact;
    };
    auto from_lane = [&](const Table &t, int src) {
        Table r;
#pragma unroll
        for (int i = 0; i < Table::kRegs; ++i) {
            r.hi[i] = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * src, (int)t.hi[i]);
            r.lo[i] = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * src, (int)t.lo[i]);
        }
        return r;
    };
    [[maybe_unused]] auto turn_round = [&](Operands &ops) {   // to inputs 8 c .. 8 c + 7 of the lane's word
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int c = 0; c < 4; ++c) *(u32x4 *)(turn_in + (16 * mt + 4 * c) * kTurnRow) = ops.x[mt][c];
        wave_handover();
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int c = 0; c < 4; ++c) ops.x[mt][c] = *(const u32x4 *)(turn_out + 16 * mt * kTurnRow + 16 * c);
        wave_handover();   // (the next step's stores)
    };
    auto multiply = [&](const Operands &ops, const Table (&tab)[kTables]) {
        Table t4[4];   // per output, or (block formats) per byte of the word
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (OWN)
                t4[i] = tab[i];
            else if constexpr (FMT == kWeightBlock)
                t4[i] = from_lane(tab[0], 16 * rg_of + 4 * kb + i);
            else
                t4[i] = from_lane(tab[0], 16 * i + li);
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            uint32_t w[NB], y[4];
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                w[b] = ops.w[b][e];
                asm volatile("" : "+v"(w[b]));   // (opaque: or the indices are kept for a second piece)
            }
            auto product = [&](int c, const u32x4 &a) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
                    acc[e][mt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, ops.x[mt][c]),
                                                                        acc[e][mt], 0, 0, 0);
            };
            // Two operands at a time save four instructions, but hold four registers more: 16-row tiles of four planes
            // and the grouped kernel, which have none left, spill more (8192x8192x4 at 4 rows 12.2 -> 12.6 us, decoding
            // a token for eight sequences 2391 -> 2470); 32-row tiles gain (8192x28672x4 42.4 -> 41.6, 11008x4096x3 14.2 ->
            // 13.7), three planes a little (4096x4096x3 at 8 rows 6.96 -> 6.81).
            if constexpr (FMT == kWeightBlock || (MT == 1 && (NB == 4 || EXTRA))) {
                sign_indices<NB, UNI>(w, y);
#pragma unroll
                for (int c = 0; c < 4; ++c) product(c, pick_weights<NB, UNI>(y[c], t4[FMT == kWeightBlock ? c : e]));
            } else {
                sign_pairs<NB, UNI>(w, y);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    u32x4 a[2];
                    pick_pair<NB, UNI>(y[2 * h], y[2 * h + 1], t4[e], a);
                    product(2 * h, a[0]);
                    product(2 * h + 1, a[1]);
                }
            }
        }
    };
    auto compute = [&](Operands &ops, int step) {
        if constexpr (!EXTRA)
            if (p.x_type == kIoBF16) {
#pragma unroll
                for (int mt = 0; mt < MT; ++mt)
#pragma unroll
                    for (int c = 0; c < 4; ++c)
#pragma unroll
                        for (int j = 0; j < 4; ++j) ops.x[mt][c][j] = halves_of_bf16(ops.x[mt][c][j]);
            }
        if constexpr (TURN) turn_round(ops);
        if (!chosen) {
            chosen = true;
            if constexpr (OWN) {
                float most = 0.0f;
#pragma unroll
                for (int i = 0; i < kTables; ++i) most = fmaxf(most, magnitude(ops, i));
                units = (__builtin_bit_cast(uint32_t, unit_for(wave_max(most))) >> 23) * 0x01010101u;
                if (ONE && any_outside(ops)) refit(ops);
            } else {
                units = unit_for(largest(ops, 0));
            }
        }
        Table tab[kTables];
        bool inexact = __builtin_amdgcn_ballot_w64(make_tables(ops, step, false, tab)) != 0ull;
        auto forget = [&]() {   // (the scales as new values: or the multipliers are kept for a second piece)
            if constexpr (OWN)
#pragma unroll
                for (int r = 0; r < Operands::kScales; ++r) asm volatile("" : "+v"(ops.s[r]));
        };
        if (!ONE && inexact) {   // (a single step has the units it chose)
            forget();
            if (any_outside(ops)) {
                forget();
                refit(ops);
                forget();
                inexact = __builtin_amdgcn_ballot_w64(make_tables(ops, step, false, tab)) != 0ull;
            }
        }
        multiply(ops, tab);
        if (inexact) {
            forget();
            (void)make_tables(ops, step, true, tab);
            multiply(ops, tab);
        }
    };

    // This wave's steps: step_begin + wave, + 8, ...  Two operand buffers alternate and
    // each step's loads are issued one compute phase ahead.  Steps are taken in pairs by
    // a counted loop with one load site per buffer (a second site makes the register
    // allocator reconcile the two with copies that wait for the loads): the first
    // iteration skips its first compute at run time, and a load beyond the wave's last
    // step re-reads that last step (the lines the wave has just asked for) and is
    // discarded, so that the waits can count it.
    Operands opA, opB;
    const int last_step = p.nsets - 1;
    const int first_step = step_begin + wave_s;
    const int n_steps = first_step < step_end ? (step_end - first_step + kMfmaWaves - 1) / kMfmaWaves : 0;
    const int own_last = n_steps > 0 ? first_step + kMfmaWaves * (n_steps - 1) : last_step;
    const int pairs = ONE ? 0 : (n_steps + 1) / 2;
    if constexpr (ONE) {
        // One round per slice: the general loop would request a second, discarded step behind
        // the first one, and a wave cannot end before those loads have come back.
        load(opA, min(first_step, last_step));
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (EXTRA)
            if (scaled) row_scales();
        __builtin_amdgcn_sched_barrier(0);
        if (n_steps > 0) compute(opA, first_step);
    }
#pragma clang loop unroll(disable)
    for (int j = 0; j < pairs; ++j) {
        // (opaque, which keeps the compiler from peeling the first iteration)
        int first = __builtin_amdgcn_readfirstlane(j == 0);
        asm volatile("" : "+s"(first));
        const int s = first_step + 2 * kMfmaWaves * j;
        load(opA, min(s, own_last));
        __builtin_amdgcn_sched_barrier(0);
        if (!first) compute(opB, s - kMfmaWaves);
        if constexpr (EXTRA)
            if (first && scaled) row_scales();
        __builtin_amdgcn_sched_barrier(0);
        load(opB, min(s + kMfmaWaves, own_last));
        __builtin_amdgcn_sched_barrier(0);
        compute(opA, s);
    }
    if (!ONE && n_steps > 0 && (n_steps & 1) == 0) compute(opB, own_last);
    if constexpr (EXTRA && !ONE)
        if (n_steps == 0 && scaled) row_scales();  // (a wave without steps still owes its rows)
    if (same) {
        const float back = chosen ? inverse_unit(unit(0)) : 1.0f;
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) acc[e][mt] *= back;
    } else {
        float back[kTables];
#pragma unroll
        for (int i = 0; i < kTables; ++i) back[i] = inverse_unit(unit(i));
        scale_sums(back, std::false_type());
    }

    // ---- the 8 waves' accumulators meet in LDS -----------------------------------
    // red[wave][j = (e*MT + mt)*4 + r][lane], rows padded to 65 words so that the
    // read-out below (consecutive threads = consecutive outputs) spreads over the banks
    float *red = (float *)xs;
    // Thread t finishes output column t & 63 of rows (t >> 6) + 8*i: a wave covers 64
    // consecutive outputs of one row, so its atomics and its fp16 read-modify-write
    // fall into whole cache lines.
    const int nl = tid & 63;
    const int n = n_base + nl;
    // What the caller had in those outputs is requested here, not where the sums are complete: the request then runs beside
    // the reduction and the atomics instead of behind them (768x3072x3 int8 exponents at 128 rows 11.1 -> 10.3 us, 4096x4096x3
    // with a bias at 16 rows 7.5 -> 6.8).  Ahead of the main loop it costs registers that the operands need (8 sequences'
    // down_proj of 4 planes 13.7 -> 14.7).  Whoever completes an output has read it before any contribution of its own, and
    // nobody writes it before all contributions are there.
    [[maybe_unused]] uint32_t init_bits[2 * MT];
    [[maybe_unused]] uint32_t next_w_bits = 0;
    if constexpr (!GATE) {
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) init_bits[i] = 0;
        if (!p.overwrite)
#pragma unroll
            for (int i = 0; i < 2 * MT; ++i)
                init_bits[i] = *(const uint16_t *)(p.init + (size_t)min(m0 + (tid >> 6) + 8 * i, p.M - 1) * p.init_stride + min(n, p.N - 1));
        if constexpr (EXTRA)
            if (p.next_w) next_w_bits = *(const uint16_t *)(p.next_w + min(n, p.N - 1));
    }
    if constexpr (TURN) __syncthreads();   // (the waves' activations lie there)
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                red[(wave * (16 * MT) + (e * MT + mt) * 4 + r) * kRedRow + lane] = acc[e][mt][r];
    __syncthreads();
    const int src_lane = (nl >> 4) * 16;            // kb of the column; + li of the row below
    const int src_j = (nl & 3) * MT * 4 + ((nl >> 2) & 3);  // e and r of the column; + mt*4 of the row
    float val[2 * MT];
    Contribution contrib[2 * MT];
    unsigned long long old[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int ml = (tid >> 6) + 8 * i;          // row within the chunk
        const int j = src_j + (ml >> 4) * 4, sl = src_lane + (ml & 15);
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < kMfmaWaves; ++w) v += red[(w * (16 * MT) + j) * kRedRow + sl];
        if (scaled) v *= row_scale[ml];
        val[i] = v;
        old[i] = 0;
        contrib[i] = Contribution{0ull, 0ull};
        const int m = m0 + ml;
        if (p.ksplit > 1 && m < p.M && n < p.N) {
            unsigned long long *word = p.accum + (size_t)m * p.N + n;
            contrib[i] = fixed_contribution(v);
            if (contrib[i].flags)
                __hip_atomic_fetch_or(word, contrib[i].flags, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            old[i] = __hip_atomic_fetch_add(word, contrib[i].add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if constexpr (GATE) {
        constexpr uint32_t kThere = 0x10000u;
        uint32_t mine[2 * MT], other[2 * MT];
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i) {
            const int m = m0 + (tid >> 6) + 8 * i;
            other[i] = 0;
            if (m < p.M && n < p.N && (p.ksplit == 1 || (int)(old[i] >> 56) == p.ksplit - 1)) {
                mine[i] = float_to_half_bits(p.ksplit == 1 ? val[i] : fixed_total((old[i] | contrib[i].flags) + contrib[i].add, p.ksplit));
                other[i] = __hip_atomic_exchange(gated.words + ((size_t)m * p.N + n), mine[i] | kThere, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (p.ksplit > 1)
                    __hip_atomic_store(p.accum + (size_t)m * p.N + n, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            }
        }
#pragma unroll
        for (int i = 0; i < 2 * MT; ++i)
            if (other[i] != 0) {
                const size_t at = (size_t)(m0 + (tid >> 6) + 8 * i) * p.N + n;
                __hip_atomic_store(gated.words + at, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const float g = half_bits_to_float(side == 0 ? mine[i] : other[i] & 0xffffu), u = half_bits_to_float(side == 0 ? other[i] & 0xffffu : mine[i]);
                gated.act[at] = __float2half_rn(__half2float(__float2half_rn(g / (1.0f + __expf(-g)))) * u);
            }
        return;
    }
    // (as new values: or they are converted, and waited for, where they were requested)
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) asm volatile("" : "+v"(init_bits[i]));
    if constexpr (EXTRA) asm volatile("" : "+v"(next_w_bits));
    [[maybe_unused]] const float next_w = half_bits_to_float(next_w_bits);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
        const int m = m0 + (tid >> 6) + 8 * i;
        [[maybe_unused]] float sq = 0.0f;  // square of the output this thread completed
        if (m < p.M && n < p.N && (p.ksplit == 1 || (int)(old[i] >> 56) == p.ksplit - 1)) {
            const float y = p.ksplit == 1 ? val[i] : fixed_total((old[i] | contrib[i].flags) + contrib[i].add, p.ksplit);
            const float sum = half_bits_to_float(init_bits[i]) + y;
            const __half y16 = __float2half_rn(sum);
            if constexpr (EXTRA)
                p.out[(size_t)m * p.N + n] = y16;
            else
                store_result(p.out, (size_t)m * p.N + n, sum, p.out_type);
            if (p.ksplit > 1)
                __hip_atomic_store(p.accum + (size_t)m * p.N + n, 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if constexpr (EXTRA) {
                const float yf = __half2float(y16);
                sq = yf * yf;
                if (p.next_in) p.next_in[(size_t)m * p.N + n] = __float2half_rn(yf * next_w);
            }
        }
        if constexpr (EXTRA) {
            // the wave's 64 columns of row m: one add into the first of their two slots
            if (p.sumsq_out) {
                const float s = wave_sum(sq);
                if (lane == 0 && m < p.M && s != 0.0f)
                    unsafeAtomicAdd(p.sumsq_out + (size_t)m * (p.N / 32) + n_base / 32, s);
            }
        }
    }
}

template <int NB, int MT, int FMT, bool OWN, bool ONE>
__global__ void __launch_bounds__(kMfmaThreads) __attribute__((amdgpu_waves_per_eu(MT == 1 ? 4 : 2, MT == 1 ? 4 : 2)))
lut_gemm_mfma_kernel(const Problem p)
{
    __shared__ __attribute__((aligned(16))) char xs[kMfmaLdsBytes<MT>];
    touch_arguments(p);
    mfma_tile<NB, MT, FMT, OWN, false, ONE>(p, (int)blockIdx.x, xs);
}

// One row-wise problem with the split-RMSNorm fields honoured.
template <int NB, int MT, bool ONE = false>
__global__ void __launch_bounds__(kMfmaThreads) __attribute__((amdgpu_waves_per_eu(MT == 1 ? 4 : 2, MT == 1 ? 4 : 2)))
lut_gemm_mfma_fused_kernel(const Problem p)
{
    __shared__ __attribute__((aligned(16))) char xs[kMfmaLdsBytes<MT>];
    touch_arguments(p);
    mfma_tile<NB, MT, kWeightRow, false, true, ONE>(p, (int)blockIdx.x, xs);
}

// Several row-wise problems in one launch; bit widths may differ.
template <int MT>
__global__ void __launch_bounds__(kMfmaThreads) __attribute__((amdgpu_waves_per_eu(MT == 1 ? 4 : 2, MT == 1 ? 4 : 2)))
lut_gemm_mfma_group_kernel(const Group g)
{
    __shared__ __attribute__((aligned(16))) char xs[kMfmaLdsBytes<MT>];
    // grid = (workgroups of the largest problem, problems)
    // (through the constant address space, which the kernel arguments live in: the fields are
    // then scalar loads that may be repeated at will instead of values to keep in registers)
    const Problem &p = *(const Problem *)((const __attribute__((address_space(4))) Problem *)&g.p[0] + blockIdx.y);
    const int b = blockIdx.x;
    touch_arguments(p);
    if (b >= p.n_blocks) return;
    switch (p.nb) {
    case 1: mfma_tile<1, MT, kWeightRow, false, true>(p, b, xs); break;
    case 2: mfma_tile<2, MT, kWeightRow, false, true>(p, b, xs); break;
    case 3: mfma_tile<3, MT, kWeightRow, false, true>(p, b, xs); break;
    default: mfma_tile<4, MT, kWeightRow, false, true>(p, b, xs); break;
    }
}

// A gate and an up projection and their product (see GATE).  The product as a launch of its own took 4.5 us of the device
// behind the 19.6 of the two projections (8 rows, 2 x 11008x4096 of 2 to 4 planes); the exchange costs 0.4.  A token for
// eight sequences, 32 of these launches, 2331 -> 2252 us.  (Tiles of half gate, half up columns, which need no exchange
// but equal widths and no K-slices, took 20.4 for 3 + 3 planes.)
template <int MT>
__global__ void __launch_bounds__(kMfmaThreads) __attribute__((amdgpu_waves_per_eu(MT == 1 ? 4 : 2, MT == 1 ? 4 : 2)))
lut_gemm_mfma_gated_kernel(const GatedProblems g)
{
    __shared__ __attribute__((aligned(16))) char xs[kMfmaLdsBytes<MT>];
    const int side = blockIdx.y;
    const Problem &p = *(const Problem *)((const __attribute__((address_space(4))) Problem *)&g.p[0] + side);
    const int b = blockIdx.x;
    touch_arguments(p);
    if (b >= p.n_blocks) return;
    switch (p.nb) {
    case 1: mfma_tile<1, MT, kWeightRow, false, true, false, true>(p, b, xs, g.pair, side); break;
    case 2: mfma_tile<2, MT, kWeightRow, false, true, false, true>(p, b, xs, g.pair, side); break;
    case 3: mfma_tile<3, MT, kWeightRow, false, true, false, true>(p, b, xs, g.pair, side); break;
    default: mfma_tile<4, MT, kWeightRow, false, true, false, true>(p, b, xs, g.pair, side); break;
    }
}

}  // namespace lutgemm

#endif
