// Glue kernels of a single-token decode step around the LUT-GEMV calls, for
// gfx950: RMSNorm (which also clears the next GEMV's accumulate-into outputs),
// rotary embedding + KV-cache append + one-query attention, and SiLU(gate)*up.
//
// A decoder block at one token per sequence is, with these, eight launches:
//   rmsnorm -> {q,k,v} GEMV -> attention -> o_proj GEMV (accumulates into the
//   residual stream) -> rmsnorm -> {gate,up} GEMV -> silu*mul -> down_proj GEMV
//   (accumulates into the residual stream).
// The reference runs the same step through HuggingFace's eager OPT decoder
// (model/opt.py:367-423 of the ShiftAddLLM checkout drives it); it has no fused
// kernels of this kind.  All of them are tiny and latency bound: they exist to
// replace some forty framework kernels per block by four.
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "lutgemm_gfx950.h"
#include "lutgemm_common.h"
#include "lutgemm_internal.h"

namespace {

constexpr int kThreads = 256;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// The value of another lane of the same row of 16, by a data-parallel-primitive move.
template <int CTRL>
__device__ __forceinline__ float dpp_lane(float v)
{
    const int vi = __builtin_bit_cast(int, v);
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(vi, vi, CTRL, 0xf, 0xf, false));
}

// Sum / maximum over the 64 lanes of a wave on the vector ALU: xor 1 and 2 inside quads, the
// mirrored quad and the mirrored half of each row of 16, then the four rows by lane reads.
template <bool MAX>
__device__ __forceinline__ float wave_reduce(float v)
{
    auto op = [](float a, float b) { return MAX ? fmaxf(a, b) : a + b; };
    v = op(v, dpp_lane<0xb1>(v));   // quad_perm [1,0,3,2]
    v = op(v, dpp_lane<0x4e>(v));   // quad_perm [2,3,0,1]
    v = op(v, dpp_lane<0x141>(v));  // row_half_mirror
    v = op(v, dpp_lane<0x140>(v));  // row_mirror
    const int vi = __builtin_bit_cast(int, v);
    const float r0 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(vi, 0));
    const float r1 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(vi, 16));
    const float r2 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(vi, 32));
    const float r3 = __builtin_bit_cast(float, __builtin_amdgcn_readlane(vi, 48));
    return op(op(r0, r1), op(r2, r3));
}

__device__ __forceinline__ float wave_sum(float v) { return wave_reduce<false>(v); }
__device__ __forceinline__ float wave_max(float v) { return wave_reduce<true>(v); }

// Sum (or max) over the 256 threads of a workgroup; `red` holds 4 floats.
template <bool MAX>
__device__ __forceinline__ float block_reduce(float v, float *red)
{
    v = MAX ? wave_max(v) : wave_sum(v);
    __syncthreads();  // `red` may still be read from a previous reduction
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
    __syncthreads();
    const float a = red[0], b = red[1], c = red[2], d = red[3];
    return MAX ? fmaxf(fmaxf(a, b), fmaxf(c, d)) : (a + b) + (c + d);
}

__device__ __forceinline__ void unpack8(const u32x4 &v, float f[8])
{
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        f[2 * i] = __half2float(__ushort_as_half((unsigned short)(w[i] & 0xffffu)));
        f[2 * i + 1] = __half2float(__ushort_as_half((unsigned short)(w[i] >> 16)));
    }
}

__device__ __forceinline__ uint32_t pack2(float lo, float hi)
{
    return (uint32_t)__half_as_ushort(__float2half_rn(lo)) |
           ((uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16);
}

// y[r] = fp16(fp16(x[r] * rsqrt(mean(x[r]^2) + eps)) * w); workgroups beyond
// `rows` only help clearing `clear_units` 16-byte units at `clear`.
__global__ void __launch_bounds__(kThreads)
rmsnorm_kernel(const __half *__restrict__ x, const __half *__restrict__ w, __half *__restrict__ y, int rows,
               int hidden, float eps, u32x4 *__restrict__ clear, long clear_units)
{
    __shared__ float red[4];
    const int tid = threadIdx.x;
    for (long u = (long)blockIdx.x * kThreads + tid; u < clear_units; u += (long)gridDim.x * kThreads)
        clear[u] = (u32x4){0u, 0u, 0u, 0u};
    const int r = blockIdx.x;
    if (r >= rows) return;
    const u32x4 *xr = (const u32x4 *)(x + (size_t)r * hidden);
    const u32x4 *wr = (const u32x4 *)w;
    u32x4 *yr = (u32x4 *)(y + (size_t)r * hidden);
    const int chunks = hidden / 8;
    // the first kHeld chunks of a thread stay in registers, with the matching weights,
    // so that rows up to 8192 wide cost one memory round trip
    constexpr int kHeld = 4;
    u32x4 xv[kHeld], wv[kHeld];
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        const int c = min(tid + kThreads * u, chunks - 1);
        xv[u] = xr[c];
        wv[u] = wr[c];
    }
    float ss = 0.0f;
#pragma unroll
    for (int u = 0; u < kHeld; ++u) {
        if (tid + kThreads * u < chunks) {
            float f[8];
            unpack8(xv[u], f);
#pragma unroll
            for (int i = 0; i < 8; ++i) ss = fmaf(f[i], f[i], ss);
        }
    }
    for (int c = tid + kThreads * kHeld; c < chunks; c += kThreads) {
        float f[8];
        unpack8(xr[c], f);
#pragma unroll
        for (int i = 0; i < 8; ++i) ss = fmaf(f[i], f[i], ss);
    }
    ss = block_reduce<false>(ss, red);
    const float scale = rsqrtf(ss / (float)hidden + eps);
    auto finish = [&](const u32x4 &xc, const u32x4 &wc) {
        float f[8], g[8];
        unpack8(xc, f);
        unpack8(wc, g);
        u32x4 o;
        uint32_t *ow = (uint32_t *)&o;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float a = __half2float(__float2half_rn(f[2 * i] * scale)) * g[2 * i];
            const float b = __half2float(__float2half_rn(f[2 * i + 1] * scale)) * g[2 * i + 1];
            ow[i] = pack2(a, b);
        }
        return o;
    };
#pragma unroll
    for (int u = 0; u < kHeld; ++u)
        if (tid + kThreads * u < chunks) yr[tid + kThreads * u] = finish(xv[u], wv[u]);
    for (int c = tid + kThreads * kHeld; c < chunks; c += kThreads) yr[c] = finish(xr[c], wr[c]);
}

// One workgroup per (sequence b, query head h).  Rotates q and the new k by the
// angle of position *pos, appends k and v to the cache (one writer per kv head),
// and attends over cache positions 0..pos, the newest one taken from LDS.
//   q [B][H*hd], k,v [B][KV*hd], cos,sin [max_pos][hd], caches [B][KV][max_pos][hd],
//   out [B][H*hd].  Dynamic LDS: (3*hd + max_pos + 4 + (256/hd)*hd) floats.
__global__ void __launch_bounds__(kThreads)
attention_kernel(const __half *__restrict__ q, const __half *__restrict__ k, const __half *__restrict__ v,
                 const __half *__restrict__ cos_t, const __half *__restrict__ sin_t, __half *__restrict__ k_cache,
                 __half *__restrict__ v_cache, const long long *__restrict__ pos_ptr, __half *__restrict__ out,
                 int H, int KV, int hd, int max_pos)
{
    extern __shared__ float lds[];
    float *q_s = lds;
    float *k_s = q_s + hd;
    float *v_s = k_s + hd;
    float *score = v_s + hd;
    float *red = score + max_pos;
    float *part = red + 4;

    const int tid = threadIdx.x;
    const int b = blockIdx.x / H, h = blockIdx.x % H;
    const int rep = H / KV, kvh = h / rep;
    int pos = (int)*pos_ptr;
    pos = min(max(pos, 0), max_pos - 1);
    const int half_d = hd / 2;
    const size_t cache_row0 = ((size_t)b * KV + kvh) * max_pos;

    for (int i = tid; i < hd; i += kThreads) {
        const float c = __half2float(cos_t[(size_t)pos * hd + i]);
        const float s = __half2float(sin_t[(size_t)pos * hd + i]);
        const __half *qh = q + ((size_t)b * H + h) * hd;
        const __half *kh = k + ((size_t)b * KV + kvh) * hd;
        const int j = i < half_d ? i + half_d : i - half_d;
        const float sign = i < half_d ? -1.0f : 1.0f;
        const __half qr = __float2half_rn(__half2float(qh[i]) * c + sign * __half2float(qh[j]) * s);
        const __half kr = __float2half_rn(__half2float(kh[i]) * c + sign * __half2float(kh[j]) * s);
        const __half vv = v[((size_t)b * KV + kvh) * hd + i];
        q_s[i] = __half2float(qr);
        k_s[i] = __half2float(kr);
        v_s[i] = __half2float(vv);
        if (h % rep == 0) {
            k_cache[(cache_row0 + pos) * hd + i] = kr;
            v_cache[(cache_row0 + pos) * hd + i] = vv;
        }
    }
    __syncthreads();

    const float scale = rsqrtf((float)hd);
    float local_max = -INFINITY;
    for (int j = tid; j <= pos; j += kThreads) {
        float dot = 0.0f;
        if (j == pos) {
            for (int i = 0; i < hd; ++i) dot = fmaf(q_s[i], k_s[i], dot);
        } else {
            const u32x4 *row = (const u32x4 *)(k_cache + (cache_row0 + j) * hd);
            for (int c = 0; c < hd / 8; ++c) {
                float f[8];
                unpack8(row[c], f);
#pragma unroll
                for (int i = 0; i < 8; ++i) dot = fmaf(q_s[8 * c + i], f[i], dot);
            }
        }
        dot *= scale;
        score[j] = dot;
        local_max = fmaxf(local_max, dot);
    }
    const float mx = block_reduce<true>(local_max, red);
    float local_sum = 0.0f;
    for (int j = tid; j <= pos; j += kThreads) {
        const float e = __expf(score[j] - mx);
        score[j] = e;
        local_sum += e;
    }
    const float inv = 1.0f / block_reduce<false>(local_sum, red);  // its barriers also publish score[]

    const int groups = kThreads / hd;  // >= 1 (hd <= 256)
    const int grp = tid / hd, d = tid % hd;
    if (grp < groups) {
        float acc = 0.0f;
        for (int j = grp; j <= pos; j += groups) {
            const float val = (j == pos) ? v_s[d] : __half2float(v_cache[(cache_row0 + j) * hd + d]);
            acc = fmaf(score[j], val, acc);
        }
        part[grp * hd + d] = acc;
    }
    __syncthreads();
    if (tid < hd) {
        float acc = 0.0f;
        for (int g = 0; g < groups; ++g) acc += part[g * hd + tid];
        out[((size_t)b * H + h) * hd + tid] = __float2half_rn(acc * inv);
    }
}

// The query heads of a kv head and how workgroups are given to them: 1 << spread (sequence, kv head) pairs, of `pairs`, side by side.
struct HeadLayout {
    int rep, KV, spread, pairs;
    uint32_t rep_reciprocal, KV_reciprocal;
};

// The same for head_dim HD in {64, 128}.  Bound by the stream of cached keys and values, and with a short
// context by the memory round trips in front of it.
//
// Thread (jg, ch) holds 16-byte chunk ch of key and value rows jg, jg + kPosGroups, ...: a wave's load
// covers whole rows.  A block of kRows rows per thread is in registers at a time; the next block's keys
// are requested as soon as the scores of this one are formed, its values once this one's are folded in, so that
// requests are in flight throughout.  Rows at and beyond *pos read as zero (the buffer descriptor ends
// there) and weigh nothing.  Every thread rotates the query chunk it multiplies itself: nothing goes through
// LDS, and no barrier stands, before the merge.  Each row of lanes keeps its own running maximum, sum of
// exponentials and weighted value sum (the "online" form of softmax); the rows of a wave are merged by lane
// exchanges, the waves through LDS.
//
// Heads of one kv head sit on one XCD, behind one L2, where place_pairs finds that no CU gets more to do for it: eight (sequence,
// kv head) pairs lie side by side, one to an XCD, and workgroups beyond the last pair leave at once.
// ONCE: cached rows are read non-temporally (read_once says for which steps, and what it gives).  A launch for eight sequences at
// position 700 19.4 -> 17.3 us.  (Heads that share rows have to sit behind one L2 for it: 14 sequences of 40 heads on 10 kv heads at
// position 1887 spread over the XCDs, a step of three blocks 524 -> 564 us.)
//
// Eight sequences of 32 heads at position 700 (92 MB): 23.1 -> 20.0 us, of which 3.3 are what position 0 takes;
// one sequence at position 255: 7.1 -> 6.4.  Before, whole blocks were fetched and then worked on, and the rotated
// query went through LDS and a barrier.
// The start is a chain of round trips: the arguments (asked for at once), the position, the first rows.  Off it since: the
// software divisions that found a workgroup's head, and, in wave 0, the new position's rows being asked for behind the
// earlier ones' (eight sequences at position 700 20.3 -> 19.4 us on the device, a token for one sequence 1402 -> 1394).
template <int HD, int T, bool ONCE>
__global__ void __launch_bounds__(T) __attribute__((amdgpu_waves_per_eu(4, 4)))
attention_hd_kernel(const __half *__restrict__ q, const __half *__restrict__ k, const __half *__restrict__ v,
                    const __half *__restrict__ cos_t, const __half *__restrict__ sin_t,
                    __half *__restrict__ k_cache, __half *__restrict__ v_cache,
                    const long long *__restrict__ pos_ptr, __half *__restrict__ out, const HeadLayout layout, int max_pos)
{
    constexpr int kChunks = HD / 8;             // 16-byte chunks of a row
    constexpr int kPosGroups = T / kChunks;     // rows that the workgroup's threads cover side by side
    constexpr int kRows = 8;
    constexpr int kBlock = kRows * kPosGroups;  // positions
    constexpr int kWaves = T / 64;
    constexpr int kNonTemporal = 2;   // (of a buffer load's cache policy)
    __shared__ float part[kWaves][HD], wave_mx[kWaves], wave_total[kWaves];

    const int tid = threadIdx.x;
    const int rep = layout.rep, KV = layout.KV, H = KV * rep;
    int pos = (int)*pos_ptr;
    asm volatile("" :: "s"(layout.spread), "s"(q), "s"(cos_t), "s"(out));   // (all of the arguments' cache lines at once)
    const int at = blockIdx.x >> layout.spread;
    int group = lutgemm::quotient(at, rep, layout.rep_reciprocal);      // (sequence, kv head) and the query head within it
    const int member = at - group * rep;
    group = (group << layout.spread) + (blockIdx.x & ((1 << layout.spread) - 1));
    if (group >= layout.pairs) return;
    const int b = lutgemm::quotient(group, KV, layout.KV_reciprocal), kvh = group - b * KV, h = kvh * rep + member;
    const int jg = tid / kChunks, ch = tid % kChunks;
    const int other = ch < kChunks / 2 ? ch + kChunks / 2 : ch - kChunks / 2;   // the chunk ch is rotated with
    const u32x4 *qh = (const u32x4 *)(q + ((size_t)b * H + h) * HD);
    const u32x4 *kh = (const u32x4 *)(k + ((size_t)b * KV + kvh) * HD);
    const u32x4 *vh = (const u32x4 *)(v + ((size_t)b * KV + kvh) * HD);
    const u32x4 q_own = qh[ch], q_other = qh[other];
    // (the new position's rows, ahead of the earlier ones': wave 0 needs them first)
    u32x4 k_own = {}, k_other = {}, v_own = {};
    if (jg == 0) {
        k_own = kh[ch];
        k_other = kh[other];
        v_own = vh[ch];
    }
    pos = min(max(pos, 0), max_pos - 1);
    const size_t cache_row0 = ((size_t)b * KV + kvh) * max_pos;
    const u32x4 cos_c = ((const u32x4 *)(cos_t + (size_t)pos * HD))[ch], sin_c = ((const u32x4 *)(sin_t + (size_t)pos * HD))[ch];

    const int live = pos * HD * 2;   // bytes of the earlier positions' rows
    auto krsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(k_cache + cache_row0 * HD), 0, live, 0x00027000);
    auto vrsrc = __builtin_amdgcn_make_buffer_rsrc((void *)(v_cache + cache_row0 * HD), 0, live, 0x00027000);
    u32x4 krow[kRows], vrow[kRows];
    auto fetch = [&](auto rsrc, u32x4 (&row)[kRows], int j0) {
#pragma unroll
        for (int u = 0; u < kRows; ++u)
            row[u] = __builtin_amdgcn_raw_buffer_load_b128(rsrc, tid * 16 + (j0 + u * kPosGroups) * (HD * 2), 0, ONCE ? kNonTemporal : 0);   // (scalar offsets escape the range check)
    };
    fetch(krsrc, krow, 0);
    fetch(vrsrc, vrow, 0);

    auto rotate = [&](const u32x4 &own, const u32x4 &partner, float (&r)[8]) {
        const float sign = ch < kChunks / 2 ? -1.0f : 1.0f;
        float x[8], y[8], c[8], s[8];
        unpack8(own, x);
        unpack8(partner, y);
        unpack8(cos_c, c);
        unpack8(sin_c, s);
#pragma unroll
        for (int i = 0; i < 8; ++i) r[i] = __half2float(__float2half_rn(x[i] * c[i] + sign * y[i] * s[i]));
    };
    auto row_sum = [](float x) {   // over a row's kChunks lanes
        x += dpp_lane<0xb1>(x);   // quad_perm [1,0,3,2]
        x += dpp_lane<0x4e>(x);   // quad_perm [2,3,0,1]
        x += dpp_lane<0x141>(x);  // row_half_mirror: the other quad of the 8
        if (kChunks == 16) x += dpp_lane<0x140>(x);  // row_mirror: the other half of the 16
        return x;
    };
    const float scale = rsqrtf((float)HD);
    float qc[8];
    rotate(q_own, q_other, qc);
    // running state of this thread's rows: maximum score, sum of exp(score - maximum), and the same
    // weights applied to the value chunks
    float run_max = -INFINITY, run_sum = 0.0f, acc[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = 0.0f;
    if (jg == 0) {
        // the new position: one row of lanes takes it, and one head of the kv head's appends it
        float kr[8], vv[8];
        rotate(k_own, k_other, kr);
        unpack8(v_own, vv);
        float dot = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            dot = fmaf(qc[i], kr[i], dot);
            acc[i] = vv[i];
        }
        run_max = row_sum(dot) * scale;
        run_sum = 1.0f;
        if (member == 0) {
            const u32x4 packed = {pack2(kr[0], kr[1]), pack2(kr[2], kr[3]), pack2(kr[4], kr[5]), pack2(kr[6], kr[7])};
            ((u32x4 *)(k_cache + (cache_row0 + pos) * HD))[ch] = packed;
            ((u32x4 *)(v_cache + (cache_row0 + pos) * HD))[ch] = v_own;
        }
    }
    for (int j0 = 0; j0 < pos; j0 += kBlock) {
        float sc[kRows], most = run_max;
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            float f[8];
            unpack8(krow[u], f);
            float dot = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; ++i) dot = fmaf(qc[i], f[i], dot);
            dot = row_sum(dot) * scale;
            sc[u] = j0 + jg + u * kPosGroups < pos ? dot : -INFINITY;
            most = fmaxf(most, sc[u]);
        }
        __builtin_amdgcn_sched_barrier(0);
        fetch(krsrc, krow, j0 + kBlock);
        __builtin_amdgcn_sched_barrier(0);
        // (no score so far, masked ones only: exponentials against 0 are zeros, against the maximum NaN)
        const float base = most == -INFINITY ? 0.0f : most;
        const float keep = __expf(run_max - base);
        run_sum *= keep;
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] *= keep;
#pragma unroll
        for (int u = 0; u < kRows; ++u) {
            const float pj = __expf(sc[u] - base);  // 0 for a masked row
            run_sum += pj;
            float f[8];
            unpack8(vrow[u], f);
#pragma unroll
            for (int i = 0; i < 8; ++i) acc[i] = fmaf(pj, f[i], acc[i]);
        }
        run_max = most;
        __builtin_amdgcn_sched_barrier(0);
        fetch(vrsrc, vrow, j0 + kBlock);
        __builtin_amdgcn_sched_barrier(0);
    }

    // ---- the rows of a wave, then the waves ------------------------------------------------------------
    auto over_rows = [](float x, auto op) {
        if (kChunks == 8) x = op(x, dpp_lane<0x128>(x));   // row_ror:8
        x = op(x, __shfl_xor(x, 16));
        return op(x, __shfl_xor(x, 32));
    };
    auto larger = [](float x, float y) { return fmaxf(x, y); };
    auto sum_of = [](float x, float y) { return x + y; };
    const int wave = tid >> 6, lane = tid & 63;
    const float wmx = over_rows(run_max, larger);
    const float weight = wmx == -INFINITY ? 0.0f : __expf(run_max - wmx);
    const float wsum = over_rows(run_sum * weight, sum_of);
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[i] = over_rows(acc[i] * weight, sum_of);
    if (lane < kChunks) {
#pragma unroll
        for (int i = 0; i < 8; ++i) part[wave][8 * ch + i] = acc[i];
        wave_mx[wave] = wmx;
        wave_total[wave] = wsum;
    }
    __syncthreads();
    if (tid < HD) {
        // (wave 0 holds the new position: the overall maximum is no -inf unless its score is)
        float mx = -INFINITY;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) mx = fmaxf(mx, wave_mx[w]);
        float sum = 0.0f, total = 0.0f;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const float e = __expf(wave_mx[w] - mx);  // 0 for a wave without rows
            total = fmaf(wave_total[w], e, total);
            sum = fmaf(part[w][tid], e, sum);
        }
        out[((size_t)b * H + h) * HD + tid] = __float2half_rn(sum / total);
    }
}

// out = fp16(fp16(silu(gate)) * up), 8 values per thread
__global__ void __launch_bounds__(kThreads)
silu_mul_kernel(const u32x4 *__restrict__ gate, const u32x4 *__restrict__ up, u32x4 *__restrict__ out, long units)
{
    const long u = (long)blockIdx.x * kThreads + threadIdx.x;
    if (u >= units) return;
    float g[8], p[8];
    unpack8(gate[u], g);
    unpack8(up[u], p);
    u32x4 o;
    uint32_t *ow = (uint32_t *)&o;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float a = __half2float(__float2half_rn(g[2 * i] / (1.0f + __expf(-g[2 * i])))) * p[2 * i];
        const float c = __half2float(__float2half_rn(g[2 * i + 1] / (1.0f + __expf(-g[2 * i + 1])))) * p[2 * i + 1];
        ow[i] = pack2(a, c);
    }
    out[u] = o;
}

// Whether the query heads of a (sequence, kv head) pair are placed on one XCD: where the fullest of its 32 CUs gets no more workgroups
// than with all spread evenly.  Rows that heads share then come from memory once and are found in one L2 (20 pairs at position 1000, 4 and 8
// query heads each, rows from memory 12.9 -> 11.4 and 18.3 -> 11.0 us, from the memory-side cache 11.6 -> 8.3 and 18.8 -> 8.5; 9 pairs of 12
// 11.7 -> 10.3 and 11.1 -> 8.2); an XCD with two workgroups to a CU beside others with one takes up to twice as long (position 1000, one
// pair of 64 8.2 -> 13.6, nine of 24 11.7 -> 14.8, nine of 48 16.4 -> 21.5).  One or two pairs of 32, which fill an XCD each and have but its
// way to memory, lose as well (8.07 -> 8.33 and 8.15 -> 8.40); of 24 they are level.
bool place_pairs(int pairs, int rep)
{
    auto rounds = [](int workgroups) { return (workgroups + 31) / 32; };
    return rep > 1 && (pairs > 2 || rep <= 24) && rounds((pairs + 7) / 8 * rep) <= rounds((pairs * rep + 7) / 8);
}

// Whether a step's cached rows are read non-temporally: where no later launch finds them in a cache, and kept there they push out what
// is found.  That is a matter of all that a token reads against the 256 MB of the memory-side cache, not of one block's rows: where
// weights and rows in use together come to less than about 400 MB, some of the rows are still there at the next token, and read so they
// are not (8 heads of 128, 8 blocks, 109 MB besides the caches, one sequence at position 2000 283 -> 341 us, eight of 2 kv heads 331 -> 382;
// four blocks, 88 MB, four sequences 182 -> 212).  The weights alone decide, since the position is the device's: from 402 MB on
// (two blocks of 32 heads, 434 MB, two sequences at positions 60, 200, 1000, 2000 167.1 -> 167.1, 167.8 -> 167.1, 186 -> 182, 215 -> 202; below
// it the early positions lose: 16 heads, 306 MB, two sequences at positions 30, 300, 1000 284 -> 287, 295 -> 306, 346 -> 349).  Caches under
// 8 MB are not worth it.  Query heads that share rows, over long contexts, drift apart and miss rows that leave L2 first: up to 64 MB
// (32 heads on 8 kv heads, 2048 positions: eight sequences, four blocks at positions 400 and 2000 297 -> 286 and 358 -> 347, sixteen
// sequences, eight blocks at position 2000 832 -> 882).
bool read_once(long cache_bytes, int rep, size_t step_bytes)
{
    return step_bytes >= (size_t)384 << 20 && cache_bytes >= 8l << 20 && (rep == 1 || cache_bytes <= 64l << 20);
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15u) == 0; }

int launch_status()
{
    hipError_t e = hipGetLastError();
    return e == hipSuccess ? LUTGEMM_OK : lutgemm_internal_hip_fail((int)e);
}

}  // namespace

extern "C" {

int lutgemm_decode_rmsnorm_f16(const void *x, const void *weight, void *y, int rows, int hidden, float eps,
                               void *clear, size_t clear_bytes, void *stream)
{
    if (!x || !weight || !y || rows < 1 || hidden < 8 || hidden % 8 != 0 || !(eps >= 0.0f)) return LUTGEMM_EINVAL;
    if (clear_bytes % 16 != 0 || (clear_bytes > 0 && !clear)) return LUTGEMM_EINVAL;
    if (!aligned16(x) || !aligned16(weight) || !aligned16(y) || !aligned16(clear)) return LUTGEMM_EALIGN;
    const long units = (long)(clear_bytes / 16);
    long extra = (units + kThreads - 1) / kThreads - rows;
    if (extra < 0) extra = 0;
    if (extra > 256) extra = 256;
    hipLaunchKernelGGL(rmsnorm_kernel, dim3((unsigned)(rows + extra)), dim3(kThreads), 0, (hipStream_t)stream,
                       (const __half *)x, (const __half *)weight, (__half *)y, rows, hidden, eps, (u32x4 *)clear,
                       units);
    return launch_status();
}

int lutgemm_describe_attention_plan(int batch, int heads, int kv_heads, int head_dim, int max_positions, size_t step_bytes,
                                    lutgemm_attention_plan *plan)
{
    if (!plan || batch < 1 || heads < 1 || kv_heads < 1 || heads % kv_heads != 0) return LUTGEMM_EINVAL;
    if (head_dim < 8 || head_dim > kThreads || head_dim % 8 != 0) return LUTGEMM_EINVAL;
    if (max_positions < 1 || max_positions > 8192) return LUTGEMM_EINVAL;
    *plan = {head_dim != 64 && head_dim != 128, batch * heads, kThreads, 0, 0};
    if (plan->general) return LUTGEMM_OK;
    const int rep = heads / kv_heads, pairs = batch * kv_heads;
    const long cache_bytes = (long)pairs * max_positions * head_dim * 4;
    plan->placed = place_pairs(pairs, rep);
    if (plan->placed) plan->workgroups = (pairs + 7) / 8 * 8 * rep;
    // With fewer workgroups than CUs eight waves each instead of four: 32 heads at position 255 6.4 us against
    // 6.7; 256 workgroups at position 700 20.4 against 20.0, where the memory is what they wait for.
    plan->threads = (long)batch * heads < 256 ? 512 : 256;
    plan->once = read_once(cache_bytes, rep, step_bytes);
    return LUTGEMM_OK;
}

int lutgemm_decode_attention_step_f16(const void *q, const void *k, const void *v, const void *cos_table,
                                      const void *sin_table, void *k_cache, void *v_cache, const int64_t *position,
                                      void *out, int batch, int heads, int kv_heads, int head_dim, int max_positions,
                                      size_t step_bytes, void *stream)
{
    if (!q || !k || !v || !cos_table || !sin_table || !k_cache || !v_cache || !position || !out)
        return LUTGEMM_EINVAL;
    lutgemm_attention_plan plan;
    const int rc = lutgemm_describe_attention_plan(batch, heads, kv_heads, head_dim, max_positions, step_bytes, &plan);
    if (rc != LUTGEMM_OK) return rc;
    if (!aligned16(k_cache) || !aligned16(v_cache)) return LUTGEMM_EALIGN;
    // (16-byte loads of every operand: others go to the general kernel)
    if (!plan.general && aligned16(q) && aligned16(k) && aligned16(v) && aligned16(cos_table) && aligned16(sin_table)) {
        const int rep = heads / kv_heads;
        const HeadLayout layout{rep, kv_heads, plan.placed ? 3 : 0, batch * kv_heads, lutgemm::reciprocal_of(rep),
                                lutgemm::reciprocal_of(kv_heads)};
        auto launch = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3((unsigned)plan.workgroups), dim3(plan.threads), 0, (hipStream_t)stream,
                               (const __half *)q, (const __half *)k, (const __half *)v, (const __half *)cos_table,
                               (const __half *)sin_table, (__half *)k_cache, (__half *)v_cache,
                               (const long long *)position, (__half *)out, layout, max_positions);
            return launch_status();
        };
        auto launch_as = [&](auto once_c) {
            constexpr bool ONCE = decltype(once_c)::value;
            const bool wide = plan.threads == 512;
            if (head_dim == 128) return wide ? launch(attention_hd_kernel<128, 512, ONCE>) : launch(attention_hd_kernel<128, 256, ONCE>);
            return wide ? launch(attention_hd_kernel<64, 512, ONCE>) : launch(attention_hd_kernel<64, 256, ONCE>);
        };
        return plan.once ? launch_as(std::true_type()) : launch_as(std::false_type());
    }
    const int groups = kThreads / head_dim;
    const size_t lds = sizeof(float) * ((size_t)3 * head_dim + max_positions + 4 + (size_t)groups * head_dim);
    hipLaunchKernelGGL(attention_kernel, dim3((unsigned)(batch * heads)), dim3(kThreads), lds, (hipStream_t)stream,
                       (const __half *)q, (const __half *)k, (const __half *)v, (const __half *)cos_table,
                       (const __half *)sin_table, (__half *)k_cache, (__half *)v_cache,
                       (const long long *)position, (__half *)out, heads, kv_heads, head_dim, max_positions);
    return launch_status();
}

int lutgemm_decode_attention_f16(const void *q, const void *k, const void *v, const void *cos_table,
                                 const void *sin_table, void *k_cache, void *v_cache, const int64_t *position,
                                 void *out, int batch, int heads, int kv_heads, int head_dim, int max_positions,
                                 void *stream)
{
    return lutgemm_decode_attention_step_f16(q, k, v, cos_table, sin_table, k_cache, v_cache, position, out, batch, heads, kv_heads,
                                             head_dim, max_positions, 0, stream);
}

int lutgemm_decode_silu_mul_f16(const void *gate, const void *up, void *out, size_t count, void *stream)
{
    if (!gate || !up || !out || count == 0 || count % 8 != 0) return LUTGEMM_EINVAL;
    if (!aligned16(gate) || !aligned16(up) || !aligned16(out)) return LUTGEMM_EALIGN;
    const long units = (long)(count / 8);
    hipLaunchKernelGGL(silu_mul_kernel, dim3((unsigned)((units + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                       (hipStream_t)stream, (const u32x4 *)gate, (const u32x4 *)up, (u32x4 *)out, units);
    return launch_status();
}

}  // extern "C"
