// Host side of liblutgemm_gfx950.so: operand validation, launch planning, the
// accumulator workspaces and the C ABI of include/lutgemm_gfx950.h.  The kernels live
// in lut_gemv_device.h (table look-ups) and lut_gemm_mfma_device.h (matrix cores).
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <stdlib.h>

#include <atomic>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "lutgemm_common.h"
#include "lutgemm_gfx950.h"
#include "lutgemm_internal.h"
#include "lutgemm_launch.h"

namespace lutgemm {
namespace {

constexpr int kMfmaWaves = 8;       // waves of a matrix-core workgroup: K-steps of a round
constexpr int kMfmaTileCols = 64;   // outputs per matrix-core workgroup
constexpr int kMfmaStepK = 128;
constexpr int kMaxDevices = 64;
constexpr int kTileMaxSlices = 16;
constexpr size_t kTileSumBytes = 64u << 20;   // GEMM kernel: sums of the K-slices of a launch, at most
constexpr size_t kTileGapBytes = kTileMaxSlices * tile_slice_stride(0, 0) * 4;   // what lies between them

thread_local int g_last_hip_error = 0;

// time-stamped build only: where the kernels leave their clock readings
std::atomic<unsigned long long *> g_stamps{nullptr};
std::atomic<long long> g_stamp_slots{0};

int hip_fail(hipError_t e)
{
    g_last_hip_error = (int)e;
    return LUTGEMM_EHIP;
}

// ---- accumulator words ------------------------------------------------------------
// K is split over workgroups; their partial sums meet in one 64-bit word per output
// (lutgemm_common.h).  Every launch leaves the words it used at zero, which is the
// state the next launch needs, so launches that are ordered on a stream can share
// one buffer.

// Fixed buffer of the entry point that may not allocate.  Zero when the code object is
// loaded; each GPU holds its own copy at its own address until the process ends.
static __device__ __align__(256) unsigned long long scratch[LUTGEMM_NOALLOC_MAX_WORDS];

std::mutex g_scratch_mutex;
unsigned long long *g_scratch_ptr[kMaxDevices] = {};

// Address of `scratch` on the current device, resolved once per device (in host code
// the array's name is a stand-in, not a device address).
int scratch_address(unsigned long long **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    if (dev < 0 || dev >= kMaxDevices) return LUTGEMM_EUNSUP;
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[dev]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return hip_fail(e);
        g_scratch_ptr[dev] = (unsigned long long *)ptr;
    }
    *out = g_scratch_ptr[dev];
    return LUTGEMM_OK;
}

struct Workspace {
    unsigned long long *accum = nullptr;
    size_t words = 0;
    std::vector<unsigned long long *> retired;  // outgrown buffers: captured graphs may still name them
    // second buffer: split activations (block-scaled kernel) or sums of K-slices (GEMM kernel) of the call in flight
    void *split = nullptr;
    size_t split_bytes = 0;
    std::vector<void *> retired_split;
};

std::mutex g_ws_mutex;
std::map<std::pair<int, hipStream_t>, Workspace> g_workspaces;

// Sizes of grown buffers are powers of two: calls of rising size cause few growths, and all outgrown buffers of a
// stream together are smaller than its largest.  (Beyond 2^48 no allocation succeeds, whatever its size.)
size_t grown(size_t wanted, size_t least)
{
    if (wanted > ((size_t)1 << 48)) return (size_t)1 << 48;
    while (least < wanted) least *= 2;
    return least;
}

// Device memory, or ENOMEM.  Callers go on without it (a smaller buffer, another kernel): the error that the runtime
// would report to their next check of a launch is taken back.
template <typename T>
int allocate(T **out, size_t bytes)
{
    const hipError_t e = hipMalloc((void **)out, bytes);
    if (e == hipSuccess) return LUTGEMM_OK;
    (void)hipGetLastError();
    g_last_hip_error = (int)e;
    return LUTGEMM_ENOMEM;
}

// Grow-only, zero-initialised accumulator words per (device, stream).  Growing
// synchronises the stream and allocates, which a stream under capture cannot do: that
// case is refused before anything is touched (reserve the words beforehand).  Without
// memory for it the buffer stays as it is.  An outgrown buffer is kept (zero, unused by
// new launches) until lutgemm_release_workspaces(): a graph captured earlier still points at it.
int stream_workspace(hipStream_t stream, size_t words, unsigned long long **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    Workspace &ws = g_workspaces[std::make_pair(dev, stream)];
    if (ws.words < words) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        e = hipStreamIsCapturing(stream, &cap);
        if (e != hipSuccess) return hip_fail(e);
        if (cap != hipStreamCaptureStatusNone) return LUTGEMM_ECAPTURE;
        const size_t want = grown(words, 1u << 18);
        unsigned long long *grown_words = nullptr;
        const int rc = allocate(&grown_words, want * sizeof(unsigned long long));
        if (rc != LUTGEMM_OK) return rc;
        e = hipStreamSynchronize(stream);  // queued work may still use the old buffer
        if (e == hipSuccess) e = hipMemsetAsync(grown_words, 0, want * sizeof(unsigned long long), stream);
        if (e == hipSuccess) e = hipStreamSynchronize(stream);
        if (e != hipSuccess) {
            (void)hipFree(grown_words);
            return hip_fail(e);
        }
        if (ws.accum) ws.retired.push_back(ws.accum);
        ws.accum = grown_words;
        ws.words = want;
    }
    *out = ws.accum;
    return LUTGEMM_OK;
}

// The same for the split activations of the block-scaled path and the sums of the GEMM kernel's K-slices (not
// zeroed: every call writes what it reads).  Calls on one stream are ordered, so they can share the buffer.
int stream_split_buffer(hipStream_t stream, size_t bytes, void **out)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    Workspace &ws = g_workspaces[std::make_pair(dev, stream)];
    if (ws.split_bytes < bytes) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        e = hipStreamIsCapturing(stream, &cap);
        if (e != hipSuccess) return hip_fail(e);
        if (cap != hipStreamCaptureStatusNone) return LUTGEMM_ECAPTURE;
        // (the gaps between slices on top of a power of two: sums that fill one would otherwise take the next)
        const size_t want = grown(bytes > kTileGapBytes ? bytes - kTileGapBytes : bytes, 1u << 20) + kTileGapBytes;
        void *grown_split = nullptr;
        const int rc = allocate(&grown_split, want);
        if (rc != LUTGEMM_OK) return rc;
        e = hipStreamSynchronize(stream);
        if (e != hipSuccess) {
            (void)hipFree(grown_split);
            return hip_fail(e);
        }
        if (ws.split) ws.retired_split.push_back(ws.split);
        ws.split = grown_split;
        ws.split_bytes = want;
    }
    *out = ws.split;
    return LUTGEMM_OK;
}

// Calls that take two launches with the second buffer between them hold this lock over both: a call of another
// host thread on the same stream would otherwise put its own first launch in between.
std::mutex g_two_launches_mutex;

// Where a call takes its accumulator words from.
struct Accum {
    hipStream_t stream;
    bool fixed = false;  // the fixed device array instead of the stream's workspace
};

int accum_words(const Accum &a, size_t words, unsigned long long **out)
{
    if (!a.fixed) return stream_workspace(a.stream, words, out);
    if (words > (size_t)LUTGEMM_NOALLOC_MAX_WORDS) return LUTGEMM_ETOOBIG;
    return scratch_address(out);
}

int env_int(const char *name, int fallback)
{
    const char *v = getenv(name);
    return (v && *v) ? atoi(v) : fallback;
}

// Tuning options (lutgemm_set_option): each starts from its environment variable, read once.
struct Option {
    const char *env;
    int fallback;
};
constexpr Option kOptions[LUTGEMM_OPTION_COUNT] = {
    {"LUTGEMM_TARGET_BLOCKS", 0}, {"LUTGEMM_FIRST_SHARE", 60}, {"LUTGEMM_MFMA_MIN_M", 3},
    {"LUTGEMM_MFMA_BLOCKS", 0},   {"LUTGEMM_PAIR_TABLES", 1},  {"LUTGEMM_SINGLE_ITEM", 1},
    {"LUTGEMM_CHAIN_BLOCKS", 0}, {"LUTGEMM_CHAIN_GRID", 0},  {"LUTGEMM_TWIN_ITEMS", 4},
    {"LUTGEMM_BLOCK_SCALED", 1}, {"LUTGEMM_POW2_CONVERT", 1},
    {"LUTGEMM_TILE_MIN_M", 0},
};
std::atomic<int> g_option[LUTGEMM_OPTION_COUNT];
std::once_flag g_option_once;

void load_options()
{
    std::call_once(g_option_once, [] {
        for (int i = 0; i < LUTGEMM_OPTION_COUNT; ++i) g_option[i].store(env_int(kOptions[i].env, kOptions[i].fallback));
    });
}

// LUTGEMM_OPTION_TARGET_BLOCKS = workgroups a look-up launch aims
// for.  74 KiB of LDS per workgroup lets two be resident per CU, and a launch above
// what is resident at once runs a second, mostly empty round that costs as much as
// the first.
// Short streams do better with ONE workgroup per CU and more items each: a workgroup's
// second and third item cost less than the start and the hand-over of another workgroup.
// Measured, one row, 256 vs 512 workgroups: 11008x4096x3 8.78 vs 9.04 us, 4096x11008x3 8.59
// vs 9.12, 13824x5120x2 8.92 vs 9.64, 8192x8192x2 8.27 vs 8.49; 8192x8192x4 11.74 vs 11.06,
// 28672x8192x2 18.75 vs 16.62.
// The block-alpha formats pay more per item (their alphas are staged per item), so a long
// range hurts them sooner: beyond four items per workgroup they take two workgroups per CU
// (13824x5120x2 in eight row groups 9.16 vs 8.58 us, 5120x13824x2 10.0 vs 8.54; 5120x5120x2,
// 1.6 items per workgroup, 5.91 vs 6.37).
int target_blocks(long sign_bytes, long items = 0, bool block_alpha = false)
{
    const int v = option(LUTGEMM_OPTION_TARGET_BLOCKS);
    if (v > 0) return v;
    if (block_alpha && items > 4 * 256) return 512;
    return sign_bytes <= (24l << 20) ? 256 : 512;  // 1 or 2 workgroups x 256 CUs
}

// Of the two workgroups that share a CU the one dispatched first runs faster (the older
// waves win the arbitration for issue slots and memory requests): with equal ranges the
// first half of a 512-workgroup grid ends 6-7 us before the second on the 132 MB shapes.
// So the first 256 workgroups get this share (per cent) of each pair's items.  Measured,
// equal ranges vs 60 %: 28672x8192x2 17.3 vs 16.3 us, 8192x28672x2 17.1 vs 15.8, 8192x28672x4
// 27.7 vs 27.0, 13824x5120x4 14.8 vs 13.1 (there mostly because 412 workgroups of 3 and 2
// items fill the CUs better than 360 of 3), 8192x8192x4 unchanged.
int first_share()
{
    return option(LUTGEMM_OPTION_FIRST_SHARE);
}

// Cut the (tile, set) items of a problem into contiguous ranges, one per workgroup,
// aiming at `want_blocks` workgroups.
// `twin`: the items are twin items, one set of inputs against a PAIR of output tiles (one table
// build for 512 outputs); n_tiles counts pairs then.
int plan_lookup(Problem &p, int mrows, long want_blocks, bool twin = false)
{
    p.n_tiles = (p.N + kTileCols - 1) / kTileCols;
    if (twin) p.n_tiles = (p.n_tiles + 1) / 2;
    p.twin = twin ? 1 : 0;
    p.mchunks = (p.M + mrows - 1) / mrows;
    const long total = (long)p.n_tiles * p.nsets;
    long wgs = want_blocks / p.mchunks;
    if (wgs < 1) wgs = 1;
    long ipw = (total + wgs - 1) / wgs;
    // an accumulator word takes at most kMaxContrib contributions: a tile of nsets items
    // overlaps at most ceil(nsets / ipw) + 1 ranges
    const long cap = (p.nsets + kMaxContrib - 2) / (kMaxContrib - 1);
    if (ipw < cap) ipw = cap;
    if (ipw > total) ipw = total;
    long n_long = (total + ipw - 1) / ipw, short_items = ipw, n_short = 0;
    // two resident workgroups per CU, one row chunk: unequal shares within each pair
    const int share = first_share();
    if (p.mchunks == 1 && want_blocks == 512 && total >= 2 * 256 * 2 && share > 50 && share < 100) {
        const long pair = (total + 255) / 256;
        long a = (pair * share + 99) / 100, b = pair - a;
        // (the smaller range may not fall below what the contribution count allows: give it
        // items of the larger one while the larger one stays the larger)
        while (b < cap && a - 1 > b + 1) {
            --a;
            ++b;
        }
        // (a split far beyond the share, 3 and 1 of 4, is worse than none: 8192x8192x4 11.4 us against 10.5)
        if (b >= 1 && b >= cap && a > b && 100 * a <= (share + 12) * pair) {
            ipw = a;
            n_long = 256;
            short_items = b;
            const long rest = total - n_long * a;
            n_short = rest > 0 ? (rest + b - 1) / b : 0;
            if (rest <= 0) n_long = (total + a - 1) / a;
        }
    }
    p.items_per_wg = (int)ipw;
    p.long_ranges = (int)n_long;
    p.short_items = (int)short_items;
    p.split_item = (int)(n_long * ipw);
    p.wgs_per_chunk = (int)(n_long + n_short);
    p.n_blocks = p.wgs_per_chunk * p.mchunks;
    p.by_items = make_divisor(p.items_per_wg);
    p.by_short_items = make_divisor(p.short_items);
    p.by_nsets = make_divisor(p.nsets);
    // the multiply-high divisions of the kernel are exact within this bound
    if (2ull * (unsigned long long)(total + p.nsets) * (unsigned long long)ipw >= (1ull << 32)) return LUTGEMM_EUNSUP;
    return LUTGEMM_OK;
}

// true when some tile is shared between ranges, i.e. accumulator words are needed
bool lookup_splits_k(const Problem &p)
{
    if (p.items_per_wg % p.nsets != 0) return true;
    return p.wgs_per_chunk > p.long_ranges && (p.short_items % p.nsets != 0 || p.split_item % p.nsets != 0);
}

int pick_mrows(int M) { return M >= 3 ? 4 : M; }

bool aligned(const void *ptr, size_t a) { return ((uintptr_t)ptr & (a - 1)) == 0; }

// Validate one problem and fill everything but the launch plan.
int fill_problem(Problem &p, int mode, const uint32_t *bW, const void *alpha, const void *qbias,
                 const void *x, void *out, int N, int K, int nb, int num_groups, int M)
{
    if (!bW || !alpha || !x || !out) return LUTGEMM_EINVAL;
    if (mode == kUniformF16 && !qbias) return LUTGEMM_EINVAL;
    if (N <= 0 || K <= 0 || M <= 0 || num_groups <= 0) return LUTGEMM_EINVAL;
    if (K % 32 != 0 || N % 4 != 0) return LUTGEMM_EINVAL;
    if (nb < 1 || nb > 4) return LUTGEMM_EINVAL;
    if (M > 65535) return LUTGEMM_EINVAL;
    if (!aligned(bW, 16) || !aligned(x, 16) || !aligned(out, 8)) return LUTGEMM_EALIGN;

    p = Problem{};
    p.W = bW;
    p.alpha = alpha;
    if (mode == kUniformF16) p.qbias = (const __half *)qbias;
    p.x = (const __half *)x;
    p.out = (__half *)out;
    p.init = p.out;
    p.init_stride = N;
    p.N = N;
    p.K = K;
    p.M = M;
    p.nb = nb;
    p.alpha_mode = mode;
    p.kwords = K / 32;
    p.nsets = (p.kwords + kSetWords - 1) / kSetWords;
    p.group_words = 1;
    if (mode == kRowF16 || mode == kUniformF16) {
        if (K % num_groups != 0) return LUTGEMM_EINVAL;
        const int gs = K / num_groups;
        if (gs % 32 != 0) return LUTGEMM_EINVAL;  // a sign word may not straddle two groups
        p.group_words = gs / 32;
        if (!aligned(alpha, 8)) return LUTGEMM_EALIGN;
        if (mode == kUniformF16 && !aligned(qbias, 8)) return LUTGEMM_EALIGN;
    } else {
        if (N % num_groups != 0) return LUTGEMM_EINVAL;
        p.R = num_groups;
        p.rows_per_group = N / num_groups;
        if (p.rows_per_group % 4 != 0) return LUTGEMM_EINVAL;
    }
    p.by_group_words = make_divisor(p.group_words);
#ifdef LUTGEMM_TIMESTAMPS
    p.stamps = g_stamps.load();
    p.stamp_slots = g_stamp_slots.load();
#endif
    // the multiply-high divisions of the kernels are exact within these bounds
    const unsigned long long tiles = (unsigned long long)(N + kTileCols - 1) / kTileCols;
    if (2ull * p.kwords * p.group_words >= (1ull << 32)) return LUTGEMM_EUNSUP;
    if (2ull * (tiles + 1) * p.nsets * p.nsets >= (1ull << 32)) return LUTGEMM_EUNSUP;
    return LUTGEMM_OK;
}

int mfma_min_rows()
{
    return option(LUTGEMM_OPTION_MFMA_MIN_M);
}

// The matrix-core path needs whole 128-input steps inside one alpha group and
// 16-output alpha runs.
bool mfma_eligible(const Problem &p, int mode)
{
    if (!(mode == kRowF16 && p.K % kMfmaStepK == 0 && p.group_words % 4 == 0 && p.N % 16 == 0 && p.N >= 16))
        return false;
    if ((unsigned long long)p.M * p.K * 2 >= (1ull << 32)) return false;   // (32-bit byte offsets)
    if (p.M >= mfma_min_rows()) return true;
    // two rows: the look-up kernel (one table set for both rows, fp16 entry pairs) wins on long sign streams.  The
    // line was drawn at 12 MB for an earlier matrix-core kernel; measured with this one (us, look-up / matrix
    // core, * = taken): 4096x4096x3 6.9 / 5.6*, 11008x4096x2 9.6 / 8.1*, 5120x5120x4 (12.5 MB) 8.7* / 8.1, 11008x4096x3
    // 10.6* / 9.5, 8192x8192x4 13.5* / 12.6, 28672x8192x4 30.8* / 33.2: it now lies between 32 and 112 MB.
    return p.M == 2 && mfma_min_rows() == 3 && (long)p.N * (p.K / 8) * p.nb <= (12l << 20);
}

// K-steps are split 8 ways inside a workgroup already; across workgroups `want` ways
// at most (whole rounds of eight steps per slice).
void plan_mfma(Problem &p, int mt, long want)
{
    p.n_tiles = (p.N + kMfmaTileCols - 1) / kMfmaTileCols;
    p.mchunks = (p.M + 16 * mt - 1) / (16 * mt);
    p.nsets = (p.K + kMfmaStepK - 1) / kMfmaStepK;  // K-steps
    if (want > (p.nsets + kMfmaWaves - 1) / kMfmaWaves) want = (p.nsets + kMfmaWaves - 1) / kMfmaWaves;
    if (want < 1) want = 1;
    if (want > kMaxSlices) want = kMaxSlices;
    p.sets_per_split = (p.nsets + (int)want - 1) / (int)want;
    p.sets_per_split = (p.sets_per_split + kMfmaWaves - 1) / kMfmaWaves * kMfmaWaves;  // whole rounds
    p.ksplit = (p.nsets + p.sets_per_split - 1) / p.sets_per_split;
    p.n_blocks = p.n_tiles * p.ksplit * p.mchunks;
    p.tiles_reciprocal = reciprocal_of(p.n_tiles);
    p.ksplit_reciprocal = reciprocal_of(p.ksplit);
}

// LUTGEMM_OPTION_MFMA_BLOCKS: workgroups a matrix-core launch aims for instead of the rules below.
int mfma_blocks_override()
{
    return option(LUTGEMM_OPTION_MFMA_BLOCKS);
}

// K-slices per tile for the problems of one launch (all get the same number, each up to
// its own limit).
//   32-row tile: as many as reach one workgroup per CU (its register count allows no second one).  Measured at 32 rows (us, slices -> time):
//   8192x28672x3: 1 -> 57.5, 2 -> 37.4, 4 -> 42.8; 8192x8192x4: 1 -> 24.1, 2 -> 19.7, 4 -> 24.0; int8 exponents 5120x13824x2: 1 -> 37.0,
//   3 -> 21.2, 4 -> 26.5; 11008x4096x3: 1 -> 13.6, 2 -> 22.1; 28672x8192x4, whose 448 tiles leave a second round a
//   quarter empty: 1 -> 48.3, 2 -> 63.8, 4 -> 71.4.
//   16-row tile: the launch ends when the busiest CU does, two workgroups share a CU.  With w =
//   ceil(workgroups / 256) workgroups on that CU and R rounds (one K-step per wave) per workgroup, the slice
//   count that minimises
//       w * R  +  0.18 * w  +  0.9 * max(0, w - 2)
//   is taken, the smaller one on ties: a workgroup's start and hand-over cost a fifth of a
//   round, and one that has to wait for a slot on its CU most of a round.  A lone workgroup
//   of four or more rounds hides its loads badly when there are many of them (more than
//   eight activation rows, or nine CUs in ten busy) and is charged 12 % more.  The constants were fitted to a
//   kernel that expanded every plane by itself; for this one they pick (us at 4 / 16 rows, slices -> time, * = taken):
//   8192x8192x4: 2 -> 12.9 / 15.4, 4* -> 12.9 / 14.6; 4096x4096x3: 2 -> 7.2 / 8.4, 4* -> 5.8 / 7.1; 5120x13824x3: 3* -> 12.3 /
//   15.3, 5 -> 14.0 / 18.9; 4096x11008x2: 3 -> 9.1 / 11.3, 4* -> 8.1 / 10.2; 28672x8192x2: 1* -> 22.8 / 27.0, 4 -> 25.4 / 30.0;
//   28672x8192x4: 1* -> 34.2 / 38.9, 4 -> 36.7 / 40.0; 22016x4096x3: 1 -> 15.6 / 18.4, 2* -> 14.7 / 17.1.  The one miss among
//   these is 11008x4096x3 at 16 rows: 1 -> 11.8, 2* -> 12.5, 4 -> 11.8 (4 rows: 1* -> 9.6).
int mfma_slices(const Group &g, int mt)
{
    constexpr long kCUs = 256;
    long tiles = 0;
    int max_rounds = 1, rows = 0;
    for (int i = 0; i < g.count; ++i) {
        const Problem &p = g.p[i];
        tiles += (long)((p.N + kMfmaTileCols - 1) / kMfmaTileCols) * ((p.M + 16 * mt - 1) / (16 * mt));
        const int rounds = ((p.K + kMfmaStepK - 1) / kMfmaStepK + kMfmaWaves - 1) / kMfmaWaves;
        if (rounds > max_rounds) max_rounds = rounds;
        if (p.M > rows) rows = p.M;
    }
    if (max_rounds > kMaxSlices) max_rounds = kMaxSlices;
    if (const int blocks = mfma_blocks_override()) return (int)(blocks / tiles > 1 ? blocks / tiles : 1);
    if (mt != 1) return (int)(kCUs / tiles > 1 ? kCUs / tiles : 1);
    int best = 1;
    double best_cost = 0.0;
    for (int ks = 1; ks <= max_rounds; ++ks) {
        long wgs = 0;
        int rounds = 0;
        for (int i = 0; i < g.count; ++i) {
            Problem q = g.p[i];
            plan_mfma(q, mt, ks);
            wgs += q.n_blocks;
            if (q.sets_per_split / kMfmaWaves > rounds) rounds = q.sets_per_split / kMfmaWaves;
        }
        const long w = (wgs + kCUs - 1) / kCUs;
        double cost = (double)w * rounds + 0.18 * (double)w + 0.9 * (double)(w > 2 ? w - 2 : 0);
        if (w == 1 && rounds >= 4 && (rows > 8 || wgs * 10 > kCUs * 9)) cost *= 1.12;
        if (ks == 1 || cost < best_cost * 0.999) {
            best = ks;
            best_cost = cost;
        }
    }
    return best;
}

// How a lone problem of more than 16 rows is cut up: the height of its tiles (mt 16-row tiles) and its K-slices, by
// the estimate in us
//     start + w * (rounds * (round + plane * nb) + wg), with several slices + cut + words * M * N * slices / 1e6,
// where w = ceil(workgroups / 256), rounds = K-steps per wave of a slice, fitted to 1100 launches timed in graphs (17 to
// 256 rows, 768 to 28672 inputs and outputs, 1 to 4 planes; 3 to 12 % rms).  32-row tiles form each weight once for twice the rows but
// pay more per round and, one workgroup per CU, wait for every accumulator word; small calls are better off with twice
// as many workgroups, large ones with few slices.  The choice is within 1 % of the best of all tried on
// average, the former one (16-row tiles only where 64 rows at most fit the chip as single rounds, slices up to a
// workgroup per CU for the rest) was 4 to 7 % off: us before / now 2048x2048x3 at 128 rows 10.5 / 7.3,
// 4096x4096x3 at 64 13.2 / 11.2, 1024x1024x3 at 256 6.3 / 5.0, int8 exponents 768x3072x3 at 96 9.4 / 7.8, 4096x4096x4 at 17 13.5 / 10.9,
// at 96 27.1 / 19.7, uniform 4096x4096x4 at 32 24.6 / 17.0, 8192x8192x4 at 64 29.3 / 27.0; of 177 calls the worst loses 4 %.
struct MfmaCost {
    double start, round, plane, wg, cut, words;
};
constexpr MfmaCost kMfmaCost[3][2] = {   // row-wise, uniform (q_bias makes every weight two pieces), block formats
    {{3.3, 0.70, 0.35, 0.00, 1.15, 3.0}, {2.05, 0.92, 0.39, 2.10, 1.6, 4.9}},
    {{4.6, 0.00, 1.71, 0.00, 0.85, 0.0}, {4.70, 0.43, 1.29, 1.43, 0.9, 6.5}},
    {{2.75, 0.30, 0.84, 0.00, 1.6, 3.1}, {1.60, 0.64, 0.88, 1.67, 2.05, 5.6}},
};

struct MfmaPlan {
    int mt, slices;
    double us;
    bool gemm;   // the GEMM kernel is the other choice: faster than 5 us + a round's worst time per round of the widest cut, or never_cut
    double gemm_us;   // gemm_estimate, where it was asked for
    bool one_launch;  // no memory here, slices there
};

MfmaPlan pick_mfma(const Problem &p, bool may_cut, bool must_cut)
{
    const MfmaCost *const cost = kMfmaCost[p.alpha_mode == kRowF16 ? 0 : p.alpha_mode == kUniformF16 ? 1 : 2];
    const int rounds = ((p.K + kMfmaStepK - 1) / kMfmaStepK + kMfmaWaves - 1) / kMfmaWaves;
    const int most = !may_cut ? 1 : rounds < kMaxSlices ? rounds : kMaxSlices;
    MfmaPlan best{};
    for (int mt = 1; mt <= 2; ++mt) {
        const MfmaCost &c = cost[mt - 1];
        const long tiles = (long)((p.N + kMfmaTileCols - 1) / kMfmaTileCols) * ((p.M + 16 * mt - 1) / (16 * mt));
        for (int ks = must_cut ? 2 : 1; ks <= most; ++ks) {
            const int own = (rounds + ks - 1) / ks;
            if ((rounds + own - 1) / own != ks) continue;
            const double us = c.start + (double)((tiles * ks + 255) / 256) * (own * (c.round + c.plane * p.nb) + c.wg) +
                              (ks > 1 ? c.cut + c.words * 1e-6 * ((double)p.M * p.N * ks) : 0.0);
            if (best.mt == 0 || us < best.us) best = MfmaPlan{mt, ks, us, false, 0.0, false};
        }
    }
    return best;
}

// Whether a call of more than 32 rows that a cut up to a workgroup per CU makes K-slices of takes none: callers that
// reserve nothing before a capture rely on which calls need accumulator words, so this line is fixed in the sizes and follows neither
// the costs above nor those of plan_tile.  It was drawn where the GEMM kernel, which needs none, was the faster choice:
// slices of four waves and steps of 1.2 us (128 rows) or 0.9 (64) alone on a CU, 2.1 or 1.6 beside another, against rounds of 3 us.
bool never_cut(const Problem &p)
{
    const int rows = p.M <= 64 ? 64 : 128;
    const long tiles = (long)((p.N + 255) / 256) * ((p.M + rows - 1) / rows), all = (p.kwords + 3) / 4 * 2;
    const double alone = rows == 128 ? 1.2 : 0.9, beside = rows == 128 ? 2.1 : 1.6;
    double best = 0.0;
    for (int ks = 1; ks <= kTileMaxSlices && (ks == 1 || 2 * ks <= all); ++ks) {
        const long steps = ((all + ks - 1) / ks + 1) & ~1l, wgs = tiles * ks, rounds = wgs / 512, rest = wgs - rounds * 512;
        const size_t sums = ks > 1 ? (size_t)ks * p.M * p.N * 4 : 0;
        if ((all + steps - 1) / steps != ks) continue;
        if (ks > 1 && (wgs > 512 || sums > kTileSumBytes)) break;
        double us = (double)rounds * (steps * beside + 5.0) + (sums ? 4.0 + 0.5e-6 * (double)sums : 0.0);
        if (rest > 0) us += steps * (rest > 256 ? beside : alone) + 5.0;
        if (ks == 1 || us < best * 0.99) best = us;
    }
    const double rounds = (double)((p.N + 63) / 64) * (double)((p.M + 31) / 32) * (double)((p.K + 1023) / 1024);
    return best < 5.0 + 3.0 * rounds / 256.0;
}

double gemm_estimate(const Problem &p, bool *sliced);

// The plan of a lone problem.  Which calls take accumulator words, and so need a reservation under capture: those that a
// cut up to a workgroup per CU makes K-slices of, beyond 32 rows less those of never_cut and less those that the GEMM kernel is
// expected to be faster for (a refit of the costs may only take calls out).  Up to 32 rows these calls keep their slices
// (uncut, the few that are faster gain under 8 %: 5120x2048x4 at 32 rows 8.1 / 8.7).
// `or_gemm`: the GEMM kernel may take the call instead; without it slices are all there is to spread a call with (4096x28672x4 at
// 64 rows, uncut 100.9 us, in two slices 65.9).
MfmaPlan mfma_plan(const Problem &p, bool or_gemm)
{
    Group one{};
    one.count = 1;
    one.p[0] = p;
    const long tiles = (p.N + kMfmaTileCols - 1) / kMfmaTileCols, rounds = ((p.K + kMfmaStepK - 1) / kMfmaStepK + kMfmaWaves - 1) / kMfmaWaves;
    const int mt = p.M <= 16 || (p.M <= 64 && tiles * ((p.M + 15) / 16) * rounds <= 512) ? 1 : 2;
    const int slices = mfma_slices(one, mt);
    plan_mfma(one.p[0], mt, slices);
    bool cut = one.p[0].ksplit > 1, gemm = false, one_launch = false;
    double gemm_us = 0.0;
    if (or_gemm && p.M > 32) {
        Problem wide = p;
        plan_mfma(wide, 2, mt == 2 ? slices : mfma_slices(one, 2));
        const double round = 1.6 + 0.32 * p.nb + (is_block(p.alpha_mode) ? 0.9 : 0.0);
        bool sliced = false;
        gemm_us = gemm_estimate(p, &sliced);
        gemm = gemm_us < 5.0 + round * (double)((wide.n_blocks + 255) / 256) * (double)(wide.sets_per_split / kMfmaWaves);
        if (cut && !gemm) gemm = never_cut(p);   // (uncut, the GEMM kernel is the other choice for these)
        one_launch = !cut && sliced;
        cut = cut && !gemm;
    }
    if (p.M <= 16 || mfma_blocks_override()) return MfmaPlan{mt, slices, 0.0, gemm, gemm_us, one_launch};
    MfmaPlan plan = pick_mfma(p, cut, cut && p.M <= 32);
    plan.gemm = gemm;
    plan.gemm_us = gemm_us;
    plan.one_launch = one_launch;
    return plan;
}

// (the grouped entry points' problems: the GEMM kernel is none of their kernels)
int run_mfma(Problem &p, const Accum &acc)
{
    const MfmaPlan plan = mfma_plan(p, false);
    const int mt = plan.mt;
    plan_mfma(p, mt, plan.slices);
    if (p.ksplit > 1) {
        int rc = accum_words(acc, (size_t)p.M * p.N, &p.accum);
        if (rc != LUTGEMM_OK) return rc;
    }
    const hipError_t e = launch_mfma(p, mt, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// Where the product of a gate and an up projection goes, and whether it went there.
struct Gated {
    __half *out;
    bool done;
};

// (returns whether some problem needs accumulator words)
bool plan_mfma_group(Group &g, int mt, int *most)
{
    const int slices = mfma_slices(g, mt);
    bool any_split = false;
    for (int i = 0; i < g.count; ++i) {
        Problem &p = g.p[i];
        plan_mfma(p, mt, slices);
        if (p.n_blocks > *most) *most = p.n_blocks;
        any_split = any_split || p.ksplit > 1;
    }
    return any_split;
}

// All problems of a group on the matrix-core kernel in one launch (they share the
// row-tile height: all M <= 16 or all M > 16).
int run_mfma_group(Group &g, const Accum &acc, Gated *gated)
{
    const int mt = g.p[0].M > 16 ? 2 : 1;
    size_t words = 0;
    for (int i = 0; i < g.count; ++i) words += (size_t)g.p[i].M * g.p[i].N;
    int begin = 0;   // grid.x: the largest problem's workgroups
    const bool any_split = plan_mfma_group(g, mt, &begin);
    // (behind the problems' words, where the launch forms a product, one 32-bit word per output)
    const size_t pair_words = gated ? ((size_t)g.p[0].M * g.p[0].N + 1) / 2 : 0;
    unsigned long long *base = nullptr;
    if (any_split || gated) {
        int rc = accum_words(acc, words + pair_words, &base);
        if (rc != LUTGEMM_OK && gated) {   // (no memory for them: the sums alone)
            gated = nullptr;
            rc = any_split ? accum_words(acc, words, &base) : LUTGEMM_OK;
        }
        if (rc != LUTGEMM_OK) return rc;
    }
    if (any_split) {
        size_t off = 0;
        for (int i = 0; i < g.count; ++i) {
            g.p[i].accum = base + off;
            off += (size_t)g.p[i].M * g.p[i].N;
        }
    }
    if (gated) {
        const GatedProblems pair{{g.p[0], g.p[1]}, {(uint32_t *)(base + words), gated->out}};
        gated->done = true;
        const hipError_t e = launch_mfma_gated(pair, mt, begin, acc.stream);
        return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
    }
    const hipError_t e = g.count == 1 ? launch_mfma_fused(g.p[0], mt, acc.stream) : launch_mfma_group(g, mt, begin, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// Which kernel a lone problem runs on and how it is cut up (no device work).
enum Kernel : int { kLookup = 0, kMatrixCore = 1 };

// The matrix-core kernel also takes the other formats, alpha groups of any length and any K; 64 outputs may
// touch four row groups at most.
bool mfma_any(const Problem &p, int mode)
{
    // (two rows: the look-up kernel, whose time is that of the sign stream, wins on longer streams; us, look-up
    // against this kernel: int8 exponents 4096x4096x3 7.3 / 6.9, 13824x5120x2 11.6 / 15.0; uniform 768x768x3
    // 5.7 / 5.1, 2048x2048x3 6.4 / 6.2, 4096x4096x4 7.6 / 8.8, where q_bias makes every weight two pieces)
    // One row as well where a look-up tile of 256 outputs touches more than two row groups and every lane would
    // fetch its own multipliers: int8 exponents 768x768x3 in 8 groups 10.0 / 5.2, 4096x4096x3 in 32 groups
    // 14.8 / 6.9, 1600x28672x4 in 8 groups 35.7 / 17.0.
    const int least = mfma_min_rows();
    if (p.M < least) {
        const long two_rows = mode == kUniformF16 ? 2l << 20 : 8l << 20;
        const bool scattered = is_block(mode) && p.rows_per_group < kTileCols;
        if (least != 3 || !(scattered || (p.M == 2 && (long)p.N * (p.K / 8) * p.nb <= two_rows))) return false;
    }
    if ((unsigned long long)p.M * p.K * 2 >= (1ull << 32)) return false;
    if (is_block(mode))
        return p.rows_per_group >= 24 && (unsigned long long)p.K / 8 * p.nb * p.R * 3 < (1ull << 32);
    return (unsigned long long)p.kwords * p.nb * p.N * 2 < (1ull << 32);
}

bool tile_possible(const Problem &p, int mode);

// `known`: tile_wanted's plan, where it made one
int plan_single(Problem &p, int mode, const MfmaPlan &known, int *kernel, int *mrows)
{
    if (known.mt || mfma_eligible(p, mode) || mfma_any(p, mode)) {
        const MfmaPlan plan = known.mt ? known : mfma_plan(p, tile_possible(p, mode));
        plan_mfma(p, plan.mt, plan.slices);
        *kernel = kMatrixCore;
        *mrows = 16 * plan.mt;
        return LUTGEMM_OK;
    }
    *kernel = kLookup;
    *mrows = pick_mrows(p.M);
    const long items = (long)((p.N + kTileCols - 1) / kTileCols) * p.nsets;
    const long want = target_blocks((long)p.N * (p.K / 8) * p.nb, items, mode != kRowF16 && mode != kUniformF16);
    int rc = plan_lookup(p, *mrows, want);
    if (rc != LUTGEMM_OK) return rc;
    // One row, per-column alphas and ranges of several items: twin items, i.e. one table build and one
    // barrier per 512 outputs instead of per 256.  A build is about a third of an item's vector
    // instructions at three bit planes, and a launch whose workgroups hold several items each is bound
    // by those; launches of one or two items per workgroup are bound by latencies that twin items would
    // lengthen (half as many ranges to spread over the chip).
    // Measured, plain against twin items (us): 28672x8192x4 27.2 / 24.7-25.1, 28672x8192x3 21.6 / 19.6-20.0;
    // with two bit planes no gain (28672x8192x2 15.0 / 15.2-15.4: bound by the stream), and none where the
    // twin plan has to give up the unequal ranges of the two workgroups of a CU (8192x28672x4 with equal
    // ranges 26.3 / 28.1) or where K is long (the same shape with ranges of 4 and 3 twin items 26.4 / 26.9).
    const int least = option(LUTGEMM_OPTION_TWIN_ITEMS);
    if (least > 0 && *mrows == 1 && (mode == kRowF16 || mode == kUniformF16) && p.nb >= 3 && p.nsets <= 64 &&
        p.short_items >= least && p.items_per_wg >= least) {
        Problem t = p;
        const bool unequal = p.items_per_wg != p.short_items;
        if (plan_lookup(t, 1, want, true) == LUTGEMM_OK && (!unequal || t.items_per_wg != t.short_items) &&
            10 * t.n_blocks >= 9 * p.n_blocks)
            p = t;
    }
    return LUTGEMM_OK;
}

// Block-scaled kernel: a workgroup takes 64 outputs, a chunk of 5, 8 or 16 rows and a K-slice of whole rounds (8 K-steps,
// one per wave); two workgroups fit a CU.  The slice length (rounds) is the one that minimises the
// rounds of the grid times the cost of a workgroup: its rounds plus a constant for its start and end
// (table build, reduction, accumulator words), in units of a round.
void plan_mx(Problem &p)
{
    constexpr long kResident = 2 * 256;
    // (measured: anything from half a round to three rounds plans the same launches for the shapes
    // tried; with no constant at all a slice is a single round and 28672x8192x4 takes 61 us instead of 34)
    constexpr double fixed_rounds = 1.0;
    p.n_tiles = (p.N + kMfmaTileCols - 1) / kMfmaTileCols;
    p.mchunks = (p.M + mx_chunk_rows(p.M) - 1) / mx_chunk_rows(p.M);
    p.nsets = p.K / kMfmaStepK;
    const int rounds = (p.nsets + kMfmaWaves - 1) / kMfmaWaves;
    int best = rounds;
    double best_cost = 0.0;
    for (int r = rounds; r >= 1; --r) {
        const int ks = (rounds + r - 1) / r;
        if (ks > kMaxSlices) break;
        const long wgs = (long)p.n_tiles * p.mchunks * ks;
        const double cost = (double)((wgs + kResident - 1) / kResident) * ((double)r + fixed_rounds);
        if (r == rounds || cost < best_cost * 0.999) {
            best = r;
            best_cost = cost;
        }
    }
    if (const int blocks = mfma_blocks_override()) {
        long want = blocks / ((long)p.n_tiles * p.mchunks);
        if (want < 1) want = 1;
        if (want > kMaxSlices) want = kMaxSlices;
        if (want > rounds) want = rounds;
        best = (rounds + (int)want - 1) / (int)want;
    }
    p.sets_per_split = best * kMfmaWaves;
    p.ksplit = (p.nsets + p.sets_per_split - 1) / p.sets_per_split;
    p.n_blocks = p.n_tiles * p.ksplit * p.mchunks;
}

// Whether a problem that may take the block-scaled kernel should.  It needs one, two or three matrix
// instructions per (bit plane, 16 outputs, 128 inputs) for up to 5, 8 or 16 rows, and a launch of its own
// that splits the activations (3 to 4 us with the gap between the launches); the fp16 kernel needs four per
// weight tile whatever the planes, and forms the weights.  Up to 5 rows from 48 MB of sign words on, up to 8 rows from
// 96 MB on: drawn for an fp16 kernel that expanded every plane (28672x8192x4: 4 rows 50.8 us).  Measured with the
// present one (us, fp16 kernel / block-scaled, * = taken):
//   28672x8192x4: 4 rows 33.7 / 33.8*, 8 rows 34.9 / 41.1*, 16 rows 38.9* / 58.8
//   28672x8192x2: 4 rows 22.5 / 23.9*, 8 rows 23.3* / 29.0;  8192x28672x4: 4 rows 33.4 / 35.3*, 8 rows 34.2 / 42.1*
//   8192x8192x4:  4 rows 12.8* / 16.0, 8 rows 13.0* / 18.6;  8192x8192x2: 4 rows 9.3* / 13.5
// so the rule no longer pays: on a par up to five rows, 20 % behind at eight.
bool mx_wanted(const Problem &p)
{
    const int how = option(LUTGEMM_OPTION_BLOCK_SCALED);
    if ((long)p.M * p.K >= (1l << 30)) return false;   // (the split kernel indexes the activations with 32 bits)
    if (how != 1) return how == 2;
    const long sign_bytes = (long)p.N * (p.K / 8) * p.nb;
    return (p.M <= 5 && sign_bytes >= (48l << 20)) || (p.M <= 8 && sign_bytes >= (96l << 20));
}

// Row-wise problem whose alphas are powers of two, with enough rows for the matrix cores: the
// block-scaled kernel (16-row tiles; more rows are further row chunks that stream the same sign
// words side by side).
int run_mx(Problem &p, const Accum &acc)
{
    plan_mx(p);
    if (p.ksplit > 1) {
        int rc = accum_words(acc, (size_t)p.M * p.N, &p.accum);
        if (rc != LUTGEMM_OK) return rc;
    }
    if (acc.fixed) return LUTGEMM_EUNSUP;
    std::lock_guard<std::mutex> lock(g_two_launches_mutex);
    void *buf = nullptr;
    int rc = stream_split_buffer(acc.stream, mx_split_bytes(p.M, p.K), &buf);
    if (rc != LUTGEMM_OK) return rc;
    const hipError_t e = launch_mx(p, buf, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// ---- GEMM kernel for many activation rows ------------------------------------------------------------
// Cut a problem into tiles of 256 outputs x 64 or 128 rows and K-slices, a workgroup each.  A workgroup is four waves,
// two workgroups per CU, or two teams of four that halve its slice (one per CU).
// The cut depends on the sizes alone, so that a call gives the same bits eagerly, under capture and through the
// entry point that allocates nothing.  Returns the time the plan should take.
// Costs in microseconds, for all formats and planes.  A step of a 128-row tile: 1.1 alone on its CU (measured 1.0 to 1.25),
// 1.95 beside another workgroup or for two teams together, 1.65 for teams while a third of the CUs are idle (clocks
// are higher); 64 rows: 0.8, 1.35 and 1.2.  A workgroup's start and end 4.6, with teams 6 (fitted when sums were added to a bias and
// stored piece by piece, 2 more than now with teams or a bias).  The sums of the slices and the launch that adds them up 6 and 0.2 per
// MB.  What they pick (us; s: slices of four waves, p: of teams, * = taken):
//   512 rows:  5120x13824x2 int8 exponents s3 105.7 s6 92.1 p2 111.6 p3* 88.3; 13824x5120x2 int8 exponents s1 106.8 s2 99.5 p1* 85.2;
//              4096x4096x3 s3 37.9 s4 34.2 p3 35.7 p4* 34.3 (s3 was taken before: 105.7, 106.6 and 42.5)
//   1024 rows: 4096x4096x3 s1 72.1 s2 51.6 p1 60.7 p2* 50.3; 5120x5120x2 blocks s1 92.1 s2 84.3 s3 76.1 p1* 72.4
//   128 rows:  8192x28672x4 s8 76.0 p4 104.4 p8* 72.9; 8192x8192x4 s8 34.2 p4 42.2 p8* 34.3; 11008x4096x3 s5 30.4 p3 34.2 p5* 29.8
//   64 rows:   8192x28672x4 s8 58.1 p4 81.7 p8* 50.2; 8192x8192x4 s8 25.6 p8* 24.2; 13824x5120x2 int8 exponents s8 30.6 p4* 29.2
double plan_tile(TileProblem &t)
{
    constexpr long kCUs = 256;
    t.tile_rows = t.M <= 64 ? 64 : 128;
    t.n_tiles = (t.N + 255) / 256;
    t.m_tiles = (t.M + t.tile_rows - 1) / t.tile_rows;
    t.steps = (t.kwords + 3) / 4 * 2;
    const long tiles = (long)t.n_tiles * t.m_tiles;
    const bool tall = t.tile_rows == 128;
    double best_cost = 0.0;
    for (int ks = 1; ks <= kTileMaxSlices && (ks == 1 || 2 * ks <= t.steps); ++ks) {
        const int steps = ((t.steps + ks - 1) / ks + 1) & ~1;
        const int slices = (t.steps + steps - 1) / steps;
        if (slices != ks) continue;
        const long wgs = tiles * slices;
        const size_t sums = ks > 1 ? ks * tile_slice_stride(t.M, t.N) * 4 : 0;
        if (ks > 1 && (wgs > 2 * kCUs || sums > kTileSumBytes)) break;
        for (int pair = 0; pair < 2; ++pair) {
            if (pair && wgs > kCUs) continue;   // (rounds of teams end together: 11008x4096x3 at 2048 rows s1 199 p1 209)
            const long rounds = wgs / (2 * kCUs), rest = wgs - rounds * 2 * kCUs;   // (of two workgroups per CU)
            const double together = tall ? 1.95 : 1.35, fixed = pair ? 6.0 : 4.6;
            const int own = pair ? (steps / 2 + 1) & ~1 : steps;
            double step = together;   // of the last, partly filled round
            if (pair) {
                const double idle = 1.0 - (double)rest / kCUs;
                step -= (tall ? 0.3 : 0.15) * (idle > 0.4 ? 1.0 : idle / 0.4);
            } else if (rest <= kCUs) {
                step = tall ? 1.1 : 0.8;
            }
            double cost = (double)rounds * (own * together + fixed);
            if (rest > 0) cost += own * step + fixed;
            if (sums) cost += 6.0 + 0.2e-6 * (double)sums;
            if ((ks == 1 && !pair) || cost < best_cost * 0.99) {
                best_cost = cost;
                t.pair = pair;
                t.ksplit = slices;
                t.slice_steps = steps;
            }
        }
    }
    return best_cost;
}

double gemm_estimate(const Problem &p, bool *sliced)
{
    TileProblem t{};
    t.N = p.N;
    t.M = p.M;
    t.kwords = p.kwords;
    const double us = plan_tile(t);
    *sliced = t.ksplit > 1;
    return us;
}

// What the GEMM kernel can take.
bool tile_possible(const Problem &p, int mode)
{
    // (32-bit byte offsets into the operands)
    const unsigned long long limit = 1ull << 32;
    if ((unsigned long long)p.kwords * p.nb * p.N * 4 >= limit || (unsigned long long)p.M * p.K * 2 >= limit) return false;
    if (is_block(mode) && (unsigned long long)p.K / 8 * p.nb * p.R * 3 >= limit) return false;
    const int least = option(LUTGEMM_OPTION_TILE_MIN_M);
    return least <= 0 || p.M >= least;
}

// What the GEMM kernel is expected to take beside the matrix-core kernel's estimate: plan_tile's costs, which know neither
// planes nor formats, scaled to what both kernels were measured to take, and 3 us that they are short of for few inputs.
// Up to 64 inputs, a single step of either kernel and outside what the estimates were fitted to, calls keep the line they had
// (us, matrix-core kernel / this one, * = taken: 6028x64x4 at 33 rows 6.4 / 8.6*, 3100x64x3 at 200 7.0* / 9.6, 13800x64x3 at 128
// 15.5 / 10.9*).
double gemm_us(const Problem &p, double estimate)
{
    if (p.K <= 64) return 0.95 * estimate;
    const double planes = p.alpha_mode == kRowF16 ? 0.55 + 0.13 * p.nb : is_block(p.alpha_mode) ? 0.62 + 0.22 * p.nb : 0.60 + 0.40 * p.nb;
    return 3.0 + planes * estimate;
}

// Whether a call takes the GEMM kernel rather than the matrix-core kernel, by the two estimates (see mfma_plan for the
// calls that may).  Drawn with 900 calls and checked on 3000 others near the line, timed on both (33 to 2048 rows, 512 to 28672
// inputs and outputs), as both kernels then were: the kernel taken was within 1.0 % of the better one on average, 6 % of the calls lost
// more than 5 %.  Closer to the line, 1000 calls that would change kernel at up to half as many rows again: 4.7 % and 22 % then,
// 5.4 % and 24 % with the present kernels, five in six of those that lose by taking the
// matrix-core kernel (most 768x17216x4 at 334 rows 72.8* / 32.8, 18192x1856x4 at 71 51.1* / 26.7).
// Measured (us, matrix-core kernel / this one, * = taken):
//   row-wise: 6464x4096x3 at 65 rows 18.0* / 22.8, 10944x5120x3 at 64 30.3* / 24.1, 6144x5120x2 at 72 18.6* / 24.4, 7680x8192x3 at 112
//   40.0 / 33.1*, 3072x3328x3 at 256 22.3* / 24.3, 24128x3072x2 at 80 45.1 / 33.5*; scales that are no powers of two 3392x6144x3 at
//   72 24.6* / 31.3, 15360x3328x3 at 33 30.0* / 37.2, 20096x1024x2 at 160 34.5 / 37.7*
//   fp16 blocks: 5056x4096x4 at 64 17.9* / 27.6, 10240x7040x3 at 56 39.7 / 28.6*, 4800x8192x2 at 512 99.5 / 62.1*, 19008x3072x3 at 72 46.1 / 35.9*
//   int8 exponents: 6144x3584x4 at 56 17.8* / 25.3, 13312x5760x3 at 36 41.5 / 29.8*, 7168x5120x3 at 128 38.6* / 32.1
//   uniform: 21888x1024x4 at 72 39.9* / 53.0, 5312x7168x3 at 112 52.7 / 40.9*, 12864x2048x3 at 128 43.4* / 38.1
// `planned`: the matrix-core kernel's plan, where one was made (mt = 0 otherwise).
bool tile_wanted(const Problem &p, int mode, MfmaPlan *planned)
{
    MfmaPlan &plan = *planned;
    plan = MfmaPlan{};
    if (!tile_possible(p, mode)) return false;
    if (option(LUTGEMM_OPTION_TILE_MIN_M) > 0) return true;
    if (!mfma_any(p, mode)) return p.M > 8;   // (the look-up kernel, four rows at a time, is the other choice)
    if (p.M <= 32) return false;
    plan = mfma_plan(p, true);
    if (!plan.gemm || plan.us == 0.0) return plan.gemm;
    // bf16 activations: the matrix-core kernel converts them on the way, 6 % (four planes) to 15 % (one) of its time; in front of the
    // GEMM kernel that is a launch of 4.2 us and 1.3 per million.  us, fp16 and bf16 of either kernel (* = taken): 13184 -> 2944
    // of 3 bits at 128 rows 31.7, 35.0* / 29.6*, 35.9; 4096 -> 4096 of 3 bits at 384 rows 34.7, 37.7* / 31.2*, 36.6; 13824 -> 5120 of 3
    // bits at 128 rows 58.8, 65.7 / 36.2*, 41.2*, at 1024 307.9, 334.1 / 165.9*, 188.7*.
    const double on_the_way = 1.18 - 0.03 * p.nb;
    const bool bf16 = p.x_type == kIoBF16;
    const double here = bf16 ? on_the_way * plan.us : plan.us;
    const double there = gemm_us(p, plan.gemm_us) + (bf16 ? 4.2 + 1.3e-6 * ((double)p.M * p.K) : 0.0);
    // One launch without memory is given up for slices only where these are expected to save an eighth, or were the choice before the
    // estimates: where their sums have no place (a capture with nothing reserved) they are taken in turn.  Of 70 calls that either rule
    // would move, those kept in one launch took 4 % more with slices, the others 12 % less, and five times as long in turn (us,
    // this kernel / slices / in turn: 13920x2560x2 at 75 rows 26.3* / 35.2 / 93, 4480x12800x3 at 34 27.1* / 29.1 / 261, 9120x9984x3 at 64 49.8 /
    // 37.6* / 194).
    if (here <= there || !plan.one_launch || here > 1.13 * there) return here > there;
    return never_cut(p);
}

int run_tile(const Problem &p, int mode, const Accum &acc)
{
    TileProblem t{};
    t.W = p.W;
    t.alpha = p.alpha;
    if (mode == kUniformF16) t.qbias = p.qbias;
    t.x = p.x;
    t.init = p.init;
    t.out = p.out;
    t.N = p.N;
    t.K = p.K;
    t.M = p.M;
    t.kwords = p.kwords;
    t.by_group_words = p.by_group_words;
    t.R = p.R;
    t.rows_per_group = p.rows_per_group;
    t.mode = mode;
    plan_tile(t);
    t.init_stride = p.init_stride;
    t.overwrite = p.overwrite;
    t.out_type = p.out_type;
    std::unique_lock<std::mutex> lock(g_two_launches_mutex, std::defer_lock);
    // Where the slices' sums have no place (a stream under capture whose buffer would have to grow, the entry
    // point that allocates nothing) a workgroup takes the slices of its tile in turn.
    if (t.ksplit > 1 && !acc.fixed) {
        void *sums = nullptr;
        lock.lock();
        const int rc = stream_split_buffer(acc.stream, t.ksplit * tile_slice_stride(t.M, t.N) * 4, &sums);
        if (rc != LUTGEMM_OK && rc != LUTGEMM_ECAPTURE) return rc;
        t.partial = (float *)sums;
    }
    const hipError_t e = launch_tile(t, p.nb, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// `bias`: null = accumulate into out; otherwise *bias is the row every output row starts from (null:
// zeros) and out is written, not read.  `x_type`, `out_type`: IoType of x and of out (then written, not read);
// the kernels that take other activations than fp16 themselves are the ones whose few rows make a launch of
// its own for the conversion dear, LUTGEMM_EUNSUP otherwise (which a caller answers by converting).
int run(int mode, const uint32_t *bW, const void *alpha, const void *qbias, const void *x,
        void *out, int N, int K, int nb, int num_groups, int M, const Accum &acc, bool alpha_pow2 = false,
        const void *const *bias = nullptr, int x_type = kIoF16, int out_type = kIoF16)
{
    Problem p;
    int rc = fill_problem(p, mode, bW, alpha, qbias, x, out, N, K, nb, num_groups, M);
    if (rc != LUTGEMM_OK) return rc;
    if (bias && *bias) {
        if (!aligned(*bias, 2)) return LUTGEMM_EALIGN;
        p.init = (const __half *)*bias;
        p.init_stride = 0;
    } else if (bias) {
        p.overwrite = 1;
    }
    p.x_type = x_type;
    p.out_type = out_type;
    // (ahead of the GEMM kernel: LUTGEMM_OPTION_BLOCK_SCALED = 2 means any number of rows)
    if (alpha_pow2 && mode == kRowF16 && mfma_eligible(p, mode) && p.M >= mfma_min_rows() && mx_wanted(p)) return run_mx(p, acc);
    MfmaPlan planned;
    if (tile_wanted(p, mode, &planned)) return x_type == kIoF16 ? run_tile(p, mode, acc) : LUTGEMM_EUNSUP;
    int kernel = kLookup, mrows = 1;
    rc = plan_single(p, mode, planned, &kernel, &mrows);
    if (rc != LUTGEMM_OK) return rc;
    if (kernel == kMatrixCore) {
        if (x_type == kIoF32) return LUTGEMM_EUNSUP;   // (a step's operands would not fit the registers)
    } else if (x_type != kIoF16 || out_type != kIoF16) {
        const bool per_column = mode == kRowF16 || mode == kUniformF16;
        if (mrows > 2 || (mrows == 2 && per_column && option(LUTGEMM_OPTION_PAIR_TABLES) == 0) ||
            (!per_column && p.rows_per_group < kTileCols))
            return LUTGEMM_EUNSUP;
    }
    if (kernel == kMatrixCore ? p.ksplit > 1 : lookup_splits_k(p)) {
        rc = accum_words(acc, (size_t)M * N, &p.accum);
        if (rc != LUTGEMM_OK) return rc;
    }
    hipError_t e;
    if (kernel == kMatrixCore)
        e = launch_mfma(p, mrows / 16, acc.stream);
    else if (mode == kRowF16 || mode == kUniformF16)
        e = launch_gemv_rowwise(p, mode, mrows, acc.stream);
    else if (p.rows_per_group >= kTileCols)  // a tile spans at most two row groups
        e = launch_gemv_block_staged(p, mode + 4, mrows, acc.stream);
    else
        e = launch_gemv_block(p, mode, mrows, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// What a workgroup of a grouped look-up launch takes, in us: an item is a table build plus look-ups in proportion to its bit
// planes.  With a workgroup per CU 0.45 + 0.13 * nb (measured).  Where two share a CU 0.10 + 0.38 * nb (one row to two of
// gate,up adds 5.4 items to each: of 2, 3 and 4 bits 4.65, 6.5 and 8.7 us), and a range that ends inside a second tile has
// another tile's sums to hand over (1.05, fitted with 100 launches of unlike widths, one and two rows, 4096 to 8192 inputs: 1.5 %
// behind the best of four sharings on average, with 0.75 to 1.5 much the same, without 4 %).  us, RMSNorm in front, with the first
// costs / with the second ones without the hand-over and kEngines below / as they are:
//   one row: gate,up 4096 -> 11008 of 1 and 3 bits 13.4 / 10.8 / 10.8; q,k,v 5120 -> 5120 of 2, 4 and 3 bits 12.3 / 11.3 / 11.1
//   two rows: q,k,v 4096 -> 4096 of 1, 4 and 3 bits 12.9 / 14.8 / 11.5, of 2, 1 and 4 bits 10.3 / 13.7 / 10.2; 5120 -> 5120 of 3, 2 and 2 bits
//   13.3 / 15.3 / 13.2; gate,up 4096 -> 11008 of 2 and 4 bits 25.0 / 21.4 / 20.8, of 3 and 4 bits 27.1 / 26.8 / 23.3, of 1 and 4 bits 20.6 / 18.3 /
//   18.2; slower: 4096 -> 14336 of 4 and 3 bits 23.0 / 26.9 / 26.6, q,k,v 5120 -> 5120 of 4, 1 and 1 bits 14.5 / 16.1 / 16.2
struct ItemCost {
    double fixed, plane, hand_over;
};
constexpr ItemCost kItemAlone{0.45, 0.13, 0.0}, kItemBeside{0.10, 0.38, 1.05};
// Workgroups are dealt to the chip's 32 shader engines in turn, the empty ones of a problem narrower than the grid as well, and
// an engine holds 16 of this kernel's; what is dealt to a full engine waits for a range to end (gate,up 4096 -> 11008 of 3 and 4
// bits at two rows: 230 + 276 workgroups, 17 on the first engines, 26.6 us; 198 + 276 23.0).
constexpr long kEngines = 32;

// Share a workgroup budget between look-up problems that run side by side so that the longest range of every problem takes
// about the same time: the problems end with their slowest workgroup, so the items per workgroup of each are what it
// takes in T, for the smallest T whose workgroups fit the budget (`by_engine`: fit every engine's part of it).
// With equal bit widths this is a share in proportion to the items, rounded down: a few
// workgroups more than can be resident run as a second, mostly empty round, and fewer
// workgroups with more items each are the better trade anyway (q,k,v of 4096x4096 as 3 x 64
// workgroups of 4 items 5.31 us per GEMV of the four-launch block, as 3 x 86 of 3 items 5.54).
struct Shares {
    int most;         // the largest workgroup count of a problem
    bool any_split;   // some problem needs accumulator words
};

struct Sharing {
    Problem *const *ps;
    int count;
    ItemCost item;
    long budget;
    bool by_engine;

    double cost(int i) const { return item.fixed + item.plane * ps[i]->nb; }
    long items(int i) const { return (long)((ps[i]->N + kTileCols - 1) / kTileCols) * ps[i]->nsets; }

    // the items of a range of problem i that takes `us`: within one tile (or of whole ones), or across two
    long within(int i, double us) const
    {
        const long across = us > 2.0 * item.hand_over ? (long)((us - 2.0 * item.hand_over) / cost(i)) : 0;
        long whole = us > item.hand_over ? (long)((us - item.hand_over) / cost(i)) : 0;
        const int nsets = ps[i]->nsets;
        if (whole >= nsets)
            whole -= whole % nsets;
        else
            while (whole > across && nsets % whole) --whole;
        return across > whole ? across : whole;
    }

    bool fits(double us) const
    {
        long wgs[kMaxGroup], all = 0, widest = 0;
        for (int i = 0; i < count; ++i) {
            const long ipw = within(i, us);
            if (ipw < 1) return false;
            wgs[i] = (items(i) + ipw - 1) / ipw * ps[i]->M;
            all += wgs[i];
            widest = wgs[i] > widest ? wgs[i] : widest;
        }
        if (!by_engine) return all <= budget;
        for (int at = 0; at < count; ++at) {   // (an engine with most of them is one that a problem begins on)
            long here = 0;
            for (int i = 0; i < count; ++i) {
                const long from = ((at - i) * widest % kEngines + kEngines) % kEngines;
                here += wgs[i] / kEngines + (from < wgs[i] % kEngines ? 1 : 0);
            }
            if (here > budget / kEngines) return false;
        }
        return true;
    }

    int plan(Shares *out) const
    {
        double lo = 0.0, hi = 0.0;
        for (int i = 0; i < count; ++i) {
            const double all = (double)items(i) * cost(i) + 2.0 * item.hand_over;
            if (all > hi) hi = all;
        }
        for (int it = 0; it < 50; ++it) {
            const double mid = 0.5 * (lo + hi);
            if (fits(mid)) hi = mid; else lo = mid;
        }
        *out = Shares{0, false};
        for (int i = 0; i < count; ++i) {
            Problem &p = *ps[i];
            long ipw = within(i, hi);
            if (ipw < 1) ipw = 1;
            const int rc = plan_lookup(p, 1, (items(i) + ipw - 1) / ipw * p.M);
            if (rc != LUTGEMM_OK) return rc;
            if (p.n_blocks > out->most) out->most = p.n_blocks;   // grid.x: the largest problem's workgroups
            out->any_split = out->any_split || lookup_splits_k(p);
        }
        return LUTGEMM_OK;
    }
};

// The shares of a grouped look-up launch.
int share_group(Problem *const *ps, int count, int xform, Shares *out)
{
    long bytes = 0;
    bool mixed = false, long_rows = true;
    for (int i = 0; i < count; ++i) {
        bytes += (long)ps[i]->N * (ps[i]->K / 8) * ps[i]->nb * ps[i]->M;
        mixed = mixed || ps[i]->nb != ps[0]->nb;
        long_rows = long_rows && ps[i]->K >= 4096;
    }
    // Two workgroups per CU also on short streams where a workgroup begins with an RMSNorm (it hides one's start behind
    // the other's) or widths differ (finer shares): us, budget of 256 against 512, one row, 4096 inputs with RMSNorm: q,k,v of
    // 2, 3 and 4 bits 10.7 / 8.9, of 3 bits 9.0 / 8.8, grouped heads (4096 + 2 x 1024 outputs) 7.8 / 7.2, two rows 10.9 / 7.9;
    // without it q,k,v of 2, 3 and 4 bits 9.9 / 8.0, of 3 bits 7.65 / 8.2.  2048 inputs: 8 MB 6.3 / 6.9, two rows 9 MB
    // 6.25 / 6.55; 3072 inputs: one row, q,k,v of 2, 4 and 3 bits 7.4 / 7.7, of 3 bits 6.8 / 7.6, gate,up of 2 and 4 bits 9.6 / 9.1, of
    // 3 bits 8.6 / 8.9 (two rows would gain there: 11.0 / 8.7, 9.2 / 8.3, 13.2 / 9.5 of 1 and 3 bits).
    const bool pairs = count > 1 && (xform == kXNorm || mixed) && long_rows && bytes >= (9l << 20) &&
                       option(LUTGEMM_OPTION_TARGET_BLOCKS) <= 0;
    const long usual = target_blocks(bytes), budget = pairs ? 512 : usual;
    // Callers that reserve nothing before a capture rely on which launches need accumulator words: none with the usual
    // budget and the costs of a workgroup alone, none now.  (That is where all its ranges are whole rows of items, nsets of
    // them or a multiple; they are not if times too short for one row of the dearest problem already fit.)
    const Sharing alone{ps, count, kItemAlone, usual, false};
    double whole = 0.0;
    for (int i = 0; i < count; ++i) {
        const double us = alone.cost(i) * ps[i]->nsets;
        whole = us > whole ? us : whole;
    }
    if (!alone.fits(whole * (1.0 - 1e-9))) {
        const int rc = alone.plan(out);
        if (rc == LUTGEMM_OK && !out->any_split) return rc;
    }
    // (inputs shorter than 4096 keep the first costs: 3072 -> 8192 of 2 and 4 bits at two rows 11.3, with the second ones 12.5)
    return Sharing{ps, count, budget == 512 && mixed && long_rows ? kItemBeside : kItemAlone, budget, budget == 512}.plan(out);
}

// Up to kMaxGroup row-wise problems in one launch of the look-up kernel.  Problems
// with enough rows for the matrix-core kernel (and no fused transform) are launched
// on that path instead.
struct GroupPlan {
    Group g;
    int xform;
    bool one_mfma, each_mfma;   // one launch of the matrix-core kernel, one per problem; neither: the look-up kernel, with
    Shares shares;
};

int plan_group(int count, const lutgemm_fused_problem *problems, const Gated *gated, GroupPlan &plan)
{
    Group &g = plan.g;
    g.count = count;
    bool plain = true, all_mfma = true;
    int &xform = plan.xform;
    xform = kXNone;
    for (int i = 0; i < count; ++i) {
        const lutgemm_fused_problem &q = problems[i];
        Problem &p = g.p[i];
        int rc = fill_problem(p, kRowF16, q.bW, q.alpha_f16, nullptr, q.x_f16, q.out_f16, q.N, q.K, q.nb,
                              q.num_groups, q.M);
        if (rc != LUTGEMM_OK) return rc;
        if (q.norm_weight_f16 && q.gate_f16) return LUTGEMM_EINVAL;
        if (q.overwrite != 0 && q.overwrite != 1) return LUTGEMM_EINVAL;
        if (q.norm_weight_f16 && !(q.norm_eps >= 0.0f)) return LUTGEMM_EINVAL;
        if (!aligned(q.norm_weight_f16, 16) || !aligned(q.gate_f16, 16)) return LUTGEMM_EALIGN;
        p.norm_w = (const __half *)q.norm_weight_f16;
        p.gate = (const __half *)q.gate_f16;
        p.norm_eps = q.norm_eps;
        p.overwrite = q.overwrite;
        // RMSNorm split over two launches
        if ((q.next_input_f16 != nullptr) != (q.next_norm_weight_f16 != nullptr)) return LUTGEMM_EINVAL;
        if (q.sumsq_out_f32 && q.N % 32 != 0) return LUTGEMM_EINVAL;
        if (q.sumsq_in_f32 && (q.sumsq_in_slots <= 0 || q.norm_weight_f16 || !(q.norm_eps >= 0.0f))) return LUTGEMM_EINVAL;
        if (!q.sumsq_in_f32 && q.sumsq_in_slots != 0) return LUTGEMM_EINVAL;
        // the slots are those a completing problem of K outputs fills (one per 32 columns); the
        // matrix-core kernel reads them four at a time
        if (q.sumsq_in_f32 && (q.K % 32 != 0 || q.sumsq_in_slots != q.K / 32)) return LUTGEMM_EINVAL;
        if (!aligned(q.next_input_f16, 2) || !aligned(q.next_norm_weight_f16, 2) || !aligned(q.sumsq_out_f32, 4) ||
            !aligned(q.sumsq_in_f32, 16))
            return LUTGEMM_EALIGN;
        p.next_w = (const __half *)q.next_norm_weight_f16;
        p.next_in = (__half *)q.next_input_f16;
        p.sumsq_out = q.sumsq_out_f32;
        p.sumsq_in = q.sumsq_in_f32;
        p.sumsq_slots = q.sumsq_in_slots;
        // one kernel instance per transform: the problems of a launch share theirs
        const int mine = p.norm_w ? kXNorm : p.gate ? kXGate : kXNone;
        if (i > 0 && mine != xform) return LUTGEMM_EUNSUP;
        xform = mine;
        plain = plain && !p.norm_w && !p.gate && !p.overwrite && !p.next_in && !p.sumsq_out && !p.sumsq_in;
        all_mfma = all_mfma && mfma_eligible(p, kRowF16);
    }
    // Every problem finishes its outputs with a plain read-modify-write, and the outputs are
    // requested early: nothing a problem of the launch writes (out, next_input, sumsq_out) may
    // overlap anything another write or a read of the launch (x, gate) touches.
    {
        struct Span {
            const char *lo, *hi;
            bool written;
        };
        Span spans[6 * kMaxGroup + 1];
        int n = 0;
        auto add = [&](const void *ptr, size_t bytes, bool written) {
            if (ptr) spans[n++] = Span{(const char *)ptr, (const char *)ptr + bytes, written};
        };
        for (int i = 0; i < count; ++i) {
            const Problem &p = g.p[i];
            const size_t mn = (size_t)p.M * p.N, mk = (size_t)p.M * p.K;
            add(p.out, mn * 2, true);
            add(p.next_in, mn * 2, true);
            add(p.sumsq_out, (size_t)p.M * (p.N / 32) * 4, true);
            add(p.x, mk * 2, false);
            add(p.gate, mk * 2, false);
            add(p.sumsq_in, (size_t)p.M * p.sumsq_slots * 4, false);
        }
        if (gated) add(gated->out, (size_t)g.p[0].M * g.p[0].N * 2, true);
        for (int i = 0; i < n; ++i)
            for (int j = i + 1; j < n; ++j)
                if ((spans[i].written || spans[j].written) && spans[i].lo < spans[j].hi && spans[j].lo < spans[i].hi)
                    return LUTGEMM_EINVAL;
    }
    // The matrix-core kernel takes plain and (as a group launch) overwriting problems.
    // Input transforms stay with the look-up kernel: there a workgroup transforms only
    // its K-slice of one row, while every 64-output workgroup of the matrix-core kernel
    // would redo the transform of all rows (measured slower than a separate kernel).
    bool same_height = true;
    for (int i = 1; i < count; ++i) same_height = same_height && ((g.p[i].M > 16) == (g.p[0].M > 16));
    plan.one_mfma = all_mfma && xform == kXNone && same_height && (count > 1 || !plain);
    plan.each_mfma = !plan.one_mfma && plain && all_mfma;
    if (plan.one_mfma || plan.each_mfma) return LUTGEMM_OK;
    Problem *ps[kMaxGroup];
    for (int i = 0; i < count; ++i) ps[i] = &g.p[i];
    return share_group(ps, count, xform, &plan.shares);
}

int run_group(int count, const lutgemm_fused_problem *problems, const Accum &acc, Gated *gated = nullptr)
{
    GroupPlan plan{};
    const int rc = plan_group(count, problems, gated, plan);
    if (rc != LUTGEMM_OK) return rc;
    Group &g = plan.g;
    if (plan.one_mfma) return run_mfma_group(g, acc, gated);
    if (plan.each_mfma) {
        for (int i = 0; i < count; ++i) {
            int rc = run_mfma(g.p[i], acc);
            if (rc != LUTGEMM_OK) return rc;
        }
        return LUTGEMM_OK;
    }
    if (plan.shares.any_split) {
        size_t words = 0;
        for (int i = 0; i < count; ++i) words += (size_t)g.p[i].M * g.p[i].N;
        unsigned long long *base = nullptr;
        int rc = accum_words(acc, words, &base);
        if (rc != LUTGEMM_OK) return rc;
        size_t off = 0;
        for (int i = 0; i < count; ++i) {
            g.p[i].accum = base + off;
            off += (size_t)g.p[i].M * g.p[i].N;
        }
    }
    const hipError_t e = count == 1 ? launch_gemv_fused(g.p[0], plan.xform, acc.stream) : launch_gemv_group(g, plan.xform, plan.shares.most, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// Row-wise problems of ONE launch that hand activations to each other through tagged rows.
// The launch's units (one workgroup's range of one problem) are numbered in the order the
// problems are given and taken in that order, so a problem that waits for a tag must come after
// the problem of the call that writes it.  Problems that wait for the same set of producers run
// side by side and share a workgroup budget (a "stage").
// Workgroups of a chained launch: all of them must be resident at once (a unit may wait for a
// unit of another workgroup), so at most what the device holds of this kernel.
int chain_grid(int *out)
{
    int resident = 0;
    const hipError_t e = chain_resident_workgroups(&resident);
    if (e != hipSuccess) return hip_fail(e);
    if (resident < 1) return LUTGEMM_EUNSUP;
    const int v = option(LUTGEMM_OPTION_CHAIN_GRID);
    *out = v > 0 && v < resident ? v : resident;
    return LUTGEMM_OK;
}

// Validate the problems of a chained launch and cut them into units (no device work when
// grid_in > 0).  On return c.g holds the planned problems, c.unit_start the units, depth[] the
// stage of every problem, *grid the workgroups of the launch.
int plan_chain(int count, const lutgemm_chain_problem *problems, int grid_in, Chain &c, int *depth, int *grid_out,
               bool *any_split_out, size_t *words_out)
{
    Group &g = c.g;
    g.count = count;
    size_t words = 0;
    unsigned direct[kMaxGroup], after[kMaxGroup], before_inputs[kMaxGroup];
    for (int i = 0; i < count; ++i) {
        const lutgemm_chain_problem &cq = problems[i];
        const lutgemm_fused_problem &q = cq.p;
        Problem &p = g.p[i];
        int rc = fill_problem(p, kRowF16, q.bW, q.alpha_f16, nullptr, q.x_f16, q.out_f16, q.N, q.K, q.nb, q.num_groups, q.M);
        if (rc != LUTGEMM_OK) return rc;
        if (q.M > LUTGEMM_CHAIN_MAX_ROWS) return LUTGEMM_EUNSUP;   // one row per workgroup: the look-up kernel only
        if (q.norm_weight_f16 && q.gate_f16) return LUTGEMM_EINVAL;
        if (q.overwrite != 0 && q.overwrite != 1) return LUTGEMM_EINVAL;
        if (q.norm_weight_f16 && !(q.norm_eps >= 0.0f)) return LUTGEMM_EINVAL;
        if (!aligned(q.norm_weight_f16, 16) || !aligned(q.gate_f16, 16)) return LUTGEMM_EALIGN;
        if (q.next_norm_weight_f16 || q.next_input_f16 || q.sumsq_out_f32 || q.sumsq_in_f32 || q.sumsq_in_slots)
            return LUTGEMM_EUNSUP;   // the RMSNorm of a chained problem is formed from the (tagged) row itself
        if (cq.x_tag < 0 || cq.x_tag > LUTGEMM_CHAIN_MAX_TAG || cq.gate_tag < 0 || cq.gate_tag > LUTGEMM_CHAIN_MAX_TAG ||
            cq.out_tag < 0 || cq.out_tag > LUTGEMM_CHAIN_MAX_TAG)
            return LUTGEMM_EINVAL;
        if (cq.gate_tag && !q.gate_f16) return LUTGEMM_EINVAL;
        // a thread holds its share of a norm row in two 16-byte registers sets: K <= 8192 when the row is tagged
        if (q.norm_weight_f16 && cq.x_tag && q.K > 8 * 2 * kThreads) return LUTGEMM_EUNSUP;
        p.norm_w = (const __half *)q.norm_weight_f16;
        p.gate = (const __half *)q.gate_f16;
        p.norm_eps = q.norm_eps;
        p.overwrite = q.overwrite;
        p.x_tag = cq.x_tag;
        p.gate_tag = cq.gate_tag;
        p.out_tag = cq.out_tag;
        words += (size_t)q.M * q.N;
        // which problems of the call this one waits for: the writers of the tags it reads
        depth[i] = 0;
        direct[i] = 0;
        auto producer = [&](const void *row, int tag) -> int {
            if (!tag) return LUTGEMM_OK;
            for (int j = 0; j < count; ++j) {
                if (problems[j].p.out_f16 != row || problems[j].out_tag != tag) continue;
                if (j >= i) return LUTGEMM_EINVAL;   // dispatched after its consumer: the wait could starve it
                direct[i] |= 1u << j;
                if (depth[j] + 1 > depth[i]) depth[i] = depth[j] + 1;
            }
            return LUTGEMM_OK;   // (no writer in the call: the row comes from elsewhere, the wait is bounded)
        };
        rc = producer(q.x_f16, cq.x_tag);
        if (rc != LUTGEMM_OK) return rc;
        rc = producer(q.gate_f16, cq.gate_tag);
        if (rc != LUTGEMM_OK) return rc;
        if (i > 0 && depth[i] < depth[i - 1]) return LUTGEMM_EINVAL;   // stages in dispatch order
        // everything this problem waits for, directly or not (after[i]), and through at least one
        // other problem (before_inputs[i])
        after[i] = direct[i];
        before_inputs[i] = 0;
        for (int j = 0; j < i; ++j)
            if (direct[i] >> j & 1u) {
                after[i] |= after[j];
                before_inputs[i] |= after[j];
            }
    }
    // What may overlap.  A problem writes an output only after contributions covering all of K
    // have arrived, each of which has waited for its inputs: when problem i writes anything, every
    // problem in after[i] has finished, and when a workgroup of i has its inputs, every problem in
    // before_inputs[i] has.  So the same tagged row may be written by several problems of a call
    // (a residual row that two GEMVs complete one after the other) and read in between, as long as
    // the waits order them; plain rows may not be shared between a writer and anyone else.
    for (int i = 0; i < count; ++i) {
        const Problem &a = g.p[i];
        const char *a0 = (const char *)a.out, *a1 = a0 + (size_t)a.M * a.N * (a.out_tag ? 4 : 2);
        auto overlaps = [&](const void *ptr, size_t bytes) {
            return ptr && a0 < (const char *)ptr + bytes && (const char *)ptr < a1;
        };
        for (int j = 0; j < count; ++j) {
            if (i == j) continue;
            const Problem &b = g.p[j];
            if (j < i && overlaps(b.out, (size_t)b.M * b.N * (b.out_tag ? 4 : 2))) {
                // an earlier writer of the same row: it must have finished before this one writes,
                // and before this one reads the row when it accumulates into it
                const bool same_row = a.out_tag && b.out_tag && a.out == b.out && a.out_tag != b.out_tag;
                const unsigned need = a.overwrite ? after[i] : before_inputs[i];
                if (!same_row || !(need >> j & 1u)) return LUTGEMM_EINVAL;
            }
            auto read_ok = [&](const __half *row, int tag, size_t bytes) {
                if (!overlaps(row, bytes)) return true;
                if (!(a.out_tag && tag && (const void *)row == (const void *)a.out)) return false;
                if (tag == a.out_tag) return i < j;             // the hand-over itself
                return (after[i] >> j & 1u) || (after[j] >> i & 1u);   // rewritten after the reader, or read after the writer
            };
            if (!read_ok(b.x, b.x_tag, (size_t)b.M * b.K * (b.x_tag ? 4 : 2))) return LUTGEMM_EINVAL;
            if (!read_ok(b.gate, b.gate_tag, (size_t)b.M * b.K * (b.gate_tag ? 4 : 2))) return LUTGEMM_EINVAL;
        }
    }
    // Plan stage by stage: the problems of a stage share one round of the grid (every workgroup
    // takes one unit of the stage) unless LUTGEMM_OPTION_CHAIN_BLOCKS says otherwise.
    int grid = grid_in;
    if (grid <= 0) {
        int rc = chain_grid(&grid);
        if (rc != LUTGEMM_OK) return rc;
    }
    const int stage_blocks = option(LUTGEMM_OPTION_CHAIN_BLOCKS) > 0 ? option(LUTGEMM_OPTION_CHAIN_BLOCKS) : grid;
    bool any_split = false;
    for (int first = 0; first < count;) {
        int last = first;
        long bytes = 0;
        Problem *ps[kMaxGroup];
        while (last < count && depth[last] == depth[first]) {
            ps[last - first] = &g.p[last];
            bytes += (long)g.p[last].N * (g.p[last].K / 8) * g.p[last].nb * g.p[last].M;
            ++last;
        }
        // a range's activations are fetched as one window of sixteen items: a stage whose units
        // would hold more takes further rounds of the grid
        constexpr int kWindowItems = kThreads / kTables;
        for (long rounds = 1;; ++rounds) {
            Shares shares;
            const int rc = Sharing{ps, last - first, kItemAlone, rounds * (long)stage_blocks, false}.plan(&shares);
            if (rc != LUTGEMM_OK) return rc;
            bool fits = true;
            for (int i = first; i < last; ++i) fits = fits && g.p[i].items_per_wg <= kWindowItems;
            if (fits) {
                any_split = any_split || shares.any_split;
                break;
            }
            if (rounds >= 4096) return LUTGEMM_EUNSUP;
        }
        first = last;
    }
    c.unit_start[0] = 0;
    for (int i = 0; i < count; ++i) c.unit_start[i + 1] = c.unit_start[i] + g.p[i].n_blocks;
    for (int i = count; i < kMaxGroup; ++i) c.unit_start[i + 1] = c.unit_start[count];
    const int total_units = c.unit_start[count];
    *grid_out = total_units < grid ? total_units : grid;
    *any_split_out = any_split;
    *words_out = words;
    return LUTGEMM_OK;
}

int run_chain(int count, const lutgemm_chain_problem *problems, const lutgemm_chain_control *ctl, const Accum &acc)
{
    if (!ctl || !ctl->status) return LUTGEMM_EINVAL;
    if (!aligned(ctl->status, 4) || !aligned(ctl->epoch, 4)) return LUTGEMM_EALIGN;
    Chain c{};
    Group &g = c.g;
    int depth[kMaxGroup], grid = 0;
    bool any_split = false;
    size_t words = 0;
    int rc = plan_chain(count, problems, 0, c, depth, &grid, &any_split, &words);
    if (rc != LUTGEMM_OK) return rc;
    if (any_split) {
        unsigned long long *base = nullptr;
        rc = accum_words(acc, words, &base);
        if (rc != LUTGEMM_OK) return rc;
        size_t off = 0;
        for (int i = 0; i < count; ++i) {
            g.p[i].accum = base + off;
            off += (size_t)g.p[i].M * g.p[i].N;
        }
    }
    c.ctl.epoch = ctl->epoch;
    c.ctl.status = ctl->status;
    const unsigned us = ctl->spin_limit_us ? ctl->spin_limit_us : 100000u;
    c.ctl.spin_ticks = (long long)us * 100;   // the wall clock ticks at 100 MHz
    const hipError_t e = launch_gemv_chain(c, grid, acc.stream);
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

// ---- tagged rows: conversions and the epoch word ---------------------------------------------
__global__ void __launch_bounds__(256) tag_rows_kernel(uint32_t *dst, const unsigned short *src, size_t n, int tag,
                                                       const uint32_t *epoch)
{
    const uint32_t t = effective_tag(tag, epoch ? *epoch : 0u) << 16;
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256) dst[i] = t | src[i];
}

__global__ void __launch_bounds__(256) untag_rows_kernel(unsigned short *dst, const uint32_t *src, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        dst[i] = (unsigned short)src[i];
}

__global__ void advance_epoch_kernel(uint32_t *epoch, uint32_t by)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *epoch += by;
}

// ---- measurement kernels ------------------------------------------------------------
__global__ void __launch_bounds__(256) copy_kernel(u32x4 *dst, const u32x4 *src, size_t n16)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < n16; i += stride) dst[i] = src[i];
}

// Reads `n16` 16-byte units and does nothing with them: what any kernel that has to
// stream that many bytes pays at least.
__global__ void __launch_bounds__(256) stream_read_kernel(const u32x4 *__restrict__ src, size_t n16, uint32_t *sink)
{
    constexpr int kUnroll = 8;
    size_t i = (size_t)blockIdx.x * 256 * kUnroll + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * 256 * kUnroll;
    u32x4 acc = {0u, 0u, 0u, 0u};
    for (; i + 256 * (kUnroll - 1) < n16; i += stride) {
        u32x4 v[kUnroll];
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) v[u] = __builtin_nontemporal_load(src + i + 256 * u);
#pragma unroll
        for (int u = 0; u < kUnroll; ++u) acc ^= v[u];
    }
    for (; i < n16; i += 256) acc ^= __builtin_nontemporal_load(src + i);
    if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x9e3779b9u && sink) sink[0] = acc.x;  // (keeps the loads alive)
}

// Same launch geometry and LDS footprint as the look-up kernel, no work.
__global__ void __launch_bounds__(kThreads) empty_kernel(uint32_t *sink)
{
    __shared__ float lds[kLutDwords + kStageDwords];
    if (sink && threadIdx.x == 0xffff) sink[0] = (uint32_t)lds[threadIdx.x];
}

}  // namespace
}  // namespace lutgemm

using namespace lutgemm;

int lutgemm_internal_hip_fail(int hip_error) { return hip_fail((hipError_t)hip_error); }

int lutgemm::option(int which)
{
    load_options();
    return g_option[which].load(std::memory_order_relaxed);
}

extern "C" {

const char *lutgemm_strerror(int code)
{
    switch (code) {
    case LUTGEMM_OK: return "ok";
    case LUTGEMM_EINVAL:
        return "invalid argument (null pointer, K % 32 != 0, N % 4 != 0, nb outside 1..4, "
               "group size not a multiple of 32, or rows per group not a multiple of 4)";
    case LUTGEMM_EALIGN: return "operand pointer is not aligned (bW, x: 16 bytes; alpha, out: 8 bytes)";
    case LUTGEMM_EUNSUP: return "unsupported configuration";
    case LUTGEMM_EHIP: return "HIP runtime error (see lutgemm_last_hip_error)";
    case LUTGEMM_ENOMEM: return "workspace allocation failed";
    case LUTGEMM_ECAPTURE:
        return "the stream is being captured and its workspace would have to grow "
               "(call lutgemm_reserve_workspace before capturing)";
    case LUTGEMM_ETIMEDOUT:
        return "a problem of a chained launch gave up waiting for a tagged row (nothing wrote it within the limit)";
    case LUTGEMM_ETOOBIG:
        return "M * N exceeds LUTGEMM_NOALLOC_MAX_WORDS, the fixed buffer of the entry point that does not allocate";
    default: return "unknown lutgemm error";
    }
}

int lutgemm_last_hip_error(void) { return g_last_hip_error; }

int lutgemm_set_timestamp_buffer(void *readings, size_t count)
{
#ifdef LUTGEMM_TIMESTAMPS
    if (!aligned(readings, 8) || (count > 0 && !readings)) return LUTGEMM_EINVAL;
    g_stamps.store((unsigned long long *)readings);
    g_stamp_slots.store((long long)count);
    return LUTGEMM_OK;
#else
    (void)readings;
    (void)count;
    return LUTGEMM_EUNSUP;   // this build of the library reads no clocks
#endif
}

int lutgemm_set_option(int which, int value)
{
    if (which < 0 || which >= LUTGEMM_OPTION_COUNT) return LUTGEMM_EINVAL;
    load_options();
    g_option[which].store(value < 0 ? env_int(kOptions[which].env, kOptions[which].fallback) : value);
    return LUTGEMM_OK;
}

int lutgemm_get_option(int which)
{
    if (which < 0 || which >= LUTGEMM_OPTION_COUNT) return LUTGEMM_EINVAL;
    return option(which);
}

int lutgemm_gemv_rowwise_f16(const uint32_t *bW, const void *alpha_f16, const void *x_f16,
                             void *out_f16, int N, int K, int nb, int num_groups, int M,
                             void *stream)
{
    return run(kRowF16, bW, alpha_f16, nullptr, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream});
}

int lutgemm_gemv_rowwise_pow2_f16(const uint32_t *bW, const void *alpha_f16, const void *x_f16,
                                  void *out_f16, int N, int K, int nb, int num_groups, int M,
                                  void *stream)
{
    return run(kRowF16, bW, alpha_f16, nullptr, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream}, true);
}

int lutgemm_gemv_rowwise_f16_noalloc(const uint32_t *bW, const void *alpha_f16, const void *x_f16,
                                     void *out_f16, int N, int K, int nb, int num_groups, int M,
                                     void *stream)
{
    if (N > 0 && M > 0 && (size_t)N * (size_t)M > (size_t)LUTGEMM_NOALLOC_MAX_WORDS) return LUTGEMM_ETOOBIG;
    // set-up on the first call on a device, whether or not this call needs the words
    unsigned long long *unused = nullptr;
    const int rc = scratch_address(&unused);
    if (rc != LUTGEMM_OK) return rc;
    return run(kRowF16, bW, alpha_f16, nullptr, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream, true});
}

int lutgemm_gemv_rowwise_f16_grouped(int count, const lutgemm_rowwise_problem *problems,
                                     void *stream_v)
{
    if (!problems || count < 1 || count > kMaxGroup) return LUTGEMM_EINVAL;
    lutgemm_fused_problem f[kMaxGroup] = {};
    for (int i = 0; i < count; ++i) {
        const lutgemm_rowwise_problem &q = problems[i];
        f[i].bW = q.bW;
        f[i].alpha_f16 = q.alpha_f16;
        f[i].x_f16 = q.x_f16;
        f[i].out_f16 = q.out_f16;
        f[i].N = q.N;
        f[i].K = q.K;
        f[i].nb = q.nb;
        f[i].num_groups = q.num_groups;
        f[i].M = q.M;
    }
    return run_group(count, f, Accum{(hipStream_t)stream_v});
}

int lutgemm_gemv_rowwise_f16_fused(int count, const lutgemm_fused_problem *problems, void *stream_v)
{
    if (!problems || count < 1 || count > kMaxGroup) return LUTGEMM_EINVAL;
    return run_group(count, problems, Accum{(hipStream_t)stream_v});
}

int lutgemm_describe_group_plan(int count, const lutgemm_fused_problem *problems, lutgemm_group_plan *plan)
{
    if (!problems || !plan || count < 1 || count > kMaxGroup) return LUTGEMM_EINVAL;
    GroupPlan group{};
    const int rc = plan_group(count, problems, nullptr, group);
    if (rc != LUTGEMM_OK) return rc;
    *plan = lutgemm_group_plan{};
    plan->kernel = group.one_mfma || group.each_mfma ? kMatrixCore : kLookup;
    plan->launches = group.each_mfma ? count : 1;
    if (group.one_mfma) {
        int most = 0;
        plan->needs_workspace = plan_mfma_group(group.g, group.g.p[0].M > 16 ? 2 : 1, &most);
    } else if (!group.each_mfma) {
        plan->needs_workspace = group.shares.any_split;
    }
    for (int i = 0; i < count; ++i) {
        Problem &p = group.g.p[i];
        if (group.each_mfma) {
            const MfmaPlan mfma = mfma_plan(p, false);
            plan_mfma(p, mfma.mt, mfma.slices);
            plan->needs_workspace |= p.ksplit > 1;
        }
        plan->workgroups[i] = p.n_blocks;
        plan->units_per_workgroup[i] = plan->kernel == kMatrixCore ? p.sets_per_split : p.items_per_wg;
    }
    return LUTGEMM_OK;
}

int lutgemm_gemv_rowwise_f16_gated(const lutgemm_fused_problem *gate_up, void *act_f16, void *stream)
{
    if (!gate_up || !act_f16) return LUTGEMM_EINVAL;
    const lutgemm_fused_problem &gate = gate_up[0], &up = gate_up[1];
    if (gate.M != up.M || gate.N != up.N || (long long)gate.M * gate.N % 8 != 0) return LUTGEMM_EINVAL;
    for (const lutgemm_fused_problem *p : {&gate, &up})
        if (p->overwrite != 1 || p->next_input_f16 || p->sumsq_out_f32) return LUTGEMM_EINVAL;
    if (!aligned(act_f16, 16) || !aligned(gate.out_f16, 16) || !aligned(up.out_f16, 16)) return LUTGEMM_EALIGN;
    Gated gated{(__half *)act_f16, false};
    const int rc = run_group(2, gate_up, Accum{(hipStream_t)stream}, &gated);
    if (rc != LUTGEMM_OK || gated.done) return rc;
    return lutgemm_decode_silu_mul_f16(gate.out_f16, up.out_f16, act_f16, (size_t)gate.M * gate.N, stream);
}

int lutgemm_gemv_rowwise_f16_chain(int count, const lutgemm_chain_problem *problems,
                                   const lutgemm_chain_control *control, void *stream_v)
{
    if (!problems || count < 1 || count > kMaxGroup) return LUTGEMM_EINVAL;
    return run_chain(count, problems, control, Accum{(hipStream_t)stream_v});
}

int lutgemm_describe_chain_plan(int count, const lutgemm_chain_problem *problems, int workgroups,
                                lutgemm_chain_plan *plan)
{
    if (!problems || !plan || count < 1 || count > kMaxGroup || workgroups < 0) return LUTGEMM_EINVAL;
    Chain c{};
    int depth[kMaxGroup], grid = 0;
    bool any_split = false;
    size_t words = 0;
    const int rc = plan_chain(count, problems, workgroups, c, depth, &grid, &any_split, &words);
    if (rc != LUTGEMM_OK) return rc;
    *plan = lutgemm_chain_plan{};
    plan->workgroups = grid;
    plan->units = c.unit_start[count];
    plan->needs_workspace = any_split;
    for (int i = 0; i < count; ++i) {
        plan->stage[i] = depth[i];
        plan->first_unit[i] = c.unit_start[i];
        plan->unit_count[i] = c.g.p[i].n_blocks;
        plan->items_per_unit[i] = c.g.p[i].items_per_wg;
    }
    return LUTGEMM_OK;
}

int lutgemm_chain_tag_rows(void *dst_tagged, const void *src_f16, size_t count, int tag, const uint32_t *epoch,
                           void *stream)
{
    if (!dst_tagged || !src_f16 || tag < 1 || tag > LUTGEMM_CHAIN_MAX_TAG) return LUTGEMM_EINVAL;
    if (!aligned(dst_tagged, 4) || !aligned(src_f16, 2) || !aligned(epoch, 4)) return LUTGEMM_EALIGN;
    if (count == 0) return LUTGEMM_OK;
    size_t blocks = (count + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(tag_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream, (uint32_t *)dst_tagged,
                       (const unsigned short *)src_f16, count, tag, epoch);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

int lutgemm_chain_untag_rows(void *dst_f16, const void *src_tagged, size_t count, void *stream)
{
    if (!dst_f16 || !src_tagged) return LUTGEMM_EINVAL;
    if (!aligned(dst_f16, 2) || !aligned(src_tagged, 4)) return LUTGEMM_EALIGN;
    if (count == 0) return LUTGEMM_OK;
    size_t blocks = (count + 255) / 256;
    if (blocks > 1024) blocks = 1024;
    hipLaunchKernelGGL(untag_rows_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (unsigned short *)dst_f16, (const uint32_t *)src_tagged, count);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

int lutgemm_chain_advance_epoch(uint32_t *epoch, uint32_t by, void *stream)
{
    if (!epoch) return LUTGEMM_EINVAL;
    if (!aligned(epoch, 4)) return LUTGEMM_EALIGN;
    hipLaunchKernelGGL(advance_epoch_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, epoch, by);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? LUTGEMM_OK : hip_fail(e);
}

int lutgemm_chain_status(const uint32_t *status, void *stream)
{
    if (!status) return LUTGEMM_EINVAL;
    uint32_t v = 0;
    hipError_t e = hipStreamSynchronize((hipStream_t)stream);
    if (e != hipSuccess) return hip_fail(e);
    e = hipMemcpy(&v, status, sizeof(v), hipMemcpyDeviceToHost);
    if (e != hipSuccess) return hip_fail(e);
    return v ? LUTGEMM_ETIMEDOUT : LUTGEMM_OK;
}

int lutgemm_gemv_uniform_f16(const uint32_t *bW, const void *alpha_f16, const void *qbias_f16,
                             const void *x_f16, void *out_f16, int N, int K, int nb,
                             int num_groups, int M, void *stream)
{
    return run(kUniformF16, bW, alpha_f16, qbias_f16, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream});
}

int lutgemm_gemv_block_f16(const uint32_t *bW, const void *alpha_f16, const void *x_f16,
                           void *out_f16, int N, int K, int nb, int num_groups, int M,
                           void *stream)
{
    return run(kBlockF16, bW, alpha_f16, nullptr, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream});
}

int lutgemm_gemv_block_shift_u16(const uint32_t *bW, const uint16_t *alpha_u16, const void *x_f16,
                                 void *out_f16, int N, int K, int nb, int num_groups,
                                 int num_apot, int M, void *stream)
{
    if (num_apot != 3) return LUTGEMM_EUNSUP;
    return run(kBlockShiftU16, bW, alpha_u16, nullptr, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream});
}

int lutgemm_gemv_block_apot_i8(const uint32_t *bW, const int8_t *alpha_i8, const void *x_f16,
                               void *out_f16, int N, int K, int nb, int num_groups, int num_apot,
                               int M, void *stream)
{
    if (num_apot != 3) return LUTGEMM_EUNSUP;
    return run(kBlockApotI8, bW, alpha_i8, nullptr, x_f16, out_f16, N, K, nb, num_groups, M,
               Accum{(hipStream_t)stream});
}

int lutgemm_linear_f16(const lutgemm_linear *layer, void *stream)
{
    if (!layer || layer->format < LUTGEMM_FORMAT_ROWWISE_F16 || layer->format > LUTGEMM_FORMAT_UNIFORM_F16) return LUTGEMM_EINVAL;
    const lutgemm_linear &c = *layer;
    if (c.x_type < kIoF16 || c.x_type > kIoF32 || c.out_type < kIoF16 || c.out_type > kIoF32) return LUTGEMM_EINVAL;
    if (c.out_type == kIoF32 && !aligned(c.out, 16)) return LUTGEMM_EALIGN;
    return run(c.format, c.bW, c.alpha, c.qbias_f16, c.x, c.out, c.N, c.K, c.nb, c.num_groups, c.M,
               Accum{(hipStream_t)stream}, c.alpha_pow2 != 0 && c.format == LUTGEMM_FORMAT_ROWWISE_F16, &c.bias_f16,
               c.x_type, c.out_type);
}

size_t lutgemm_algorithmic_bytes(int N, int K, int nb, int M, size_t alpha_entries,
                                 int alpha_bytes_per_entry)
{
    const size_t signs = (size_t)K / 8 * (size_t)N * (size_t)nb;
    const size_t alphas = alpha_entries * (size_t)alpha_bytes_per_entry;
    const size_t xin = 2u * (size_t)M * (size_t)K;
    const size_t yio = 2u * 2u * (size_t)M * (size_t)N;  // read (accumulate) + write
    return signs + alphas + xin + yio;
}

// The problem of a describe call, without operands (nothing is dereferenced while planning: any aligned
// non-null address will do).
static int fill_described(Problem &p, int format, int N, int K, int nb, int groups, int M)
{
    alignas(16) static const uint64_t dummy[2] = {0, 0};
    return fill_problem(p, format, (const uint32_t *)dummy, dummy, dummy, dummy, (void *)dummy, N, K, nb, groups, M);
}

int lutgemm_describe_plan(int format, int N, int K, int nb, int groups, int M, lutgemm_plan *plan)
{
    if (!plan || format < LUTGEMM_FORMAT_ROWWISE_F16 || format > LUTGEMM_FORMAT_UNIFORM_F16) return LUTGEMM_EINVAL;
    Problem p;
    int rc = fill_described(p, format, N, K, nb, groups, M);
    if (rc != LUTGEMM_OK) return rc;
    *plan = lutgemm_plan{};
    MfmaPlan planned;
    if (tile_wanted(p, format, &planned)) {
        TileProblem t{};
        t.N = N;
        t.M = M;
        t.kwords = p.kwords;
        plan_tile(t);
        plan->kernel = 3;
        plan->workgroups = t.n_tiles * t.m_tiles * t.ksplit;
        plan->rows_per_pass = t.tile_rows;
        plan->row_chunks = t.m_tiles;
        plan->tiles = t.n_tiles;
        plan->tile_columns = 256;
        plan->k_units = t.steps;
        plan->k_slices = t.ksplit;
        plan->units_per_slice = t.slice_steps;
        plan->ranges = t.pair ? 2 : 1;
        return LUTGEMM_OK;
    }
    int kernel = kLookup, mrows = 1;
    rc = plan_single(p, format, planned, &kernel, &mrows);
    if (rc != LUTGEMM_OK) return rc;
    plan->kernel = kernel;
    plan->workgroups = p.n_blocks;
    plan->rows_per_pass = mrows;
    plan->row_chunks = p.mchunks;
    plan->tiles = p.n_tiles;
    plan->k_units = p.nsets;
    if (kernel == kMatrixCore) {
        plan->tile_columns = kMfmaTileCols;
        plan->k_slices = p.ksplit;
        plan->units_per_slice = p.sets_per_split;
        plan->needs_workspace = p.ksplit > 1;
    } else {
        plan->tile_columns = p.twin ? 2 * kTileCols : kTileCols;
        plan->long_ranges = p.long_ranges;
        plan->items_per_long_range = p.items_per_wg;
        plan->items_per_short_range = p.short_items;
        plan->ranges = p.wgs_per_chunk;
        plan->needs_workspace = lookup_splits_k(p);
    }
    return LUTGEMM_OK;
}

int lutgemm_describe_pow2_plan(int N, int K, int nb, int groups, int M, lutgemm_plan *plan)
{
    if (!plan) return LUTGEMM_EINVAL;
    Problem p;
    const int rc = fill_described(p, kRowF16, N, K, nb, groups, M);
    if (rc != LUTGEMM_OK) return rc;
    if (!(mfma_eligible(p, kRowF16) && p.M >= mfma_min_rows() && mx_wanted(p)))
        return lutgemm_describe_plan(LUTGEMM_FORMAT_ROWWISE_F16, N, K, nb, groups, M, plan);
    plan_mx(p);
    *plan = lutgemm_plan{};
    plan->kernel = 2;
    plan->workgroups = p.n_blocks;
    plan->rows_per_pass = mx_chunk_rows(p.M);
    plan->row_chunks = p.mchunks;
    plan->tiles = p.n_tiles;
    plan->tile_columns = kMfmaTileCols;
    plan->k_units = p.nsets;
    plan->k_slices = p.ksplit;
    plan->units_per_slice = p.sets_per_split;
    plan->needs_workspace = p.ksplit > 1;
    return LUTGEMM_OK;
}

int lutgemm_describe_tile_plan(int format, int N, int K, int nb, int groups, int M, lutgemm_plan *plan)
{
    return lutgemm_describe_plan(format, N, K, nb, groups, M, plan);
}

size_t lutgemm_workspace_words(int N, int M)
{
    if (N <= 0 || M <= 0) return 0;
    return (size_t)N * (size_t)M;
}

int lutgemm_reserve_workspace(void *stream, size_t words)
{
    unsigned long long *unused = nullptr;
    const int rc = stream_workspace((hipStream_t)stream, words, &unused);
    if (rc != LUTGEMM_OK) return rc;
    // the sums of the GEMM kernel's K-slices: at most sixteen per output and what lies between them, 64 MB in all (plan_tile)
    void *sums = nullptr;
    return stream_split_buffer((hipStream_t)stream, words < (kTileSumBytes - kTileGapBytes) / 64 ? words * 64 + kTileGapBytes : kTileSumBytes, &sums);
}

int lutgemm_copy_bytes(void *dst, const void *src, size_t bytes, void *stream)
{
    if (!dst || !src || bytes % 16 != 0) return LUTGEMM_EINVAL;
    if (!aligned(dst, 16) || !aligned(src, 16)) return LUTGEMM_EALIGN;
    if (bytes == 0) return LUTGEMM_OK;
    const size_t n16 = bytes / 16;
    size_t blocks = (n16 + 255) / 256;
    if (blocks > 256 * 16) blocks = 256 * 16;
    hipLaunchKernelGGL(copy_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (u32x4 *)dst, (const u32x4 *)src, n16);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e);
    return LUTGEMM_OK;
}

int lutgemm_measure_stream_read(const void *src, size_t bytes, void *sink, void *stream)
{
    if (!src || bytes % 16 != 0) return LUTGEMM_EINVAL;
    if (!aligned(src, 16)) return LUTGEMM_EALIGN;
    if (bytes == 0) return LUTGEMM_OK;
    const size_t n16 = bytes / 16;
    size_t blocks = (n16 + 256 * 8 - 1) / (256 * 8);
    if (blocks > 2048) blocks = 2048;
    hipLaunchKernelGGL(stream_read_kernel, dim3((unsigned)blocks), dim3(256), 0, (hipStream_t)stream,
                       (const u32x4 *)src, n16, (uint32_t *)sink);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e);
    return LUTGEMM_OK;
}

int lutgemm_measure_empty_launch(int workgroups, void *stream)
{
    if (workgroups < 1 || workgroups > 65535) return LUTGEMM_EINVAL;
    hipLaunchKernelGGL(empty_kernel, dim3((unsigned)workgroups), dim3(kThreads), 0, (hipStream_t)stream,
                       (uint32_t *)nullptr);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return hip_fail(e);
    return LUTGEMM_OK;
}

int lutgemm_release_workspaces(void)
{
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return hip_fail(e);
    e = hipDeviceSynchronize();
    if (e != hipSuccess) return hip_fail(e);
    std::lock_guard<std::mutex> lock(g_ws_mutex);
    for (auto it = g_workspaces.begin(); it != g_workspaces.end();) {
        if (it->first.first == dev) {
            if (it->second.accum) (void)hipFree(it->second.accum);
            for (unsigned long long *old : it->second.retired) (void)hipFree(old);
            if (it->second.split) (void)hipFree(it->second.split);
            for (void *old : it->second.retired_split) (void)hipFree(old);
            it = g_workspaces.erase(it);
        } else {
            ++it;
        }
    }
    return LUTGEMM_OK;
}

}  // extern "C"
