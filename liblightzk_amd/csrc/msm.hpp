// MSM plan, batch descriptors and entry points shared by the C ABI, the
// batcher and the prover.
#pragma once
#include <cstddef>
#include <cstdint>
#include <hip/hip_runtime.h>

struct hzk_ctx;

namespace hzk {

constexpr int MSM_MIN_C = 4;
constexpr int MSM_MAX_C = 16;         // a caller's window sizes and the autotuner's
constexpr int MSM_PLAN_MAX_C = 17;    // tuned plans (msm_widen)

struct MsmPlan {
    int c;          // window bits
    int W;          // windows, ceil(255 / c)
    uint32_t NB;    // buckets per window, 2^(c-1)
    uint32_t K;     // sorted entries per accumulation lane (chunk length)
    uint32_t g;     // buckets per bucket-reduction run
    bool fit = false;   // a tuned plan (built in, autotuned or loaded): msm_fit_chunks may move K, msm_widen c
};
// Tuned plans from MSM_WIDE_N G1 points on take 17-bit windows, one more than a
// caller may ask for: 15 of them instead of 16 save that part of the
// accumulation and the sort, for twice the buckets: 2^23 points 10.89 -> 10.45
// ms, 2^24 20.83 -> 20.14, 7 million 9.11 -> 8.89; 2^22 and less gain under 1 %.
// From 2^25 points on, above the classes of the shipped table, plans are the
// heuristic's (16 bits) unless a tuned one is loaded.
constexpr size_t MSM_WIDE_N = (size_t)1 << 22;
inline void msm_widen(int g2, size_t n, MsmPlan& p) {
    if (!g2 && p.c == 16 && n >= MSM_WIDE_N) p.c = MSM_PLAN_MAX_C, p.W = 15, p.NB = 1u << 16;
}
// Plan for n points: autotuned entry for the size class if one is loaded,
// else the built-in heuristic; force_c / force_g override (0 = automatic).
MsmPlan msm_plan(size_t n, int force_c, int force_g);
// plan regimes: an MSM with the GPU to itself, or an instance of a wide
// batch: two or more instances whose digits total at least
// MSM_WIDE_BATCH_ENTRIES, or many instances (MSM_WIDE_BATCH_COUNT, G1 / G2)
// totalling MSM_WIDE_BATCH_MIN_ENTRIES (measured on served-like batches: a
// batch of 16 G1 or 16 G2 MSMs of mixed sizes already runs faster on the
// throughput plans, while the 4 G1 MSMs of one 2^18 proof do not)
constexpr int MSM_REGIME_SINGLE = 0, MSM_REGIME_BATCH = 1;
constexpr uint64_t MSM_WIDE_BATCH_ENTRIES = (uint64_t)1 << 26;
constexpr uint64_t MSM_WIDE_BATCH_MIN_ENTRIES = (uint64_t)1 << 24;
constexpr size_t MSM_WIDE_BATCH_COUNT[2] = {8, 16};
inline bool msm_wide_batch(int g2, size_t count, uint64_t entries) {
    if (count < 2) return false;
    return entries >= MSM_WIDE_BATCH_ENTRIES ||
           (count >= MSM_WIDE_BATCH_COUNT[g2 ? 1 : 0] && entries >= MSM_WIDE_BATCH_MIN_ENTRIES);
}
MsmPlan msm_plan_ctx(hzk_ctx* ctx, int g2, size_t n, int force_c, int regime = MSM_REGIME_SINGLE);
// the built-in plan of a regime (no context overrides)
MsmPlan msm_plan_builtin(int g2, size_t n, int regime);

// Work spaces of the batched stages; each instance owns a contiguous range
// [begin[s][i], begin[s][i+1]) of every space.
enum MsmSpace {
    SP_TILE = 0,    // one workgroup per tile of scalars (recode)
    SP_TILEWG,      // one workgroup per (tile, window) (coarse scatter)
    SP_CNT,         // W * CG * T + 1 coarse counts, then starts
    SP_SCANTILE,    // scan tiles over them
    SP_GROUP,       // W * CG + 1 coarse groups
    SP_SUB,         // pieces of MSM_SUB entries of a group (upper bound)
    SP_ROW,         // FB counters per piece
    SP_SMALL,       // one workgroup per window of a small instance
    SP_KEY,         // nk + 1 entries per instance (offsets, bucket sums)
    SP_CHUNK,       // accumulation chunks of K sorted entries (upper bound)
    SP_BRED,        // windows (two result points each)
    SP_WIN,         // window-sum partials (S per window)
    SP_ENTRY,       // n * W digit / sorted-entry slots
    SP_COUNT
};

// Device-side descriptor of one MSM instance of a batch.
struct MsmInst {
    const void* scalars;   // Fr[n], Montgomery
    const void* bases;     // affine points
    uint32_t n, c, W, NB, nk, K, g, G, T, tile;
    uint32_t S;            // window-sum workgroups per window
    // Level tables: nd scalars with Wd digit windows over a table of Lg levels
    // (point t*nd + i = 2^(c t) P_i, t < Lg); each bucket set ("window" of the
    // pipeline) serves Lg consecutive digit windows, so W = ceil(Wd / Lg) and
    // n = nd * Lg virtual points. Plain bases: nd = n, Wd = W, Lg = 1.
    uint32_t nd, Wd, Lg;
    uint32_t CG, FB;       // coarse groups per window, buckets per group (powers of two, CG * FB = NB)
    uint32_t small;        // 1: sorted by one workgroup per window (CG = 1)
    uint32_t ctile;        // tiles per coarse-scatter workgroup
    uint32_t ib;           // bits of a point index where it shares a coarse entry's word with the bucket, else 0
    // Digit window j covers bits [j*wb + min(j, wx), +wb + (j < wx)): the 255
    // bits of a signed recoding of a scalar < 2^254 split as evenly as the W
    // windows allow (widths c and c - 1), so the top window is not a sliver
    // of a few bits whose digits pile into a handful of buckets. Level tables
    // keep uniform windows of c bits (wb = c, wx = 0).
    uint32_t wb, wx;
    void* dest;            // the result (device), for the device-side combine
};

struct MsmBatchDev {
    const MsmInst* inst;      // [ninst]
    const uint64_t* begin;    // [SP_COUNT][ninst + 1]
    uint32_t ninst;
    uint32_t* stats;          // per instance {entries, chunks, largest bucket, 0}
};

// Limits of the two-level sort. Coarse groups: 256 keep the runs that a round
// of the coarse scatter writes at 128 bytes (512 only where that lets an entry
// fit one word); FB counters of a group times three and a round of the fine
// scatter share the LDS. A piece is two rounds.
constexpr uint32_t MSM_MAX_COARSE = 512, MSM_MAX_FINE = 2048;
constexpr uint32_t MSM_MAX_GROUPS = 8192;   // W * CG counters of the recode
constexpr uint32_t MSM_SUB = 16384;
static_assert((1u << (MSM_PLAN_MAX_C - 1)) <= MSM_MAX_COARSE * MSM_MAX_FINE, "a window's buckets fit the two levels");
// Small instances take one workgroup per window instead of the two levels'
// seven launches: up to 2^15 points, or 2^17 in a wide batch, whose windows
// fill the GPU together
constexpr uint32_t MSM_SMALL_N = 1u << 15, MSM_SMALL_BATCH_N = 1u << 17, MSM_SMALL_NB = 1u << 13;
inline uint32_t msm_log2_ceil(uint64_t n) {
    uint32_t k = 0;
    while (((uint64_t)1 << k) < n) ++k;
    return k;
}
// point index, bucket of the group and sign in one 32-bit word
inline bool msm_packs(uint64_t n, uint32_t FB) { return msm_log2_ceil(n) + msm_log2_ceil(FB) <= 31; }
// coarse groups per window: about 4096 entries each, within the limits
inline uint32_t msm_coarse_groups(uint64_t n, uint32_t NB, uint32_t W) {
    uint32_t cg = 1;
    while (cg < 256 && cg < NB && n / cg > 4096 && W * cg * 2 <= MSM_MAX_GROUPS) cg *= 2;
    while (NB / cg > MSM_MAX_FINE) cg *= 2;
    while (cg < MSM_MAX_COARSE && cg < NB && !msm_packs(n, NB / cg) && W * cg * 2 <= MSM_MAX_GROUPS) cg *= 2;
    return cg;
}
// tiles of scalars: about 256 each, at most 512 of them (their counts are scanned)
inline uint32_t msm_tiles(uint64_t nd) {
    const uint64_t t = (nd + 255) / 256;
    return (uint32_t)(t < 512 ? t : 512);
}

// Launch the scalar-side stages (recode, scans, scatters) for a whole batch.
// Buffers are indexed through the work spaces above.
struct MsmScalarBufs {
    uint32_t* digits;    // SP_ENTRY
    uint32_t* count;     // SP_CNT
    uint64_t* tiles;     // SP_SCANTILE
    uint32_t* sub;       // SP_GROUP
    uint32_t* rows;      // SP_ROW
    uint32_t* cidx;      // SP_ENTRY coarse entries: point index and sign
    uint16_t* ckey;      // SP_ENTRY: bucket within the group
    uint32_t* offs;      // SP_KEY
    uint32_t* sorted;    // SP_ENTRY
};
// largest of the batch, for the launches' LDS
struct MsmSortMax { uint32_t groups = 1, fine = 1, small_nb = 1, tile = 1; };
void msm_launch_scalar_stages(hzk_ctx* ctx, const MsmBatchDev& b, const uint64_t* host_totals, const MsmSortMax& mx,
                              const MsmScalarBufs& bufs);
constexpr uint32_t MSM_SCAN_TILE = 1024;
// one-time kernel attribute setup (call outside graph capture)
void msm_prepare();

// levels != 0: bases is a level table (see MsmJob)
int msm_g1(hzk_ctx* ctx, const void* scalars, const void* bases, size_t n, size_t win_siz, void* dest, uint32_t levels = 0);
int msm_g2(hzk_ctx* ctx, const void* scalars, const void* bases, size_t n, size_t win_siz, void* dest, uint32_t levels = 0);

// Batched MSM: out[i] (device or host pointer per dests_on_host) receives the
// normalised Jacobian result of instance i. capture != 0 records the device
// stages into a hipGraph on first use of this batch shape and replays it.
struct MsmJob {
    const void* scalars;
    const void* bases;
    size_t n;
    void* dest;
    uint32_t win_siz;
    uint32_t levels;   // 0 or 1: affine bases; else levels per bucket set of a level table (<= ceil(255 / win_siz))
    uint32_t form = 0; // 0 affine bases, 1 bases already converted by msm_convert_g1 / _g2 (kept by the prover)
};
// device_combine: the window combine runs as a kernel into device dests and
// the call returns without waiting (HZK_BATCH_DEVICE_COMBINE)
int msm_batch_g1(hzk_ctx* ctx, const MsmJob* jobs, size_t count, int dests_on_host, int capture, int device_combine = 0);
// G1 affine bases -> the form the G1 bucket accumulation reads (field29.hpp's
// 2^261 Montgomery coordinates, infinity marked), n points, on ctx's stream;
// dst may equal src
int msm_convert_g1(hzk_ctx* ctx, const void* src, void* dst, size_t n);
// the same for G2 affine bases (128 bytes each)
int msm_convert_g2(hzk_ctx* ctx, const void* src, void* dst, size_t n);
int msm_batch_g2(hzk_ctx* ctx, const MsmJob* jobs, size_t count, int dests_on_host, int capture, int device_combine = 0);

}  // namespace hzk
