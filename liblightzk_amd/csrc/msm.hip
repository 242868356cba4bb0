// Pippenger multi-scalar multiplication for alt_bn128 G1 and G2 on gfx950:
// scalar-side stages, batched over any number of MSM instances.
//
// Replaces the reference's operator (include/operator/msm.cuh:77-248: one
// counting sort of n*win_cnt (bucket, point) pairs into 2^c buckets with
// global atomics and a serial <<<1,1>>> scan, one 32-lane warp per bucket,
// fixed <<<128,1024>>> geometry valid only for c = 12) with a two-level
// counting sort per window (coarse groups of FB = NB / CG consecutive buckets,
// then the buckets of each group):
//
//  1. recode   one lane per scalar: leave Montgomery form, signed c-bit digits
//              d_j in [-2^(c-1), 2^(c-1)] over W = ceil(255/c) windows (the
//              top window cannot carry because scalars are < r < 2^254),
//              written window-major; digit 0 is dropped (the reference
//              accumulates bucket 0 and scales it by 0, msm.cuh:121-161). The
//              workgroup counts its tile's digits by (window, coarse group) in
//              LDS on the way.
//  2. scan     exclusive scan of those counts in (window, group, tile) order:
//              where every tile's entries of a group start; per group the
//              pieces of MSM_SUB entries that the fine level works on.
//  3. coarse scatter  workgroup per (tile, window): entries to their group,
//              counting-sorted in LDS first so that consecutive lanes write
//              consecutive addresses.
//  4. fine level  workgroup per piece counts its entries by bucket, workgroup
//              per group turns the counts into bucket offsets, workgroup per
//              piece scatters. A group that one digit value fills (the ones of
//              a witness) is many pieces, so no workgroup has more to do than
//              the others; a histogram over all buckets of a window is never
//              needed, so a window may have more buckets than LDS has counters.
//  1'-4'. instances of at most MSM_SMALL_N points with few buckets: the recode,
//              then one workgroup per window sorts it whole in LDS.
//  5-8 (msm_impl.hpp) chunked accumulation with boundary fix-up, bucket
//              reduction, window sums;
//  9. window combine on the host (Horner with c doublings per window) and
//              normalisation; see host_ec.hpp for why this tail runs on the CPU.
//
// Per-instance totals (entries, chunks, largest bucket) land in device stats,
// so no stage waits for the host. No device-scope atomics per entry: on a
// multi-XCD part they resolve past the per-XCD L2 and ran at ~5 G/s.
//
// Every stage is one launch over the whole batch: each instance owns a
// contiguous range of every work space (MsmSpace), and a lane finds its
// instance by binary search over the range starts. A single MSM is a batch of
// one; a batch of uneven sizes fills the GPU where one small MSM cannot.
#include <algorithm>
#include <cstring>
#include <mutex>
#include "common.hpp"
#include "curve.hpp"
#include "msm.hpp"

namespace hzk {

static constexpr uint32_t DIGIT_NEG = 0x80000000u;
static constexpr int SCAN_ITEMS = 4;
static constexpr int SCAN_THREADS = 256;
static_assert(SCAN_ITEMS * SCAN_THREADS == MSM_SCAN_TILE, "scan tile");

// largest i < ninst with beg[i] <= gid (beg[0] = 0 <= gid < beg[ninst])
HZK_DEV uint32_t find_inst(const uint64_t* __restrict__ beg, uint32_t ninst, uint64_t gid) {
    uint32_t lo = 0, hi = ninst;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (beg[mid] <= gid) lo = mid; else hi = mid;
    }
    return lo;
}
HZK_DEV const uint64_t* space(const MsmBatchDev& b, int s) { return b.begin + (size_t)s * (b.ninst + 1); }

// exclusive scan of n LDS counters by a workgroup of T threads; returns the total
template <int T>
HZK_DEV uint32_t lds_exclusive_scan(const uint32_t* cnt, uint32_t* out, uint32_t* part, uint32_t n) {
    const uint32_t t = threadIdx.x, per = (n + T - 1) / T, lo = min(n, t * per), hi = min(n, lo + per);
    uint32_t s = 0;
    for (uint32_t i = lo; i < hi; ++i) s += cnt[i];
    // inclusive scan of the threads' sums: in the wave, then over the waves
    uint32_t x = s;
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if ((t & 63) >= off) x += y;
    }
    if ((t & 63) == 63) part[t >> 6] = x;
    __syncthreads();
    uint32_t run = x - s, total = 0;
    for (uint32_t w = 0; w < T / 64; ++w) {
        if (w < (t >> 6)) run += part[w];
        total += part[w];
    }
    for (uint32_t i = lo; i < hi; ++i) {
        const uint32_t v = cnt[i];
        out[i] = run;
        run += v;
    }
    __syncthreads();
    return total;
}

// ------------------------------------------------------------------ 1. digits
// digits[j * n + i] = |d_ij| | sign << 31, or 0 for a zero digit. For a level
// table of Lg levels the same array is, window by window of the pipeline, the
// digits of Lg consecutive digit windows over nd * Lg virtual points
// 2^(c (j mod Lg)) P_i, so Lg digit windows share one bucket set.
// Workgroup per tile of scalars; its counts by (bucket set, coarse group) go
// to count[(set * CG + group) * T + tile].
// 1024 threads, or 256 where every tile of the launch is small (more
// workgroups for a small MSM).
__global__ void __launch_bounds__(1024) k_msm_digits(MsmBatchDev b, uint32_t* __restrict__ digits, uint32_t* __restrict__ count) {
    extern __shared__ uint32_t cnt[];
    const uint64_t* beg = space(b, SP_TILE);
    const uint32_t ii = find_inst(beg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    // the instance's fields in registers: stores could alias them
    const uint32_t t = (uint32_t)(blockIdx.x - beg[ii]), CG = d.CG, groups = d.W * CG, fshift = __ffs(d.FB) - 1;
    const uint32_t nd = d.nd, Lg = d.Lg, Wd = d.Wd, windows = d.W * Lg, wb = d.wb, wx = d.wx;
    const fr_t* scalars = (const fr_t*)d.scalars;
    uint32_t* const dig = digits + space(b, SP_ENTRY)[ii];
    for (uint32_t x = threadIdx.x; x < groups; x += blockDim.x) cnt[x] = 0;
    if (t == 0 && threadIdx.x < 4) b.stats[4 * ii + threadIdx.x] = 0;
    __syncthreads();
    const uint32_t i1 = min(nd, (t + 1) * d.tile);
    for (uint32_t idx = t * d.tile + threadIdx.x; idx < i1; idx += blockDim.x) {
        fr_t s = scalars[idx].from_mont();
        uint32_t carry = 0;
        uint32_t* out = dig + idx;
        // window j: the next wj bits, wj = wb + 1 for j < wx, then wb (<= c);
        // digits in [-2^(wj-1), 2^(wj-1)]. The scalar is shifted down in
        // registers (words in LDS and two loads a window took 1.8 times as long)
        uint32_t wj = wb + (wx ? 1u : 0u), level = 0, set = 0;
        uint32_t half = 1u << (wj - 1), mask = (1u << wj) - 1;
        for (uint32_t j = 0; j < windows; ++j) {   // level tables: windows past Wd pad the last set
            uint32_t dg = 0;
            if (j == wx && wx) {
                wj = wb;
                half = 1u << (wj - 1);
                mask = (1u << wj) - 1;
            }
            if (j < Wd) {
                const uint32_t raw = (s.l[0] & mask) + carry;
#pragma unroll
                for (int w = 0; w < 7; ++w) s.l[w] = __builtin_amdgcn_alignbit(s.l[w + 1], s.l[w], wj);
                s.l[7] >>= wj;
                if (raw > half) { carry = 1; dg = (2 * half - raw) | DIGIT_NEG; }
                else { carry = 0; dg = raw; }
                const uint32_t m = dg & ~DIGIT_NEG;
                if (!m) dg = 0;
                if (CG > 1) {
                    if (m) atomicAdd(&cnt[set * CG + ((m - 1) >> fshift)], 1u);
                } else {   // one counter per set: one addition per wave
                    const uint64_t some = __ballot(m != 0);
                    if (some && (threadIdx.x & 63) == (uint32_t)__builtin_ctzll(__ballot(1))) atomicAdd(&cnt[set], (uint32_t)__popcll(some));
                }
            }
            out[(size_t)j * nd] = dg;   // window j of scalar idx (level tables: set j / Lg, point (j % Lg) nd + idx)
            if (++level == Lg) level = 0, ++set;
        }
    }
    __syncthreads();
    uint32_t* row = count + space(b, SP_CNT)[ii] + t;
    for (uint32_t x = threadIdx.x; x < groups; x += blockDim.x) row[(size_t)x * d.T] = cnt[x];
}

// ------------------------------------------------------------------ 2. scans
// exclusive scan, in place, of an instance's W * CG * T counts (and one more
// place for the total). One block per scan tile: tile sum
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_tiles(MsmBatchDev b, const uint32_t* __restrict__ count, uint64_t* __restrict__ tile_sum) {
    __shared__ uint64_t red[SCAN_THREADS];
    const uint64_t* tbeg = space(b, SP_SCANTILE);
    uint32_t ii = find_inst(tbeg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint64_t kbase = space(b, SP_CNT)[ii];
    const uint32_t n = d.W * d.CG * d.T, base = (uint32_t)(blockIdx.x - tbeg[ii]) * MSM_SCAN_TILE;
    uint64_t s = 0;
    for (int t = 0; t < SCAN_ITEMS; ++t) {
        uint32_t k = base + threadIdx.x + t * SCAN_THREADS;
        if (k < n) s += count[kbase + k];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    for (int off = SCAN_THREADS / 2; off > 0; off >>= 1) {
        if ((int)threadIdx.x < off) red[threadIdx.x] += red[threadIdx.x + off];
        __syncthreads();
    }
    if (threadIdx.x == 0) tile_sum[blockIdx.x] = red[0];
}

// one block per instance: exclusive scan of its tile sums
__global__ void __launch_bounds__(1024) k_scan_top(MsmBatchDev b, uint64_t* __restrict__ tile_sum) {
    __shared__ uint64_t part[1024];
    const uint64_t* tbeg = space(b, SP_SCANTILE);
    const uint32_t ii = blockIdx.x;
    const uint64_t t0 = tbeg[ii];
    const uint32_t ntiles = (uint32_t)(tbeg[ii + 1] - t0);
    if (ntiles == 0) return;
    uint32_t per = (ntiles + 1023) / 1024;
    uint32_t lo = min(ntiles, threadIdx.x * per), hi = min(ntiles, lo + per);
    uint64_t s = 0;
    for (uint32_t i = lo; i < hi; ++i) s += tile_sum[t0 + i];
    part[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < 1024; off <<= 1) {
        uint64_t v = (int)threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += v;
        __syncthreads();
    }
    uint64_t run = threadIdx.x ? part[threadIdx.x - 1] : 0;
    for (uint32_t i = lo; i < hi; ++i) { uint64_t v = tile_sum[t0 + i]; tile_sum[t0 + i] = run; run += v; }
}

// per tile: exclusive scan in place; place n takes the total
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_apply(MsmBatchDev b, uint32_t* __restrict__ count, const uint64_t* __restrict__ tile_sum) {
    __shared__ uint64_t part[SCAN_THREADS];
    const uint64_t* tbeg = space(b, SP_SCANTILE);
    uint32_t ii = find_inst(tbeg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint64_t kbase = space(b, SP_CNT)[ii];
    const uint32_t n = d.W * d.CG * d.T;
    const uint32_t base = (uint32_t)(blockIdx.x - tbeg[ii]) * MSM_SCAN_TILE + threadIdx.x * SCAN_ITEMS;
    uint64_t v[SCAN_ITEMS];
    uint64_t s = 0;
    for (int t = 0; t < SCAN_ITEMS; ++t) {
        uint32_t k = base + t;
        v[t] = k < n ? count[kbase + k] : 0;
        s += v[t];
    }
    part[threadIdx.x] = s;
    __syncthreads();
    for (int off = 1; off < SCAN_THREADS; off <<= 1) {
        uint64_t x = (int)threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += x;
        __syncthreads();
    }
    uint64_t run = tile_sum[blockIdx.x] + (threadIdx.x ? part[threadIdx.x - 1] : 0);
    for (int t = 0; t < SCAN_ITEMS; ++t) {
        uint32_t k = base + t;
        if (k <= n) count[kbase + k] = (uint32_t)run;
        run += v[t];
    }
}

// one block per instance: pieces of each group, sub[g] = pieces before group
// g, sub[W CG] = all; entry totals to stats
__global__ void __launch_bounds__(1024) k_msm_pieces(MsmBatchDev b, const uint32_t* __restrict__ start, uint32_t* __restrict__ sub,
                                                     uint32_t* __restrict__ offs) {
    __shared__ uint32_t part[16];
    const uint32_t ii = blockIdx.x;
    const MsmInst& d = b.inst[ii];
    if (d.small) return;
    const uint32_t groups = d.W * d.CG, per = (groups + 1023) / 1024, t = threadIdx.x;
    const uint32_t* st = start + space(b, SP_CNT)[ii];
    uint32_t* out = sub + space(b, SP_GROUP)[ii];
    const uint32_t lo = min(groups, t * per), hi = min(groups, lo + per);
    auto pieces = [&](uint32_t g) { return (st[(size_t)(g + 1) * d.T] - st[(size_t)g * d.T] + MSM_SUB - 1) / MSM_SUB; };
    uint32_t s = 0;
    for (uint32_t g = lo; g < hi; ++g) s += pieces(g);
    uint32_t x = s;
    for (uint32_t off = 1; off < 64; off <<= 1) {
        const uint32_t y = __shfl_up(x, off, 64);
        if ((t & 63) >= off) x += y;
    }
    if ((t & 63) == 63) part[t >> 6] = x;
    __syncthreads();
    uint32_t run = x - s;
    for (uint32_t w = 0; w < (t >> 6); ++w) run += part[w];
    for (uint32_t g = lo; g < hi; ++g) {
        out[g] = run;
        run += pieces(g);
    }
    if (t == 1023) {
        out[groups] = run;
        const uint32_t entries = st[(size_t)groups * d.T];
        b.stats[4 * ii + 0] = entries;
        b.stats[4 * ii + 1] = (entries + d.K - 1) / d.K;
        offs[space(b, SP_KEY)[ii] + d.nk] = entries;
    }
}

// ------------------------------------------------------------------ 3. coarse scatter
// A round of SC_ROUND entries is counting-sorted in LDS first, so consecutive
// lanes write consecutive addresses of one group. 8192-entry rounds give a
// group of 256 about 32 entries (128 B) per round; 4096 left half-filled lines
// (both levels of a 2^24 MSM 2.18 ms with 4096, 1.84 ms with 8192, slower again
// with 16384 and its single workgroup per CU). An entry is its point index
// (sign in bit 31) and its bucket within the group.
static constexpr uint32_t SC_ROUND = 8192;
static constexpr uint32_t SC_THREADS = 1024;
static constexpr uint32_t SC_PER = SC_ROUND / SC_THREADS;
static constexpr uint32_t SC_NONE = 0xffffffffu;

__global__ void __launch_bounds__(SC_THREADS) k_msm_scatter_coarse(MsmBatchDev b, const uint32_t* __restrict__ digits,
                                                                   const uint32_t* __restrict__ start, uint32_t* __restrict__ cidx,
                                                                   uint16_t* __restrict__ ckey) {
    __shared__ uint32_t cur[MSM_MAX_COARSE], cnt[MSM_MAX_COARSE], lstart[MSM_MAX_COARSE], part[SC_THREADS / 64];
    __shared__ uint32_t stage[SC_ROUND], skey[SC_ROUND];
    const uint64_t* beg = space(b, SP_TILEWG);
    const uint32_t ii = find_inst(beg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t local = (uint32_t)(blockIdx.x - beg[ii]);
    // the instance's fields in registers: stores could alias them
    const uint32_t T = d.T, ctile = d.ctile, CG = d.CG, fmask = d.FB - 1, fshift = __ffs(d.FB) - 1, ib = d.ib, nd = d.nd, Lg = d.Lg, n = d.n;
    const uint32_t per = (T + ctile - 1) / ctile;   // workgroups per window, ctile tiles each
    const uint32_t t = (local % per) * ctile, j = local / per;
    const uint32_t tid = threadIdx.x;
    const uint32_t* st = start + space(b, SP_CNT)[ii] + (size_t)j * CG * T + t;
    for (uint32_t h = tid; h < CG; h += SC_THREADS) cur[h] = st[(size_t)h * T];
    const uint32_t i0 = min(nd, t * d.tile), i1 = min(nd, i0 + ctile * d.tile);
    const uint64_t ebase = space(b, SP_ENTRY)[ii];
    uint32_t* oi = cidx + ebase;
    uint16_t* ok = ckey + ebase;
    for (uint32_t level = 0; level < Lg; ++level) {
        const uint32_t first = level * nd;
        const uint32_t* dj = digits + ebase + (size_t)j * n + first;
        for (uint32_t base = i0; base < i1; base += SC_ROUND) {
            for (uint32_t h = tid; h < CG; h += SC_THREADS) cnt[h] = 0;
            __syncthreads();
            uint32_t dg[SC_PER], key[SC_PER], rank[SC_PER];
#pragma unroll
            for (uint32_t k = 0; k < SC_PER; ++k) {   // all loads before the first use
                const uint32_t i = base + tid + k * SC_THREADS;
                dg[k] = i < i1 ? dj[i] : 0;
            }
#pragma unroll
            for (uint32_t k = 0; k < SC_PER; ++k) {
                key[k] = (dg[k] & ~DIGIT_NEG) - 1;
                rank[k] = dg[k] ? atomicAdd(&cnt[key[k] >> fshift], 1u) : SC_NONE;
            }
            __syncthreads();
            const uint32_t total = lds_exclusive_scan<SC_THREADS>(cnt, lstart, part, CG);
#pragma unroll
            for (uint32_t k = 0; k < SC_PER; ++k) {
                if (rank[k] == SC_NONE) continue;
                const uint32_t p = lstart[key[k] >> fshift] + rank[k];
                const uint32_t val = (first + base + tid + k * SC_THREADS) | (dg[k] & DIGIT_NEG);
                stage[p] = ib ? val | ((key[k] & fmask) << ib) : val;
                skey[p] = key[k];
            }
            __syncthreads();
            for (uint32_t p = tid; p < total; p += SC_THREADS) {
                const uint32_t key2 = skey[p], h = key2 >> fshift, to = cur[h] + (p - lstart[h]);
                oi[to] = stage[p];
                if (!ib) ok[to] = (uint16_t)(key2 & fmask);
            }
            __syncthreads();
            for (uint32_t h = tid; h < CG; h += SC_THREADS) cur[h] += cnt[h];
            __syncthreads();
        }
    }
}

// ------------------------------------------------------------------ 4. fine level
struct MsmPiece { uint32_t group, e0, e1; };   // entries [e0, e1) of a group
// the piece of an instance's local piece number, or group = UINT32_MAX past the last
HZK_DEV MsmPiece find_piece(const MsmInst& d, const uint32_t* __restrict__ sub, const uint32_t* __restrict__ start, uint32_t local) {
    uint32_t lo = 0, hi = d.W * d.CG;
    if (local >= sub[hi]) return {UINT32_MAX, 0, 0};
    while (hi - lo > 1) {   // sub[lo] <= local < sub[hi]; empty groups are skipped by taking the last such lo
        const uint32_t mid = (lo + hi) >> 1;
        if (sub[mid] <= local) lo = mid; else hi = mid;
    }
    const uint32_t g0 = start[(size_t)lo * d.T], g1 = start[(size_t)(lo + 1) * d.T], e0 = g0 + (local - sub[lo]) * MSM_SUB;
    return {lo, e0, min(g1, e0 + MSM_SUB)};
}

// workgroup per piece: counts by bucket of the group
__global__ void __launch_bounds__(512) k_msm_fine_count(MsmBatchDev b, const uint32_t* __restrict__ start, const uint32_t* __restrict__ sub,
                                                        const uint32_t* __restrict__ cidx, const uint16_t* __restrict__ ckey,
                                                        uint32_t* __restrict__ rows) {
    extern __shared__ uint32_t dyn[];
    const uint64_t* beg = space(b, SP_SUB);
    const uint32_t ii = find_inst(beg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t local = (uint32_t)(blockIdx.x - beg[ii]);
    const MsmPiece p = find_piece(d, sub + space(b, SP_GROUP)[ii], start + space(b, SP_CNT)[ii], local);
    if (p.group == UINT32_MAX) return;
    for (uint32_t f = threadIdx.x; f < d.FB; f += 512) dyn[f] = 0;
    __syncthreads();
    const uint64_t ebase = space(b, SP_ENTRY)[ii];   // a multiple of 64 entries
    const uint32_t ib = d.ib, fmask = d.FB - 1;
    if (ib) {
        // 16-byte loads over the aligned middle, single entries at the ends
        const uint32_t* in = cidx + ebase;
        auto count = [&](uint32_t w) { atomicAdd(&dyn[(w >> ib) & fmask], 1u); };
        const uint32_t ea = min(p.e1, (p.e0 + 3) & ~3u), nv = (p.e1 - ea) / 4, eb = ea + 4 * nv;
        if (p.e0 + threadIdx.x < ea) count(in[p.e0 + threadIdx.x]);
        if (eb + threadIdx.x < p.e1) count(in[eb + threadIdx.x]);
        const uint4* in4 = (const uint4*)(in + ea);
        for (uint32_t q = threadIdx.x; q < nv; q += 512) {
            const uint4 w = in4[q];
            count(w.x);
            count(w.y);
            count(w.z);
            count(w.w);
        }
    } else {
        const uint16_t* key = ckey + ebase;
        for (uint32_t e = p.e0 + threadIdx.x; e < p.e1; e += 512) atomicAdd(&dyn[key[e]], 1u);
    }
    __syncthreads();
    uint32_t* row = rows + space(b, SP_ROW)[ii] + (size_t)local * d.FB;
    for (uint32_t f = threadIdx.x; f < d.FB; f += 512) row[f] = dyn[f];
}

// workgroup per group: bucket offsets; the pieces' counts become where each
// piece's entries of a bucket start
__global__ void __launch_bounds__(256) k_msm_fine_offsets(MsmBatchDev b, const uint32_t* __restrict__ start, const uint32_t* __restrict__ sub,
                                                          uint32_t* __restrict__ rows, uint32_t* __restrict__ offs) {
    extern __shared__ uint32_t dyn[];   // FB totals, FB starts
    __shared__ uint32_t part[4], mx;
    const uint64_t* beg = space(b, SP_GROUP);
    const uint32_t ii = find_inst(beg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t g = (uint32_t)(blockIdx.x - beg[ii]);
    if (d.small || g >= d.W * d.CG) return;
    const uint32_t* su = sub + beg[ii];
    const uint32_t s0 = su[g], s1 = su[g + 1], g0 = start[space(b, SP_CNT)[ii] + (size_t)g * d.T];
    uint32_t* row = rows + space(b, SP_ROW)[ii];
    uint32_t *tot = dyn, *at = dyn + d.FB;
    uint32_t largest = 0;
    if (threadIdx.x == 0) mx = 0;
    for (uint32_t f = threadIdx.x; f < d.FB; f += 256) {
        uint32_t s = 0;
        for (uint32_t q = s0; q < s1; ++q) s += row[(size_t)q * d.FB + f];
        tot[f] = s;
        largest = max(largest, s);
    }
    __syncthreads();
    lds_exclusive_scan<256>(tot, at, part, d.FB);
    atomicMax(&mx, largest);
    uint32_t* of = offs + space(b, SP_KEY)[ii] + (size_t)g * d.FB;   // g = window * CG + group
    for (uint32_t f = threadIdx.x; f < d.FB; f += 256) {
        uint32_t run = g0 + at[f];
        of[f] = run;
        for (uint32_t q = s0; q < s1; ++q) {
            const uint32_t v = row[(size_t)q * d.FB + f];
            row[(size_t)q * d.FB + f] = run;
            run += v;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0 && mx) atomicMax(&b.stats[4 * ii + 2], mx);
}

// workgroup per piece: entries to their bucket, staged in LDS as in the coarse scatter
__global__ void __launch_bounds__(SC_THREADS) k_msm_scatter_fine(MsmBatchDev b, const uint32_t* __restrict__ start,
                                                                 const uint32_t* __restrict__ sub, const uint32_t* __restrict__ rows,
                                                                 const uint32_t* __restrict__ cidx, const uint16_t* __restrict__ ckey,
                                                                 uint32_t* __restrict__ sorted) {
    extern __shared__ uint32_t dyn[];   // per bucket of the group: cursor, count, start in the round
    __shared__ uint32_t stage[SC_ROUND], part[SC_THREADS / 64];
    __shared__ uint16_t skey[SC_ROUND];
    const uint64_t* beg = space(b, SP_SUB);
    const uint32_t ii = find_inst(beg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t local = (uint32_t)(blockIdx.x - beg[ii]);
    const MsmPiece pc = find_piece(d, sub + space(b, SP_GROUP)[ii], start + space(b, SP_CNT)[ii], local);
    if (pc.group == UINT32_MAX) return;
    const uint32_t FB = d.FB, ib = d.ib, tid = threadIdx.x;
    uint32_t *cur = dyn, *cnt = dyn + FB, *lstart = dyn + 2 * FB;
    const uint32_t* row = rows + space(b, SP_ROW)[ii] + (size_t)local * FB;
    for (uint32_t f = tid; f < FB; f += SC_THREADS) cur[f] = row[f];
    const uint64_t ebase = space(b, SP_ENTRY)[ii];
    const uint32_t* in = cidx + ebase;
    const uint16_t* ik = ckey + ebase;
    uint32_t* out = sorted + ebase;
    for (uint32_t base = pc.e0; base < pc.e1; base += SC_ROUND) {
        for (uint32_t f = tid; f < FB; f += SC_THREADS) cnt[f] = 0;
        __syncthreads();
        uint32_t v[SC_PER], key[SC_PER], rank[SC_PER];
        const uint32_t e0 = base + tid, e1 = pc.e1;
#pragma unroll
        for (uint32_t k = 0; k < SC_PER; ++k) v[k] = e0 + k * SC_THREADS < e1 ? in[e0 + k * SC_THREADS] : 0;   // all loads before the first use
        if (ib) {
#pragma unroll
            for (uint32_t k = 0; k < SC_PER; ++k) {
                key[k] = (v[k] >> ib) & (FB - 1);
                v[k] &= 0x80000000u | ((1u << ib) - 1);
            }
        } else {
#pragma unroll
            for (uint32_t k = 0; k < SC_PER; ++k) key[k] = e0 + k * SC_THREADS < e1 ? ik[e0 + k * SC_THREADS] : 0;
        }
#pragma unroll
        for (uint32_t k = 0; k < SC_PER; ++k) rank[k] = e0 + k * SC_THREADS < e1 ? atomicAdd(&cnt[key[k]], 1u) : SC_NONE;
        __syncthreads();
        const uint32_t total = lds_exclusive_scan<SC_THREADS>(cnt, lstart, part, FB);
#pragma unroll
        for (uint32_t k = 0; k < SC_PER; ++k) {
            if (rank[k] == SC_NONE) continue;
            const uint32_t p = lstart[key[k]] + rank[k];
            stage[p] = v[k];
            skey[p] = (uint16_t)key[k];
        }
        __syncthreads();
        for (uint32_t p = tid; p < total; p += SC_THREADS) {
            const uint32_t f = skey[p];
            out[cur[f] + (p - lstart[f])] = stage[p];
        }
        __syncthreads();
        for (uint32_t f = tid; f < FB; f += SC_THREADS) cur[f] += cnt[f];
        __syncthreads();
    }
}

// ------------------------------------------------------------------ 4'. small instances
// workgroup per bucket set: counts, offsets and order in LDS; count holds the
// recode's entries per (set, tile)
__global__ void __launch_bounds__(1024) k_msm_sort_small(MsmBatchDev b, const uint32_t* __restrict__ digits, const uint32_t* __restrict__ count,
                                                         uint32_t* __restrict__ offs, uint32_t* __restrict__ sorted) {
    extern __shared__ uint32_t dyn[];   // NB counts, NB cursors
    __shared__ uint32_t part[16], before, all, mx;
    const uint64_t* beg = space(b, SP_SMALL);
    const uint32_t ii = find_inst(beg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t j = (uint32_t)(blockIdx.x - beg[ii]), tid = threadIdx.x, n = d.n;
    uint32_t *cnt = dyn, *cur = dyn + d.NB;
    for (uint32_t x = tid; x < d.NB; x += 1024) cnt[x] = 0;
    if (tid == 0) before = all = mx = 0;
    __syncthreads();
    const uint32_t* ct = count + space(b, SP_CNT)[ii];
    uint32_t s0 = 0, s1 = 0;
    for (uint32_t q = tid; q < d.W * d.T; q += 1024) {
        const uint32_t v = ct[q];
        s1 += v;
        if (q < j * d.T) s0 += v;
    }
    if (s1) atomicAdd(&all, s1);
    if (s0) atomicAdd(&before, s0);
    const uint64_t ebase = space(b, SP_ENTRY)[ii];
    const uint32_t* dj = digits + ebase + (size_t)j * n;
    // the thread's nonzero digits, eight loads at a time
    auto each = [&](auto f) {
        for (uint32_t base = tid; base < n; base += 8 * 1024) {
            uint32_t dg[8];
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k) dg[k] = base + k * 1024 < n ? dj[base + k * 1024] : 0;
#pragma unroll
            for (uint32_t k = 0; k < 8; ++k)
                if (dg[k]) f(base + k * 1024, dg[k]);
        }
    };
    each([&](uint32_t, uint32_t dg) { atomicAdd(&cnt[(dg & ~DIGIT_NEG) - 1], 1u); });
    __syncthreads();
    lds_exclusive_scan<1024>(cnt, cur, part, d.NB);
    uint32_t* of = offs + space(b, SP_KEY)[ii] + (size_t)j * d.NB;
    uint32_t largest = 0;
    for (uint32_t x = tid; x < d.NB; x += 1024) {
        cur[x] += before;
        of[x] = cur[x];
        largest = max(largest, cnt[x]);
    }
    if (largest) atomicMax(&mx, largest);
    __syncthreads();
    if (tid == 0) {
        if (mx) atomicMax(&b.stats[4 * ii + 2], mx);
        if (j + 1 == d.W) {
            of[d.NB] = all;
            b.stats[4 * ii + 0] = all;
            b.stats[4 * ii + 1] = (all + d.K - 1) / d.K;
        }
    }
    uint32_t* out = sorted + ebase;
    each([&](uint32_t i, uint32_t dg) { out[atomicAdd(&cur[(dg & ~DIGIT_NEG) - 1], 1u)] = i | (dg & DIGIT_NEG); });
}

// ------------------------------------------------------------------ host side
void msm_prepare() {
    static std::once_flag once;
    std::call_once(once, [] {
        auto allow = [](const void* k, size_t bytes) { (void)hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes); };
        allow((const void*)k_msm_scatter_fine, 12 * MSM_MAX_FINE);
        allow((const void*)k_msm_sort_small, 8 * MSM_SMALL_NB);
    });
}

void msm_launch_scalar_stages(hzk_ctx* ctx, const MsmBatchDev& b, const uint64_t* tot, const MsmSortMax& mx, const MsmScalarBufs& bufs) {
    hipStream_t st = ctx->stream;
    const uint64_t ntiles = tot[SP_SCANTILE];
    {
        TimedLaunch tl(ctx, "msm_digits");
        hipLaunchKernelGGL(k_msm_digits, dim3((unsigned)tot[SP_TILE]), dim3(mx.tile < 1024 ? 256 : 1024), 4 * mx.groups, st, b,
                           bufs.digits, bufs.count);
    }
    if (ntiles) {
        TimedLaunch tl(ctx, "msm_scan");
        hipLaunchKernelGGL(k_scan_tiles, dim3((unsigned)ntiles), dim3(SCAN_THREADS), 0, st, b, (const uint32_t*)bufs.count, bufs.tiles);
        hipLaunchKernelGGL(k_scan_top, dim3(b.ninst), dim3(1024), 0, st, b, bufs.tiles);
        hipLaunchKernelGGL(k_scan_apply, dim3((unsigned)ntiles), dim3(SCAN_THREADS), 0, st, b, bufs.count, (const uint64_t*)bufs.tiles);
        hipLaunchKernelGGL(k_msm_pieces, dim3(b.ninst), dim3(1024), 0, st, b, (const uint32_t*)bufs.count, bufs.sub, bufs.offs);
    }
    TimedLaunch tl(ctx, "msm_scatter");
    if (ntiles) {
        hipLaunchKernelGGL(k_msm_scatter_coarse, dim3((unsigned)tot[SP_TILEWG]), dim3(SC_THREADS), 0, st, b, (const uint32_t*)bufs.digits,
                           (const uint32_t*)bufs.count, bufs.cidx, bufs.ckey);
        hipLaunchKernelGGL(k_msm_fine_count, dim3((unsigned)tot[SP_SUB]), dim3(512), 4 * mx.fine, st, b, (const uint32_t*)bufs.count,
                           (const uint32_t*)bufs.sub, (const uint32_t*)bufs.cidx, (const uint16_t*)bufs.ckey, bufs.rows);
        hipLaunchKernelGGL(k_msm_fine_offsets, dim3((unsigned)tot[SP_GROUP]), dim3(256), 8 * mx.fine, st, b, (const uint32_t*)bufs.count,
                           (const uint32_t*)bufs.sub, bufs.rows, bufs.offs);
        hipLaunchKernelGGL(k_msm_scatter_fine, dim3((unsigned)tot[SP_SUB]), dim3(SC_THREADS), 12 * mx.fine, st, b,
                           (const uint32_t*)bufs.count, (const uint32_t*)bufs.sub, (const uint32_t*)bufs.rows, (const uint32_t*)bufs.cidx,
                           (const uint16_t*)bufs.ckey, bufs.sorted);
    }
    if (tot[SP_SMALL])
        hipLaunchKernelGGL(k_msm_sort_small, dim3((unsigned)tot[SP_SMALL]), dim3(1024), 8 * mx.small_nb, st, b,
                           (const uint32_t*)bufs.digits, (const uint32_t*)bufs.count, bufs.offs, bufs.sorted);
}

// Built-in plan (autotuned entries override it per size class).
// c minimises n*W (bucket entries, one mixed addition each) + 3*W*2^(c-1)
// (bucket reduction: two full additions per bucket plus its share of the run
// weights). K makes the accumulation about
// 2^18..2^19 lanes (4 waves per SIMD on every CU), each adding exactly K
// entries.
MsmPlan msm_plan(size_t n, int force_c, int force_g) {
    MsmPlan p;
    const int cmax = MSM_MAX_C;
    int c = MSM_MIN_C;
    double best = -1;
    for (int cc = MSM_MIN_C; cc <= cmax; ++cc) {
        double w = (double)((255 + cc - 1) / cc);
        double cost = (double)n * w + 3.0 * w * (double)(1u << (cc - 1));
        if (best < 0 || cost < best) { best = cost; c = cc; }
    }
    if (force_c) c = force_c;
    p.c = c;
    p.W = (255 + c - 1) / c;
    p.NB = 1u << (c - 1);
    size_t L = n * (size_t)p.W;
    uint32_t K = 4;   // multiple of 4: the accumulation reads indices in groups of four
    while (K < 4096 && L / (2 * (size_t)K) >= ((size_t)1 << 18)) K <<= 1;
    p.K = K;
    uint32_t g = p.NB / 512;
    if (g < 4) g = 4;
    if (g > 16) g = 16;
    if (g > p.NB) g = p.NB;
    if (force_g) g = force_g;
    if (g > p.NB) g = p.NB;   // a run never spans more buckets than a window has
    p.g = g;
    return p;
}

// plans measured by the autotuner on an MI355X (liblightzk_amd/tune/mi355x.json),
// [regime][G1, G2][log2 n]
static const hzk_tune_entry BUILTIN_PLANS[2][2][32] = {
#include "tune_table.inc"
};

static int size_class(size_t n) {
    int cls = 0;
    while (((size_t)1 << (cls + 1)) <= n) ++cls;
    return cls < 32 ? cls : 31;
}

static bool plan_from_entry(const hzk_tune_entry& t, size_t n, int force_g, MsmPlan* out) {
    if (!t.c) return false;
    MsmPlan q = msm_plan(n, t.c, t.g ? (int)t.g : force_g);
    if (t.K) q.K = t.K;
    *out = q;
    return true;
}

MsmPlan msm_plan_builtin(int g2, size_t n, int regime) {
    MsmPlan p = msm_plan(n, 0, 0);
    const int cls = size_class(n);
    if (regime == MSM_REGIME_BATCH && plan_from_entry(BUILTIN_PLANS[1][g2 ? 1 : 0][cls], n, 0, &p)) return p;
    plan_from_entry(BUILTIN_PLANS[0][g2 ? 1 : 0][cls], n, 0, &p);
    return p;
}

// plan for an MSM of n points: the context's tuned entry for the regime and
// size class, else the built-in measured plan of the regime; a batch-regime
// class with neither falls back to the single-MSM plan, and that one to the
// heuristic. A caller-forced window size (or hzk_set_tuning) bypasses the
// tables.
MsmPlan msm_plan_ctx(hzk_ctx* ctx, int g2, size_t n, int force_c, int regime) {
    MsmPlan p = msm_plan(n, force_c ? force_c : ctx->force_window, ctx->force_seg);
    if (!force_c && !ctx->force_window) {
        const int cls = size_class(n), gi = g2 ? 1 : 0;
        for (int r = regime; r >= MSM_REGIME_SINGLE; --r) {
            hzk_tune_entry t = ctx->tune[r][gi][cls];
            if (!t.c && !ctx->force_seg) {
                t = BUILTIN_PLANS[r][gi][cls];
                t.fit = true;
            }
            if (plan_from_entry(t, n, ctx->force_seg, &p)) {
                p.fit = t.fit;
                break;
            }
        }
    }
    return p;
}

}  // namespace hzk
