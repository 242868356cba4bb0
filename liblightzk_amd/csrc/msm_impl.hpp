// Group-generic MSM stages 5-8 and the batched driver (G1 over Fq, G2 over
// Fq2); included by msm_g1.hip and msm_g2.hip, one instantiation per
// translation unit. Stages 1-4 and the batch layout are described in msm.hip.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstring>
#include <map>
#include <vector>
#include "common.hpp"
#include "curve.hpp"
#include "field29.hpp"
#include "host_ec.hpp"
#include "host_pool.hpp"
#include "lanes29.hpp"
#include "msm.hpp"

namespace hzk {

static constexpr uint32_t HOT = 64;         // a bucket spanning more chunks than this is summed by k_msm_hot_sum first
static constexpr uint32_t HOT_LIST = 256;   // hot instances a hot-sum block lists in LDS

HZK_DEV uint32_t find_inst_g(const uint64_t* __restrict__ beg, uint32_t ninst, uint64_t gid) {
    uint32_t lo = 0, hi = ninst;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (beg[mid] <= gid) lo = mid; else hi = mid;
    }
    return lo;
}
HZK_DEV const uint64_t* space_g(const MsmBatchDev& b, int s) { return b.begin + (size_t)s * (b.ninst + 1); }

// the key whose entries [offs[k], offs[k+1]) contain entry e (offs[nk] > e)
HZK_DEV uint32_t find_key(const uint32_t* __restrict__ offs, uint32_t nk, uint32_t e) {
    uint32_t lo = 0, hi = nk;   // invariant: offs[lo] <= e < offs[hi]
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (offs[mid] <= e) lo = mid; else hi = mid;
    }
    return lo;
}

// the next non-empty key after k, whose entries end at entry e (offs[nk] > e);
// next: where its own end. Empty keys come in long runs: the upper half of
// the buckets of a window one bit narrower than the others, scalars with few
// distinct values. A walk through 2048 of them, one dependent load each, held
// its wave for 200 us (13-bit windows, 2^16 points: 16 entries a chunk: accumulation 308 -> 136 us).
HZK_DEV uint32_t next_key(const uint32_t* __restrict__ offs, uint32_t nk, uint32_t k, uint32_t e, uint32_t& next) {
    next = offs[k + 2];
    if (next > e) return k + 1;
    uint32_t lo = k + 1, step = 1;   // offs[lo + 1] <= e
    while (lo + step < nk - 1 && offs[lo + step + 1] <= e) lo += step, step <<= 1;
    uint32_t hi = min(lo + step, nk - 1);   // offs[hi + 1] > e
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (offs[mid + 1] <= e) lo = mid; else hi = mid;
    }
    next = offs[hi + 1];
    return hi;
}

// ------------------------------------------------------------------ 5. accumulate
// Lane per chunk of K consecutive sorted entries; a chunk crosses bucket
// boundaries freely, so every lane does exactly K mixed additions (the last
// chunk of an instance fewer). The running XYZZ sum is flushed at each bucket
// end: a bucket that lies wholly inside the chunk is final and goes straight
// to bucket[k]; the partial of a bucket that began in an earlier chunk goes
// to carry[2c] (head), that of a bucket continuing into the next chunk to
// carry[2c+1] (tail). Persistent grid over the whole batch's chunk space.
// G1: the additions in 29-bit-limb arithmetic (field29.hpp) over the bases converted
// to its Montgomery form by k_msm_convert_g1. Bucket sums and chunk partials
// are stored as raw accumulator states (g1acc29::store_raw), the form the
// fix-up and the bucket reduction work in. At least two waves per SIMD (the
// G2 lane state does not fit twice in 512 registers otherwise).
static __global__ void __launch_bounds__(256, 2) k_msm_accumulate_g1(MsmBatchDev b, const uint32_t* __restrict__ sorted,
                                                           const uint32_t* __restrict__ offs, uint4* __restrict__ bucket,
                                                           uint4* __restrict__ carry, uint32_t* __restrict__ chunk2key) {
    constexpr int RW = g1acc29::RAW_WORDS / 4;   // uint4 per raw point
    const uint64_t* cbeg = space_g(b, SP_CHUNK);
    const uint64_t total = cbeg[b.ninst];
    for (uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total; gid += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t ii = find_inst_g(cbeg, b.ninst, gid);
        const MsmInst& d = b.inst[ii];
        const uint32_t E = b.stats[4 * ii];
        const uint32_t e0 = (uint32_t)(gid - cbeg[ii]) * d.K;
        if (e0 >= E) continue;
        const uint32_t e1 = min(e0 + d.K, E);
        const uint64_t kb = space_g(b, SP_KEY)[ii];
        const uint32_t* of = offs + kb;
        uint32_t k = find_key(of, d.nk, e0);
        chunk2key[gid] = k;
        uint32_t next = of[k + 1];
        bool before = of[k] < e0;
        const uint4* srt4 = (const uint4*)(sorted + space_g(b, SP_ENTRY)[ii]);
        const uint4* bases = (const uint4*)d.bases;   // converted: x | y, 8 x 32-bit limbs each
        g1acc29 acc;
        acc.set_inf();
        uint4 q = srt4[e0 >> 2];
        uint32_t idx = q.x;
        uint4 p0, p1, p2, p3;
        {
            const uint4* bp = bases + 4 * (size_t)(idx & 0x7fffffffu);
            p0 = bp[0], p1 = bp[1], p2 = bp[2], p3 = bp[3];
        }
        for (uint32_t e = e0; e < e1; ++e) {
            const bool neg = idx >> 31;
            const uint4 x0 = p0, x1 = p1, y0 = p2, y1 = p3;
            const bool inf = p1.w == 0xffffffffu;   // the converter's mark for the point at infinity
            if (e + 1 < e1) {   // prefetch the next base while this one is added
                const uint32_t t = (e + 1) & 3;
                if (t == 0) q = srt4[(e + 1) >> 2];
                idx = t == 0 ? q.x : (t == 1 ? q.y : (t == 2 ? q.z : q.w));
                const uint4* bp = bases + 4 * (size_t)(idx & 0x7fffffffu);
                p0 = bp[0], p1 = bp[1], p2 = bp[2], p3 = bp[3];
            }
            if (!inf) {
                acc.add_affine(fq29::unpack(x0, x1), fq29::negate_if(fq29::unpack(y0, y1), neg));
            }
            if (e + 1 == next || e + 1 == e1) {
                if (before) acc.store_raw(carry + RW * (2 * gid));
                else if (next > e1) acc.store_raw(carry + RW * (2 * gid + 1));
                else acc.store_raw(bucket + RW * (kb + k));
                if (e + 1 < e1) {   // next non-empty bucket
                    k = next_key(of, d.nk, k, e + 1, next);
                    before = false;
                    acc.set_inf();
                }
            }
        }
    }
}

// G2: the same walk over Fq2 = Fq[u]/(u^2 + 1) in 29-bit-limb components
// (g2acc29), bases converted by k_msm_convert (128 bytes: x.c0 | x.c1 |
// y.c0 | y.c1)
static __global__ void __launch_bounds__(256, 2) k_msm_accumulate_g2(MsmBatchDev b, const uint32_t* __restrict__ sorted,
                                                           const uint32_t* __restrict__ offs, uint4* __restrict__ bucket,
                                                           uint4* __restrict__ carry, uint32_t* __restrict__ chunk2key) {
    constexpr int RW = g2acc29::RAW_WORDS / 4;
    const uint64_t* cbeg = space_g(b, SP_CHUNK);
    const uint64_t total = cbeg[b.ninst];
    for (uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total; gid += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t ii = find_inst_g(cbeg, b.ninst, gid);
        const MsmInst& d = b.inst[ii];
        const uint32_t E = b.stats[4 * ii];
        const uint32_t e0 = (uint32_t)(gid - cbeg[ii]) * d.K;
        if (e0 >= E) continue;
        const uint32_t e1 = min(e0 + d.K, E);
        const uint64_t kb = space_g(b, SP_KEY)[ii];
        const uint32_t* of = offs + kb;
        uint32_t k = find_key(of, d.nk, e0);
        chunk2key[gid] = k;
        uint32_t next = of[k + 1];
        bool before = of[k] < e0;
        const uint4* srt4 = (const uint4*)(sorted + space_g(b, SP_ENTRY)[ii]);
        const uint4* bases = (const uint4*)d.bases;
        g2acc29 acc;
        acc.set_inf();
        uint4 q = srt4[e0 >> 2];
        uint32_t idx = q.x;
        for (uint32_t e = e0; e < e1; ++e) {
            const bool neg = idx >> 31;
            const uint4* bp = bases + 8 * (size_t)(idx & 0x7fffffffu);
            const uint4 p0 = bp[0], p1 = bp[1], p2 = bp[2], p3 = bp[3], p4 = bp[4], p5 = bp[5], p6 = bp[6], p7 = bp[7];
            if (e + 1 < e1) {
                const uint32_t t = (e + 1) & 3;
                if (t == 0) q = srt4[(e + 1) >> 2];
                idx = t == 0 ? q.x : (t == 1 ? q.y : (t == 2 ? q.z : q.w));
            }
            if (p3.w != 0xffffffffu) {   // the converter's mark for the point at infinity
                const fq2_29 x{fq29::unpack(p0, p1), fq29::unpack(p2, p3)};
                const fq2_29 y{fq29::unpack(p4, p5), fq29::unpack(p6, p7)};
                acc.add_affine(x, fq2_29::negate_if(y, neg));
            }
            if (e + 1 == next || e + 1 == e1) {
                if (before) acc.store_raw(carry + RW * (2 * gid));
                else if (next > e1) acc.store_raw(carry + RW * (2 * gid + 1));
                else acc.store_raw(bucket + RW * (kb + k));
                if (e + 1 < e1) {
                    k = next_key(of, d.nk, k, e + 1, next);
                    before = false;
                    acc.set_inf();
                }
            }
        }
    }
}

// one base array to convert for the G1 accumulation: count affine points
// from src into dst, as items [begin, next begin) of the conversion space
struct MsmConvTask {
    const void* src;
    void* dst;
    uint64_t begin;
};

// x, y -> x 2^5, y 2^5 mod p (the 2^261 Montgomery form of field29.hpp),
// canonical, 8 x 32-bit limbs; the point at infinity (all zero) becomes
// x word 7 = 0xffffffff, a value no canonical coordinate has
HZK_DEV void convert_point_g1(const uint4* __restrict__ sp, uint4* __restrict__ dp) {
    const uint4 a = sp[0], b2 = sp[1], c = sp[2], e = sp[3];
    const uint32_t any = a.x | a.y | a.z | a.w | b2.x | b2.y | b2.z | b2.w | c.x | c.y | c.z | c.w | e.x | e.y | e.z | e.w;
    if (!any) {
        dp[0] = make_uint4(0, 0, 0, 0);
        dp[1] = make_uint4(0, 0, 0, 0xffffffffu);
        dp[2] = make_uint4(0, 0, 0, 0);
        dp[3] = make_uint4(0, 0, 0, 0);
        return;
    }
    const uint32_t xw[8] = {a.x, a.y, a.z, a.w, b2.x, b2.y, b2.z, b2.w};
    const uint32_t yw[8] = {c.x, c.y, c.z, c.w, e.x, e.y, e.z, e.w};
    uint32_t xo[8], yo[8];
    const fq29 xi = fq29::unpack(xw), yi = fq29::unpack(yw), to = fq29::konst(fq29::TO);
    fq29 x, y;
    scan29(Mul29<Fq29Mod>(x, xi, to), Mul29<Fq29Mod>(y, yi, to));
    x.canonical().pack(xo);
    y.canonical().pack(yo);
    dp[0] = make_uint4(xo[0], xo[1], xo[2], xo[3]);
    dp[1] = make_uint4(xo[4], xo[5], xo[6], xo[7]);
    dp[2] = make_uint4(yo[0], yo[1], yo[2], yo[3]);
    dp[3] = make_uint4(yo[4], yo[5], yo[6], yo[7]);
}

// G2: x.c0 | x.c1 | y.c0 | y.c1 -> the same conversion per Fq component;
// infinity (all zero) marked by x.c1 word 7 = 0xffffffff
HZK_DEV void convert_point_g2(const uint4* __restrict__ sp, uint4* __restrict__ dp) {
    uint4 v[8];
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        v[i] = sp[i];
        any |= v[i].x | v[i].y | v[i].z | v[i].w;
    }
    if (!any) {
#pragma unroll
        for (int i = 0; i < 8; ++i) dp[i] = make_uint4(0, 0, 0, i == 3 ? 0xffffffffu : 0);
        return;
    }
#pragma unroll
    for (int c = 0; c < 4; c += 2) {
        const uint32_t a[8] = {v[2 * c].x, v[2 * c].y, v[2 * c].z, v[2 * c].w, v[2 * c + 1].x, v[2 * c + 1].y, v[2 * c + 1].z, v[2 * c + 1].w};
        const uint32_t b[8] = {v[2 * c + 2].x, v[2 * c + 2].y, v[2 * c + 2].z, v[2 * c + 2].w,
                               v[2 * c + 3].x, v[2 * c + 3].y, v[2 * c + 3].z, v[2 * c + 3].w};
        const fq29 xi = fq29::unpack(a), yi = fq29::unpack(b), to = fq29::konst(fq29::TO);
        fq29 x, y;
        scan29(Mul29<Fq29Mod>(x, xi, to), Mul29<Fq29Mod>(y, yi, to));
        uint32_t xo[8], yo[8];
        x.canonical().pack(xo);
        y.canonical().pack(yo);
        dp[2 * c] = make_uint4(xo[0], xo[1], xo[2], xo[3]);
        dp[2 * c + 1] = make_uint4(xo[4], xo[5], xo[6], xo[7]);
        dp[2 * c + 2] = make_uint4(yo[0], yo[1], yo[2], yo[3]);
        dp[2 * c + 3] = make_uint4(yo[4], yo[5], yo[6], yo[7]);
    }
}

static __global__ void __launch_bounds__(256) k_msm_convert_g2(const MsmConvTask* __restrict__ tasks, uint32_t ntasks, uint64_t total) {
    for (uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total; gid += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = ntasks;
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (tasks[mid].begin <= gid) lo = mid; else hi = mid;
        }
        const MsmConvTask& t = tasks[lo];
        const uint64_t i = gid - t.begin;
        convert_point_g2((const uint4*)t.src + 8 * i, (uint4*)t.dst + 8 * i);
    }
}

static __global__ void __launch_bounds__(256) k_msm_convert_g1(const MsmConvTask* __restrict__ tasks, uint32_t ntasks, uint64_t total) {
    for (uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; gid < total; gid += (uint64_t)gridDim.x * blockDim.x) {
        uint32_t lo = 0, hi = ntasks;   // tasks[lo].begin <= gid < tasks[hi].begin
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (tasks[mid].begin <= gid) lo = mid; else hi = mid;
        }
        const MsmConvTask& t = tasks[lo];
        const uint64_t i = gid - t.begin;
        convert_point_g1((const uint4*)t.src + 4 * i, (uint4*)t.dst + 4 * i);
    }
}

// one array, in place or not
static __global__ void __launch_bounds__(256) k_msm_convert_g1_array(const uint4* src, uint4* dst, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        convert_point_g1(src + 4 * i, dst + 4 * i);
}
static __global__ void __launch_bounds__(256) k_msm_convert_g2_array(const uint4* src, uint4* dst, uint64_t n) {
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        convert_point_g2(src + 8 * i, dst + 8 * i);
}

// ------------------------------------------------------------------ 6. fix-up
// The 29-bit accumulator of each group; bucket sums, chunk partials and run
// sums live in memory as its raw states (RW uint4 per point).
template <class F> struct Acc29;
template <> struct Acc29<fq_t> { using A = g1acc29; };
template <> struct Acc29<fq2_t> { using A = g2acc29; };
template <class F> using acc29_t = typename Acc29<F>::A;
template <class F> constexpr int raw_vec() { return acc29_t<F>::RAW_WORDS / 4; }

// Hot buckets (more than HOT chunks): the head partials carry[2c] of chunks
// f+1..l (f, l: first and last chunk of the bucket) are summed in place,
// HOT_SEG slots' worth of them per workgroup and level, into the segment's
// first; one or two levels leave the whole sum in carry[2(f+1)].
template <class F> constexpr uint32_t hot_seg() { return 16 * LdsLanes<F, 256>::SLOTS; }

// the segment starting at chunk c of instance ii at this level, or 0: number
// of elements (stride chunks apart)
template <class F>
HZK_DEV uint32_t hot_segment(const MsmBatchDev& b, const uint32_t* __restrict__ offs, const uint32_t* __restrict__ chunk2key,
                             uint64_t stride, uint32_t ii, uint32_t c) {
    const MsmInst& d = b.inst[ii];
    if ((uint64_t)c * d.K >= b.stats[4 * ii]) return 0;
    const uint32_t* of = offs + space_g(b, SP_KEY)[ii];
    const uint32_t k = chunk2key[space_g(b, SP_CHUNK)[ii] + c], start = of[k];
    if (start >= c * d.K) return 0;   // chunk c holds no head partial
    const uint32_t f = start / d.K, l = (of[k + 1] - 1) / d.K;
    if (l - f <= HOT) return 0;
    const uint64_t rel = c - (f + 1), span = l - f;
    if (rel % (stride * hot_seg<F>()) != 0) return 0;
    const uint64_t left = (span - rel + stride - 1) / stride;
    return (uint32_t)(left < hot_seg<F>() ? left : hot_seg<F>());
}

template <class F>
__global__ void __launch_bounds__(256) k_msm_hot_sum(MsmBatchDev b, const uint32_t* __restrict__ offs,
                                                     const uint32_t* __restrict__ chunk2key, uint64_t stride,
                                                     uint32_t* __restrict__ carry) {
    using A = LanePoint<F>;
    using S = LdsLanes<F, 256>;
    __shared__ uint32_t shw[S::WORDS];
    __shared__ uint32_t hot[HOT_LIST];
    __shared__ uint64_t hbeg[HOT_LIST + 1];
    __shared__ uint64_t wmask[4];
    __shared__ uint32_t nhot;
    __shared__ uint32_t seg_inst[256], seg_chunk[256], seg_cnt[256], nseg;
    const S sh{shw};
    // Most instances have no hot bucket. Each block lists the instances that
    // do (largest bucket > HOT chunks), in instance order, with the prefix
    // sums of their chunk counts, all in LDS; the grid then strides over the
    // concatenated chunks of the hot instances only (over all chunks when the
    // list overflows), 256 chunks at a time: each thread looks whether a
    // segment starts at its chunk, then the whole block sums the found ones.
    const uint64_t* cbeg = space_g(b, SP_CHUNK);
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) nhot = 0;
    __syncthreads();
    for (uint32_t i0 = 0; i0 < b.ninst; i0 += 256) {
        const uint32_t ii = i0 + threadIdx.x;
        const bool h = ii < b.ninst && b.stats[4 * ii + 2] > HOT * b.inst[ii].K;
        const uint64_t m = __ballot(h);
        if (lane == 0) wmask[wave] = m;
        __syncthreads();
        uint32_t pos = nhot + __popcll(m & ((1ull << lane) - 1));
        for (uint32_t w = 0; w < wave; ++w) pos += __popcll(wmask[w]);
        if (h && pos < HOT_LIST) hot[pos] = ii;
        __syncthreads();
        if (threadIdx.x == 0) nhot += __popcll(wmask[0]) + __popcll(wmask[1]) + __popcll(wmask[2]) + __popcll(wmask[3]);
        __syncthreads();
    }
    const uint32_t nh = nhot;
    if (nh == 0) return;
    const bool listed = nh <= HOT_LIST;
    if (listed && threadIdx.x == 0) {
        uint64_t t = 0;
        for (uint32_t h = 0; h < nh; ++h) { hbeg[h] = t; t += cbeg[hot[h] + 1] - cbeg[hot[h]]; }
        hbeg[nh] = t;
    }
    __syncthreads();
    const uint64_t total = listed ? hbeg[nh] : cbeg[b.ninst];
    const uint32_t slot = threadIdx.x / A::LANES;
    for (uint64_t base = (uint64_t)blockIdx.x * 256; base < total; base += (uint64_t)gridDim.x * 256) {
        if (threadIdx.x == 0) nseg = 0;
        __syncthreads();
        const uint64_t g = base + threadIdx.x;
        if (g < total) {
            uint32_t ii, c;
            if (listed) {
                uint32_t lo = 0, hi = nh;   // hbeg[lo] <= g < hbeg[hi]
                while (hi - lo > 1) {
                    const uint32_t mid = (lo + hi) >> 1;
                    if (hbeg[mid] <= g) lo = mid; else hi = mid;
                }
                ii = hot[lo], c = (uint32_t)(g - hbeg[lo]);
            } else {
                ii = find_inst_g(cbeg, b.ninst, g), c = (uint32_t)(g - cbeg[ii]);
            }
            const uint32_t cnt = hot_segment<F>(b, offs, chunk2key, stride, ii, c);
            if (cnt > 1) {
                const uint32_t at = atomicAdd(&nseg, 1u);
                seg_inst[at] = ii, seg_chunk[at] = c, seg_cnt[at] = cnt;
            }
        }
        __syncthreads();
        const uint32_t ns = nseg;
        for (uint32_t q = 0; q < ns; ++q) {
            const uint32_t cnt = seg_cnt[q];
            uint32_t* first = carry + (size_t)A::RAW_WORDS * 2 * (cbeg[seg_inst[q]] + seg_chunk[q]);
            const size_t step = (size_t)A::RAW_WORDS * 2 * stride;
            A acc;
            acc.set_inf();
            for (uint32_t i = slot; i < cnt; i += S::SLOTS) acc.add(A::load_raw(first + step * i));
            sh.tree_sum(acc, S::SLOTS);
            if (slot == 0) acc.store_raw(first);
        }
        __syncthreads();
    }
}

// Buckets that span chunks f..l (f < l): bucket = tail(f) + heads(f+1..l), a
// lane group per bucket. The groups are numbered by bucket where there are
// fewer buckets than chunks and by chunk (the bucket's second one works)
// otherwise, so that few groups of a wave idle. A group adds its first
// FIX_OWN heads itself; beyond those its wave sums whole runs together where
// that takes fewer steps than the longest one alone. Against a group per chunk
// that adds up to 16 heads one after the other: 2^24 G1 points 357 -> 209 us,
// 200003 G2 points (chunks of 16) 413 -> 157, 15000 G1 points 82 -> 46.
static constexpr uint32_t FIX_OWN = 4;

template <class F, bool BY_KEY>
__global__ void __launch_bounds__(256) k_msm_fixup(MsmBatchDev b, const uint32_t* __restrict__ offs,
                                                   const uint32_t* __restrict__ chunk2key, const uint32_t* __restrict__ carry,
                                                   uint32_t* __restrict__ bucket) {
    using A = LanePoint<F>;
    constexpr int RW = A::RAW_WORDS, LANES = A::LANES, GROUPS = 64 / LANES;
    const uint64_t* beg = space_g(b, BY_KEY ? SP_KEY : SP_CHUNK);
    const uint64_t gid = ((uint64_t)blockIdx.x * blockDim.x + threadIdx.x) / LANES;
    A acc;
    acc.set_inf();
    uint32_t left = 0;                // heads to add, the next one at head
    const uint32_t* head = nullptr;
    uint32_t* dst = nullptr;
    if (gid < beg[b.ninst]) {
        const uint32_t ii = find_inst_g(beg, b.ninst, gid), at = (uint32_t)(gid - beg[ii]);
        const MsmInst& d = b.inst[ii];
        const uint64_t kb = space_g(b, SP_KEY)[ii];
        const bool any = BY_KEY ? at < d.nk : (uint64_t)at * d.K < b.stats[4 * ii];
        if (any) {
            const uint32_t k = BY_KEY ? at : chunk2key[gid], start = offs[kb + k], end = offs[kb + k + 1];
            const uint32_t f = start / d.K, l = end > start ? (end - 1) / d.K : f;
            if (f < l && (BY_KEY || at == f + 1)) {
                const uint32_t* base = carry + (size_t)RW * 2 * space_g(b, SP_CHUNK)[ii];
                acc = A::load_raw(base + (size_t)RW * (2 * f + 1));
                head = base + (size_t)RW * 2 * (f + 1);
                left = l - f > HOT ? 1 : l - f;   // hot: their sum stands in the first
                dst = bucket + (size_t)RW * (kb + k);
            }
        }
    }
    const auto add_own = [&](uint32_t steps) {
        for (uint32_t i = 0; i < steps; ++i) {
            A x;
            if (i < left) x = A::load_raw(head + (size_t)RW * 2 * i);
            else x.set_inf();
            acc.add(x);
        }
    };
    uint32_t most = left;
    for (int m = 32; m >= LANES; m >>= 1) most = max(most, (uint32_t)__shfl_xor((int)most, m));
    if (most == 0) return;   // the whole wave
    add_own(min(most, FIX_OWN));
    if (most > FIX_OWN) {
        most -= FIX_OWN;
        left -= min(left, FIX_OWN);
        head += (size_t)RW * 2 * FIX_OWN;
        constexpr uint32_t TREE = LANES == 4 ? 4 : 3;   // log2 GROUPS
        uint32_t together = left ? (left + GROUPS - 1) / GROUPS + TREE + 1 : 0;
        for (int m = 32; m >= LANES; m >>= 1) together += (uint32_t)__shfl_xor((int)together, m);
        if (most <= together) {
            add_own(most);
        } else {
            const uint32_t lane = threadIdx.x & 63, group = lane / LANES;
            for (uint64_t m = __ballot(left > 0 && lane % LANES == 0); m; m &= m - 1) {
                const int src = __ffsll((unsigned long long)m) - 1;
                const uint32_t n = (uint32_t)__shfl((int)left, src);
                const uint64_t p = (uint64_t)head;
                const uint32_t* run = (const uint32_t*)((uint64_t)(uint32_t)__shfl((int)(uint32_t)p, src) |
                                                        (uint64_t)(uint32_t)__shfl((int)(uint32_t)(p >> 32), src) << 32);
                A x;
                x.set_inf();
                for (uint32_t i = 0; i < n; i += GROUPS) {
                    A y;
                    if (i + group < n) y = A::load_raw(run + (size_t)RW * 2 * (i + group));
                    else y.set_inf();
                    x.add(y);
                }
                for (int off = 32; off >= LANES; off >>= 1) x.add(x.from_lane((int)lane + off));   // group 0 has the sum
                A y = x.from_lane((int)(lane % LANES));
                if (group != (uint32_t)src / LANES) y.set_inf();
                acc.add(y);
            }
        }
    }
    if (dst) acc.store_raw(dst);
}

// ------------------------------------------------------------------ 7. bucket reduction
// log2 of the buckets of a part where a window has several, else 0
__host__ __device__ inline uint32_t window_part_log(const MsmInst& d) {
    uint32_t k = 0;
    if (d.S > 1) while ((1u << k) < d.NB / d.S) ++k;
    return k;
}

// A window's value is sum_{d=1..NB} d * B_d. Workgroup per (window, part of
// NB / S buckets), each lane group (slot) of it takes the g consecutive
// buckets t*g .. t*g + g-1 of the part: with A_t = sum_q (q+1) B and R_t =
// sum_q B by running sums (2g additions, no scalar multiplication) the part's
// value, weights relative to its first bucket, is
//     sum_t [ A_t + g * t * R_t ] = sum_t A_t + g * sum_{t>=1} X_t,
// X_t the suffix sums of R, one LDS scan. Each part yields its value P_p and
// its bucket sum RS_p; the window is sum_p P_p + (NB / S) * sum_p p RS_p. Both
// sums (k_window_value) leave as R = 2^256 XYZZ points; the factor is applied
// among the doublings between windows.
// T = 256 threads for single MSMs, 64 in wide batches (fewer scan and tree
// steps per bucket; the batch fills the GPU by itself).
template <class F, int T>
__global__ void __launch_bounds__(T) k_window_sum(MsmBatchDev b, const uint32_t* __restrict__ bucket, const uint32_t* __restrict__ offs,
                                                  uint32_t* __restrict__ parts, xyzz_t<F>* __restrict__ wval) {
    using A = LanePoint<F>;
    using S = LdsLanes<F, T>;
    constexpr int RW = A::RAW_WORDS;
    __shared__ uint32_t shw[S::WORDS];
    const S sh{shw};
    const uint64_t* wbeg = space_g(b, SP_WIN);
    const uint32_t ii = find_inst_g(wbeg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t local = (uint32_t)(blockIdx.x - wbeg[ii]);
    const uint32_t j = local / d.S, part = local % d.S, PB = d.NB / d.S;   // buckets of the part
    const uint32_t n = PB < (uint32_t)S::SLOTS ? PB : (uint32_t)S::SLOTS, m = PB / n;   // slots, buckets per slot
    const uint32_t slot = threadIdx.x / A::LANES;
    A a, run;
    a.set_inf();
    run.set_inf();
    if (slot < n) {
        const uint64_t kb = space_g(b, SP_KEY)[ii];
        const uint32_t key0 = j * d.NB + part * PB + slot * m;
        const uint32_t* of = offs + kb + key0;
        const uint32_t* bk = bucket + (size_t)RW * (kb + key0);
        auto load = [&](uint32_t q) {
            A p;
            if (of[q + 1] != of[q]) p = A::load_raw(bk + (size_t)RW * q);
            else p.set_inf();
            return p;
        };
        A next = load(m - 1);
        for (int q = (int)m - 1; q >= 0; --q) {
            run.add(next);
            if (q > 0) next = load(q - 1);
            a.add(run);
        }
    }
    // inclusive suffix scan of the slots' bucket sums
    for (uint32_t off = 1; off < n; off <<= 1) {
        __syncthreads();
        sh.put(run);
        __syncthreads();
        if (slot + off < n) run.add(sh.get(off));
    }
    uint32_t* out = parts + (size_t)RW * 2 * blockIdx.x;   // P_p, RS_p
    if (slot == 0) {
        if (d.S > 1) run.store_raw(out + RW);
        run.set_inf();
    }
    for (uint32_t k = 1; k < m; k <<= 1) run.dbl();
    a.add(run);
    sh.tree_sum(a, n);
    if (slot == 0) {
        if (d.S > 1) a.store_raw(out);
        else a.store_xyzz(wval + 2 * (space_g(b, SP_BRED)[ii] + j));
    }
}

// The parts of a window as two points, workgroup per window: sum_p P_p and
// sum_p p RS_p (the suffix sums of RS over p >= 1, summed). S slots scan RS
// while S others sum P in the same steps, then a tree: 2 log2 S additions one
// after the other, 31 us at 32 parts of G1 and 76 us at 64 parts of G2. The
// host's 3 S additions a window, shared by a worker pool, with a copy of 2 S
// points took longer: 2^16 points 559 -> 506 us, 200003 of G2 1705 -> 1500,
// 32 G1 MSMs of a batch 3754 -> 3500.
template <class F>
constexpr int WINDOW_VALUE_T = 128 * LanePoint<F>::LANES;   // 2 x 64 parts
template <class F>
__global__ void __launch_bounds__(WINDOW_VALUE_T<F>) k_window_value(MsmBatchDev b, const uint32_t* __restrict__ parts,
                                                                    xyzz_t<F>* __restrict__ wval) {
    using A = LanePoint<F>;
    constexpr int RW = A::RAW_WORDS;
    __shared__ uint32_t shw[LdsLanes<F, WINDOW_VALUE_T<F>>::WORDS];
    const LdsLanes<F, WINDOW_VALUE_T<F>> sh{shw};
    const uint64_t* vbeg = space_g(b, SP_BRED);
    const uint32_t ii = find_inst_g(vbeg, b.ninst, blockIdx.x);
    const MsmInst& d = b.inst[ii];
    const uint32_t S = d.S, j = (uint32_t)(blockIdx.x - vbeg[ii]);
    if (S == 1) return;   // written by k_window_sum
    const uint32_t slot = threadIdx.x / A::LANES;
    const bool sums = slot >= S;               // the half that sums P
    const uint32_t p = sums ? slot - S : slot;
    A x;
    x.set_inf();
    if (p < S) x = A::load_raw(parts + (size_t)RW * (2 * (space_g(b, SP_WIN)[ii] + (size_t)j * S + p) + (sums ? 0 : 1)));
    for (uint32_t off = 1; off < S; off <<= 1) {
        const uint32_t step = sums ? S / 2 / off : off;
        __syncthreads();
        sh.put(x);
        __syncthreads();
        if (sums ? p < step : p + step < S) x.add(sh.get(step));
    }
    if (slot == S) x.store_xyzz(wval + 2 * blockIdx.x);
    if (slot == 0) x.set_inf();
    sh.tree_sum(x, S);
    if (slot == 0) x.store_xyzz(wval + 2 * blockIdx.x + 1);
}

// ------------------------------------------------------------------ 8. device-side combine (optional)
// The host's combine as a kernel, in the 29-bit accumulator arithmetic: lane
// per instance, Horner over the windows (the dependent doublings that make
// this path slower than the host's), then the normalised Jacobian (x, y, 1) or
// (0, 1, 0): the bytes the host writes.
template <class F>
HZK_DEV acc29_t<F> acc_from_xyzz(const xyzz_t<F>& p);
template <>
HZK_DEV g1acc29 acc_from_xyzz<fq_t>(const xyzz_t<fq_t>& p) {
    auto to = [](const fq_t& v) { return fq29::mul(fq29::unpack(v.l), fq29::konst(fq29::TO)); };
    return {to(p.X), to(p.Y), to(p.ZZ), to(p.ZZZ), p.ZZ.is_zero()};
}
template <>
HZK_DEV g2acc29 acc_from_xyzz<fq2_t>(const xyzz_t<fq2_t>& p) {
    auto to = [](const fq2_t& v) -> fq2_29 {
        const fq29 k = fq29::konst(fq29::TO);
        return {fq29::mul(fq29::unpack(v.c0.l), k), fq29::mul(fq29::unpack(v.c1.l), k)};
    };
    return {to(p.X), to(p.Y), to(p.ZZ), to(p.ZZZ), p.ZZ.is_zero()};
}

template <class F>
__global__ void __launch_bounds__(64) k_msm_combine_horner(MsmBatchDev b, const xyzz_t<F>* __restrict__ wval) {
    using A = acc29_t<F>;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= b.ninst) return;
    const MsmInst& d = b.inst[i];
    const xyzz_t<F>* v = wval + 2 * space_g(b, SP_BRED)[i];
    const uint32_t k = window_part_log(d);
    A acc;
    acc.set_inf();
    for (int j = (int)d.W - 1; j >= 0; --j) {
        const uint32_t shift = d.Lg > 1 ? d.c * d.Lg : d.wb + ((uint32_t)j < d.wx ? 1u : 0u);
        for (uint32_t q = k; q < shift; ++q) acc.dbl();
        if (d.S > 1) acc.add(acc_from_xyzz<F>(v[2 * j + 1]));
        for (uint32_t q = 0; q < k; ++q) acc.dbl();
        acc.add(acc_from_xyzz<F>(v[2 * j]));
    }
    const xyzz_t<F> r = acc.to_xyzz();
    F* out = (F*)d.dest;
    if (r.is_inf()) {
        out[0] = F::zero(), out[1] = F::one(), out[2] = F::zero();
        return;
    }
    const F inv = (r.ZZ * r.ZZZ).inverse();   // 1 / (ZZ ZZZ)
    out[0] = r.X * (r.ZZZ * inv);             // X / ZZ
    out[1] = r.Y * (r.ZZ * inv);              // Y / ZZZ
    out[2] = F::one();
}

// ------------------------------------------------------------------ driver
struct MsmBatchLayout {
    std::vector<MsmInst> inst;
    std::vector<uint64_t> begin;   // [SP_COUNT][ninst + 1]
    uint64_t tot[SP_COUNT];
    MsmSortMax sort_max;
    uint32_t max_parts = 1;        // parts per window
    uint32_t hot_levels = 0;       // levels of k_msm_hot_sum (upper bound)
    bool two_level = false;        // some instance is sorted in two levels
    bool unpacked = false;         // some coarse entries take two arrays
    int regime = 0;                // plan regime (MSM_REGIME_*)
    size_t bytes = 0;              // scratch needed
    // scratch offsets
    size_t o_inst, o_begin, o_stats, o_digits, o_count, o_tiles, o_sub, o_rows, o_cidx, o_ckey, o_offs, o_sorted, o_chunk2key, o_bucket,
        o_carry, o_parts, o_wval;
    // base arrays converted for the accumulation, one per distinct source
    // array (its largest referenced point count), and which one each instance reads
    std::vector<MsmConvTask> conv;     // dst holds the offset into the scratch until run time
    std::vector<uint32_t> conv_of;     // instance -> task
    uint64_t conv_total = 0;
    size_t o_conv = 0, o_convdesc = 0;
    size_t o_upload_end = 0, o_download_end = 0;
};

// Chunk lengths between 3/4 and 2 times the plans' that give the SIMDs equal
// work. The accumulation issues one wave's instructions at a time on a SIMD,
// so it takes K additions times the waves of the fullest SIMD (a wave alone
// issues 1.2 times slower), and a chunk more costs the fix-up about 4.5
// additions of a wave per 64. The plans are tuned at one size of a class of
// [2^k, 2^(k+1)); at others a last, nearly empty round cost up to a third:
// G2 65536 points 806 -> 745 us, 131072 1077 -> 996; G1 50000 399 -> 382, 420000
// 1031 -> 949; 32 G1 MSMs of a batch 3300 -> 2910. How many digits
// are zero is known on the GPU only: the cost is that of all and of the third
// that a witness of 0/1 flags leaves (2^20 witness by the first alone: 1133 ->
// 1252). Above 16 waves a SIMD it gains less than the model knows.
static constexpr double MSM_SPARSE = 0.32;
static void msm_fit_chunks(const hzk_ctx* ctx, MsmInst* inst, const uint8_t* fit, size_t count) {
    const auto scaled = [&](size_t i, uint32_t q) {
        return fit[i] ? (inst[i].K * q / 16 + 3) & ~3u : inst[i].K;   // a multiple of 4, as the plans are
    };
    const auto cost = [&](uint32_t q, double share) {   // share: digits that are not zero
        uint64_t entries = 0, chunks = 0;
        for (size_t i = 0; i < count; ++i) {
            const uint64_t e = (uint64_t)inst[i].n * inst[i].W, K = scaled(i, q);
            entries += e;
            chunks += (e + K - 1) / K;
        }
        const double waves = share * (double)((chunks + 255) / 256) / ctx->num_cus;   // per SIMD
        return (double)entries / chunks * (waves <= 1 ? 1.2 : std::ceil(waves)) + 4.5 * waves;
    };
    uint64_t chunks = 0;
    for (size_t i = 0; i < count; ++i) chunks += (uint64_t)inst[i].n * inst[i].W / inst[i].K;
    if (chunks > (uint64_t)ctx->num_cus * 256 * 16) return;
    uint32_t best = 16;
    double least = 0.97 * (cost(16, 1) + cost(16, MSM_SPARSE));
    for (uint32_t q = 12; q <= 32; ++q) {
        const double c = cost(q, 1) + cost(q, MSM_SPARSE);
        if (c < least) least = c, best = q;
    }
    for (size_t i = 0; i < count; ++i) inst[i].K = scaled(i, best);
}

// longer: chunks of that many times the plans' length (less scratch)
template <class F>
static MsmBatchLayout msm_layout(hzk_ctx* ctx, const MsmJob* jobs, size_t count, uint32_t longer = 1) {
    MsmBatchLayout L;
    L.inst.resize(count);
    L.begin.assign((size_t)SP_COUNT * (count + 1), 0);
    const int g2 = sizeof(F) == 32 ? 0 : 1;
    // regime: a wide batch (msm_wide_batch, digits counted under the
    // single-MSM plans) fills the GPU by itself, so its instances take the
    // throughput plans (fewer buckets, longer runs)
    int regime = ctx->force_regime;
    if (regime < 0) {
        uint64_t e = 0;
        for (size_t i = 0; i < count; ++i) {
            const MsmPlan q = msm_plan_ctx(ctx, g2, jobs[i].n, (int)jobs[i].win_siz, MSM_REGIME_SINGLE);
            e += (uint64_t)jobs[i].n * (uint64_t)q.W;
        }
        regime = msm_wide_batch(g2, count, e) ? MSM_REGIME_BATCH : MSM_REGIME_SINGLE;
    }
    L.regime = regime;
    std::vector<uint8_t> fit(count);
    for (size_t i = 0; i < count; ++i) {
        MsmPlan p = msm_plan_ctx(ctx, g2, jobs[i].n, (int)jobs[i].win_siz, regime);
        if (p.fit) msm_widen(g2, jobs[i].n, p);
        MsmInst& d = L.inst[i];
        d.scalars = jobs[i].scalars;
        d.bases = jobs[i].bases;
        d.dest = jobs[i].dest;
        d.n = (uint32_t)jobs[i].n;
        d.c = (uint32_t)p.c;
        d.W = (uint32_t)p.W;
        d.NB = p.NB;
        d.nk = d.W * d.NB;
        d.K = p.K;
        d.g = p.g;
        d.G = p.NB / p.g;
        d.nd = d.n;
        d.Wd = d.W;
        d.Lg = 1;
        d.wb = 255 / d.W;   // balanced windows (c = ceil(255 / W) >= every width)
        d.wx = 255 % d.W;
        if (jobs[i].levels > 1) {
            // level table: every bucket set serves Lg digit windows over nd * Lg
            // virtual points; fewer bucket sets to reduce, larger buckets
            d.wb = d.c;   // the table's levels are 2^(c t) multiples: uniform windows
            d.wx = 0;
            d.Lg = jobs[i].levels;
            d.W = (d.Wd + d.Lg - 1) / d.Lg;
            d.n = d.nd * d.Lg;
            d.nk = d.W * d.NB;
            const uint64_t entries = (uint64_t)d.n * d.W;
            uint32_t K = 4;
            while (K < 4096 && entries / (2 * (uint64_t)K) >= ((uint64_t)1 << 18)) K <<= 1;
            d.K = K;
        }
        fit[i] = p.fit && jobs[i].levels <= 1;
        d.K *= longer;
    }
    if (longer == 1) msm_fit_chunks(ctx, L.inst.data(), fit.data(), count);
    for (size_t i = 0; i < count; ++i) {
        MsmInst& d = L.inst[i];
        // parts per window: one run of g buckets per slot of a window-sum
        // workgroup, at most 64 parts (host combine, lanes of the device combine)
        const uint32_t slots = regime == MSM_REGIME_BATCH ? LdsLanes<F, 64>::SLOTS : LdsLanes<F, 256>::SLOTS;
        d.S = 1;
        while (d.S < 64 && d.G / d.S > slots) d.S *= 2;
        L.max_parts = std::max(L.max_parts, d.S);
        d.T = msm_tiles(d.nd);
        d.tile = (d.nd + d.T - 1) / d.T;
        d.small = d.n <= (regime == MSM_REGIME_BATCH ? MSM_SMALL_BATCH_N : MSM_SMALL_N) && d.NB <= MSM_SMALL_NB;
        d.CG = d.small ? 1 : msm_coarse_groups(d.n, d.NB, d.W);
        d.FB = d.NB / d.CG;
        // at least a round of the coarse scatter per workgroup, and about 2048 workgroups
        d.ctile = std::max({1u, 8192 / d.tile, d.T * d.W / 2048});
        d.ib = msm_packs(d.n, d.FB) ? std::max(1u, msm_log2_ceil(d.n)) : 0;
        L.sort_max.tile = std::max(L.sort_max.tile, d.tile);
        L.sort_max.groups = std::max(L.sort_max.groups, d.W * d.CG);
        if (d.small) L.sort_max.small_nb = std::max(L.sort_max.small_nb, d.NB);
        else L.sort_max.fine = std::max(L.sort_max.fine, d.FB), L.two_level = true, L.unpacked |= !d.ib;
        uint64_t entries = (uint64_t)d.n * d.W;
        const uint64_t groups = (uint64_t)d.W * d.CG;
        uint64_t sz[SP_COUNT];
        sz[SP_TILE] = d.T;
        sz[SP_TILEWG] = d.small ? 0 : (uint64_t)((d.T + d.ctile - 1) / d.ctile) * d.W;
        sz[SP_CNT] = groups * d.T + 1;
        sz[SP_SCANTILE] = d.small ? 0 : (groups * d.T + MSM_SCAN_TILE) / MSM_SCAN_TILE;
        sz[SP_GROUP] = d.small ? 0 : groups + 1;
        sz[SP_SUB] = d.small ? 0 : entries / MSM_SUB + groups;
        sz[SP_ROW] = sz[SP_SUB] * d.FB;
        sz[SP_SMALL] = d.small ? d.W : 0;
        sz[SP_KEY] = (uint64_t)d.nk + 1;
        sz[SP_CHUNK] = (entries + d.K - 1) / d.K;
        sz[SP_BRED] = (uint64_t)d.W;
        sz[SP_WIN] = (uint64_t)d.W * d.S;
        sz[SP_ENTRY] = (entries + 63) & ~(uint64_t)63;   // 256-B aligned per instance (vector index loads)
        for (int s = 0; s < SP_COUNT; ++s) L.begin[(size_t)s * (count + 1) + i + 1] = L.begin[(size_t)s * (count + 1) + i] + sz[s];
        uint64_t maxspan = (d.n + d.K - 1) / d.K + 1;   // a bucket holds at most n entries
        uint32_t lv = 0;
        if (maxspan > HOT)
            for (uint64_t stride = 1; stride < maxspan; stride *= hot_seg<F>()) ++lv;
        if (lv > L.hot_levels) L.hot_levels = lv;
    }
    for (int s = 0; s < SP_COUNT; ++s) L.tot[s] = L.begin[(size_t)s * (count + 1) + count];
    {
        std::map<const void*, uint64_t> need;   // source array -> points referenced (virtual points of level tables)
        for (size_t i = 0; i < count; ++i)
            if (jobs[i].form == 0) need[L.inst[i].bases] = std::max<uint64_t>(need[L.inst[i].bases], L.inst[i].n);
        std::map<const void*, uint32_t> task_of;
        uint64_t pts = 0;
        for (const auto& kv : need) {
            task_of[kv.first] = (uint32_t)L.conv.size();
            L.conv.push_back({kv.first, (void*)(uintptr_t)(pts * (g2 ? 128 : 64)), pts});
            pts += kv.second;
        }
        L.conv_total = pts;
        L.conv_of.assign(count, UINT32_MAX);   // UINT32_MAX: bases already converted
        for (size_t i = 0; i < count; ++i)
            if (jobs[i].form == 0) L.conv_of[i] = task_of[L.inst[i].bases];
    }
    size_t off = 0;
    auto take = [&off](size_t bytes) { size_t o = (off + 255) & ~size_t(255); off = o + bytes; return o; };
    // descriptors, uploaded in one copy (o_inst .. o_upload_end)
    L.o_inst = take(count * sizeof(MsmInst));
    L.o_begin = take(L.begin.size() * 8);
    L.o_convdesc = take(L.conv.size() * sizeof(MsmConvTask));
    L.o_upload_end = off;
    L.o_digits = take(L.tot[SP_ENTRY] * 4);
    L.o_count = take(L.tot[SP_CNT] * 4);
    L.o_tiles = take(L.tot[SP_SCANTILE] * 8);
    L.o_sub = take(L.tot[SP_GROUP] * 4);
    L.o_rows = take(L.tot[SP_ROW] * 4);
    L.o_cidx = take(L.two_level ? L.tot[SP_ENTRY] * 4 : 0);
    L.o_ckey = take(L.unpacked ? L.tot[SP_ENTRY] * 2 : 0);
    L.o_offs = take(L.tot[SP_KEY] * 4);
    L.o_sorted = take(L.tot[SP_ENTRY] * 4);
    const size_t raw = (size_t)raw_vec<F>() * 16;   // bytes per raw accumulator state
    L.o_chunk2key = take(L.tot[SP_CHUNK] * 4);
    L.o_bucket = take(L.tot[SP_KEY] * raw);
    L.o_carry = take(2 * L.tot[SP_CHUNK] * raw);             // head and tail partial per chunk
    L.o_parts = take(2 * L.tot[SP_WIN] * raw);               // P_p, RS_p per part of a window
    // results for the host, downloaded in one copy (o_stats .. o_download_end)
    L.o_stats = take(count * 16);
    L.o_wval = take(2 * L.tot[SP_BRED] * sizeof(xyzz_t<F>));   // two points per window (R = 2^256, for the host)
    L.o_download_end = off;
    L.o_conv = take(L.conv_total * (g2 ? 128 : 64));
    L.bytes = off + 256;
    return L;
}

// device stages 1-8 for a laid-out batch (all launches on ctx->stream; no host waits)
template <class F>
static void msm_device_stages(hzk_ctx* ctx, const MsmBatchLayout& L, char* base) {
    const size_t ninst = L.inst.size();
    MsmBatchDev b;
    b.inst = (const MsmInst*)(base + L.o_inst);
    b.begin = (const uint64_t*)(base + L.o_begin);
    b.ninst = (uint32_t)ninst;
    b.stats = (uint32_t*)(base + L.o_stats);
    MsmScalarBufs sb;
    sb.digits = (uint32_t*)(base + L.o_digits);
    sb.count = (uint32_t*)(base + L.o_count);
    sb.tiles = (uint64_t*)(base + L.o_tiles);
    sb.sub = (uint32_t*)(base + L.o_sub);
    sb.rows = (uint32_t*)(base + L.o_rows);
    sb.cidx = (uint32_t*)(base + L.o_cidx);
    sb.ckey = (uint16_t*)(base + L.o_ckey);
    sb.offs = (uint32_t*)(base + L.o_offs);
    sb.sorted = (uint32_t*)(base + L.o_sorted);
    uint32_t* chunk2key = (uint32_t*)(base + L.o_chunk2key);
    uint4* bucket = (uint4*)(base + L.o_bucket);
    uint4* carry = (uint4*)(base + L.o_carry);
    uint32_t* parts = (uint32_t*)(base + L.o_parts);
    xyzz_t<F>* wval = (xyzz_t<F>*)(base + L.o_wval);
    hipStream_t st = ctx->stream;

    if (L.conv_total) {
        TimedLaunch tl(ctx, "msm_convert");
        const uint64_t blocks = (L.conv_total + 255) / 256, cap = (uint64_t)ctx->num_cus * 32;
        const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
        const MsmConvTask* tasks = (const MsmConvTask*)(base + L.o_convdesc);
        if constexpr (sizeof(F) == 32)
            hipLaunchKernelGGL(k_msm_convert_g1, grid, dim3(256), 0, st, tasks, (uint32_t)L.conv.size(), L.conv_total);
        else
            hipLaunchKernelGGL(k_msm_convert_g2, grid, dim3(256), 0, st, tasks, (uint32_t)L.conv.size(), L.conv_total);
    }
    msm_launch_scalar_stages(ctx, b, L.tot, L.sort_max, sb);
    {
        TimedLaunch tl(ctx, "msm_accumulate");
        uint64_t blocks = (L.tot[SP_CHUNK] + 255) / 256;
        uint64_t cap = (uint64_t)ctx->num_cus * 16;   // persistent grid: 16 waves per CU
        const dim3 grid((unsigned)(blocks < cap ? blocks : cap));
        if constexpr (sizeof(F) == 32)
            hipLaunchKernelGGL(k_msm_accumulate_g1, grid, dim3(256), 0, st, b, (const uint32_t*)sb.sorted, (const uint32_t*)sb.offs,
                               bucket, carry, chunk2key);
        else
            hipLaunchKernelGGL(k_msm_accumulate_g2, grid, dim3(256), 0, st, b, (const uint32_t*)sb.sorted, (const uint32_t*)sb.offs,
                               bucket, carry, chunk2key);
    }
    {
        TimedLaunch tl(ctx, "msm_fixup");
        uint64_t stride = 1;
        for (uint32_t lv = 0; lv < L.hot_levels; ++lv, stride *= hot_seg<F>())
            hipLaunchKernelGGL(k_msm_hot_sum<F>, dim3(std::min<unsigned>(blocks_for(L.tot[SP_CHUNK], 256), 1024)), dim3(256), 0, st, b,
                               (const uint32_t*)sb.offs, (const uint32_t*)chunk2key, stride, (uint32_t*)carry);
        const bool by_key = L.tot[SP_KEY] < L.tot[SP_CHUNK];
        hipLaunchKernelGGL((by_key ? k_msm_fixup<F, true> : k_msm_fixup<F, false>),
                           dim3(blocks_for(std::min(L.tot[SP_KEY], L.tot[SP_CHUNK]) * LanePoint<F>::LANES, 256)), dim3(256), 0, st, b,
                           (const uint32_t*)sb.offs, (const uint32_t*)chunk2key, (const uint32_t*)carry, (uint32_t*)bucket);
    }
    {
        TimedLaunch tl(ctx, "msm_bucket_reduce");
        if (L.regime == MSM_REGIME_BATCH)
            hipLaunchKernelGGL((k_window_sum<F, 64>), dim3((unsigned)L.tot[SP_WIN]), dim3(64), 0, st, b, (const uint32_t*)bucket,
                               (const uint32_t*)sb.offs, parts, wval);
        else
            hipLaunchKernelGGL((k_window_sum<F, 256>), dim3((unsigned)L.tot[SP_WIN]), dim3(256), 0, st, b, (const uint32_t*)bucket,
                               (const uint32_t*)sb.offs, parts, wval);
        if (L.max_parts > 1)
            hipLaunchKernelGGL(k_window_value<F>, dim3((unsigned)L.tot[SP_BRED]),
                               dim3(std::max<unsigned>(64, 2 * L.max_parts * LanePoint<F>::LANES)), 0, st, b, (const uint32_t*)parts, wval);
    }
}

template <class F>
static void msm_launch_combine(hzk_ctx* ctx, const MsmBatchLayout& L, char* base) {
    MsmBatchDev b;
    b.inst = (const MsmInst*)(base + L.o_inst);
    b.begin = (const uint64_t*)(base + L.o_begin);
    b.ninst = (uint32_t)L.inst.size();
    b.stats = (uint32_t*)(base + L.o_stats);
    TimedLaunch tl(ctx, "msm_combine");
    hipLaunchKernelGGL(k_msm_combine_horner<F>, dim3(blocks_for(L.inst.size(), 64)), dim3(64), 0, ctx->stream, b,
                       (const xyzz_t<F>*)(base + L.o_wval));
}

template <class F>
static std::string shape_key(const MsmBatchLayout& L, bool combine) {
    std::string k(sizeof(F) == 32 ? "g1:" : "g2:");
    k += L.regime == MSM_REGIME_BATCH ? "b:" : "s:";
    if (combine) k += "dev:";
    k += std::to_string(L.conv.size()) + "/" + std::to_string(L.conv_total) + ":";
    for (const MsmInst& d : L.inst) {
        char buf[64];
        snprintf(buf, sizeof buf, "%u/%u/%u/%u/%u/%u;", d.n, d.c, d.K, d.g, d.T, d.Lg);
        k += buf;
    }
    return k;
}

// bytes from p to the end of the allocation that it lies in (0: unknown). Two
// allocations may be neighbours, and a copy into both is refused.
inline size_t allocation_left(const void* p) {
    hipDeviceptr_t base = nullptr;
    size_t size = 0;
    if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) != hipSuccess) {
        (void)hipGetLastError();
        return 0;
    }
    return (size_t)((char*)base + size - (const char*)p);
}

// ext_scratch != null: run on that device buffer (ext_bytes long) instead of
// the context's arena, with pageable host staging; nothing is allocated on
// the device or pinned on the host (no graph capture in this mode)
template <class F, class HostPt>
int msm_batch_run(hzk_ctx* ctx, const MsmJob* jobs, size_t count, int dests_on_host, int capture, void* ext_scratch = nullptr,
                  size_t ext_bytes = 0, int device_combine = 0) {
    HZK_CHECK(ctx, count > 0 && jobs, HZK_ERR_INVALID, "msm: empty batch");
    for (size_t i = 0; i < count; ++i) {
        HZK_CHECK(ctx, jobs[i].n > 0 && jobs[i].n < (1ull << 31), HZK_ERR_INVALID, "msm: n=%zu out of range [1, 2^31)", jobs[i].n);
        HZK_CHECK(ctx, jobs[i].levels <= 1 || (jobs[i].win_siz && jobs[i].levels <= (255 + jobs[i].win_siz - 1) / jobs[i].win_siz),
                  HZK_ERR_INVALID, "msm: a level table needs win_siz and at most ceil(255 / win_siz) levels (%u)", jobs[i].levels);
        HZK_CHECK(ctx, (uint64_t)jobs[i].n * (jobs[i].levels ? jobs[i].levels : 1) < (1ull << 31), HZK_ERR_UNSUPPORTED,
                  "msm: n=%zu x %u levels exceeds 2^31 table points", jobs[i].n, jobs[i].levels);
        HZK_CHECK(ctx, jobs[i].scalars && jobs[i].bases && jobs[i].dest, HZK_ERR_INVALID, "msm: null pointer in job %zu", i);
        HZK_CHECK(ctx, jobs[i].form <= 1, HZK_ERR_INVALID, "msm: base form %u", jobs[i].form);
        HZK_CHECK(ctx, jobs[i].win_siz == 0 || (jobs[i].win_siz >= (uint32_t)MSM_MIN_C && jobs[i].win_siz <= (uint32_t)MSM_MAX_C),
                  HZK_ERR_INVALID, "msm: win_siz=%u unsupported (0 or %d..%d)", jobs[i].win_siz, MSM_MIN_C, MSM_MAX_C);
    }
    HZK_CHECK(ctx, !(device_combine && dests_on_host), HZK_ERR_INVALID, "msm: the device-side combine needs device dests");
    msm_prepare();
    MsmBatchLayout L = msm_layout<F>(ctx, jobs, count);
    for (size_t i = 0; i < count; ++i)   // bucket offsets are 32-bit
        HZK_CHECK(ctx, (uint64_t)L.inst[i].n * L.inst[i].W <= 0xffff0000ull, HZK_ERR_UNSUPPORTED,
                  "msm: n=%u with %u windows exceeds 2^32 bucket entries", L.inst[i].n, L.inst[i].W);
    int rc = 0;
    if (ext_scratch) {   // longer chunks need less
        for (uint32_t longer = 2; L.bytes > ext_bytes && longer <= 4; longer *= 2) L = msm_layout<F>(ctx, jobs, count, longer);
        HZK_CHECK(ctx, L.bytes <= ext_bytes && !capture, HZK_ERR_UNSUPPORTED,
                  "msm: this MSM needs %zu bytes of scratch, the static buffer holds %zu", L.bytes, ext_bytes);
    } else {
        rc = ensure_scratch(ctx, L.bytes);
        if (rc) return rc;
    }
    // staging: the descriptors as they lie in the scratch, the downloaded
    // window sums and statistics, the results
    const size_t up_bytes = L.o_upload_end - L.o_inst, down_bytes = L.o_download_end - L.o_stats;
    const size_t s_down = (up_bytes + 255) & ~size_t(255), s_out = (s_down + down_bytes + 255) & ~size_t(255);
    const size_t host_bytes = s_out + count * 3 * sizeof(F);
    char* pin;
    int slot = -1;
    std::vector<char> pageable;
    if (ext_scratch) {
        pageable.resize(host_bytes);
        pin = pageable.data();
    } else {
        rc = stage_acquire(ctx, host_bytes, &pin, &slot);
        if (rc) return rc;
    }
    char* base = ext_scratch ? (char*)ext_scratch : (char*)ctx->scratch;
    hipStream_t st = ctx->stream;
    // G1: instances read their converted base arrays in the scratch
    for (MsmConvTask& t : L.conv) t.dst = base + L.o_conv + (size_t)(uintptr_t)t.dst;
    for (size_t i = 0; i < L.conv_of.size(); ++i)
        if (L.conv_of[i] != UINT32_MAX) L.inst[i].bases = L.conv[L.conv_of[i]].dst;
    // descriptors and work-space starts
    std::memcpy(pin, L.inst.data(), count * sizeof(MsmInst));
    std::memcpy(pin + (L.o_begin - L.o_inst), L.begin.data(), L.begin.size() * 8);
    if (!L.conv.empty()) std::memcpy(pin + (L.o_convdesc - L.o_inst), L.conv.data(), L.conv.size() * sizeof(MsmConvTask));
    HZK_HIP(ctx, hipMemcpyAsync(base + L.o_inst, pin, up_bytes, hipMemcpyHostToDevice, st));

    if (capture) {
        std::string key = shape_key<F>(L, device_combine != 0);
        hzk_graph_entry& g = ctx->graphs[key];
        if (!g.exec || g.generation != ctx->scratch_generation) {
            if (g.exec) { (void)hipGraphExecDestroy(g.exec); g.exec = nullptr; }
            hipGraph_t graph;
            bool timing = ctx->timing;
            ctx->timing = false;
            HZK_HIP(ctx, hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            msm_device_stages<F>(ctx, L, base);
            if (device_combine) msm_launch_combine<F>(ctx, L, base);
            hipError_t e = hipStreamEndCapture(st, &graph);
            ctx->timing = timing;
            HZK_HIP(ctx, e);
            e = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            HZK_HIP(ctx, e);
            g.generation = ctx->scratch_generation;
        }
        TimedLaunch tl(ctx, "msm_graph");
        HZK_HIP(ctx, hipGraphLaunch(g.exec, st));
    } else {
        msm_device_stages<F>(ctx, L, base);
        if (device_combine) msm_launch_combine<F>(ctx, L, base);
    }
    HZK_HIP(ctx, hipGetLastError());
    if (device_combine) {   // results are written by the device; nothing comes back to the host
        if (slot >= 0) return stage_fence(ctx, slot);
        HZK_HIP(ctx, hipStreamSynchronize(st));   // pageable staging (no-alloc scratch): wait for the copies
        return 0;
    }
    const uint32_t* hstats = (const uint32_t*)(pin + s_down);
    const char* hval = pin + s_down + (L.o_wval - L.o_stats);
    HZK_HIP(ctx, hipMemcpyAsync(pin + s_down, base + L.o_stats, down_bytes, hipMemcpyDeviceToHost, st));
    if (slot >= 0) {   // a slot that an error leaves early is free once the download is done
        rc = stage_fence(ctx, slot);
        if (rc) return rc;
    }
    HZK_HIP(ctx, hipStreamSynchronize(st));

    // Horner over windows, instances in parallel
    char* const out = pin + s_out;   // pinned: a copy from pageable memory goes through a staging copy and a wait of its own
    const uint64_t* vbeg = L.begin.data() + (size_t)SP_BRED * (count + 1);
    parallel_for((long)count, [&](long i) {
        const MsmInst& d = L.inst[i];
        const uint32_t k = window_part_log(d);
        HostPt acc = HostPt::inf();
        for (int j = (int)d.W - 1; j >= 0; --j) {
            // a window is sum_p P_p + 2^k sum_p p RS_p: the second sum joins k
            // doublings early. A bucket set spans Lg digit windows of c bits;
            // plain windows are wb or wb + 1 bits, either more than k
            const char* v = hval + 2 * (vbeg[i] + j) * sizeof(xyzz_t<F>);
            const uint32_t shift = d.Lg > 1 ? d.c * d.Lg : d.wb + ((uint32_t)j < d.wx ? 1u : 0u);
            acc = acc.dbl_n(shift - k);
            if (d.S > 1) acc = acc.add(HostPt::load_xyzz(v + sizeof(xyzz_t<F>)));
            acc = acc.dbl_n(k).add(HostPt::load_xyzz(v));
        }
        acc.store_jacobian(&out[i * 3 * sizeof(F)]);
    });
    // results whose places follow one another in one allocation go in one copy:
    // 32 of a batch were 32 copies, 110 us (2800 -> 2685 us with one)
    for (size_t i = 0, k = 1; i < count; i = k++) {
        constexpr size_t B = 3 * sizeof(F);
        if (dests_on_host) {
            std::memcpy(jobs[i].dest, &out[i * B], B);
            continue;
        }
        const auto follows = [&] { return k < count && (char*)jobs[k].dest == (char*)jobs[i].dest + (k - i) * B; };
        if (follows())
            for (const size_t room = allocation_left(jobs[i].dest); follows() && (k - i + 1) * B <= room;) ++k;
        HZK_HIP(ctx, hipMemcpyAsync(jobs[i].dest, &out[i * B], (k - i) * B, hipMemcpyHostToDevice, st));
    }
    if (!dests_on_host) HZK_HIP(ctx, hipStreamSynchronize(st));
    const MsmInst& d0 = L.inst[count - 1];
    ctx->last_msm[0] = hstats[4 * (count - 1)];
    ctx->last_msm[1] = hstats[4 * (count - 1) + 1];
    ctx->last_msm[2] = hstats[4 * (count - 1) + 2];
    ctx->last_msm[3] = d0.c;
    ctx->last_msm[4] = d0.W;
    return 0;
}

template <class F, class HostPt>
int msm_run(hzk_ctx* ctx, const void* scalars, const void* bases, size_t n, size_t win_siz, void* dest, uint32_t levels) {
    HZK_CHECK(ctx, win_siz <= (size_t)MSM_MAX_C, HZK_ERR_INVALID, "msm: win_siz=%zu unsupported (0 or %d..%d)", win_siz,
              MSM_MIN_C, MSM_MAX_C);
    MsmJob j{scalars, bases, n, dest, (uint32_t)win_siz, levels};
    return msm_batch_run<F, HostPt>(ctx, &j, 1, 0, 0);
}

}  // namespace hzk
