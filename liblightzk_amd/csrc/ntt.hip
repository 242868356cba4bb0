// Fr number-theoretic transforms on gfx950: NTT, inverse NTT and coset NTT.
//
// Replaces number_theory_transformation (include/operator/poly.cuh:65-73:
// one launch and one full HBM read+write per radix-2 stage, half the lanes
// idle, then a bit-reverse launch and a scaling launch) while keeping its
// semantics exactly: natural-order input and output,
//   out[k] = factor * sum_j in[j] * w^(j k),   w = omega_powers[1],
// with omega_powers[e] = w^e for e < deg/2 (the table layout of ntt_setup,
// include/protocol/groth16-operator.cuh:6-32) and the same decimation-in-
// frequency butterfly (a, b) -> (a + b, (a - b) w^((j mod h) 2^s)).
//
// Here the log2(deg) stages are grouped into passes. A pass covers R
// consecutive stages over tiles of 2^R rows x 2^g columns (2^10 elements); rows
// or columns are contiguous in HBM, so loads and stores stay coalesced.
// Inside a tile every thread holds 4 elements in registers: the 2^2 rows
// that two consecutive stages pair up, runs those stages' 4 butterflies there,
// and trades its elements with the other threads through LDS before the next
// two stages. 8 elements a thread (as many products, a third fewer exchanges)
// need 256 registers and spill; 4 take 146, three waves a SIMD, and 37 KB of
// LDS a workgroup.
//
// Elements are nine signed 29-bit limbs (limb29.hpp) from the load of a pass
// to its store, LDS included: a difference is nine subtractions, carries are
// propagated every second stage, and a multiple of r is subtracted once or
// twice a pass (values grow to at most 2^9.4 r, the capacity of nine limbs).
// The issue of the multiply-adds bounds the passes (a product is 162 of them,
// 330 us of a coset transform of 2^22 points). Measured on the MI355X against
// 32-bit limbs, canonical after every butterfly, and a permutation of its own:
// that transform 687 -> 472 us, 48 transforms of 2^10..2^20 1549 -> 1110 us, a
// lone 2^20 181 -> 118 us, 2^18 52.7 -> 45 us, 2^12 21.9 -> 17.5 us.
//
// Decimation in frequency (DIF, the reference's butterfly) takes natural
// order to bit-reversed order; running the same stages backwards with the
// transposed butterfly (a, b) -> (a + t b, a - t b) (decimation in time,
// DIT) takes bit-reversed order back to natural order. The operator keeps
// the reference's natural-in, natural-out contract: its last pass takes the
// columns of a tile from the top bits of the index, which the bit reversal
// makes the lowest ones, and stores every element at its natural place (out
// of a workspace that the pass before wrote: the permutation costs no pass
// over memory of its own). The Groth16 H pipeline needs no permutation at
// all: DIF for its inverse transforms, DIT for its coset transform, with the
// coset powers and 1/n folded into the first load or the last store of a
// pass, and the quotient h left in bit-reversed order, matched by a
// bit-reversed copy of the H query points.
#include <algorithm>
#include <mutex>
#include <string>
#include <vector>
#include "common.hpp"
#include "field.hpp"
#include "fr29.hpp"
#include "host_ec.hpp"
#include "limb29.hpp"

namespace hzk {

// Tiles of 2^TB elements, TB = 9 or 10, 2^(TB-LE) threads each holding 2^LE
// elements: LE = 2 where that gives every SIMD two waves, else LE = 1 (a lone
// transform below 2^19 points: a lone 2^18 takes 45 us with 2 elements a
// thread, 58 with 4; 2^19 73 and 67). The largest tile that still gives every
// CU two workgroups (LE = 2), or one (LE = 1); 2^11 elements leave room for
// fewer waves and ran a third slower.
static constexpr int NTT_TILE_BITS = 10;   // largest tile
template <int TB, int LE>
constexpr int ntt_threads() { return (1 << TB) >> LE; }
static constexpr int NTT_MAX_LOG = 26;

// Tables are in the 2^261 Montgomery form (value * 2^261 mod r), so that a
// product with an element in the library's 2^256 form keeps that form. A
// caller's own tables are in the 2^256 form and are scaled as they are read.
constexpr int NTT_DIT = 1;    // stages backwards, transposed butterfly
constexpr int NTT_REV = 2;    // store at bit-reversed places (dst other than src unless one tile holds the transform)
constexpr int NTT_RAW = 4;    // tw is a caller's table
constexpr int NTT_LAST = 8;   // last pass: canonical values

// one pass of one transform over its tiles [tile_begin, next tile_begin)
struct NttPassDesc {
    const fr_t* src;
    fr_t* dst;
    const fr_t* tw;      // w^e (or w^-e), e < n/2
    const fr_t* pre;     // x[j] *= pre[j] as the pass loads (first pass only), or null
    const fr_t* post;    // x[p] *= post[p], p the place stored to (last pass only), or null
    const fr_t* scale;   // every element times this factor (2^256 form; last pass only), or null
    int k, s0, R, gl, hb, flags;
    uint64_t tile_begin;
};

// ---- elements
HZK_DEV limbs29 fr_unpack(const fr_t& x) {
    return limbs29::unpack(make_uint4(x.l[0], x.l[1], x.l[2], x.l[3]), make_uint4(x.l[4], x.l[5], x.l[6], x.l[7]));
}
HZK_DEV fr_t fr_pack(const limbs29& v) {
    uint4 a, b;
    v.pack(a, b);
    fr_t x;
    x.l[0] = a.x, x.l[1] = a.y, x.l[2] = a.z, x.l[3] = a.w, x.l[4] = b.x, x.l[5] = b.y, x.l[6] = b.z, x.l[7] = b.w;
    return x;
}
// 32 x, reduced: a 2^256-form factor made a 2^261-form one
HZK_DEV limbs29 fr_times32(const limbs29& x) {
    limbs29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = x.l[i] << 2;
    r = r.norm();
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] <<= 2;
    r = r.norm();
    return fr_reduce(r.twice());
}
// a twiddle read from the pass's table
HZK_DEV limbs29 fr_twiddle(const fr_t& t, int flags) {
    limbs29 w = fr_unpack(t);
    if (flags & NTT_RAW) w = fr_times32(w);
    return w;
}
HZK_DEV void fr_mul(limbs29& r, const limbs29& a, const limbs29& b) {
    __builtin_amdgcn_sched_barrier(0);
    scan29(Mul29<Fr29Mod>(r, a, b));
    __builtin_amdgcn_sched_barrier(0);
}
HZK_DEV void fr_mul2(limbs29& r0, const limbs29& a0, const limbs29& b0, limbs29& r1, const limbs29& a1, const limbs29& b1) {
    scan29(Mul29<Fr29Mod>(r0, a0, b0), Mul29<Fr29Mod>(r1, a1, b1));
}

// LDS slot of tile element e: two 16-byte planes and a 4-byte one (limbs 0-3,
// 4-7, 8), so lanes reading consecutive elements touch consecutive words; the
// low 3 bits are XOR-ed with the next 3 so that lanes that hold 4 (or 2)
// consecutive elements each, in the lowest stages, spread over the banks
HZK_DEV uint32_t lds_slot(uint32_t e) { return e ^ ((e >> 3) & 7); }
template <int TB>
constexpr int ntt_lds_vecs() { return (2 << TB) + (1 << (TB - 2)); }   // uint4 of a tile's LDS
template <int TB>
HZK_DEV void lds_put(uint4* sh, uint32_t e, const limbs29& v) {
    const uint32_t s = lds_slot(e);
    sh[s] = make_uint4(v.l[0], v.l[1], v.l[2], v.l[3]);
    sh[s + (1u << TB)] = make_uint4(v.l[4], v.l[5], v.l[6], v.l[7]);
    ((int32_t*)(sh + (2u << TB)))[s] = v.l[8];
}
template <int TB>
HZK_DEV limbs29 lds_get(const uint4* sh, uint32_t e) {
    const uint32_t s = lds_slot(e);
    const uint4 a = sh[s], b = sh[s + (1u << TB)];
    return {{(int32_t)a.x, (int32_t)a.y, (int32_t)a.z, (int32_t)a.w, (int32_t)b.x, (int32_t)b.y, (int32_t)b.z, (int32_t)b.w,
             ((const int32_t*)(sh + (2u << TB)))[s]}};
}

// Between the writes and the reads of an exchange. A slot is written by the
// thread that last read it, so no barrier is needed before the writes; and
// none at all when every element stays in its wave (LDS accesses of a wave
// are in order), which is the case while the register bits of both chunks lie
// below the wave's part of the tile index.
HZK_DEV void lds_exchange(bool in_wave) {
    if (in_wave) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    else __syncthreads();
}

// Geometry of one tile of a pass (stages s0 .. s0+R-1 of a 2^k transform).
// Tile element e = (h, m, g): row m (R bits, the butterfly dimension) above
// gl column bits g taken from the bits below the rows, or below hb column bits
// h taken from the top bits of the index (last pass with bit-reversed stores).
// The DIF stage s0 + st pairs rows differing in bit R - 1 - st, i.e. tile bit
// gl + R - 1 - st, with twiddle w^((((m & mask) << low) | column) << s).
struct NttTile {
    int k, s0, R, gl, hb, low, TB;
    uint32_t colbase, base;   // indices fit 32 bits (k <= 26)
    HZK_DEV NttTile(const NttPassDesc& d, uint32_t b) : k(d.k), s0(d.s0), R(d.R), gl(d.gl), hb(d.hb) {
        low = k - s0 - R;
        TB = R + gl + hb;
        const uint32_t lchunks = (1u << low) >> gl;
        const uint32_t hi = b / lchunks, lc = b % lchunks;
        base = (hi << (k - s0)) | (lc << gl);
        colbase = lc << gl;
    }
    HZK_DEV uint32_t row(uint32_t e) const { return (e >> gl) & ((1u << R) - 1); }
    HZK_DEV uint32_t gidx(uint32_t e) const {
        return base + (row(e) << low) + (e & ((1u << gl) - 1)) + (hb ? (e >> (gl + R)) << (k - hb) : 0);
    }
    // twiddle exponent of the butterfly of local stage st whose lower element is e
    HZK_DEV uint32_t texp(uint32_t e, int st) const {
        const int mp = R - 1 - st;
        const uint32_t m = (e >> gl) & ((1u << mp) - 1);
        return ((m << low) | colbase | (e & ((1u << gl) - 1))) << (s0 + st);
    }
    HZK_DEV uint32_t out(uint32_t e, int flags) const {
        const uint32_t i = gidx(e);
        return (flags & NTT_REV) ? __brev(i) >> (32 - k) : i;
    }
};

// Two stages over the thread's four elements (tile indices eb | i << L): the
// first pairs (0, 2) and (1, 3) with twiddles w0, w1, the second (0, 1) and
// (2, 3), both with w2. A product's operand may hold a sum or difference of
// two normalized values; elements leave normalized. One product at a time:
// three waves share the SIMD, and the registers saved are what lets them.
HZK_DEV void ntt_dif2(limbs29* v, const fr_t& t0, const fr_t& t1, const fr_t& t2, int flags) {
    limbs29 d = v[0] - v[2], e = v[1] - v[3];
    v[0] = v[0] + v[2];
    v[1] = v[1] + v[3];
    fr_mul(v[2], d, fr_twiddle(t0, flags));
    fr_mul(v[3], e, fr_twiddle(t1, flags));
    d = v[0] - v[1];
    e = v[2] - v[3];
    v[0] = (v[0] + v[1]).norm();
    v[2] = (v[2] + v[3]).norm();
    const limbs29 w = fr_twiddle(t2, flags);
    fr_mul(v[1], d, w);
    fr_mul(v[3], e, w);
}
HZK_DEV void ntt_dit2(limbs29* v, const fr_t& t0, const fr_t& t1, const fr_t& t2, int flags) {
    limbs29 p;
    {
        const limbs29 w = fr_twiddle(t2, flags);
        fr_mul(p, v[1], w);
        v[1] = v[0] - p, v[0] = v[0] + p;
        fr_mul(p, v[3], w);
        v[3] = v[2] - p, v[2] = v[2] + p;
    }
    fr_mul(p, v[2], fr_twiddle(t0, flags));
    v[2] = (v[0] - p).norm(), v[0] = (v[0] + p).norm();
    fr_mul(p, v[3], fr_twiddle(t1, flags));
    v[3] = (v[1] - p).norm(), v[1] = (v[1] + p).norm();
}
// one stage pairing bit IB of the element number, twiddles t0, t1
template <bool DIT, int IB>
HZK_DEV void ntt_one(limbs29* v, const fr_t& t0, const fr_t& t1, int flags) {
    constexpr int lo[2] = {0, IB ? 1 : 2}, step = 1 << IB;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        limbs29 &a = v[lo[j]], &b = v[lo[j] + step];
        const limbs29 w = fr_twiddle(j ? t1 : t0, flags);
        if (!DIT) {
            const limbs29 d = a - b;
            a = (a + b).norm();
            fr_mul(b, d, w);
        } else {
            limbs29 p;
            fr_mul(p, b, w);
            b = (a - p).norm(), a = (a + p).norm();
        }
    }
}
// The last two stages of a DIF over the library's tables: of the four
// butterflies' twiddles only w (the 4th root of unity) is not one
HZK_DEV void ntt_last4(limbs29* v, const fr_t* __restrict__ tw, int k) {
    const limbs29 w = fr_unpack(tw[1u << (k - 2)]), d0 = v[0] - v[2], d1 = v[1] - v[3];
    const limbs29 s0 = v[0] + v[2], s1 = v[1] + v[3];
    limbs29 p;
    fr_mul(p, d1, w);
    v[0] = s0 + s1, v[1] = s0 - s1, v[2] = d0 + p, v[3] = d0 - p;
}

// x[i] *= tab[i] for the thread's 2^LE elements, interleaved in pairs
template <int LE>
HZK_DEV void mul_pre(limbs29* v, const NttTile& T, const fr_t* __restrict__ tab, uint32_t eb, int L) {
#pragma unroll
    for (int i = 0; i < (1 << LE); i += 2) {
        const limbs29 a = fr_unpack(tab[T.gidx(eb | ((uint32_t)i << L))]), b = fr_unpack(tab[T.gidx(eb | ((uint32_t)(i + 1) << L))]);
        fr_mul2(v[i], v[i], a, v[i + 1], v[i + 1], b);
    }
}

// the thread's 2^LE elements to memory: [0, 2r) between passes, canonical
// (after the optional factors) at the end
template <int LE>
HZK_DEV void ntt_store(limbs29* v, const NttPassDesc& d, const NttTile& T, uint32_t eb, int L) {
    uint32_t p[1 << LE];
#pragma unroll
    for (int i = 0; i < (1 << LE); ++i) p[i] = T.out(eb | ((uint32_t)i << L), d.flags);
    if (d.post)
#pragma unroll
        for (int i = 0; i < (1 << LE); i += 2) {
            const limbs29 a = fr_unpack(d.post[p[i]]), b = fr_unpack(d.post[p[i + 1]]);
            v[i] = v[i].norm(), v[i + 1] = v[i + 1].norm();
            fr_mul2(v[i], v[i], a, v[i + 1], v[i + 1], b);
        }
    if (d.scale) {
        const limbs29 f = fr_times32(fr_unpack(*d.scale));
#pragma unroll
        for (int i = 0; i < (1 << LE); i += 2) {
            v[i] = v[i].norm(), v[i + 1] = v[i + 1].norm();
            fr_mul2(v[i], v[i], f, v[i + 1], v[i + 1], f);
        }
    }
#pragma unroll
    for (int i = 0; i < (1 << LE); ++i) {
        limbs29 r = fr_reduce(v[i]);
        if (d.flags & NTT_LAST) r = fr_canonical(r);
        d.dst[p[i]] = fr_pack(r);
    }
}

// One tile of a pass: stages in chunks of two. DIF runs local stages 0..R-1
// from the first chunk (tile bits TB-1..) down; DIT runs them in reverse. A
// thread's 4 elements for a chunk span the 2 tile bits [L, L + 2) that contain
// the chunk's stage bits; its other tile bits come from the thread index (low
// bits first, so a wave's lanes read consecutive elements wherever L > 0). A
// chunk's twiddles are loaded before the exchange that leads to it.
// Bounds, in units of r: an element enters in [0, 2). DIF sums double in both
// directions; a product of a difference (-2^(s+1), 2^(s+1)) after s stages lies
// above -2^(s+1)/169 (twice that with a caller's table), so after eight stages
// sums stay in (-4, 512). The last two stages over the library's tables leave
// differences unmultiplied: after six stages sums of two are in (-2, 256), their
// differences in (-258, 258). A pass of more than eight stages reduces every
// element after the sixth. DIT elements grow by less than 1.7 a stage.
template <bool DIT, int TB>
HZK_DEV void ntt_tile(const NttPassDesc& d, uint32_t b, uint4* sh) {
    constexpr int LE = 2, E = 4;
    const NttTile T(d, b);
    const uint32_t t = threadIdx.x;
    const bool active = t < (1u << (T.TB - LE));
    limbs29 v[E];
    fr_t t0, t1, t2;
    const int R = d.R, nch = (R + 1) / 2;
    // chunk c: first DIF stage stA, len stages, element bits [L, L + 2)
    int stA, len, L;
    uint32_t eb;
    auto chunk = [&](int c) {
        stA = DIT ? max(0, R - 2 * (c + 1)) : 2 * c;
        len = DIT ? R - 2 * c - stA : min(2, R - stA);
        const int blo = T.gl + R - stA - len;
        L = min(blo, T.TB - LE);
        eb = (t & ((1u << L) - 1)) | ((t >> L) << (L + LE));
    };
    auto twiddles = [&]() {
        if (!active) return;
        const bool low = len == 1 && T.gl + R - 1 - stA == L;   // one stage on the lower element bit
        t0 = d.tw[T.texp(eb, stA)];
        t1 = d.tw[T.texp(eb | ((low ? 2u : 1u) << L), stA)];
        if (len == 2) t2 = d.tw[T.texp(eb, stA + 1)];
    };
    chunk(0);
    if (active) {
#pragma unroll
        for (int i = 0; i < E; ++i) v[i] = fr_unpack(d.src[T.gidx(eb | ((uint32_t)i << L))]);
        twiddles();
        if (d.pre) mul_pre<LE>(v, T, d.pre, eb, L);
    }
    for (int c = 0;; ++c) {
        if (active) {
            if (!DIT && R > 8 && c == 3) {
#pragma unroll
                for (int i = 0; i < E; ++i) v[i] = fr_reduce(v[i]);
            }
            if (len == 2) {
                if constexpr (DIT) ntt_dit2(v, t0, t1, t2, d.flags);
                else if (L == 0 && d.s0 + R == d.k && !(d.flags & NTT_RAW)) ntt_last4(v, d.tw, d.k);
                else ntt_dif2(v, t0, t1, t2, d.flags);
            } else {
                if (T.gl + R - 1 - stA == L) ntt_one<DIT, 0>(v, t0, t1, d.flags);
                else ntt_one<DIT, 1>(v, t0, t1, d.flags);
            }
        }
        if (c + 1 == nch) break;
        const uint32_t eb_prev = eb;
        const int L_prev = L;
        chunk(c + 1);
        twiddles();
        if (active)
#pragma unroll
            for (int i = 0; i < E; ++i) lds_put<TB>(sh, eb_prev | ((uint32_t)i << L_prev), v[i]);
        lds_exchange(max(L, L_prev) <= 6);
        if (active)
#pragma unroll
            for (int i = 0; i < E; ++i) v[i] = lds_get<TB>(sh, eb | ((uint32_t)i << L));
    }
    if (active) ntt_store<LE>(v, d, T, eb, L);
}

// The same pass with two elements per thread (one butterfly per stage, an
// exchange between stages), for lone transforms that are latency-bound: each
// stage's twiddle is loaded one stage ahead, so no butterfly waits for a
// global load. DIF sums are reduced every third stage.
template <bool DIT, int TB>
HZK_DEV void ntt_tile_r2(const NttPassDesc& d, uint32_t b, uint4* sh) {
    const NttTile T(d, b);
    const uint32_t t = threadIdx.x;
    const bool active = t < (1u << (T.TB - 1));
    const int R = d.R;
    // executed step i runs local stage st(i) on tile bit L(i) = gl + R - 1 - st(i);
    // the thread's pair is (eb(i), eb(i) | 2^L(i))
    auto stage_of = [&](int i) { return DIT ? R - 1 - i : i; };
    auto bit_of = [&](int i) { return T.gl + R - 1 - stage_of(i); };
    auto pair_base = [&](int L) { return (t & ((1u << L) - 1)) | ((t >> L) << (L + 1)); };
    limbs29 v[2];
    fr_t w, wn;
    uint32_t eb = 0;
    int L = 0;
    if (active) w = d.tw[T.texp(pair_base(bit_of(0)), stage_of(0))];
    for (int i = 0; i < R; ++i) {
        const int Li = bit_of(i);
        const uint32_t ebi = pair_base(Li);
        if (active && i + 1 < R) wn = d.tw[T.texp(pair_base(bit_of(i + 1)), stage_of(i + 1))];
        if (i == 0) {
            if (active) {
                v[0] = fr_unpack(d.src[T.gidx(ebi)]);
                v[1] = fr_unpack(d.src[T.gidx(ebi | (1u << Li))]);
                if (d.pre) mul_pre<1>(v, T, d.pre, ebi, Li);
            }
        } else if (min(L, Li) < 6) {
            // the pair bits of this stage and the last differ by one; the
            // threads that trade elements differ in thread bit pb = min(L, Li)
            // and share a wave: swap one element across lanes, no barrier.
            // Thread bit pb = b keeps v_b and receives the partner's element
            // into v_(1-b) (both for DIF, pb = Li, and DIT, pb = L).
            const int pb = min(L, Li);
            const bool hi = (t >> pb) & 1;
#pragma unroll
            for (int q = 0; q < 9; ++q) {
                const int32_t got = __shfl_xor(hi ? v[0].l[q] : v[1].l[q], 1 << pb, 64);
                v[0].l[q] = hi ? got : v[0].l[q];
                v[1].l[q] = hi ? v[1].l[q] : got;
            }
        } else {
            if (active) {
                lds_put<TB>(sh, eb, v[0]);
                lds_put<TB>(sh, eb | (1u << L), v[1]);
            }
            __syncthreads();
            if (active) {
                v[0] = lds_get<TB>(sh, ebi);
                v[1] = lds_get<TB>(sh, ebi | (1u << Li));
            }
        }
        if (active) {
            const limbs29 wl = fr_twiddle(w, d.flags);
            if (!DIT) {
                const limbs29 df = v[0] - v[1], s = v[0] + v[1];
                // the very last stage's twiddles are one
                if (d.s0 + stage_of(i) + 1 == d.k && !(d.flags & NTT_RAW)) v[1] = df;
                else fr_mul(v[1], df, wl);
                v[0] = i % 3 == 2 ? fr_reduce(s) : s.norm();
            } else {
                limbs29 p;
                fr_mul(p, v[1], wl);
                v[1] = (v[0] - p).norm();
                v[0] = (v[0] + p).norm();
            }
        }
        w = wn;
        eb = ebi;
        L = Li;
    }
    if (active) ntt_store<1>(v, d, T, eb, L);
}

template <class D>
HZK_DEV uint32_t find_desc(const D* d, uint32_t nd, uint64_t gid) {
    uint32_t lo = 0, hi = nd;
    while (hi - lo > 1) {
        uint32_t mid = (lo + hi) >> 1;
        if (d[mid].tile_begin <= gid) lo = mid; else hi = mid;
    }
    return lo;
}

template <bool DIT, int TB, int LE>
__global__ void __launch_bounds__((ntt_threads<TB, LE>()), LE == 2 ? 3 : 2) k_ntt_pass(NttPassDesc d) {
    __shared__ uint4 sh[ntt_lds_vecs<TB>()];
    if constexpr (LE == 1) ntt_tile_r2<DIT, TB>(d, blockIdx.x, sh);
    else ntt_tile<DIT, TB>(d, blockIdx.x, sh);
}

template <int TB, int LE>
__global__ void __launch_bounds__((ntt_threads<TB, LE>()), LE == 2 ? 3 : 2) k_ntt_pass_batch(const NttPassDesc* __restrict__ pd, uint32_t npd) {
    __shared__ uint4 sh[ntt_lds_vecs<TB>()];
    const NttPassDesc& d = pd[find_desc(pd, npd, blockIdx.x)];
    const uint32_t b = (uint32_t)(blockIdx.x - d.tile_begin);
    if constexpr (LE == 1) {
        if (d.flags & NTT_DIT) ntt_tile_r2<true, TB>(d, b, sh);
        else ntt_tile_r2<false, TB>(d, b, sh);
    } else {
        if (d.flags & NTT_DIT) ntt_tile<true, TB>(d, b, sh);
        else ntt_tile<false, TB>(d, b, sh);
    }
}

// transforms of 1, 2 and 4 points, natural order with all factors: a lane per
// element, so a launch waits for one product per stage and factor. 64 scaled
// transforms in a captured batch: 301 -> 161 us for 2 points and 642 -> 228 for
// 4, against one lane for all elements.
__global__ void __launch_bounds__(64) k_ntt_tiny(NttPassDesc d) {
    const int n = 1 << d.k, j = threadIdx.x;
    if (j >= n) return;
    fr29 v = fr29::unpack(d.src[j]);
    if (d.pre) v = fr29::mul(v, fr29::unpack(d.pre[j]));
    for (int h = n / 2, s = 0; h > 0; h >>= 1, ++s) {
        fr29 o;
#pragma unroll
        for (int i = 0; i < 9; ++i) o.l[i] = (uint32_t)__shfl_xor((int)v.l[i], h);
        if (j & h) {
            v = fr29::sub2(o, v);
            if (h > 1 || (d.flags & NTT_RAW)) {   // the library's last twiddle is one
                fr29 w = fr29::unpack(d.tw[(j & (h - 1)) << s]);
                if (d.flags & NTT_RAW) w = w.times32();
                v = fr29::mul(v, w);
            }
        } else {
            v = fr29::add(v, o);
        }
        v = v.reduce();
    }
    const int p = d.k == 2 ? ((j & 1) << 1) | (j >> 1) : j;
    if (d.post) v = fr29::mul(v, fr29::unpack(d.post[p]));
    if (d.scale) v = fr29::mul(v, fr29::unpack(*d.scale).times32());
    d.dst[p] = v.canonical().pack();
}

// In-place bit-reverse permutation of one transform (k >= 8) with the factors
// that a last pass would have applied, for calls that cannot use the workspace
// (no room for it, or the caller captures the stream). In 16 x 16 blocks
// through LDS: index i = (a, m, b) with a its top 4 bits, b its low 4 and m the
// k - 8 bits between, so rev(i) = (rev b, rev m, rev a): block m (every a, b)
// and block rev(m) trade places, transposed, and every global access is a run
// of 16 consecutive elements. One workgroup per m; the one with m > rev(m) has
// nothing to do.
__global__ void __launch_bounds__(256) k_ntt_permute(NttPassDesc d) {
    __shared__ fr_t blk[2][16 * 17];   // rows padded to 17 elements
    const int k = d.k, mb = k - 8;
    const uint32_t m = blockIdx.x, mr = mb ? __brev(m) >> (32 - mb) : 0;
    if (m > mr) return;
    const uint32_t t = threadIdx.x, a = t >> 4, b = t & 15;
    const size_t stride_a = (size_t)1 << (k - 4);
    auto at = [&](uint32_t aa, uint32_t mm, uint32_t bb) { return (size_t)aa * stride_a + ((size_t)mm << 4) + bb; };
    blk[0][a * 17 + b] = d.dst[at(a, m, b)];
    blk[1][a * 17 + b] = d.dst[at(a, mr, b)];
    __syncthreads();
    auto put = [&](size_t p, const fr_t& x) {
        fr29 v = fr29::unpack(x);
        if (d.post) v = fr29::mul(v, fr29::unpack(d.post[p]));
        if (d.scale) v = fr29::mul(v, fr29::unpack(*d.scale).times32());
        d.dst[p] = v.canonical().pack();
    };
    // destination (a, mr, b) takes source (rev b, m, rev a), and (a, m, b) takes (rev b, mr, rev a)
    const uint32_t src = (__brev(b) >> 28) * 17 + (__brev(a) >> 28);
    put(at(a, mr, b), blk[0][src]);
    if (m != mr) put(at(a, m, b), blk[1][src]);
}

// out[p] = tab[rev_k(p)] * scale: a bit-reversed copy of a coset table
__global__ void __launch_bounds__(256) k_bitrev_table(fr_t* __restrict__ out, const fr_t* __restrict__ tab, int k,
                                                      const fr_t* __restrict__ scale) {
    size_t p = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= ((size_t)1 << k)) return;
    size_t r = k ? (size_t)(__brev((uint32_t)p) >> (32 - k)) : 0;
    out[p] = scale ? tab[r] * *scale : tab[r];
}

// out[e] = c w^e for e < n, from sq[b] = w^(2^b), sq[63] = c
__global__ void __launch_bounds__(256) k_powers(fr_t* __restrict__ out, size_t n, const fr_t* __restrict__ sq) {
    size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= n) return;
    fr_t acc = sq[63];
    for (int b = 0; (e >> b) != 0; ++b)
        if ((e >> b) & 1) acc = acc * sq[b];
    out[e] = acc;
}

// ------------------------------------------------------------------ host side
// Fr constants in Montgomery form: primitive 2^k-th roots of unity
// w_k = 5^((r-1)/2^k) (5 generates Fr*, alt_bn128_init.cu:50) and inverses
// are derived on the host from w_28, the value the reference stores as
// root_of_unity (alt_bn128_init.cu:51).
static host::Fr fr_from_u64(uint64_t v) {
    host::Fr t{{v, 0, 0, 0}};
    host::Fr r2;
    std::memcpy(r2.v, host::FR.r2, 32);
    return t * r2;
}
static host::Fr root_of_unity(int k) {
    // w_28 = 5^t, t = (r-1)/2^28
    static const uint64_t t[4] = {0x9b9709143e1f593fULL, 0x181585d2833e8487ULL, 0x131a029b85045b68ULL, 0x000000030644e72eULL};
    host::Fr w = fr_from_u64(5).pow(t);
    for (int i = 28; i > k; --i) w = w.sqr();
    return w;
}

// per transform size, in the 2^261 form: forward / inverse twiddles (n/2
// each), coset powers g^j and g^-j / n (n each), and (built when the Groth16 H
// pipeline first asks) the bit-reversed coset tables g^rev(p) / n and g^-rev(p)
// / n; 1/n in the 2^256 form. Built on first use, kept for the context
struct NttTables {
    fr_t* tw[2] = {nullptr, nullptr};
    fr_t* coset[2] = {nullptr, nullptr};
    fr_t* coset_rev[2] = {nullptr, nullptr};
    fr_t* ninv = nullptr;
};
struct NttCache {
    NttTables t[NTT_MAX_LOG + 1];
};

static NttCache& cache_of(hzk_ctx* ctx) {
    if (!ctx->ntt_cache) ctx->ntt_cache = new NttCache();
    return *(NttCache*)ctx->ntt_cache;
}

void ntt_release(hzk_ctx* ctx) {
    if (ctx->ntt_ws) {
        (void)hipFreeAsync(ctx->ntt_ws, ctx->stream);
        (void)hipStreamSynchronize(ctx->stream);
        ctx->ntt_ws = nullptr;
        ctx->ntt_ws_bytes = 0;
    }
    if (!ctx->ntt_cache) return;
    NttCache& c = *(NttCache*)ctx->ntt_cache;
    for (auto& t : c.t)
        for (auto p : {t.tw[0], t.tw[1], t.coset[0], t.coset[1], t.coset_rev[0], t.coset_rev[1], t.ninv})
            if (p) (void)hipFree(p);
    delete &c;
    ctx->ntt_cache = nullptr;
}

// out[e] = c w^e, e < n
static int fill_powers(hzk_ctx* ctx, fr_t* out, size_t n, host::Fr w, host::Fr c) {
    std::vector<host::Fr> sq(64);
    for (int b = 0; b < 63; ++b) { sq[b] = w; w = w.sqr(); }
    sq[63] = c;
    fr_t* dsq = nullptr;
    HZK_HIP(ctx, hipMalloc(&dsq, 64 * 32));
    HZK_HIP(ctx, hipMemcpy(dsq, sq.data(), 64 * 32, hipMemcpyHostToDevice));
    hipLaunchKernelGGL(k_powers, dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, out, n, (const fr_t*)dsq);
    HZK_HIP(ctx, hipGetLastError());
    HZK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    HZK_HIP(ctx, hipFree(dsq));
    return 0;
}

static int ensure_tables(hzk_ctx* ctx, int logn, NttTables** out) {
    NttTables& t = cache_of(ctx).t[logn];
    *out = &t;
    if (t.ninv) return 0;
    size_t n = (size_t)1 << logn;
    size_t half = n / 2 ? n / 2 : 1;
    host::Fr w = root_of_unity(logn), wi = w.inverse();
    host::Fr g = fr_from_u64(5), gi = g.inverse();
    host::Fr ninv = fr_from_u64(n).inverse();
    const host::Fr to261 = fr_from_u64(32);
    for (int d = 0; d < 2; ++d) {
        HZK_HIP(ctx, device_malloc(ctx, (void**)&t.tw[d], half * 32));
        HZK_HIP(ctx, device_malloc(ctx, (void**)&t.coset[d], n * 32));
        int rc = fill_powers(ctx, t.tw[d], half, d ? wi : w, to261);
        if (rc) return rc;
        rc = fill_powers(ctx, t.coset[d], n, d ? gi : g, d ? to261 * ninv : to261);
        if (rc) return rc;
    }
    fr_t* ni = nullptr;
    HZK_HIP(ctx, hipMalloc(&ni, 32));
    HZK_HIP(ctx, hipMemcpy(ni, ninv.v, 32, hipMemcpyHostToDevice));
    t.ninv = ni;
    return 0;
}

static int ensure_rev_tables(hzk_ctx* ctx, int logn, NttTables* t) {
    if (t->coset_rev[0]) return 0;
    const size_t n = (size_t)1 << logn;
    for (int d = 0; d < 2; ++d) {
        HZK_HIP(ctx, device_malloc(ctx, (void**)&t->coset_rev[d], n * 32));
        hipLaunchKernelGGL(k_bitrev_table, dim3(blocks_for(n, 256)), dim3(256), 0, ctx->stream, t->coset_rev[d],
                           (const fr_t*)t->coset[d], logn, d ? (const fr_t*)nullptr : (const fr_t*)t->ninv);
        HZK_HIP(ctx, hipGetLastError());
    }
    HZK_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return 0;
}

static int log2_exact(size_t n) {
    int k = 0;
    while (((size_t)1 << k) < n) ++k;
    return ((size_t)1 << k) == n ? k : -1;
}

// one pass: stages s0 .. s0+R-1, columns as in NttTile
struct NttPlanPass { int s0, R, gl, hb; };

// Pass plan of a 2^k transform in DIF order over tiles of 2^TB elements. rev:
// natural order out, the last pass storing bit-reversed from tiles of 2^hb
// runs of 2^R elements (hb = TB - R, at least 2 so that it stores runs of 128
// bytes or more, 1 where that saves a pass); the passes before it keep as
// many columns. Otherwise the lowest min(k, TB) stages (contiguous rows) form
// the last pass, the rest split evenly into passes of <= TB - 2 stages. A DIT
// run executes the same passes in reverse order. 3 <= k <= NTT_MAX_LOG, TB >= 9
// or k <= TB; returns the number of passes.
static constexpr int NTT_MAX_PASSES = 4;
static int plan_passes(int k, int TB, bool rev, NttPlanPass* out) {
    if (k <= TB) {
        out[0] = {0, k, 0, 0};
        return 1;
    }
    const int last = rev ? 0 : TB, rest = k - last;
    int np = (rest + TB - 3) / (TB - 2);
    if (rev && (rest + TB - 2) / (TB - 1) < np) np = (rest + TB - 2) / (TB - 1);
    int s0 = 0;
    for (int p = 0; p < np; ++p) {
        const int R = rest / np + (p < rest % np ? 1 : 0);
        if (rev && p + 1 == np) {
            out[p] = {s0, R, 0, std::min(TB - R, s0)};
            return np;
        }
        out[p] = {s0, R, std::min(TB - R, k - s0 - R), 0};
        s0 += R;
    }
    out[np] = {s0, last, 0, 0};
    return np + 1;
}
static_assert((NTT_MAX_LOG - 9 + 6) / 7 + 1 <= NTT_MAX_PASSES && (NTT_MAX_LOG + 7) / 8 <= NTT_MAX_PASSES, "passes over tiles of 2^9");

// elements per thread (2^LE) of a launch over `elems` elements: 4 while
// that still gives every SIMD two waves, else 2 (more threads and more
// exchanges: such transforms are latency-bound, not issue-bound)
static int elem_bits_for(hzk_ctx* ctx, uint64_t elems) {
    const uint64_t want = 2ull * 4 * 64 * (uint64_t)ctx->num_cus;   // threads for two waves per SIMD
    return (elems >> 2) >= want ? 2 : 1;
}
// tile bits of such a launch: the largest tile that gives every CU two
// workgroups (LE = 2) or one (LE = 1: fewer passes count for more)
static int tile_bits_for(hzk_ctx* ctx, uint64_t elems, int le) {
    int TB = NTT_TILE_BITS;
    while (TB > 9 && (elems >> TB) < (uint64_t)le * (uint64_t)ctx->num_cus) --TB;
    return TB;
}

// The transform's passes as descriptors (tile_begin 0). Natural-order output
// (rev) of more than one pass goes through ws (n elements): the first pass
// writes it, the last reads it. ws null: everything stays in place, the last
// descriptor of *permute (k > 0) is left to k_ntt_permute.
static void build_passes(fr_t* x, int k, int TB, bool dit, bool rev, const fr_t* tw, bool raw, const fr_t* pre, const fr_t* post,
                         const fr_t* scale, fr_t* ws, std::vector<NttPassDesc>& out, NttPassDesc* permute) {
    NttPlanPass plan[NTT_MAX_PASSES];
    const int m = plan_passes(k, TB, rev && (ws || k <= TB), plan);
    if (dit) std::reverse(plan, plan + m);
    const bool swap = rev && m > 1 && ws, later = rev && m > 1 && !ws;
    permute->k = 0;
    for (int p = 0; p < m; ++p) {
        const bool first = p == 0, last = p + 1 == m;
        NttPassDesc d{};
        d.src = swap && !first ? ws : x;
        d.dst = swap && !last ? ws : x;
        d.tw = tw;
        d.pre = first ? pre : nullptr;
        d.k = k, d.s0 = plan[p].s0, d.R = plan[p].R, d.gl = plan[p].gl, d.hb = plan[p].hb;
        d.flags = (dit ? NTT_DIT : 0) | (raw ? NTT_RAW : 0);
        if (last) {
            d.flags |= NTT_LAST | (rev && !later ? NTT_REV : 0);
            if (!later) d.post = post, d.scale = scale;
        }
        out.push_back(d);
    }
    if (later) {
        *permute = NttPassDesc{};
        permute->dst = x, permute->k = k, permute->post = post, permute->scale = scale;
    }
}

// workspace of `elems` elements on ctx's stream, grown stream-ordered; null
// when the device has no room for it, and while the caller captures the
// stream (its graph must not hold a pointer that a later call may free)
static fr_t* ntt_workspace(hzk_ctx* ctx, uint64_t elems) {
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(ctx->stream, &capture) != hipSuccess || capture != hipStreamCaptureStatusNone) return nullptr;
    const size_t bytes = (size_t)elems * 32;
    if (ctx->ntt_ws_bytes >= bytes) return (fr_t*)ctx->ntt_ws;
    const size_t doubled = 2 * ctx->ntt_ws_bytes;   // slowly growing calls settle after a few steps
    if (ctx->ntt_ws) (void)hipFreeAsync(ctx->ntt_ws, ctx->stream);
    ctx->ntt_ws = nullptr;
    ctx->ntt_ws_bytes = 0;
    for (const size_t want : {std::max(bytes, doubled), bytes}) {
        if (hipMallocAsync(&ctx->ntt_ws, want, ctx->stream) == hipSuccess) {
            ctx->ntt_ws_bytes = want;
            return (fr_t*)ctx->ntt_ws;
        }
        (void)hipGetLastError();
        ctx->ntt_ws = nullptr;
    }
    return nullptr;
}

static uint64_t pass_tiles(const NttPassDesc& d) { return (uint64_t)1 << (d.k - d.R - d.gl - d.hb); }

template <int TB>
static void launch_pass(int le, hipStream_t st, const NttPassDesc& d) {
    const dim3 grid((unsigned)pass_tiles(d));
    const bool dit = d.flags & NTT_DIT;
    if (le == 1) {
        if (dit) hipLaunchKernelGGL((k_ntt_pass<true, TB, 1>), grid, dim3(ntt_threads<TB, 1>()), 0, st, d);
        else hipLaunchKernelGGL((k_ntt_pass<false, TB, 1>), grid, dim3(ntt_threads<TB, 1>()), 0, st, d);
    } else {
        if (dit) hipLaunchKernelGGL((k_ntt_pass<true, TB, 2>), grid, dim3(ntt_threads<TB, 2>()), 0, st, d);
        else hipLaunchKernelGGL((k_ntt_pass<false, TB, 2>), grid, dim3(ntt_threads<TB, 2>()), 0, st, d);
    }
}

// In-place transform with twiddle table tw (w^e, e < n/2; raw: a caller's, in
// the 2^256 form) and the reference's natural-in, natural-out contract;
// optional factor tables (2^261 form) and device factor (2^256 form).
static int ntt_run(hzk_ctx* ctx, fr_t* x, int k, const fr_t* tw, bool raw, const fr_t* pre, const fr_t* post, const fr_t* scale) {
    hipStream_t st = ctx->stream;
    TimedLaunch tl(ctx, "ntt_pass");
    if (k < 3) {
        NttPassDesc d{};
        d.src = d.dst = x, d.tw = tw, d.pre = pre, d.post = post, d.scale = scale, d.k = k, d.flags = raw ? NTT_RAW : 0;
        if (k > 0 || pre || post || scale) hipLaunchKernelGGL(k_ntt_tiny, dim3(1), dim3(64), 0, st, d);
        HZK_HIP(ctx, hipGetLastError());
        return 0;
    }
    const int le = elem_bits_for(ctx, (uint64_t)1 << k);
    const int TB = std::max(3, std::min(k, tile_bits_for(ctx, (uint64_t)1 << k, le)));
    std::vector<NttPassDesc> passes;
    NttPassDesc permute;
    build_passes(x, k, TB, false, true, tw, raw, pre, post, scale, k > TB ? ntt_workspace(ctx, (uint64_t)1 << k) : nullptr, passes,
                 &permute);
    for (const NttPassDesc& d : passes) {
        const int tb = d.R + d.gl + d.hb;   // the kernel's tile holds 2^tb <= 2^TB elements
        if (tb <= 9) launch_pass<9>(le, st, d);
        else launch_pass<10>(le, st, d);
    }
    if (permute.k) hipLaunchKernelGGL(k_ntt_permute, dim3(1u << (k - 8)), dim3(256), 0, st, permute);
    HZK_HIP(ctx, hipGetLastError());
    return 0;
}

int ntt_standard(hzk_ctx* ctx, fr_t* x, size_t deg, int inverse) {
    int k = log2_exact(deg);
    HZK_CHECK(ctx, k >= 0 && k <= NTT_MAX_LOG && k <= 28, HZK_ERR_INVALID, "ntt: deg %zu is not a power of two <= 2^%d", deg,
              NTT_MAX_LOG);
    NttTables* t;
    int rc = ensure_tables(ctx, k, &t);
    if (rc) return rc;
    return ntt_run(ctx, x, k, t->tw[inverse ? 1 : 0], false, nullptr, nullptr, inverse ? t->ninv : nullptr);
}

int coset_ntt(hzk_ctx* ctx, fr_t* x, size_t deg, int inverse) {
    int k = log2_exact(deg);
    HZK_CHECK(ctx, k >= 0 && k <= NTT_MAX_LOG, HZK_ERR_INVALID, "coset_ntt: deg %zu is not a power of two <= 2^%d", deg,
              NTT_MAX_LOG);
    NttTables* t;
    int rc = ensure_tables(ctx, k, &t);
    if (rc) return rc;
    // the coset powers ride on the first pass's loads, or (with 1/n) on the last pass's stores
    if (!inverse) return ntt_run(ctx, x, k, t->tw[0], false, t->coset[0], nullptr, nullptr);
    return ntt_run(ctx, x, k, t->tw[1], false, nullptr, t->coset[1], nullptr);
}

// Batched transforms. kind 0 NTT, 1 inverse NTT (scaled 1/n), 2 coset NTT,
// 3 coset inverse NTT, all natural order in and out; and, for the Groth16
// H pipeline (no permutation): 4 inverse NTT, natural in, bit-reversed out,
// unscaled; 5 coset NTT of bit-reversed coefficients c scaled by 1/n on the
// way in (x[p] * g^rev(p) / n), natural out; 6 coset inverse NTT, natural
// in, bit-reversed out, with g^-rev(p) / n applied on the way out. Pass p of
// every transform runs in round p, each round one launch over the tiles of
// every transform in it.
int ntt_batch(hzk_ctx* ctx, const NttJob* jobs, size_t count, int capture) {
    HZK_CHECK(ctx, jobs && count > 0, HZK_ERR_INVALID, "ntt batch: empty");
    std::vector<int> ks(count);
    std::vector<NttTables*> tabs(count);
    uint64_t all = 0;
    for (size_t i = 0; i < count; ++i) all += jobs[i].deg;
    const int LE = elem_bits_for(ctx, all);
    const int TB = tile_bits_for(ctx, all, LE);
    uint64_t ws_elems = 0;
    for (size_t i = 0; i < count; ++i) {
        HZK_CHECK(ctx, jobs[i].x && jobs[i].kind >= 0 && jobs[i].kind <= 6, HZK_ERR_INVALID, "ntt batch: bad job %zu", i);
        int k = log2_exact(jobs[i].deg);
        HZK_CHECK(ctx, k >= 0 && k <= NTT_MAX_LOG, HZK_ERR_INVALID, "ntt batch: deg %zu of job %zu is not a power of two <= 2^%d",
                  jobs[i].deg, i, NTT_MAX_LOG);
        HZK_CHECK(ctx, jobs[i].kind <= 3 || k >= 3, HZK_ERR_INVALID, "ntt batch: kind %d needs deg >= 8", jobs[i].kind);
        ks[i] = k;
        int rc = ensure_tables(ctx, k, &tabs[i]);
        if (!rc && jobs[i].kind >= 5) rc = ensure_rev_tables(ctx, k, tabs[i]);
        if (rc) return rc;
        if (jobs[i].kind <= 3 && k > TB) ws_elems += jobs[i].deg;
    }
    fr_t* const ws = ws_elems ? ntt_workspace(ctx, ws_elems) : nullptr;
    // the passes of each transform, one after the other; tiny ones and (without a workspace) permutations are launched singly
    std::vector<NttPassDesc> passes;
    std::vector<size_t> pass_begin(count + 1, 0);
    passes.reserve(2 * count);
    std::vector<NttPassDesc> tiny, permutes;
    size_t rounds = 0;
    uint64_t ws_at = 0;
    for (size_t i = 0; i < count; ++i) {
        const int kind = jobs[i].kind, inv = kind == 1 || kind == 3 || kind == 4 || kind == 6;
        const NttTables& t = *tabs[i];
        const fr_t* pre = kind == 2 ? t.coset[0] : kind == 5 ? t.coset_rev[0] : nullptr;
        const fr_t* post = kind == 3 ? t.coset[1] : kind == 6 ? t.coset_rev[1] : nullptr;
        const fr_t* scale = kind == 1 ? t.ninv : nullptr;
        fr_t* x = (fr_t*)jobs[i].x;
        pass_begin[i + 1] = passes.size();
        if (ks[i] < 3) {
            NttPassDesc d{};
            d.src = d.dst = x, d.tw = t.tw[inv], d.pre = pre, d.post = post, d.scale = scale, d.k = ks[i];
            tiny.push_back(d);
            continue;
        }
        NttPassDesc permute;
        fr_t* w = nullptr;
        if (kind <= 3 && ks[i] > TB && ws) {
            w = ws + ws_at;
            ws_at += jobs[i].deg;
        }
        build_passes(x, ks[i], TB, kind == 5, kind <= 3, t.tw[inv], false, pre, post, scale, w, passes, &permute);
        if (permute.k) permutes.push_back(permute);
        pass_begin[i + 1] = passes.size();
        rounds = std::max(rounds, pass_begin[i + 1] - pass_begin[i]);
    }
    // pass descriptors, round by round
    std::vector<NttPassDesc> pds;
    pds.reserve(passes.size());
    std::vector<size_t> round_begin(rounds + 1, 0);
    std::vector<uint64_t> round_tiles(rounds, 0);
    for (size_t r = 0; r < rounds; ++r) {
        round_begin[r] = pds.size();
        uint64_t tiles = 0;
        for (size_t i = 0; i < count; ++i) {
            if (pass_begin[i] + r >= pass_begin[i + 1]) continue;
            pds.push_back(passes[pass_begin[i] + r]);
            pds.back().tile_begin = tiles;
            tiles += pass_tiles(pds.back());
        }
        round_tiles[r] = tiles;
    }
    round_begin[rounds] = pds.size();
    const NttPassDesc* dpd = nullptr;
    if (!pds.empty()) {
        const void* dev = nullptr;
        int rc = upload_desc(ctx, pds.data(), pds.size() * sizeof(NttPassDesc), &dev);
        if (rc) return rc;
        dpd = (const NttPassDesc*)dev;
    }
    hipStream_t st = ctx->stream;
    auto stages = [&]() {
        for (const NttPassDesc& d : tiny) hipLaunchKernelGGL(k_ntt_tiny, dim3(1), dim3(64), 0, st, d);
        for (size_t r = 0; r < rounds; ++r) {
            uint32_t np = (uint32_t)(round_begin[r + 1] - round_begin[r]);
            const dim3 grid((unsigned)round_tiles[r]);
            const NttPassDesc* rp = dpd + round_begin[r];
            if (LE == 1) {
                if (TB == 9) hipLaunchKernelGGL((k_ntt_pass_batch<9, 1>), grid, dim3(ntt_threads<9, 1>()), 0, st, rp, np);
                else hipLaunchKernelGGL((k_ntt_pass_batch<10, 1>), grid, dim3(ntt_threads<10, 1>()), 0, st, rp, np);
            } else {
                if (TB == 9) hipLaunchKernelGGL((k_ntt_pass_batch<9, 2>), grid, dim3(ntt_threads<9, 2>()), 0, st, rp, np);
                else hipLaunchKernelGGL((k_ntt_pass_batch<10, 2>), grid, dim3(ntt_threads<10, 2>()), 0, st, rp, np);
            }
        }
        for (const NttPassDesc& d : permutes)
            hipLaunchKernelGGL(k_ntt_permute, dim3(1u << (d.k - 8)), dim3(256), 0, st, d);
    };
    if (capture) {
        std::string key = "ntt:" + std::to_string(TB) + "/" + std::to_string(LE) + "/" + std::to_string(ws_elems && !ws) + ":";
        for (size_t i = 0; i < count; ++i) {
            key += std::to_string(ks[i]) + "/" + std::to_string(jobs[i].kind) + ";";
            // launched with direct arguments
            if (ks[i] < 3 || (ws_elems && !ws)) key += std::to_string((uintptr_t)jobs[i].x) + ";";
        }
        hzk_graph_entry& g = ctx->graphs[key];
        if (!g.exec || g.generation != ctx->desc_generation) {
            if (g.exec) { (void)hipGraphExecDestroy(g.exec); g.exec = nullptr; }
            hipGraph_t graph;
            HZK_HIP(ctx, hipStreamBeginCapture(st, hipStreamCaptureModeThreadLocal));
            stages();
            hipError_t e = hipStreamEndCapture(st, &graph);
            HZK_HIP(ctx, e);
            e = hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0);
            (void)hipGraphDestroy(graph);
            HZK_HIP(ctx, e);
            g.generation = ctx->desc_generation;
        }
        TimedLaunch tl(ctx, "ntt_graph");
        HZK_HIP(ctx, hipGraphLaunch(g.exec, st));
    } else {
        TimedLaunch tl(ctx, "ntt_batch");
        stages();
    }
    HZK_HIP(ctx, hipGetLastError());
    return 0;
}

int ntt_standard_raw(hzk_ctx* ctx, void* x, size_t deg, int inverse) { return ntt_standard(ctx, (fr_t*)x, deg, inverse); }
int coset_ntt_raw(hzk_ctx* ctx, void* x, size_t deg, int inverse) { return coset_ntt(ctx, (fr_t*)x, deg, inverse); }

}  // namespace hzk

using namespace hzk;

extern "C" {

int hzk_ntt(hzk_ctx* ctx, void* coeffs, size_t deg, const void* omega_powers, int inverse, const void* factor) {
    if (!ctx) return HZK_ERR_INVALID;
    HZK_CHECK(ctx, coeffs != nullptr, HZK_ERR_INVALID, "ntt: null coefficients");
    if (!omega_powers) {
        if (factor) {
            int k = log2_exact(deg);
            HZK_CHECK(ctx, k >= 0 && k <= NTT_MAX_LOG, HZK_ERR_INVALID, "ntt: deg %zu invalid", deg);
            NttTables* t;
            int rc = ensure_tables(ctx, k, &t);
            if (rc) return rc;
            return ntt_run(ctx, (fr_t*)coeffs, k, t->tw[inverse ? 1 : 0], false, nullptr, nullptr, (const fr_t*)factor);
        }
        return ntt_standard(ctx, (fr_t*)coeffs, deg, inverse);
    }
    int k = log2_exact(deg);
    HZK_CHECK(ctx, k >= 0 && k <= NTT_MAX_LOG, HZK_ERR_INVALID, "ntt: deg %zu is not a power of two <= 2^%d", deg, NTT_MAX_LOG);
    return ntt_run(ctx, (fr_t*)coeffs, k, (const fr_t*)omega_powers, true, nullptr, nullptr, (const fr_t*)factor);
}

int hzk_ntt_batch(hzk_ctx* ctx, const hzk_ntt_desc* d, size_t count, uint32_t flags) {
    if (!ctx) return HZK_ERR_INVALID;
    HZK_CHECK(ctx, d && count > 0, HZK_ERR_INVALID, "ntt batch: empty");
    HZK_CHECK(ctx, (flags & ~HZK_BATCH_GRAPH) == 0, HZK_ERR_INVALID, "ntt batch: bad flags %u", flags);
    std::vector<NttJob> jobs(count);
    for (size_t i = 0; i < count; ++i) jobs[i] = {d[i].coeffs, d[i].deg, d[i].kind};
    return ntt_batch(ctx, jobs.data(), count, (flags & HZK_BATCH_GRAPH) ? 1 : 0);
}

// The reference's twiddle table for an M-point interpolation domain and its
// 2M-point evaluation domain (ntt_setup, include/protocol/groth16-operator.cuh:
// 6-32), on the host: w_M^i and w_M^-i (i < M), M^-1, w_2M^i and w_2M^-i
// (i < 2M), then (4M)^-1 at 6M + 1, the entry the reference writes there
// (its layout comment, groth16.cuh:32-33, names (2M)^-1).
int hzk_ntt_setup(size_t M, void* host_out) {
    int lg = log2_exact(M);
    if (lg < 0 || lg + 2 > 28 || !host_out) return HZK_ERR_INVALID;
    host::Fr* t = (host::Fr*)host_out;
    const host::Fr w[4] = {root_of_unity(lg), root_of_unity(lg).inverse(), root_of_unity(lg + 1),
                           root_of_unity(lg + 1).inverse()};
    const size_t base[4] = {0, M, 2 * M + 1, 4 * M + 1}, len[4] = {M, M, 2 * M, 2 * M};
    const size_t chunk = 4096;
    for (int s = 0; s < 4; ++s) {
        const long nchunks = (long)((len[s] + chunk - 1) / chunk);
#pragma omp parallel for schedule(static)
        for (long c = 0; c < nchunks; ++c) {
            size_t i0 = (size_t)c * chunk, i1 = std::min(len[s], i0 + chunk);
            uint64_t e[4] = {(uint64_t)i0, 0, 0, 0};
            host::Fr acc = w[s].pow(e);
            for (size_t i = i0; i < i1; ++i) {
                t[base[s] + i] = acc;
                acc = acc * w[s];
            }
        }
    }
    host::Fr two_inv = fr_from_u64(2).inverse();
    host::Fr mi = host::Fr::one(), m4i;
    for (int i = 0; i < lg; ++i) mi = mi * two_inv;
    m4i = mi * two_inv * two_inv;
    t[2 * M] = mi;
    t[6 * M + 1] = m4i;
    return 0;
}

int hzk_coset_ntt(hzk_ctx* ctx, void* coeffs, size_t deg, int inverse) {
    if (!ctx) return HZK_ERR_INVALID;
    HZK_CHECK(ctx, coeffs != nullptr, HZK_ERR_INVALID, "coset_ntt: null coefficients");
    return coset_ntt(ctx, (fr_t*)coeffs, deg, inverse);
}

}  // extern "C"
