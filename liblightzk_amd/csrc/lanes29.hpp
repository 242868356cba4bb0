// XYZZ points spread over the lanes of a group, for the MSM stages that are
// chains of dependent full additions (fix-up, hot buckets, bucket reduction).
//
// Bound: one lane adds two points in 14 dependent-enough products, about 7 us
// (G1) and 20 us (G2, Fq2 products) on an MI355X whatever the occupancy, and
// those stages are chains of 20 to 40 additions on few lanes. Here a G1 point
// takes four lanes, one coordinate (X, Y, ZZ, ZZZ) each, and an addition four
// steps of four products side by side; a G2 point takes eight lanes (the c0
// components in one quad, the c1 components in the next) with one reduced sum
// of two products per lane and step. Operands change lanes by DPP moves inside
// the quad (and its mirror for the other component). 14 of the 16 product
// slots do work, so throughput is close to the one-lane form, a lane's state is
// 9 registers instead of 36 or 72, and the latency of an addition falls 3.5
// times (G1) and 7 times (G2). Measured on the MI355X, one-lane form against
// this, same plans: a 1000-point G1 MSM 470 -> 325 us (its fix-up of 16 chunks
// a bucket 170 -> 79), the bucket reduction of a 200003-point G2 MSM 620 -> 360
// us and its fix-up 188 -> 113, the hot bucket of a 2^20 MSM with 70 % 0/1
// scalars 310 -> 100, the reduction of 32 G1 MSMs in a batch 995 -> 430.
//
// All lanes of a group must be active and take the same branches.
#pragma once
#include "field29.hpp"

namespace hzk {

// lane c of each quad takes x from lane L_c of its quad
template <int L0, int L1, int L2, int L3>
HZK_DEV int32_t quad_get(int32_t x) {
    return __builtin_amdgcn_mov_dpp(x, L0 | (L1 << 2) | (L2 << 4) | (L3 << 6), 0xf, 0xf, true);
}
template <int L0, int L1, int L2, int L3>
HZK_DEV limbs29 quad_get(const limbs29& v) {
    limbs29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = quad_get<L0, L1, L2, L3>(v.l[i]);
    return r;
}
template <int L>
HZK_DEV bool quad_flag(bool f) { return quad_get<L, L, L, L>((int32_t)f) != 0; }
// the same lane of the other quad of eight: mirrored quad, then mirrored eight
HZK_DEV int32_t pair_get(int32_t x) {
    constexpr int ROW_HALF_MIRROR = 0x141;
    return __builtin_amdgcn_mov_dpp(quad_get<3, 2, 1, 0>(x), ROW_HALF_MIRROR, 0xf, 0xf, true);
}
HZK_DEV limbs29 sel(bool f, const limbs29& a, const limbs29& b) {
    limbs29 r;
#pragma unroll
    for (int i = 0; i < 9; ++i) r.l[i] = f ? a.l[i] : b.l[i];
    return r;
}

// the lane's part of a field: G1 one Fq element per lane, G2 one component of
// an Fq2 element per lane (bit 2 of the lane)
struct LaneFq {
    static constexpr int LANES = 4;
    static HZK_DEV int word() { return 9 * (threadIdx.x & 3); }      // first word of the lane in a raw state
    static HZK_DEV int elem() { return threadIdx.x & 3; }            // field element of the lane in an XYZZ point
    static HZK_DEV bool both(bool f) { return f; }
    static HZK_DEV void mul(limbs29& r, const limbs29& a, const limbs29& b) { scan29(Mul29<Fq29Mod>(r, a, b)); }
};
struct LaneFq2 {
    static constexpr int LANES = 8;
    static HZK_DEV bool c1() { return threadIdx.x & 4; }
    static HZK_DEV int word() { return 18 * (threadIdx.x & 3) + (c1() ? 9 : 0); }
    static HZK_DEV int elem() { return 2 * (threadIdx.x & 3) + c1(); }
    static HZK_DEV bool both(bool f) { return ((int32_t)f & pair_get((int32_t)f)) != 0; }
    // c0 lanes a0 b0 + a1 (-b1), c1 lanes a1 b0 + a0 b1
    static HZK_DEV void mul(limbs29& r, const limbs29& a, const limbs29& b) {
        limbs29 ao, x, y;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int32_t bo = pair_get(b.l[i]);
            ao.l[i] = pair_get(a.l[i]);
            x.l[i] = c1() ? bo : b.l[i];
            y.l[i] = c1() ? b.l[i] : -bo;
        }
        const limbs29 own = a;
        scan29(Sum29<Fq29Mod>(r, own, x, ao, y));
    }
};
template <class F> struct LaneOf;
template <> struct LaneOf<fq_t> { using T = LaneFq; };
template <> struct LaneOf<fq2_t> { using T = LaneFq2; };

// the lane's coordinate of an accumulator (bounds as in g1acc29, Y in (-2, 2):
// here it is the difference of two reduced products), normalized; inf is the
// same in every lane of the group
template <class F>
struct LanePoint {
    using L = typename LaneOf<F>::T;
    static constexpr int LANES = L::LANES;
    static constexpr int RAW_WORDS = 9 * LANES;
    limbs29 v;
    bool inf;

    HZK_DEV void set_inf() { v = limbs29::zero(), inf = true; }
    static HZK_DEV bool zz_zero(const limbs29& v) {
        int32_t t = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) t |= v.l[i];
        return L::both(quad_flag<2>(t == 0));
    }
    // raw states as g1acc29 / g2acc29 store them
    static HZK_DEV LanePoint load_raw(const uint32_t* state) {
        LanePoint p;
        const uint32_t* w = state + L::word();
#pragma unroll
        for (int i = 0; i < 9; ++i) p.v.l[i] = (int32_t)w[i];
        p.inf = zz_zero(p.v);
        return p;
    }
    HZK_DEV void store_raw(uint32_t* state) const {
        uint32_t* w = state + L::word();
#pragma unroll
        for (int i = 0; i < 9; ++i) w[i] = inf ? 0u : (uint32_t)v.l[i];
    }
    // the lane's element of the R = 2^256 XYZZ point
    HZK_DEV void store_xyzz(xyzz_t<F>* out) const {
        fq_t r = fq_t::zero();
        if (!inf) r = fq29(v).to_r256();
        ((fq_t*)out)[L::elem()] = r;
    }

    // the point of the group that lane `lane` (this one's place in it) belongs to
    HZK_DEV LanePoint from_lane(int lane) const {
        LanePoint p;
#pragma unroll
        for (int i = 0; i < 9; ++i) p.v.l[i] = __shfl(v.l[i], lane);
        p.inf = __shfl((int)inf, lane) != 0;
        return p;
    }

    // this += q (add-2008-s), every special case handled as in g1acc29::add
    HZK_DEV void add(const LanePoint& q) {
        const bool live = !inf && !q.inf;
        if (__ballot(live) == 0) {   // nothing to add in any group of the wave
            if (inf) *this = q;
            return;
        }
        const int c = threadIdx.x & 3;
        limbs29 w, d, a, b, e, f, g;
        L::mul(w, v, quad_get<2, 3, 0, 1>(q.v));          // U1, S1, U2, S2
        d = quad_get<2, 3, 0, 1>(w) - w;                  // P, R, -P, -R
        const bool z = L::both(fq29(d).is_zero_mod_p());
        const bool pz = quad_flag<0>(z), rz = quad_flag<1>(z), dbl = live && pz && rz;
        a = sel(c < 2, d, v);
        b = sel(c < 2, d, q.v);
        if (dbl) {                                        // P = 2Y, R = 3X^2, U1 = X, S1 = Y, ZZ, ZZZ as they are
            a = doubling(d);
            b = a, w = v;
        }
        tail(v, w, d, a, b, dbl, dbl, e, f, g);
        const bool keep = q.inf, take = inf;
        inf = inf && q.inf;
        if (live && pz && !rz) inf = true;
#pragma unroll
        for (int i = 0; i < 9; ++i) v.l[i] = keep ? v.l[i] : (take ? q.v.l[i] : g.l[i]);
    }
    HZK_DEV void dbl() {
        if (__ballot(!inf) == 0) return;
        limbs29 d, e, f, g;
        const limbs29 a = doubling(d);
        tail(v, v, d, a, a, true, true, e, f, g);
        v = g;
    }

private:
    // d = P, R of a doubling in lanes 0, 1 (P = 2Y, R = 3X^2); its factor operand
    HZK_DEV limbs29 doubling(limbs29& d) const {
        limbs29 x = quad_get<0, 0, 0, 0>(v), xx;
        L::mul(xx, x, x);
        xx = (xx + xx + xx).norm();
        const limbs29 y2 = quad_get<1, 1, 1, 1>(v).twice().norm();
        d = sel((threadIdx.x & 3) == 0, y2, xx);
        return d;
    }
    // e = a b (PP, RR, ZZ12, ZZZ12; lanes 2, 3 keep st's when keep_zz), then
    // Q, PPP, ZZ3 and R D, S1 PPP, ZZZ3; the new coordinates in g. w: U1, S1 in
    // lanes 0, 1. no_ppp: a doubling's X3.
    static HZK_DEV void tail(const limbs29& st, const limbs29& w, const limbs29& d, const limbs29& a, const limbs29& b, bool keep_zz,
                             bool no_ppp, limbs29& e, limbs29& f, limbs29& g) {
        const int c = threadIdx.x & 3;
        L::mul(e, a, b);
        e = sel(keep_zz && c >= 2, st, e);
        const limbs29 p0 = quad_get<0, 0, 0, 0>(d), r1 = quad_get<1, 1, 1, 1>(d);
        L::mul(f, sel(c == 0, w, sel(c == 1, p0, e)), quad_get<0, 0, 0, 0>(e));
        const limbs29 ppp = quad_get<1, 1, 1, 1>(f), rr = quad_get<1, 1, 1, 1>(e);
        limbs29 x3;
#pragma unroll
        for (int i = 0; i < 9; ++i) x3.l[i] = rr.l[i] - (no_ppp ? 0 : ppp.l[i]) - (f.l[i] << 1);
        x3 = x3.norm();
        L::mul(g, sel(c == 0, r1, sel(c == 1, w, e)), sel(c == 0, f - x3, ppp));
        const limbs29 y3 = (quad_get<0, 0, 0, 0>(g) - g).norm();
        g = sel(c == 0, x3, sel(c == 1, y3, sel(c == 2, f, g)));
    }
};

// Group accumulators of a workgroup of T threads in LDS: lane-linear words, so
// a wave's accesses touch consecutive words
template <class F, int T>
struct LdsLanes {
    using A = LanePoint<F>;
    static constexpr int SLOTS = T / A::LANES;
    static constexpr int WORDS = 10 * T;
    uint32_t* sh;
    HZK_DEV void put(const A& p) const {
#pragma unroll
        for (int i = 0; i < 9; ++i) sh[i * T + threadIdx.x] = (uint32_t)p.v.l[i];
        sh[9 * T + threadIdx.x] = p.inf;
    }
    // the point of slot (own + off)
    HZK_DEV A get(uint32_t off) const {
        const uint32_t t = threadIdx.x + off * A::LANES;
        A p;
#pragma unroll
        for (int i = 0; i < 9; ++i) p.v.l[i] = (int32_t)sh[i * T + t];
        p.inf = sh[9 * T + t] != 0;
        return p;
    }
    // slots [0, n) (n a power of two) summed into slot 0; every thread calls
    HZK_DEV void tree_sum(A& x, uint32_t n) const {
        const uint32_t slot = threadIdx.x / A::LANES;
        for (uint32_t off = n / 2; off > 0; off >>= 1) {
            __syncthreads();
            put(x);
            __syncthreads();
            if (slot < off) x.add(get(off));
        }
    }
};

}  // namespace hzk
