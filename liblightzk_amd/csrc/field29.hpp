// Fq in nine signed 29-bit limbs (limb29.hpp) and the XYZZ accumulators of the
// MSM in that form: mixed additions of the bucket accumulation (the MSM's hot
// loop), full additions and doublings of the later stages.
//
// Montgomery radix 2^261; the bases are converted to it once (fq29::TO), the
// window sums leave it (to_r256). Measured on the MI355X against unsigned
// limbs with one reduction per product, multiples of p added to differences
// and Karatsuba in Fq2: 2^24 G1 accumulation 19.1 -> 17.2 ms (1467 instead of
// 1548 multiply-adds per mixed addition, 141 instead of 152 registers), that
// of a 200003-point G2 MSM 0.97 -> 0.65 ms. The G1 loop issues a wave's
// addition in about 10000 cycles, 7800 of them multiply-adds at their
// measured rate: what is left to gain is fewer additions. Four G1 waves per
// SIMD (128 registers, 68 B of scratch) run 3 % slower than three, three G2
// waves (168 registers) 15 % slower than two. Values are lazily reduced: the bounds (in
// units of p) stand at each formula, and every operand of a product is either
// normalized or a difference of two normalized values.
#pragma once
#include "curve.hpp"
#include "field.hpp"
#include "limb29.hpp"

namespace hzk {

struct fq29 : limbs29 {
    typedef Fq29Mod M;
    static constexpr uint32_t MASK = MASK29;
    static constexpr uint32_t ONE[9] = {0x157ccc21, 0x141c2758, 0x185230d3, 0x014c0419, 0x0aa36fb9,
                                        0x1d4240ce, 0x11d54c07, 0x052ac7a8, 0x000dc836};   // 2^261 mod p
    static constexpr uint32_t TO[9] = {0x13349ca1, 0x1a5d84a8, 0x0a3e5cac, 0x100249e0, 0x12b951e8,
                                       0x0e92d304, 0x14cb95b3, 0x041b9d3d, 0x00058003};    // 2^266 mod p
    static constexpr uint32_t FROM[9] = {0x058f0d9d, 0x1aea1c6e, 0x11c2cf74, 0x11d651eb, 0x1462c0a7,
                                         0x11b7bc3c, 0x1cbd99ba, 0x183340fb, 0x000e0a77};  // 2^256 mod p

    fq29() = default;
    HZK_DEV fq29(const limbs29& v) : limbs29(v) {}
    static HZK_DEV fq29 zero() { return limbs29::zero(); }
    static HZK_DEV fq29 one() { return konst(ONE); }
    static HZK_DEV fq29 konst(const uint32_t* c) { fq29 r; for (int i = 0; i < 9; ++i) r.l[i] = (int32_t)c[i]; return r; }

    // repack 8 x 32-bit limbs (a value < 2^256) into 9 x 29-bit limbs
    static HZK_DEV fq29 unpack(const uint32_t* w) {
        return unpack(make_uint4(w[0], w[1], w[2], w[3]), make_uint4(w[4], w[5], w[6], w[7]));
    }
    static HZK_DEV fq29 unpack(const uint4& lo, const uint4& hi) { return limbs29::unpack(lo, hi); }
    // a canonical value back to 8 x 32-bit limbs
    HZK_DEV void pack(uint32_t* w) const {
        uint4 lo, hi;
        limbs29::pack(lo, hi);
        w[0] = lo.x, w[1] = lo.y, w[2] = lo.z, w[3] = lo.w, w[4] = hi.x, w[5] = hi.y, w[6] = hi.z, w[7] = hi.w;
    }
    // y or p - y for y in [0, p], normalized
    static HZK_DEV fq29 negate_if(const fq29& y, bool neg) {
        fq29 r;
        int32_t c = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            const int32_t v = (int32_t)M::P[i] - y.l[i] + c;
            r.l[i] = neg ? (i < 8 ? v & (int32_t)MASK : v) : y.l[i];
            c = v >> 29;
        }
        return r;
    }

    static HZK_DEV fq29 mul(const fq29& a, const fq29& b) { fq29 r; scan29(Mul29<M>(r, a, b)); return r; }

    // the canonical representative of a normalized value in [-p, 2p)
    HZK_DEV fq29 canonical() const {
        fq29 v = *this;
        if (v.l[8] < 0) v = add_p(1);
        const fq29 d = v.add_p(-1);
        return d.l[8] < 0 ? v : d;
    }
    // + k p, normalized (|k| < 16)
    HZK_DEV fq29 add_p(int32_t k) const {
        fq29 r;
        int64_t c = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            c += (int64_t)l[i] + (int64_t)k * (int32_t)M::P[i];
            r.l[i] = (int32_t)c & (int32_t)MASK;
            c >>= 29;
        }
        r.l[8] = l[8] + k * (int32_t)M::P[8] + (int32_t)c;
        return r;
    }

    // value = 0 mod p, for a value in (-16p, 16p), limbs of either sign: a
    // multiple k p has k = value p^-1 mod 2^29, so unless that is small
    // (almost never: 33 of 2^29) the value is none
    HZK_DEV bool is_zero_mod_p() const {
        const uint32_t k = ((uint32_t)l[0] * M::PINV + 16) & MASK;
        if (k > 32) return false;
        const fq29 d = add_p(16 - (int32_t)k);
        int32_t t = 0;
        for (int i = 0; i < 9; ++i) t |= d.l[i];
        return t == 0;
    }

    // canonical, in the R = 2^256 form
    HZK_DEV fq_t to_r256() const {
        const fq29 v = mul(*this, konst(FROM)).canonical();
        fq_t r;
        v.pack(r.l);
        return r;
    }
};

// G1 accumulator over fq29 in XYZZ coordinates, with the point at infinity as
// a flag. Bounds (in units of p): X in (-4, 2), Y in (-1, 2), ZZ, ZZZ in
// (-1, 1.2), all normalized; affine inputs in [0, 1).
struct g1acc29 {
    typedef Fq29Mod M;
    fq29 X, Y, ZZ, ZZZ;
    bool inf;

    HZK_DEV void set_inf() { inf = true; }
    HZK_DEV void set_affine(const fq29& x, const fq29& y) {
        X = x, Y = y, ZZ = fq29::one(), ZZZ = fq29::one();
        inf = false;
    }
    // this += (x, y) for a finite affine point (madd-2008-s), every special
    // case handled. When (x, y) equals this point (P = R = 0) the same code
    // doubles it: dbl-2008-s-1 on the XYZZ state is madd-2008-s with P = 2Y,
    // R = 3X^2 and no PPP term in X3, so the rare case costs one squaring and
    // a select instead of a second formula's registers.
    HZK_DEV void add_affine(const fq29& x, const fq29& y) {
        if (inf) { set_affine(x, y); return; }
        fq29 U2, S2;
        scan29(Mul29<M>(U2, x, ZZ), Mul29<M>(S2, y, ZZZ));   // (-0.1, 1.2) each
        fq29 P = U2 - X, R = S2 - Y;                         // (-2.1, 5.2), (-2.1, 2.2)
        bool d = false;
        if (P.is_zero_mod_p()) {
            if (!R.is_zero_mod_p()) { set_inf(); return; }
            P = Y.twice().norm();
            fq29 xx;
            scan29(Sqr29<M>(xx, X));
            R = (xx + xx + xx).norm();
            d = true;
        }
        finish(P, R, X, Y, ZZ, ZZZ, d);
    }
    // the R = 2^256 XYZZ point (canonical coordinates; infinity = all zero)
    HZK_DEV xyzz_t<fq_t> to_xyzz() const {
        if (inf) return xyzz_t<fq_t>::inf();
        return {X.to_r256(), Y.to_r256(), ZZ.to_r256(), ZZZ.to_r256()};
    }
    // The raw state, 36 words (X, Y, ZZ, ZZZ limbs; infinity has ZZ = 0, which
    // a finite point's ZZ = Z^2 never is): a plain store, so a lane that
    // finishes a bucket in the middle of its chunk holds the others up for a
    // few instructions instead of four conversions. The later stages (bucket
    // fix-up and reduction) read and write this form too, a coordinate per lane
    // (LanePoint::load_raw); only the window sums leave it.
    static constexpr int RAW_WORDS = 36;
    HZK_DEV void to_words(uint32_t* w) const {
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            w[i] = X.l[i], w[9 + i] = Y.l[i], w[18 + i] = inf ? 0 : ZZ.l[i], w[27 + i] = ZZZ.l[i];
        }
    }
    static HZK_DEV g1acc29 from_words(const uint32_t* w) {
        g1acc29 a;
        uint32_t zz = 0;
#pragma unroll
        for (int i = 0; i < 9; ++i) {
            a.X.l[i] = w[i], a.Y.l[i] = w[9 + i], a.ZZ.l[i] = w[18 + i], a.ZZZ.l[i] = w[27 + i];
            zz |= w[18 + i];
        }
        a.inf = zz == 0;
        return a;
    }
    HZK_DEV void store_raw(uint4* dst) const {
        uint32_t w[RAW_WORDS];
        to_words(w);
#pragma unroll
        for (int q = 0; q < RAW_WORDS / 4; ++q) dst[q] = make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
    }

    // this += q for two states under the bounds (add-2008-s); when q equals
    // this point the same tail doubles it (dbl-2008-s-1 as in add_affine: U1
    // -> X, S1 -> Y, the ZZ, ZZZ products -> this point's)
    HZK_DEV void add(const g1acc29& q) {
        if (q.inf) return;
        if (inf) { *this = q; return; }
        fq29 U1, U2, ZZ12, S1, S2, ZZZ12;
        scan29(Mul29<M>(U1, X, q.ZZ), Mul29<M>(U2, q.X, ZZ), Mul29<M>(ZZ12, ZZ, q.ZZ));
        scan29(Mul29<M>(S1, Y, q.ZZZ), Mul29<M>(S2, q.Y, ZZZ), Mul29<M>(ZZZ12, ZZZ, q.ZZZ));
        fq29 P = U2 - U1, R = S2 - S1;                       // (-1.3, 1.3)
        bool d = false;
        if (P.is_zero_mod_p()) {
            if (!R.is_zero_mod_p()) { set_inf(); return; }
            P = Y.twice().norm();
            fq29 xx;
            scan29(Sqr29<M>(xx, X));
            R = (xx + xx + xx).norm();
            U1 = X, S1 = Y, ZZ12 = ZZ, ZZZ12 = ZZZ;
            d = true;
        }
        finish(P, R, U1, S1, ZZ12, ZZZ12, d);
    }
    HZK_DEV void dbl() {
        if (inf) return;
        fq29 xx;
        scan29(Sqr29<M>(xx, X));
        finish(Y.twice().norm(), (xx + xx + xx).norm(), X, Y, ZZ, ZZZ, true);
    }
    // the common tail, P in (-6, 6), R in (-4, 4), U1 in (-4, 2), S1 in (-1,
    // 2), ZZ12, ZZZ12 in (-1, 1.2): PP in (0, 1.4), PPP, Q in (-0.1, 1.2), X3
    // = RR - PPP - 2Q in (-3.7, 1.6), Y3 = R (Q - X3) - S1 PPP in (-0.2, 1.4);
    // X3 is reduced with its addend, Y3 as one sum of two products
    HZK_DEV void finish(const fq29& P, const fq29& R, const fq29& U1, const fq29& S1, const fq29& ZZ12, const fq29& ZZZ12, bool d) {
        fq29 PP, PPP, Q;
        scan29(Sqr29<M>(PP, P));
        const fq29 u = U1, s = S1;
        scan29(Mul29<M>(PPP, P, PP), Mul29<M>(Q, u, PP), Mul29<M>(ZZ, ZZ12, PP));
        const fq29 F = -PPP;
        const fq29 T = (d ? fq29::zero() : F) - Q.twice();
        scan29(SqrAdd29<M>(X, R, T), Mul29<M>(ZZZ, ZZZ12, PPP));
        const fq29 D = Q - X;
        scan29(Sum29<M>(Y, R, D, s, F));
    }
};

// Fq2 = Fq[u]/(u^2 + 1) over fq29 components. Products as two reduced sums of
// two products each (a0 b0 - a1 b1, a0 b1 + a1 b0): as many multiply-adds as
// Karatsuba's three products with their three reductions, and no additions or
// corrections around them.
struct fq2_29 {
    typedef Fq29Mod M;
    fq29 c0, c1;
    static HZK_DEV fq2_29 one() { return {fq29::one(), fq29::zero()}; }
    static HZK_DEV fq2_29 zero() { return {fq29::zero(), fq29::zero()}; }
    friend HZK_DEV fq2_29 operator+(const fq2_29& a, const fq2_29& b) { return {a.c0 + b.c0, a.c1 + b.c1}; }
    friend HZK_DEV fq2_29 operator-(const fq2_29& a, const fq2_29& b) { return {a.c0 - b.c0, a.c1 - b.c1}; }
    HZK_DEV fq2_29 operator-() const { return {-c0, -c1}; }
    HZK_DEV fq2_29 twice() const { return {c0.twice(), c1.twice()}; }
    HZK_DEV fq2_29 norm() const { return {c0.norm(), c1.norm()}; }
    HZK_DEV bool is_zero_mod_p() const { return c0.is_zero_mod_p() && c1.is_zero_mod_p(); }
    static HZK_DEV fq2_29 negate_if(const fq2_29& y, bool neg) { return {fq29::negate_if(y.c0, neg), fq29::negate_if(y.c1, neg)}; }
    static HZK_DEV void mul(fq2_29& r, const fq2_29& a, const fq2_29& b) {
        const fq29 n = -b.c1;
        fq2_29 t;
        scan29(Sum29<M>(t.c0, a.c0, b.c0, a.c1, n), Sum29<M>(t.c1, a.c0, b.c1, a.c1, b.c0));
        r = t;
    }
    // a0^2 - a1^2 and (2 a0) a1
    static HZK_DEV void sqr(fq2_29& r, const fq2_29& a) {
        const fq29 a2 = a.c0.twice();
        scan29(SqrDiff29<M>(r.c0, a.c0, a.c1), Mul29<M>(r.c1, a2, a.c1));
    }
    // a^2 + t
    static HZK_DEV void sqr_add(fq2_29& r, const fq2_29& a, const fq2_29& t) {
        const fq29 a2 = a.c0.twice();
        scan29(SqrDiffAdd29<M>(r.c0, a.c0, a.c1, t.c0), MulAdd29<M>(r.c1, a2, a.c1, t.c1));
    }
    // r d - s f, each component one reduced sum of four products. Columns (in
    // units of 2^58, eight full-size products a pair): s and f have no
    // negative limbs 0..7, so r0 d0 - r1 d1 - s0 f0 + s1 f1 stays within
    // (-24, 24 + 8) and r0 d1 + r1 d0 - s0 f1 - s1 f0 within (-32, 16 + 8):
    // 32 (2^29 - 1)^2 is 2^35 short of 2^63, more than the carry between columns.
    static HZK_DEV void mul_sub(fq2_29& o, const fq2_29& r, const fq2_29& d, const fq2_29& s, const fq2_29& f) {
        const fq29 nd = -d.c1, n0 = -s.c0, n1 = -s.c1, s1 = s.c1;
        scan29(Sum4_29<M>(o.c0, r.c0, d.c0, r.c1, nd, n0, f.c0, s1, f.c1),
               Sum4_29<M>(o.c1, r.c0, d.c1, r.c1, d.c0, n0, f.c1, n1, f.c0));
    }
};

// G2 accumulator over fq2_29, infinity as a flag. Component bounds (in units
// of p): X in (-4, 2), Y in (-1, 2), ZZ, ZZZ in (-1, 1.3), all normalized;
// affine inputs in [0, 1].
struct g2acc29 {
    fq2_29 X, Y, ZZ, ZZZ;
    bool inf;

    HZK_DEV void set_inf() { inf = true; }
    HZK_DEV void set_affine(const fq2_29& x, const fq2_29& y) {
        X = x, Y = y, ZZ = fq2_29::one(), ZZZ = fq2_29::one();
        inf = false;
    }
    // this += (x, y), every special case handled; a doubling (x, y equal to
    // this point) runs the same code with P = 2Y, R = 3X^2 and no PPP term in
    // X3 (dbl-2008-s-1)
    HZK_DEV void add_affine(const fq2_29& x, const fq2_29& y) {
        if (inf) { set_affine(x, y); return; }
        fq2_29 P, R;
        fq2_29::mul(P, x, ZZ);      // U2 in (-0.1, 1.2)
        P = P - X;                  // (-2.1, 5.2)
        fq2_29::mul(R, y, ZZZ);     // S2
        R = R - Y;                  // (-2.1, 2.2)
        bool d = false;
        if (P.is_zero_mod_p()) {
            if (!R.is_zero_mod_p()) { set_inf(); return; }
            P = Y.twice().norm();
            fq2_29 xx;
            fq2_29::sqr(xx, X);
            R = (xx + xx + xx).norm();
            d = true;
        }
        finish(P, R, X, Y, ZZ, ZZZ, d);
    }
    // raw state: 72 words, infinity has ZZ = 0 (read back by LanePoint::load_raw)
    static constexpr int RAW_WORDS = 72;
    HZK_DEV void to_words(uint32_t* w) const {
        const fq29* c[8] = {&X.c0, &X.c1, &Y.c0, &Y.c1, &ZZ.c0, &ZZ.c1, &ZZZ.c0, &ZZZ.c1};
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int i = 0; i < 9; ++i) w[9 * k + i] = (inf && (k == 4 || k == 5)) ? 0 : c[k]->l[i];
    }
    static HZK_DEV g2acc29 from_words(const uint32_t* w) {
        g2acc29 a;
        fq29* c[8] = {&a.X.c0, &a.X.c1, &a.Y.c0, &a.Y.c1, &a.ZZ.c0, &a.ZZ.c1, &a.ZZZ.c0, &a.ZZZ.c1};
        uint32_t zz = 0;
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int i = 0; i < 9; ++i) c[k]->l[i] = w[9 * k + i];
#pragma unroll
        for (int i = 0; i < 18; ++i) zz |= w[36 + i];
        a.inf = zz == 0;
        return a;
    }
    HZK_DEV void store_raw(uint4* dst) const {
        uint32_t w[RAW_WORDS];
        to_words(w);
#pragma unroll
        for (int q = 0; q < RAW_WORDS / 4; ++q) dst[q] = make_uint4(w[4 * q], w[4 * q + 1], w[4 * q + 2], w[4 * q + 3]);
    }
    // the R = 2^256 XYZZ point (canonical components; infinity = all zero)
    HZK_DEV xyzz_t<fq2_t> to_xyzz() const {
        if (inf) return xyzz_t<fq2_t>::inf();
        return {{X.c0.to_r256(), X.c1.to_r256()}, {Y.c0.to_r256(), Y.c1.to_r256()},
                {ZZ.c0.to_r256(), ZZ.c1.to_r256()}, {ZZZ.c0.to_r256(), ZZZ.c1.to_r256()}};
    }

    // this += q for two states under the bounds (add-2008-s); when q equals
    // this point the same tail doubles it (dbl-2008-s-1 with U1 -> X, S1 -> Y
    // and the ZZ, ZZZ products -> this point's)
    HZK_DEV void add(const g2acc29& q) {
        if (q.inf) return;
        if (inf) { *this = q; return; }
        fq2_29 U1, S1, P, R;
        fq2_29::mul(U1, X, q.ZZ);
        fq2_29::mul(P, q.X, ZZ);
        P = P - U1;                 // (-1.4, 1.4)
        fq2_29::mul(S1, Y, q.ZZZ);
        fq2_29::mul(R, q.Y, ZZZ);
        R = R - S1;
        bool d = false;
        if (P.is_zero_mod_p()) {
            if (!R.is_zero_mod_p()) { set_inf(); return; }
            P = Y.twice().norm();
            fq2_29 xx;
            fq2_29::sqr(xx, X);
            R = (xx + xx + xx).norm();
            U1 = X, S1 = Y;
            d = true;
        }
        fq2_29 ZZ12 = ZZ, ZZZ12 = ZZZ;
        if (!d) {
            fq2_29::mul(ZZ12, ZZ, q.ZZ);
            fq2_29::mul(ZZZ12, ZZZ, q.ZZZ);
        }
        finish(P, R, U1, S1, ZZ12, ZZZ12, d);
    }
    HZK_DEV void dbl() {
        if (inf) return;
        fq2_29 xx;
        fq2_29::sqr(xx, X);
        finish(Y.twice().norm(), (xx + xx + xx).norm(), X, Y, ZZ, ZZZ, true);
    }
    // the common tail: component bounds as in g1acc29::finish (an Fq2 product
    // adds two limb-product sums before its reduction, so every bound there
    // holds with at most 0.3 more on either side)
    HZK_DEV void finish(const fq2_29& P, const fq2_29& R, const fq2_29& U1, const fq2_29& S1, const fq2_29& ZZ12,
                        const fq2_29& ZZZ12, bool d) {
        fq2_29 PP, PPP, Q;
        fq2_29::sqr(PP, P);
        fq2_29::mul(PPP, P, PP);
        fq2_29::mul(Q, U1, PP);
        fq2_29::mul(ZZ, ZZ12, PP);
        const fq2_29 S = S1;
        fq2_29::mul(ZZZ, ZZZ12, PPP);
        const fq2_29 T = d ? -Q.twice() : -PPP - Q.twice();
        fq2_29::sqr_add(X, R, T);
        fq2_29::mul_sub(Y, R, Q - X, S, PPP);
    }
};

}  // namespace hzk
