// Host-side alt_bn128 arithmetic for the sequential tails of the GPU path:
// the MSM window combine (c doublings per window, Horner), affine
// normalisation of results, and the Groth16 phase-6 assembly, which the
// reference also performs on the host (include/protocol/groth16.cuh:210-215).
// These are a few thousand dependent field operations per call: one GPU wave
// needs ~1 us per 256-bit Montgomery product, a CPU core ~20 ns, so they run
// here. Values use the same 32-byte Montgomery layout as the device.
#pragma once
#include <cstdint>
#include <cstring>
#include <vector>

namespace hzk {
namespace host {

typedef unsigned __int128 u128;

struct Params { uint64_t p[4]; uint64_t inv; uint64_t one[4]; uint64_t r2[4]; };
inline constexpr Params FQ = {
    {0x3c208c16d87cfd47ULL, 0x97816a916871ca8dULL, 0xb85045b68181585dULL, 0x30644e72e131a029ULL},
    0x87d20782e4866389ULL,
    {0xd35d438dc58f0d9dULL, 0x0a78eb28f5c70b3dULL, 0x666ea36f7879462cULL, 0x0e0a77c19a07df2fULL},
    {0xf32cfc5b538afa89ULL, 0xb5e71911d44501fbULL, 0x47ab1eff0a417ff6ULL, 0x06d89f71cab8351fULL}};
inline constexpr Params FR = {
    {0x43e1f593f0000001ULL, 0x2833e84879b97091ULL, 0xb85045b68181585dULL, 0x30644e72e131a029ULL},
    0xc2e1f593efffffffULL,
    {0xac96341c4ffffffbULL, 0x36fc76959f60cd29ULL, 0x666ea36f7879462eULL, 0x0e0a77c19a07df2fULL},
    {0x1bb8e645ae216da7ULL, 0x53fe3ab1e35c59e3ULL, 0x8c49833d53bb8085ULL, 0x0216d0b17f4e44a5ULL}};

template <const Params& P>
struct Fp {
    uint64_t v[4];
    static Fp zero() { return Fp{{0, 0, 0, 0}}; }
    static Fp one() { Fp r; std::memcpy(r.v, P.one, 32); return r; }
    static Fp load(const void* src) { Fp r; std::memcpy(r.v, src, 32); return r; }
    void store(void* dst) const { std::memcpy(dst, v, 32); }
    bool is_zero() const { return (v[0] | v[1] | v[2] | v[3]) == 0; }
    bool operator==(const Fp& o) const { return std::memcmp(v, o.v, 32) == 0; }
    bool operator!=(const Fp& o) const { return !(*this == o); }

    // t - p where t >= p, else t (t < 2p), without a branch: the comparison is
    // a coin toss, and a mispredicted one costs as much as a product
    static Fp reduced(uint64_t t0, uint64_t t1, uint64_t t2, uint64_t t3) {
        uint64_t d[4], bw = 0;
        const uint64_t t[4] = {t0, t1, t2, t3};
        for (int i = 0; i < 4; ++i) { u128 x = (u128)t[i] - P.p[i] - bw; d[i] = (uint64_t)x; bw = (uint64_t)(x >> 64) & 1; }
        const uint64_t keep = 0 - bw;   // all ones: t < p
        Fp r;
        for (int i = 0; i < 4; ++i) r.v[i] = (t[i] & keep) | (d[i] & ~keep);
        return r;
    }
    // Montgomery product, operand scanning with interleaved reduction; both
    // carry words stay below 2^64 because the top word of p is below 2^62
    friend Fp operator*(const Fp& a, const Fp& b) {
        uint64_t t0 = 0, t1 = 0, t2 = 0, t3 = 0;
#pragma GCC unroll 4
        for (int i = 0; i < 4; ++i) {
            const uint64_t y = b.v[i];
            u128 x = (u128)a.v[0] * y + t0;
            const uint64_t lo = (uint64_t)x, m = lo * P.inv;
            uint64_t ca = (uint64_t)(x >> 64);
            u128 z = (u128)m * P.p[0] + lo;
            uint64_t cm = (uint64_t)(z >> 64);
            x = (u128)a.v[1] * y + t1 + ca;
            ca = (uint64_t)(x >> 64);
            z = (u128)m * P.p[1] + (uint64_t)x + cm;
            t0 = (uint64_t)z, cm = (uint64_t)(z >> 64);
            x = (u128)a.v[2] * y + t2 + ca;
            ca = (uint64_t)(x >> 64);
            z = (u128)m * P.p[2] + (uint64_t)x + cm;
            t1 = (uint64_t)z, cm = (uint64_t)(z >> 64);
            x = (u128)a.v[3] * y + t3 + ca;
            ca = (uint64_t)(x >> 64);
            z = (u128)m * P.p[3] + (uint64_t)x + cm;
            t2 = (uint64_t)z;
            t3 = (uint64_t)(z >> 64) + ca;
        }
        return reduced(t0, t1, t2, t3);
    }
    friend Fp operator+(const Fp& a, const Fp& b) {
        uint64_t t[4];
        u128 c = 0;
        for (int i = 0; i < 4; ++i) { c += (u128)a.v[i] + b.v[i]; t[i] = (uint64_t)c; c >>= 64; }
        return reduced(t[0], t[1], t[2], t[3]);   // a + b < 2p < 2^255
    }
    friend Fp operator-(const Fp& a, const Fp& b) {
        uint64_t t[4], bw = 0;
        for (int i = 0; i < 4; ++i) { u128 d = (u128)a.v[i] - b.v[i] - bw; t[i] = (uint64_t)d; bw = (uint64_t)(d >> 64) & 1; }
        const uint64_t add = 0 - bw;
        u128 c = 0;
        Fp r;
        for (int i = 0; i < 4; ++i) { c += (u128)t[i] + (P.p[i] & add); r.v[i] = (uint64_t)c; c >>= 64; }
        return r;
    }
    Fp neg() const { return zero() - *this; }
    Fp dbl() const { return *this + *this; }
    Fp sqr() const { return *this * *this; }
    Fp pow(const uint64_t e[4]) const {
        Fp acc = one();
        for (int i = 255; i >= 0; --i) { acc = acc.sqr(); if ((e[i / 64] >> (i % 64)) & 1) acc = acc * *this; }
        return acc;
    }
    // 1/a; 0 -> 0. T. Pornin, "Optimized Binary GCD for Modular Inversion"
    // (2020): 17 rounds of 31 halvings (2 * 254 - 1 are enough) on 64-bit
    // stand-ins for a and b, their low 31 and leading 33 bits, after which the
    // recorded factors update a, b exactly and u, v modulo p. 2.5 us against
    // 13 us for a^(p-2).
    Fp inverse() const {
        uint64_t a[4], b[4];
        std::memcpy(a, v, 32);
        std::memcpy(b, P.p, 32);
        Fp u{{1, 0, 0, 0}}, w = zero();
        for (int round = 0; round < 17; ++round) {
            uint64_t x, y;
            {
                int k = 3;
                while (k > 0 && !(a[k] | b[k])) --k;
                if (k == 0) x = a[0], y = b[0];
                else {
                    const int sh = __builtin_clzll(a[k] | b[k]);
                    const uint64_t ha = sh ? (a[k] << sh) | (a[k - 1] >> (64 - sh)) : a[k];
                    const uint64_t hb = sh ? (b[k] << sh) | (b[k - 1] >> (64 - sh)) : b[k];
                    const uint64_t low = 0x7fffffffu;
                    x = (a[0] & low) | (ha & ~low);
                    y = (b[0] & low) | (hb & ~low);
                }
            }
            int64_t f0 = 1, g0 = 0, f1 = 0, g1 = 1;
            for (int i = 0; i < 31; ++i) {
                const uint64_t odd = 0 - (x & 1), swap = odd & (0 - (uint64_t)(x < y));
                const uint64_t tx = (x ^ y) & swap;
                x ^= tx, y ^= tx;
                const int64_t tf = (f0 ^ f1) & (int64_t)swap, tg = (g0 ^ g1) & (int64_t)swap;
                f0 ^= tf, f1 ^= tf, g0 ^= tg, g1 ^= tg;
                x = (x - (y & odd)) >> 1;
                f0 -= f1 & (int64_t)odd, g0 -= g1 & (int64_t)odd;
                f1 *= 2, g1 *= 2;
            }
            uint64_t na[4], nb[4];
            if (combine(na, a, b, f0, g0)) f0 = -f0, g0 = -g0;
            if (combine(nb, a, b, f1, g1)) f1 = -f1, g1 = -g1;
            std::memcpy(a, na, 32);
            std::memcpy(b, nb, 32);
            const Fp nu = combine_mod(u, w, f0, g0);
            w = combine_mod(u, w, f1, g1);
            u = nu;
        }
        // w = 2^(17 (31 - 64)) / this; times 2^(768 + 17 * 33) / 2^256 is 2^512 / this
        static const Fp undo = [] {
            Fp t = one();   // 2^256
            for (int i = 0; i < 512 + 17 * 33; ++i) t = t + t;
            return t;
        }();
        return w * undo;
    }

private:
    // r = |f a + g b| / 2^31 (an exact division), true when the sum was negative
    static bool combine(uint64_t r[4], const uint64_t a[4], const uint64_t b[4], int64_t f, int64_t g) {
        uint64_t t[5];
        __int128 c = 0;
        for (int i = 0; i < 4; ++i) {   // |f|, |g| <= 2^31: the sum of both products and the carry fits
            c += (__int128)f * a[i] + (__int128)g * b[i];
            t[i] = (uint64_t)c;
            c >>= 64;
        }
        t[4] = (uint64_t)c;
        const uint64_t neg = 0 - (t[4] >> 63);
        u128 d = neg & 1;
        for (int i = 0; i < 5; ++i) { d += t[i] ^ neg; t[i] = (uint64_t)d; d >>= 64; }
        for (int i = 0; i < 4; ++i) r[i] = (t[i] >> 31) | (t[i + 1] << 33);
        return neg;
    }
    // (f u + g w) / 2^64 modulo p
    static Fp combine_mod(const Fp& u, const Fp& w, int64_t f, int64_t g) {
        const Fp x = f < 0 ? u.neg() : u, y = g < 0 ? w.neg() : w;
        const uint64_t m0 = f < 0 ? 0 - (uint64_t)f : (uint64_t)f, m1 = g < 0 ? 0 - (uint64_t)g : (uint64_t)g;
        uint64_t t[5];
        u128 c = 0;
        for (int i = 0; i < 4; ++i) { c += (u128)m0 * x.v[i] + (u128)m1 * y.v[i]; t[i] = (uint64_t)c; c >>= 64; }
        t[4] = (uint64_t)c;
        const uint64_t m = t[0] * P.inv;
        c = ((u128)m * P.p[0] + t[0]) >> 64;
        for (int i = 1; i < 4; ++i) { c += (u128)m * P.p[i] + t[i]; t[i - 1] = (uint64_t)c; c >>= 64; }
        t[3] = (uint64_t)(c + t[4]);
        return reduced(t[0], t[1], t[2], t[3]);
    }

public:
    void canonical(uint64_t out[4]) const {   // leave Montgomery form
        Fp one_raw{{1, 0, 0, 0}};
        Fp r = *this * one_raw;
        std::memcpy(out, r.v, 32);
    }
};
typedef Fp<FQ> Fq;
typedef Fp<FR> Fr;

struct Fq2 {
    Fq c0, c1;
    static Fq2 zero() { return {Fq::zero(), Fq::zero()}; }
    static Fq2 one() { return {Fq::one(), Fq::zero()}; }
    static Fq2 load(const void* s) { const char* p = (const char*)s; return {Fq::load(p), Fq::load(p + 32)}; }
    void store(void* d) const { char* p = (char*)d; c0.store(p); c1.store(p + 32); }
    bool is_zero() const { return c0.is_zero() && c1.is_zero(); }
    bool operator==(const Fq2& o) const { return c0 == o.c0 && c1 == o.c1; }
    friend Fq2 operator+(const Fq2& a, const Fq2& b) { return {a.c0 + b.c0, a.c1 + b.c1}; }
    friend Fq2 operator-(const Fq2& a, const Fq2& b) { return {a.c0 - b.c0, a.c1 - b.c1}; }
    friend Fq2 operator*(const Fq2& a, const Fq2& b) {
        Fq aa = a.c0 * b.c0, bb = a.c1 * b.c1;
        return {aa - bb, (a.c0 + a.c1) * (b.c0 + b.c1) - aa - bb};
    }
    Fq2 neg() const { return {c0.neg(), c1.neg()}; }
    Fq2 dbl() const { return {c0.dbl(), c1.dbl()}; }
    Fq2 sqr() const { Fq ab = c0 * c1; return {(c0 + c1) * (c0 - c1), ab.dbl()}; }
    Fq2 inverse() const { Fq t = (c0.sqr() + c1.sqr()).inverse(); return {c0 * t, (c1 * t).neg()}; }
    static constexpr int BYTES = 64;
};

// Field-generic XYZZ point (x = X/ZZ, y = Y/ZZZ; infinity ZZ = 0), the same
// coordinates the device buckets use, so device partial sums load verbatim.
template <class F>
struct Xyzz {
    F X, Y, ZZ, ZZZ;
    static Xyzz inf() { return {F::zero(), F::zero(), F::zero(), F::zero()}; }
    bool is_inf() const { return ZZ.is_zero(); }
    static Xyzz from_affine(const F& x, const F& y) {
        if (x.is_zero() && y.is_zero()) return inf();
        return {x, y, F::one(), F::one()};
    }
    Xyzz dbl() const {
        if (is_inf()) return *this;
        F U = Y.dbl(), V = U.sqr(), W = U * V, S = X * V, xx = X.sqr();
        F M = xx.dbl() + xx;
        F X3 = M.sqr() - S.dbl();
        F Y3 = M * (S - X3) - W * Y;
        return {X3, Y3, V * ZZ, W * ZZZ};
    }
    // 2^k times this. The doublings run on Jacobian coordinates, 7 products
    // each against 9 (dbl-2009-l, a = 0; 0.80 against 0.87 us on Fq2, within 5 % on Fq,
    // where the chain of three products bounds both): (X ZZ, Y ZZZ, ZZ) is the same point
    // with Z = ZZ, since ZZ^3 = ZZZ^2, and (X, Y, Z^2, Z^3) leads back.
    Xyzz dbl_n(unsigned k) const {
        if (is_inf() || k == 0) return *this;
        if (k == 1) return dbl();
        F x = X * ZZ, y = Y * ZZZ, z = ZZ;
        for (; k; --k) {
            const F A = x.sqr(), B = y.sqr(), C = B.sqr();
            const F D = (x * B).dbl().dbl(), E = A.dbl() + A;
            z = (y * z).dbl();
            x = E.sqr() - D.dbl();
            y = E * (D - x) - C.dbl().dbl().dbl();
        }
        const F zz = z.sqr();
        return {x, y, zz, zz * z};
    }
    Xyzz add(const Xyzz& o) const {
        if (o.is_inf()) return *this;
        if (is_inf()) return o;
        F U1 = X * o.ZZ, U2 = o.X * ZZ, S1 = Y * o.ZZZ, S2 = o.Y * ZZZ;
        F P = U2 - U1, R = S2 - S1;
        if (P.is_zero()) return R.is_zero() ? dbl() : inf();
        F PP = P.sqr(), PPP = P * PP, Q = U1 * PP;
        F X3 = R.sqr() - PPP - Q.dbl();
        F Y3 = R * (Q - X3) - S1 * PPP;
        return {X3, Y3, ZZ * o.ZZ * PP, ZZZ * o.ZZZ * PPP};
    }
    Xyzz neg() const { return {X, Y.neg(), ZZ, ZZZ}; }
    // k * this for a canonical little-endian scalar
    Xyzz mul(const uint64_t k[4]) const {
        Xyzz acc = inf();
        for (int i = 255; i >= 0; --i) { acc = acc.dbl(); if ((k[i / 64] >> (i % 64)) & 1) acc = acc.add(*this); }
        return acc;
    }
    // affine (x, y); false for infinity
    bool to_affine(F& x, F& y) const {
        if (is_inf()) { x = F::zero(); y = F::zero(); return false; }
        F inv = (ZZ * ZZZ).inverse();      // 1/(ZZ ZZZ)
        x = X * (inv * ZZZ);                 // X / ZZ
        y = Y * (inv * ZZ);                  // Y / ZZZ
        return true;
    }
    // normalised Jacobian (x, y, 1) or libff's infinity (0, 1, 0)
    void store_jacobian(void* dst) const {
        char* d = (char*)dst;
        const int B = sizeof(F);
        F x, y;
        if (to_affine(x, y)) { x.store(d); y.store(d + B); F::one().store(d + 2 * B); }
        else { F::zero().store(d); F::one().store(d + B); F::zero().store(d + 2 * B); }
    }
    void store_affine(void* dst) const {
        char* d = (char*)dst;
        F x, y;
        to_affine(x, y);
        x.store(d); y.store(d + sizeof(F));
    }
    static Xyzz load_affine(const void* src) {
        const char* s = (const char*)src;
        return from_affine(F::load(s), F::load(s + sizeof(F)));
    }
    static Xyzz load_xyzz(const void* src) {
        const char* s = (const char*)src;
        const int B = sizeof(F);
        return {F::load(s), F::load(s + B), F::load(s + 2 * B), F::load(s + 3 * B)};
    }
};

// k * P for a point P fixed for many products (a proving key's delta and
// beta): 32 byte windows, entry (w, b) = b 2^(8w) P for b = 1..255, so a
// product is at most 32 additions and no doublings (double-and-add: 256
// doublings and ~128 additions)
template <class F>
struct FixedBase {
    std::vector<Xyzz<F>> t;   // 32 x 256 entries, b = 0 unused
    void build(const Xyzz<F>& p) {
        t.assign(32 * 256, Xyzz<F>::inf());
        Xyzz<F> base = p;
        for (int w = 0; w < 32; ++w) {
            Xyzz<F> acc = Xyzz<F>::inf();
            for (int b = 1; b < 256; ++b) {
                acc = acc.add(base);
                t[w * 256 + b] = acc;
            }
            for (int q = 0; q < 8; ++q) base = base.dbl();
        }
    }
    bool ready() const { return !t.empty(); }
    Xyzz<F> mul(const uint64_t k[4]) const {
        Xyzz<F> acc = Xyzz<F>::inf();
        for (int w = 0; w < 32; ++w) {
            const uint32_t b = (uint32_t)(k[w / 8] >> (8 * (w % 8))) & 0xffu;
            if (b) acc = acc.add(t[w * 256 + b]);
        }
        return acc;
    }
};

typedef Xyzz<Fq> G1x;
typedef Xyzz<Fq2> G2x;

// Generators (libff alt_bn128_init.cu:130-132, :191-195), Montgomery form.
inline G1x g1_generator() {
    Fq x = Fq::one();
    Fq y = x.dbl();
    return G1x::from_affine(x, y);
}
inline Fq fq_from_canonical(const uint64_t c[4]) { Fq t; std::memcpy(t.v, c, 32); Fq r2; std::memcpy(r2.v, FQ.r2, 32); return t * r2; }
inline G2x g2_generator() {
    static const uint64_t xc0[4] = {0x46debd5cd992f6edULL, 0x674322d4f75edaddULL, 0x426a00665e5c4479ULL, 0x1800deef121f1e76ULL};
    static const uint64_t xc1[4] = {0x97e485b7aef312c2ULL, 0xf1aa493335a9e712ULL, 0x7260bfb731fb5d25ULL, 0x198e9393920d483aULL};
    static const uint64_t yc0[4] = {0x4ce6cc0166fa7daaULL, 0xe3d1e7690c43d37bULL, 0x4aab71808dcb408fULL, 0x12c85ea5db8c6debULL};
    static const uint64_t yc1[4] = {0x55acdadcd122975bULL, 0xbc4b313370b38ef3ULL, 0xec9e99ad690c3395ULL, 0x090689d0585ff075ULL};
    Fq2 x{fq_from_canonical(xc0), fq_from_canonical(xc1)};
    Fq2 y{fq_from_canonical(yc0), fq_from_canonical(yc1)};
    return G2x::from_affine(x, y);
}

// Montgomery's trick: affine (x, y) of every point with one inversion.
template <class F>
void batch_affine(const std::vector<Xyzz<F>>& pts, std::vector<F>& xs, std::vector<F>& ys) {
    size_t n = pts.size();
    xs.assign(n, F::zero());
    ys.assign(n, F::zero());
    std::vector<F> pre(n);
    F acc = F::one();
    for (size_t i = 0; i < n; ++i) {
        pre[i] = acc;
        if (!pts[i].is_inf()) acc = acc * (pts[i].ZZ * pts[i].ZZZ);
    }
    F inv = acc.inverse();
    for (size_t i = n; i-- > 0;) {
        if (pts[i].is_inf()) continue;
        F d = pts[i].ZZ * pts[i].ZZZ;
        F di = inv * pre[i];   // 1 / (ZZ ZZZ)
        inv = inv * d;
        xs[i] = pts[i].X * (di * pts[i].ZZZ);
        ys[i] = pts[i].Y * (di * pts[i].ZZ);
    }
}

}  // namespace host
}  // namespace hzk
