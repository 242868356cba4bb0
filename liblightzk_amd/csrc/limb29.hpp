// Montgomery arithmetic on nine signed 29-bit limbs (radix 2^261), the form
// the MSM's point additions and the throughput NTT compute in.
//
// Bound: the integer multiply. On the MI355X a v_mad_i64_i32 (like every
// three-operand VALU instruction) issues in four cycles a wave and more (5.3
// measured at 2.4 GHz nominal over a full chip, 4.2-4.7 for bfe, alignbit,
// 64-bit shifts), a two-operand one (v_sub, v_and) in two (2.4-3.1), and a
// chain of dependent multiply-adds runs as fast as independent ones. So what
// counts is the number of multiply-adds, then of other three-operand steps:
//
//  * 29-bit limbs: a column of up to 18 limb products, 9 reduction products and
//    a carry fits a signed 64-bit accumulator, so every partial product is one
//    v_mad_i64_i32 and nothing else (32-bit limbs need a carry fold each).
//  * Signed limbs: a difference is nine two-operand subtractions, with no
//    multiple of p added and no carries propagated; products take it as it is
//    (limbs in (-2^29, 2^29), value negative or not) and normalise.
//  * Sums of products (a b + c d, a^2 - b^2, with an addend at the result's
//    scale) are reduced once: 81 multiply-adds, 9 masks and 17 shifts less for
//    every product that shares a reduction.
//  * Reduction digits without a multiplication: with N = p (-p^-1 mod 2^29),
//    N = -1 mod 2^29, the digit of a column is its low 29 bits, and adding
//    digit * N clears the column and adds digit * (N + 1) / 2^29 one column
//    up. Eight of the nine digits go that way (together they add less than
//    0.51 p to the result); the last uses p itself, which keeps the result
//    small.
//
// A result is normalized: limbs 0..7 in [0, 2^29), limb 8 signed. For operands
// a, b (values in units of p) it lies between a b / 169 and a b / 169 + 1 +
// NPR, NPR = (N + 1) / 2^29 p = 0.142 for Fq, 0.5 for Fr (2^261 / p > 169.2 for
// both); a sum of products likewise with its sum for a b.
//
// Column bound: |limb product| <= (2^29 - 1)^2, at most eight full-size
// products per column and operand pair (limb 8 holds at most 25 bits), at most
// eight full-size reduction products, carry < 2^35: two products with limbs in
// (-2^29, 2^29) make at most 16 + 8 units of 2^58, below the 32 of a signed
// 64-bit column. A doubled operand counts twice.
#pragma once
#include <utility>
#include "field.hpp"

namespace hzk {

static constexpr uint32_t MASK29 = (1u << 29) - 1;

struct Fq29Mod {
    static constexpr uint32_t P[9] = {0x187cfd47, 0x010460b6, 0x1c72a34f, 0x02d522d0, 0x1585d978,
                                      0x02db40c0, 0x00a6e141, 0x0e5c2634, 0x0030644e};
    static constexpr uint32_t M0 = 0x04866389;     // -p^-1 mod 2^29
    static constexpr uint32_t PINV = 0x1b799c77;   // p^-1 mod 2^29
    // (p M0 + 1) / 2^29
    static constexpr uint32_t NP[9] = {0x17789a9f, 0x05ffc3dc, 0x0d6bde42, 0x1cf152e3, 0x18eb055f,
                                       0x0ed815e2, 0x016626d2, 0x0b8bab0f, 0x0006d7c4};
};

struct Fr29Mod {
    static constexpr uint32_t P[9] = {0x10000001, 0x1f0fac9f, 0x0e5c2450, 0x07d090f3, 0x1585d283,
                                      0x02db40c0, 0x00a6e141, 0x0e5c2634, 0x0030644e};   // r
    static constexpr uint32_t M0 = 0x0fffffff;     // -r^-1 mod 2^29
    // (r M0 + 1) / 2^29
    static constexpr uint32_t NP[9] = {0x18f05361, 0x012bb1fe, 0x0f5d8135, 0x1e6275f6, 0x07e7a880,
                                       0x10c6bf1f, 0x11f74a6c, 0x06fdaecb, 0x00183227};
};

// acc += sum_i x[i] * y[i]: one v_mad_i64_i32 each, addend and sum in place.
// As plain C++ the compiler re-associates a column into partial chains joined
// by extra 64-bit adds. S: y are constants, held in scalar registers.
template <int N, bool S = false>
HZK_DEV void mads(int64_t& acc, const int32_t (&x)[N], const int32_t (&y)[N]) {
    static_assert(N >= 1 && N <= 9, "one to nine products");
    if constexpr (N == 1) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]) : "vcc");
    }
    else if constexpr (N == 2) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]) : "vcc");
    }
    else if constexpr (N == 3) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]) : "vcc");
    }
    else if constexpr (N == 4) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]), "v"(x[3]), "s"(y[3]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]), "v"(x[3]), "v"(y[3]) : "vcc");
    }
    else if constexpr (N == 5) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]), "v"(x[3]), "s"(y[3]), "v"(x[4]), "s"(y[4]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]), "v"(x[3]), "v"(y[3]), "v"(x[4]), "v"(y[4]) : "vcc");
    }
    else if constexpr (N == 6) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]), "v"(x[3]), "s"(y[3]), "v"(x[4]), "s"(y[4]), "v"(x[5]), "s"(y[5]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]), "v"(x[3]), "v"(y[3]), "v"(x[4]), "v"(y[4]), "v"(x[5]), "v"(y[5]) : "vcc");
    }
    else if constexpr (N == 7) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %13, %14, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]), "v"(x[3]), "s"(y[3]), "v"(x[4]), "s"(y[4]), "v"(x[5]), "s"(y[5]), "v"(x[6]), "s"(y[6]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %13, %14, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]), "v"(x[3]), "v"(y[3]), "v"(x[4]), "v"(y[4]), "v"(x[5]), "v"(y[5]), "v"(x[6]), "v"(y[6]) : "vcc");
    }
    else if constexpr (N == 8) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %13, %14, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %15, %16, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]), "v"(x[3]), "s"(y[3]), "v"(x[4]), "s"(y[4]), "v"(x[5]), "s"(y[5]), "v"(x[6]), "s"(y[6]), "v"(x[7]), "s"(y[7]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %13, %14, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %15, %16, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]), "v"(x[3]), "v"(y[3]), "v"(x[4]), "v"(y[4]), "v"(x[5]), "v"(y[5]), "v"(x[6]), "v"(y[6]), "v"(x[7]), "v"(y[7]) : "vcc");
    }
    else if constexpr (N == 9) {
        if constexpr (S) asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %13, %14, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %15, %16, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %17, %18, %0"
            : "+v"(acc) : "v"(x[0]), "s"(y[0]), "v"(x[1]), "s"(y[1]), "v"(x[2]), "s"(y[2]), "v"(x[3]), "s"(y[3]), "v"(x[4]), "s"(y[4]), "v"(x[5]), "s"(y[5]), "v"(x[6]), "s"(y[6]), "v"(x[7]), "s"(y[7]), "v"(x[8]), "s"(y[8]) : "vcc");
        else asm("v_mad_i64_i32 %0, vcc, %1, %2, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %3, %4, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %5, %6, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %7, %8, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %9, %10, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %11, %12, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %13, %14, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %15, %16, %0\n\t"
            "v_mad_i64_i32 %0, vcc, %17, %18, %0"
            : "+v"(acc) : "v"(x[0]), "v"(y[0]), "v"(x[1]), "v"(y[1]), "v"(x[2]), "v"(y[2]), "v"(x[3]), "v"(y[3]), "v"(x[4]), "v"(y[4]), "v"(x[5]), "v"(y[5]), "v"(x[6]), "v"(y[6]), "v"(x[7]), "v"(y[7]), "v"(x[8]), "v"(y[8]) : "vcc");
    }
}
// acc += x
HZK_DEV void mad_one(int64_t& acc, int32_t x) { asm("v_mad_i64_i32 %0, vcc, %1, 1, %0" : "+v"(acc) : "v"(x) : "vcc"); }

// nine signed limbs; see the header for which functions take limbs of either sign
struct limbs29 {
    int32_t l[9];
    static HZK_DEV limbs29 zero() { return {{0, 0, 0, 0, 0, 0, 0, 0, 0}}; }
    // 8 x 32-bit limbs (a value < 2^256) from two 16-byte words (low, high); no
    // array in between: a small private array indexed in a loop can be placed
    // in LDS by the compiler
    static HZK_DEV limbs29 unpack(const uint4& lo, const uint4& hi) {
        limbs29 r;
        r.l[0] = lo.x & MASK29;
        r.l[1] = ((lo.x >> 29) | (lo.y << 3)) & MASK29;
        r.l[2] = ((lo.y >> 26) | (lo.z << 6)) & MASK29;
        r.l[3] = ((lo.z >> 23) | (lo.w << 9)) & MASK29;
        r.l[4] = ((lo.w >> 20) | (hi.x << 12)) & MASK29;
        r.l[5] = ((hi.x >> 17) | (hi.y << 15)) & MASK29;
        r.l[6] = ((hi.y >> 14) | (hi.z << 18)) & MASK29;
        r.l[7] = ((hi.z >> 11) | (hi.w << 21)) & MASK29;
        r.l[8] = hi.w >> 8;
        return r;
    }
    // a normalized value in [0, 2^256) back
    HZK_DEV void pack(uint4& lo, uint4& hi) const {
        uint32_t u[9];
#pragma unroll
        for (int i = 0; i < 9; ++i) u[i] = (uint32_t)l[i];
        lo = make_uint4(u[0] | (u[1] << 29), (u[1] >> 3) | (u[2] << 26), (u[2] >> 6) | (u[3] << 23), (u[3] >> 9) | (u[4] << 20));
        hi = make_uint4((u[4] >> 12) | (u[5] << 17), (u[5] >> 15) | (u[6] << 14), (u[6] >> 18) | (u[7] << 11), (u[7] >> 21) | (u[8] << 8));
    }
    // limb by limb, no carries
    friend HZK_DEV limbs29 operator+(const limbs29& a, const limbs29& b) {
        limbs29 r;
#pragma unroll
        for (int i = 0; i < 9; ++i) r.l[i] = a.l[i] + b.l[i];
        return r;
    }
    friend HZK_DEV limbs29 operator-(const limbs29& a, const limbs29& b) {
        limbs29 r;
#pragma unroll
        for (int i = 0; i < 9; ++i) r.l[i] = a.l[i] - b.l[i];
        return r;
    }
    HZK_DEV limbs29 operator-() const {
        limbs29 r;
#pragma unroll
        for (int i = 0; i < 9; ++i) r.l[i] = -l[i];
        return r;
    }
    HZK_DEV limbs29 twice() const {
        limbs29 r;
#pragma unroll
        for (int i = 0; i < 9; ++i) r.l[i] = l[i] << 1;
        return r;
    }
    // carries propagated: the same value normalized (limbs within +-2^30)
    HZK_DEV limbs29 norm() const {
        limbs29 r;
        int32_t c = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int32_t v = l[i] + c;
            r.l[i] = v & (int32_t)MASK29;
            c = v >> 29;
        }
        r.l[8] = l[8] + c;
        return r;
    }
};

// ---- one reduced sum of products; column k of the scan is vv<k> (the limb
// products), red<k> (the reduction products), fin<k> (digit or result limb)
template <class M>
struct Scan29 {
    limbs29& r;
    int64_t acc = 0;
    int32_t m[9];
    HZK_DEV explicit Scan29(limbs29& out) : r(out) {}
    static constexpr int lo(int k) { return k > 8 ? k - 8 : 0; }
    static constexpr int terms(int k) { return k < 9 ? k + 1 : 17 - k; }
    template <int k>
    HZK_DEV void mul_col(const limbs29& a, const limbs29& b) {
        constexpr int n = terms(k);
        int32_t x[n], y[n];
#pragma unroll
        for (int i = 0; i < n; ++i) x[i] = a.l[lo(k) + i], y[i] = b.l[k - lo(k) - i];
        mads<n>(acc, x, y);
    }
    // sum_j a_j a_(k-j) as sum_(j < k-j) (2 a_j) a_(k-j) + a_(k/2)^2; d = 2 a
    template <int k>
    HZK_DEV void sqr_col(const limbs29& d, const limbs29& a) {
        constexpr int n = (terms(k) + 1) / 2;
        int32_t x[n], y[n];
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const int j = lo(k) + i;
            x[i] = 2 * j == k ? a.l[j] : d.l[j], y[i] = a.l[k - j];
        }
        mads<n>(acc, x, y);
    }
    template <int k>
    HZK_DEV void red() {
        if constexpr (k > 0) {
            constexpr int j0 = k < 9 ? 0 : k - 9, n = k < 9 ? k : 18 - k;   // digits j0 .. (7 by NP, 8 by P)
            int32_t x[n], y[n];
#pragma unroll
            for (int i = 0; i < n; ++i) {
                const int j = j0 + i;
                x[i] = m[j], y[i] = (int32_t)(j < 8 ? M::NP[k - 1 - j] : M::P[k - 8]);
            }
            mads<n, true>(acc, x, y);
        }
    }
    template <int k>
    HZK_DEV void fin() {
        if constexpr (k < 8) {
            m[k] = (int32_t)((uint32_t)acc & MASK29);
        } else if constexpr (k == 8) {
            m[8] = (int32_t)(((uint32_t)acc * M::M0) & MASK29);
            const int32_t x[1] = {m[8]}, y[1] = {(int32_t)M::P[0]};
            mads<1, true>(acc, x, y);
        } else {
            r.l[k - 9] = (int32_t)((uint32_t)acc & MASK29);
        }
        acc >>= 29;
        if constexpr (k == 16) r.l[8] = (int32_t)acc;
    }
    HZK_DEV void end() {}
};
// r = a b
template <class M>
struct Mul29 : Scan29<M> {
    const limbs29 &a, &b;
    HZK_DEV Mul29(limbs29& r, const limbs29& a_, const limbs29& b_) : Scan29<M>(r), a(a_), b(b_) {}
    template <int k>
    HZK_DEV void vv() { this->template mul_col<k>(a, b); }
};
// r = a^2
template <class M>
struct Sqr29 : Scan29<M> {
    const limbs29& a;
    limbs29 d;
    HZK_DEV Sqr29(limbs29& r, const limbs29& a_) : Scan29<M>(r), a(a_), d(a_.twice()) {}
    template <int k>
    HZK_DEV void vv() { this->template sqr_col<k>(d, a); }
};
// r = a^2 + t (t at the result's scale: 9 multiply-adds by one, no carry pass of its own)
template <class M>
struct SqrAdd29 : Sqr29<M> {
    const limbs29& t;
    HZK_DEV SqrAdd29(limbs29& r, const limbs29& a_, const limbs29& t_) : Sqr29<M>(r, a_), t(t_) {}
    template <int k>
    HZK_DEV void vv() {
        Sqr29<M>::template vv<k>();
        if constexpr (k >= 9) mad_one(this->acc, t.l[k - 9]);
    }
    HZK_DEV void end() { this->r.l[8] += t.l[8]; }
};
// r = a b + c d
template <class M>
struct Sum29 : Scan29<M> {
    const limbs29 &a, &b, &c, &d;
    HZK_DEV Sum29(limbs29& r, const limbs29& a_, const limbs29& b_, const limbs29& c_, const limbs29& d_)
        : Scan29<M>(r), a(a_), b(b_), c(c_), d(d_) {}
    template <int k>
    HZK_DEV void vv() {
        this->template mul_col<k>(a, b);
        this->template mul_col<k>(c, d);
    }
};
// r = a b + t
template <class M>
struct MulAdd29 : Mul29<M> {
    const limbs29& t;
    HZK_DEV MulAdd29(limbs29& r, const limbs29& a_, const limbs29& b_, const limbs29& t_) : Mul29<M>(r, a_, b_), t(t_) {}
    template <int k>
    HZK_DEV void vv() {
        Mul29<M>::template vv<k>();
        if constexpr (k >= 9) mad_one(this->acc, t.l[k - 9]);
    }
    HZK_DEV void end() { this->r.l[8] += t.l[8]; }
};
// r = a^2 - b^2 (+ t)
template <class M>
struct SqrDiff29 : Scan29<M> {
    const limbs29 &a, &b;
    limbs29 da, nb, ndb;
    HZK_DEV SqrDiff29(limbs29& r, const limbs29& a_, const limbs29& b_)
        : Scan29<M>(r), a(a_), b(b_), da(a_.twice()), nb(-b_), ndb(nb.twice()) {}
    template <int k>
    HZK_DEV void vv() {
        this->template sqr_col<k>(da, a);
        constexpr int n = (Scan29<M>::terms(k) + 1) / 2;
        int32_t x[n], y[n];
#pragma unroll
        for (int i = 0; i < n; ++i) {
            const int j = Scan29<M>::lo(k) + i;
            x[i] = 2 * j == k ? nb.l[j] : ndb.l[j], y[i] = b.l[k - j];
        }
        mads<n>(this->acc, x, y);
    }
};
template <class M>
struct SqrDiffAdd29 : SqrDiff29<M> {
    const limbs29& t;
    HZK_DEV SqrDiffAdd29(limbs29& r, const limbs29& a_, const limbs29& b_, const limbs29& t_) : SqrDiff29<M>(r, a_, b_), t(t_) {}
    template <int k>
    HZK_DEV void vv() {
        SqrDiff29<M>::template vv<k>();
        if constexpr (k >= 9) mad_one(this->acc, t.l[k - 9]);
    }
    HZK_DEV void end() { this->r.l[8] += t.l[8]; }
};
// r = a b + c d + e f + g h
template <class M>
struct Sum4_29 : Scan29<M> {
    const limbs29 &a, &b, &c, &d, &e, &f, &g, &h;
    HZK_DEV Sum4_29(limbs29& r, const limbs29& a_, const limbs29& b_, const limbs29& c_, const limbs29& d_, const limbs29& e_,
                    const limbs29& f_, const limbs29& g_, const limbs29& h_)
        : Scan29<M>(r), a(a_), b(b_), c(c_), d(d_), e(e_), f(f_), g(g_), h(h_) {}
    template <int k>
    HZK_DEV void vv() {
        this->template mul_col<k>(a, b);
        this->template mul_col<k>(c, d);
        this->template mul_col<k>(e, f);
        this->template mul_col<k>(g, h);
    }
};

template <int k, class... J>
HZK_DEV void scan29_col(J&... j) {
    (j.template vv<k>(), ...);
    (j.template red<k>(), ...);
    (j.template fin<k>(), ...);
}
template <int... k, class... J>
HZK_DEV void scan29_all(std::integer_sequence<int, k...>, J&... j) {
    (scan29_col<k>(j...), ...);
}
// the scans column by column side by side: an independent scan's block stands
// between a block and the one that reads its accumulator, where the compiler
// would otherwise put a wait state after inline asm. A result may be an
// operand too: limb k - 9 is written after column k, its last use.
template <class... J>
HZK_DEV void scan29(J&&... j) {
    scan29_all(std::make_integer_sequence<int, 17>{}, j...);
    (j.end(), ...);
}

}  // namespace hzk
