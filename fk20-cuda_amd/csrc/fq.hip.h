// Fp arithmetic of the G1 kernels: Montgomery form, 13 signed digits of 30 bits in VGPRs.
//
// What bounds every G1 kernel is the issue of v_mad_u64_u32 / v_mad_i64_i32 (one per 4 cycles and
// SIMD, about 2.0 ns under their own power limit; 32-bit VOP2 adds and masks issue at twice that
// rate, 64-bit shifts and VOP3 operations at the same).  So the representation is chosen for the
// fewest of them:
//  * 13 digits instead of the 14 unsigned limbs of fp.hip.h.  Digits are balanced (|d| about
//    2^29), products below 2^58.1, so a column of 13 + 13 of them stays below 2^63 and is
//    accumulated by v_mad_i64_i32 without carry flags: 338 multiply-adds a product against 392,
//    260 a square against 301, 507 a sum of two products against 588.
//  * Quotient digits without a multiplication.  With c = p^-1 mod 2^30 = 0x30003, -c p has
//    digit 0 equal to -1, so the quotient digit of column k < 12 is the column's low 30 bits and
//    the shift drops it.  Only the last digit uses p itself (|quotient| <= 2^29), which keeps
//    the result within +-(1/2 + 2^-12) p of a b / R.
//  * Balanced output digits without rounding: digit k is (column mod 2^30) - FQ_BETA[k]; the
//    offset's value is cancelled mod p by the constant FQ_K0 the lowest column starts from
//    (gen_constants.py).
// Values are signed and lazy: a product of |a b| <= M p^2 is below (0.54 + M / 630) p in
// absolute value (R = 630 p); sums and differences need no multiple of p added.
//
// Digit bounds.  "Balanced" digits (outputs of products and of fq_norm / fq_lin, negations of
// those): |d| <= FQ_BAL = 554 000 000 < 1.032 * 2^29, top digit < 2^27.  "Wide" (a sum or
// difference of two balanced values, digit by digit): twice that.  A product takes one balanced
// and one wide operand (12 * 2 * BAL^2 + 2^30 * sum of the positive or of the negative digits of
// -c p, 0.16 * 2^63: together below 0.97 * 2^63); a square and a pair of products (fq_mul2) take
// balanced operands only.  Tested at the extremes (tests/test_fq_host.py).
//
// Memory form: 12 x 32-bit words holding the value plus 4 p (fq_pack / fq_unpack, |value| < 4 p).
// Functions are __host__ __device__, so the kernels' code also runs in the CPU tests.
#pragma once
#include <stdint.h>

#include "constants.hip.h"

#ifndef FK20_HD
#define FK20_HD __host__ __device__ __forceinline__
#endif

// Hides a value from the optimiser, which would otherwise replace single multiply-adds by
// sequences: a factor known to be non-negative splits a column into a signed and an unsigned chain
// (an extra 64-bit addition per column, 6% of a product), a constant that is a power of two
// becomes a 64-bit shift and a subtraction with borrow.
#ifdef __HIP_DEVICE_COMPILE__
#define FQ_OPAQUE_V(x) asm("" : "+v"(x))
#define FQ_OPAQUE_S(x) asm("" : "+s"(x))
#else
#define FQ_OPAQUE_V(x)
#define FQ_OPAQUE_S(x)
#endif

namespace fk20 {

struct fq {
    int32_t l[FQ_N];
};

// ---------------------------------------------------------------- linear operations

FK20_HD void fq_set(fq &z, const int32_t *c) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = c[i];
}

FK20_HD void fq_zero(fq &z) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = 0;
}

FK20_HD void fq_one(fq &z) { fq_set(z, FQ_ONE); }

// Digit by digit, no carries: wide if both are balanced.
FK20_HD void fq_addw(fq &z, const fq &a, const fq &b) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = a.l[i] + b.l[i];
}

FK20_HD void fq_subw(fq &z, const fq &a, const fq &b) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = a.l[i] - b.l[i];
}

// -a: balanced if a is.
FK20_HD void fq_neg(fq &z, const fq &a) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = -a.l[i];
}

// Balanced digits of the same value, from wide ones: every digit hands its rounded quotient to
// the next, in parallel (no ripple).
FK20_HD void fq_norm(fq &z, const fq &a) {
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++) {
        const int32_t t = a.l[i] + (1 << 29);
        z.l[i] = (int32_t)((uint32_t)t & FQ_MASK) - (1 << 29) + c;
        c = t >> 30;
    }
    z.l[FQ_N - 1] = a.l[FQ_N - 1] + c;
}

FK20_HD void fq_add(fq &z, const fq &a, const fq &b) {
    fq_addw(z, a, b);
    fq_norm(z, z);
}

FK20_HD void fq_sub(fq &z, const fq &a, const fq &b) {
    fq_subw(z, a, b);
    fq_norm(z, z);
}

// a - b - c, balanced (three balanced digits and the rounding constant can pass 2^31: the
// quotient is taken from half the digit)
FK20_HD void fq_sub2(fq &z, const fq &a, const fq &b, const fq &c) {
    int32_t k = 0;
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++) {
        const int32_t t = a.l[i] - b.l[i] - c.l[i];
        z.l[i] = (int32_t)(((uint32_t)t + (1u << 29)) & FQ_MASK) - (1 << 29) + k;
        k = ((t >> 1) + (1 << 28)) >> 29;
    }
    z.l[FQ_N - 1] = a.l[FQ_N - 1] - b.l[FQ_N - 1] - c.l[FQ_N - 1] + k;
}

// One digit of a linear combination: t (any 64-bit value whose quotient by 2^30 is below 2^24)
// plus the carry c of the digit below; c receives this digit's.
FK20_HD int32_t fq_lin_digit(int64_t t, int32_t &c) {
    const int32_t z = (int32_t)((uint32_t)t & FQ_MASK) - (1 << 29) + c;
    c = (int32_t)(t >> 30);
    return z;
}

// Balanced digits of A a, A a + B b, A a + B b + C c for small constants: one multiply-add per
// term and digit, the rounding constant as the first one's addend.
template <int A>
FK20_HD void fq_lin(fq &z, const fq &a) {
    int32_t k = 0, ca = A;
    FQ_OPAQUE_S(ca);
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++) z.l[i] = fq_lin_digit((int64_t)a.l[i] * ca + (1 << 29), k);
    z.l[FQ_N - 1] = a.l[FQ_N - 1] * A + k;
}

template <int A, int B>
FK20_HD void fq_lin(fq &z, const fq &a, const fq &b) {
    int32_t k = 0, ca = A, cb = B;
    FQ_OPAQUE_S(ca);
    FQ_OPAQUE_S(cb);
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++)
        z.l[i] = fq_lin_digit((int64_t)b.l[i] * cb + ((int64_t)a.l[i] * ca + (1 << 29)), k);
    z.l[FQ_N - 1] = a.l[FQ_N - 1] * A + b.l[FQ_N - 1] * B + k;
}

template <int A, int B, int C>
FK20_HD void fq_lin(fq &z, const fq &a, const fq &b, const fq &c) {
    int32_t k = 0, ca = A, cb = B, cc = C;
    FQ_OPAQUE_S(ca);
    FQ_OPAQUE_S(cb);
    FQ_OPAQUE_S(cc);
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++)
        z.l[i] = fq_lin_digit((int64_t)c.l[i] * cc + ((int64_t)b.l[i] * cb + ((int64_t)a.l[i] * ca + (1 << 29))), k);
    z.l[FQ_N - 1] = a.l[FQ_N - 1] * A + b.l[FQ_N - 1] * B + c.l[FQ_N - 1] * C + k;
}

// ---------------------------------------------------------------- products

// Montgomery reduction, product scanning: `col(acc, k)` adds column k of the product (k < 25).
template <class Col>
FK20_HD void fq_reduce(fq &z, const Col &col) {
    int32_t q[FQ_N];
    int64_t acc = FQ_K0;
#pragma unroll
    for (int k = 0; k < FQ_N - 1; k++) {
        acc = col(acc, k);
#pragma unroll
        for (int i = 0; i < k; i++) acc += (int64_t)q[i] * FQ_PT[k - i];
        q[k] = (int32_t)((uint32_t)acc & FQ_MASK);  // times digit 0 of -c p: removed by the shift
        FQ_OPAQUE_V(q[k]);
        acc >>= 30;
    }
    acc = col(acc, FQ_N - 1);
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++) acc += (int64_t)q[i] * FQ_PT[FQ_N - 1 - i];
    q[FQ_N - 1] = (int32_t)((uint32_t)acc * FQ_PINV4) >> 2;
    acc += (int64_t)q[FQ_N - 1] * FQ_P[0];
    acc >>= 30;
#pragma unroll
    for (int k = FQ_N; k < 2 * FQ_N - 1; k++) {
        acc = col(acc, k);
#pragma unroll
        for (int i = k - FQ_N; i < FQ_N - 1; i++) acc += (int64_t)q[i] * FQ_PT[k - i];
        acc += (int64_t)q[FQ_N - 1] * FQ_P[k - FQ_N + 1];
        z.l[k - FQ_N] = (int32_t)((uint32_t)acc & FQ_MASK) - FQ_BETA[k - FQ_N];
        acc >>= 30;
    }
    z.l[FQ_N - 1] = (int32_t)acc - FQ_BETA[FQ_N - 1];
}

FK20_HD int64_t fq_col_mul(int64_t acc, int k, const fq &a, const fq &b) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++)
        if (k - i >= 0 && k - i < FQ_N) acc += (int64_t)a.l[i] * b.l[k - i];
    return acc;
}

// column k of a * b for b proportional to a digit by digit, given d = 2 a: the cross terms once
FK20_HD int64_t fq_col_sqr(int64_t acc, int k, const fq &a, const fq &d, const fq &b) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++)
        if (2 * i < k && k - i < FQ_N) acc += (int64_t)d.l[i] * b.l[k - i];
    if (k % 2 == 0) acc += (int64_t)a.l[k / 2] * b.l[k / 2];
    return acc;
}

struct fq_cols_mul {
    const fq &a, &b;
    FK20_HD int64_t operator()(int64_t acc, int k) const { return fq_col_mul(acc, k, a, b); }
};
struct fq_cols_sqr {
    const fq &a, &d;
    FK20_HD int64_t operator()(int64_t acc, int k) const { return fq_col_sqr(acc, k, a, d, a); }
};
struct fq_cols_mul2 {
    const fq &a, &b, &c, &d;
    FK20_HD int64_t operator()(int64_t acc, int k) const { return fq_col_mul(fq_col_mul(acc, k, a, b), k, c, d); }
};
struct fq_cols_mulsubsqr {
    const fq &a, &b, &c, &d, &n;
    FK20_HD int64_t operator()(int64_t acc, int k) const { return fq_col_sqr(fq_col_mul(acc, k, a, b), k, c, d, n); }
};

// z = a b / 2^390; one operand balanced, the other balanced or wide.
FK20_HD void fq_mul(fq &z, const fq &a, const fq &b) {
    fq r;
    fq_reduce(r, fq_cols_mul{a, b});
    z = r;
}

// z = a^2 / 2^390, a balanced.
FK20_HD void fq_sqr(fq &z, const fq &a) {
    fq r, d;
    fq_addw(d, a, a);
    fq_reduce(r, fq_cols_sqr{a, d});
    z = r;
}

// z = (a b + c d) / 2^390 with one reduction; balanced operands.
FK20_HD void fq_mul2(fq &z, const fq &a, const fq &b, const fq &c, const fq &d) {
    fq r;
    fq_reduce(r, fq_cols_mul2{a, b, c, d});
    z = r;
}

// z = (a b - c^2) / 2^390 with one reduction; balanced operands.
FK20_HD void fq_mulsubsqr(fq &z, const fq &a, const fq &b, const fq &c) {
    fq r, d, n;
    fq_addw(d, c, c);
    fq_neg(n, c);
    fq_reduce(r, fq_cols_mulsubsqr{a, b, c, d, n});
    z = r;
}

// ---------------------------------------------------------------- packing

// Non-negative 30-bit digits of a value in [0, 2^390), from any digits below 2^31 - 2^8.
FK20_HD void fq_ripple(fq &z, const fq &a) {
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < FQ_N - 1; i++) {
        const int32_t t = a.l[i] + c;
        z.l[i] = (int32_t)((uint32_t)t & FQ_MASK);
        c = t >> 30;
    }
    z.l[FQ_N - 1] = a.l[FQ_N - 1] + c;
}

// non-negative 30-bit digits of a value below 2^384 <-> 12 x 32-bit words
FK20_HD void fq_digits_to_words(uint32_t *w, const fq &a) {
#pragma unroll
    for (int j = 0; j < 12; j++) {
        const int bit = 32 * j, li = bit / 30, off = bit % 30;
        uint32_t v = (uint32_t)a.l[li] >> off;
        v |= (uint32_t)a.l[li + 1] << (30 - off);
        if (off == 29 && li + 2 < FQ_N) v |= (uint32_t)a.l[li + 2] << 31;
        w[j] = v;
    }
}

FK20_HD void fq_words_to_digits(fq &z, const uint32_t *w) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) {
        const int bit = 30 * i, wd = bit >> 5, off = bit & 31;
        const uint64_t v = ((uint64_t)(wd + 1 < 12 ? w[wd + 1] : 0u) << 32) | w[wd];
        z.l[i] = (int32_t)((uint32_t)(v >> off) & FQ_MASK);
    }
}

// |a| < 4 p (balanced) -> words of a + 4 p
FK20_HD void fq_pack(uint32_t *w, const fq &a) {
    fq t;
#pragma unroll
    for (int i = 0; i < FQ_N; i++) t.l[i] = a.l[i] + FQ_4P[i];
    fq_ripple(t, t);
    fq_digits_to_words(w, t);
}

FK20_HD void fq_unpack(fq &z, const uint32_t *w) {
    fq t;
    fq_words_to_digits(t, w);
#pragma unroll
    for (int i = 0; i < FQ_N; i++) t.l[i] -= FQ_4P[i];
    fq_norm(z, t);
}

// words of a value in [0, 2^384), as it is (no offset)
FK20_HD void fq_unpack_raw(fq &z, const uint32_t *w) {
    fq t;
    fq_words_to_digits(t, w);
    fq_norm(z, t);
}

// ---------------------------------------------------------------- conversions

// |a| < p -> non-negative digits of a mod p in [0, p)
FK20_HD void fq_canon_digits(fq &z, const fq &a) {
    fq t, u;
#pragma unroll
    for (int i = 0; i < FQ_N; i++) t.l[i] = a.l[i] + FQ_P[i];
    fq_ripple(t, t);  // in (0, 2 p)
#pragma unroll
    for (int i = 0; i < FQ_N; i++) u.l[i] = t.l[i] - FQ_P[i];
    fq_ripple(u, u);
    const bool neg = u.l[FQ_N - 1] < 0;
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = neg ? t.l[i] : u.l[i];
}

// Montgomery value (balanced, |a| < 200 p) -> 12 words of the canonical standard form in [0, p)
FK20_HD void fq_to_std(uint32_t *w, const fq &a) {
    fq one, t;
    fq_zero(one);
    one.l[0] = 1;
    fq_mul(t, a, one);
    fq_canon_digits(t, t);
    fq_digits_to_words(w, t);
}

// words of any standard-form value below 2^384 -> Montgomery (|z| < 0.6 p)
FK20_HD void fq_from_std(fq &z, const uint32_t *w) {
    fq t, r2;
    fq_unpack_raw(t, w);
    fq_set(r2, FQ_R2);
    fq_mul(z, t, r2);
}

// Montgomery value (balanced, |a| < 200 p) -> 12 words of the canonical Montgomery value in [0, p)
FK20_HD void fq_canon_words(uint32_t *w, const fq &a) {
    fq one, t;
    fq_one(one);
    fq_mul(t, a, one);
    fq_canon_digits(t, t);
    fq_digits_to_words(w, t);
}

// whether a = 0 mod p (balanced, |a| < 200 p)
FK20_HD bool fq_is_zero(const fq &a) {
    fq one, t;
    fq_one(one);
    fq_mul(t, a, one);
    fq_canon_digits(t, t);
    uint32_t acc = 0;
#pragma unroll
    for (int i = 0; i < FQ_N; i++) acc |= (uint32_t)t.l[i];
    return acc == 0;
}

// ---------------------------------------------------------------- inversion
//
// 1 / a by divsteps (Bernstein and Yang, "Fast constant-time gcd computation and modular
// inversion", TCHES 2019), 30 of them per pass over the digits, starting from delta = 1/2.  A
// division step needs only the low bits of f and g, so a pass runs 30 on one word of each with
// 32-bit adds and masks (the instructions that issue at twice the rate of a multiply-add),
// collects them in a 2 x 2 matrix and applies it to f, g and to the cofactors d, e (whose
// division by 2^30 mod p takes one quotient digit).  |d|, |e| grow by at most p / 2 a pass,
// which the digits hold without reduction.  About 30 passes of 900 instructions, the lanes of a
// wave together until the last is done, against 610 products by Fermat's theorem: 262 144
// affine points in 0.24 ms instead of 1.35, 512 in 0.066 instead of 0.47.

#ifdef __HIP_DEVICE_COMPILE__
#define FQ_ANY(x) __any(x)
#else
#define FQ_ANY(x) (x)
#endif

// 30 division steps on the low words: 2^30 (f', g') = (u f + v g, q f + r g).  D = 2 delta.
struct fq_divsteps {
    int32_t u, v, q, r;
    FK20_HD void run(int32_t &D, uint32_t f, uint32_t g) {
        u = 1, v = 0, q = 0, r = 1;
#pragma unroll 6
        for (int i = 0; i < 30; i++) {
            const int32_t odd = -(int32_t)(g & 1);
            int32_t pos = (-D) >> 31;  // delta > 0: subtract f (and swap if g is odd), else add
            g += (((uint32_t)f ^ (uint32_t)pos) - (uint32_t)pos) & (uint32_t)odd;
            q += ((u ^ pos) - pos) & odd;
            r += ((v ^ pos) - pos) & odd;
            pos &= odd;
            D = (D ^ pos) - pos + 2;
            f += g & (uint32_t)pos;
            u += q & pos;
            v += r & pos;
            g >>= 1;
            u = (int32_t)((uint32_t)u << 1);
            v = (int32_t)((uint32_t)v << 1);
        }
    }
};

// Inverse of a Montgomery value (balanced, |a| < 200 p), Montgomery; 0 gives 0.
FK20_HD void fq_inv(fq &z, const fq &a) {
    // non-negative 30-bit digits below a signed top digit
    fq f, g, d, e;
    fq_one(e);
    fq_mul(g, a, e);
    fq_canon_digits(g, g);
    fq_set(f, FQ_P);
    fq_ripple(f, f);
    fq_zero(d);
    fq_zero(e);
    e.l[0] = 1;
    int32_t D = 1;
    // 381-bit values are done after at most 37 passes (1102 steps); the bound only ends the loop
#pragma unroll 1
    for (int pass = 0; pass < 40; pass++) {
        uint32_t nz = 0;
#pragma unroll
        for (int i = 0; i < FQ_N; i++) nz |= (uint32_t)g.l[i];
        if (!FQ_ANY(nz != 0)) break;
        fq_divsteps t;
        t.run(D, (uint32_t)f.l[0] | (uint32_t)f.l[1] << 30, (uint32_t)g.l[0] | (uint32_t)g.l[1] << 30);
        int64_t cf = (int64_t)t.u * f.l[0] + (int64_t)t.v * g.l[0];
        int64_t cg = (int64_t)t.q * f.l[0] + (int64_t)t.r * g.l[0];
        int64_t cd = (int64_t)t.u * d.l[0] + (int64_t)t.v * e.l[0];
        int64_t ce = (int64_t)t.q * d.l[0] + (int64_t)t.r * e.l[0];
        const int32_t md = (int32_t)((uint32_t)cd * FQ_PINV4) >> 2, me = (int32_t)((uint32_t)ce * FQ_PINV4) >> 2;
        cd += (int64_t)md * FQ_P[0];
        ce += (int64_t)me * FQ_P[0];
        cf >>= 30, cg >>= 30, cd >>= 30, ce >>= 30;
#pragma unroll
        for (int i = 1; i < FQ_N; i++) {
            const int32_t fi = f.l[i], gi = g.l[i], di = d.l[i], ei = e.l[i];
            cf += (int64_t)t.u * fi + (int64_t)t.v * gi;
            cg += (int64_t)t.q * fi + (int64_t)t.r * gi;
            cd += (int64_t)t.u * di + (int64_t)t.v * ei + (int64_t)md * FQ_P[i];
            ce += (int64_t)t.q * di + (int64_t)t.r * ei + (int64_t)me * FQ_P[i];
            f.l[i - 1] = (int32_t)((uint32_t)cf & FQ_MASK);
            g.l[i - 1] = (int32_t)((uint32_t)cg & FQ_MASK);
            d.l[i - 1] = (int32_t)((uint32_t)cd & FQ_MASK);
            e.l[i - 1] = (int32_t)((uint32_t)ce & FQ_MASK);
            FQ_OPAQUE_V(f.l[i - 1]);
            FQ_OPAQUE_V(g.l[i - 1]);
            FQ_OPAQUE_V(d.l[i - 1]);
            FQ_OPAQUE_V(e.l[i - 1]);
            cf >>= 30, cg >>= 30, cd >>= 30, ce >>= 30;
        }
        f.l[FQ_N - 1] = (int32_t)cf;
        g.l[FQ_N - 1] = (int32_t)cg;
        d.l[FQ_N - 1] = (int32_t)cd;
        e.l[FQ_N - 1] = (int32_t)ce;
    }
    // f = +-1 (or p for a = 0, where d = 0): 1 / (x R) = f d, times R^3 / R
    const int32_t s = f.l[FQ_N - 1] >> 31;
    fq_norm(d, d);
#pragma unroll
    for (int i = 0; i < FQ_N; i++) d.l[i] = (d.l[i] ^ s) - s;
    fq_set(e, FQ_R3);
    fq_mul(z, d, e);
}

}  // namespace fk20
