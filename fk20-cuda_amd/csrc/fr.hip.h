// Fr arithmetic (BLS12-381 scalar field) on gfx950: Montgomery form, 8 x 32-bit limbs,
// canonical values in [0, r).
//
// Replaces the reference's standard-form Fr (fr_mul.cu:13 schoolbook + Barrett,
// fr_addsub.cu:18, fr_add.cuh, fr_sub.cuh).  This is a plain CIOS with carry chains, for the
// element-wise operations and the programs' checks; the transforms run on the 9 signed
// 29-bit digits of fn below.
#pragma once
#include <stdint.h>

#include "constants.hip.h"

#ifndef FK20_HD
#define FK20_HD __host__ __device__ __forceinline__
#endif

// Hides a value from the optimiser (see fq.hip.h).
#ifndef FK20_OPAQUE_V
#ifdef __HIP_DEVICE_COMPILE__
#define FK20_OPAQUE_V(x) asm("" : "+v"(x))
#else
#define FK20_OPAQUE_V(x)
#endif
#endif

namespace fk20 {

struct fs {
    uint32_t l[8];
};

FK20_HD uint32_t addc32(uint32_t a, uint32_t b, uint32_t cin, uint32_t &cout) {
    uint64_t s = (uint64_t)a + b + cin;
    cout = (uint32_t)(s >> 32);
    return (uint32_t)s;
}

FK20_HD uint32_t subb32(uint32_t a, uint32_t b, uint32_t bin, uint32_t &bout) {
    uint64_t d = (uint64_t)a - b - bin;
    bout = (uint32_t)(d >> 63);
    return (uint32_t)d;
}

// z = z - r if z >= r (z < 2r)
FK20_HD void fs_cond_sub(fs &z, uint32_t top) {
    fs t;
    uint32_t br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) t.l[i] = subb32(z.l[i], FR_R[i], br, br);
    // keep t unless the subtraction borrowed past the extra top word
    const bool keep = (top != 0) || (br == 0);
#pragma unroll
    for (int i = 0; i < 8; i++) z.l[i] = keep ? t.l[i] : z.l[i];
}

FK20_HD void fs_add(fs &z, const fs &a, const fs &b) {
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) z.l[i] = addc32(a.l[i], b.l[i], c, c);
    fs_cond_sub(z, c);
}

FK20_HD void fs_sub(fs &z, const fs &a, const fs &b) {
    uint32_t br = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) z.l[i] = subb32(a.l[i], b.l[i], br, br);
    // add r back if negative
    uint32_t c = 0;
    const uint32_t mask = 0u - br;
#pragma unroll
    for (int i = 0; i < 8; i++) z.l[i] = addc32(z.l[i], FR_R[i] & mask, c, c);
}

// CIOS Montgomery product, inputs < r (or a < 2^256 and b < r), output < r.
FK20_HD void fs_mul(fs &z, const fs &a, const fs &b) {
    uint32_t t[10];
#pragma unroll
    for (int j = 0; j < 10; j++) t[j] = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        uint32_t c = 0;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            uint64_t s = (uint64_t)a.l[j] * b.l[i] + t[j] + c;
            t[j] = (uint32_t)s;
            c = (uint32_t)(s >> 32);
        }
        uint64_t s = (uint64_t)t[8] + c;
        t[8] = (uint32_t)s;
        t[9] = (uint32_t)(s >> 32);
        const uint32_t m = t[0] * FR_RINV;
        s = (uint64_t)m * FR_R[0] + t[0];
        c = (uint32_t)(s >> 32);
#pragma unroll
        for (int j = 1; j < 8; j++) {
            s = (uint64_t)m * FR_R[j] + t[j] + c;
            t[j - 1] = (uint32_t)s;
            c = (uint32_t)(s >> 32);
        }
        s = (uint64_t)t[8] + c;
        t[7] = (uint32_t)s;
        t[8] = t[9] + (uint32_t)(s >> 32);
    }
#pragma unroll
    for (int j = 0; j < 8; j++) z.l[j] = t[j];
    fs_cond_sub(z, t[8]);
}

FK20_HD void fs_set(fs &z, const uint32_t *c) {
#pragma unroll
    for (int i = 0; i < 8; i++) z.l[i] = c[i];
}

FK20_HD void fs_zero(fs &z) {
#pragma unroll
    for (int i = 0; i < 8; i++) z.l[i] = 0;
}

// any 256-bit standard-form value -> its canonical representative in [0, r): 2^256 < 3 r, so
// at most two subtractions of r
FK20_HD void fs_reduce_std(fs &z) {
    fs_cond_sub(z, 0);
    fs_cond_sub(z, 0);
}

// standard form (any 256-bit value) -> canonical Montgomery
FK20_HD void fs_to_mont(fs &z, const fs &a) {
    fs r2;
    fs_set(r2, FR_R2);
    fs_mul(z, a, r2);
}

// canonical Montgomery -> canonical standard form
FK20_HD void fs_from_mont(fs &z, const fs &a) {
    fs one;
    fs_zero(one);
    one.l[0] = 1;
    fs_mul(z, a, one);
}

// ---------------------------------------------------------------- transforms
//
// The scalar transforms are bound by the issue of the products' instructions too.  Their form is 9
// signed digits of 29 bits: columns of 9 + 8 products of at most 2^59 need no carries, r = 1
// (mod 2^32) makes a quotient digit the column's low 29 bits, so a product is 153 multiply-adds
// and 34 masks and shifts, against about 420 instructions of the carry-chained 8 x 32-bit form
// above; and sums need no reduction.  The data stays in standard form (the factors are in
// Montgomery form), so there is no conversion.
//
// Digits: a product's are in [0, 2^29) under a signed top digit; sums and differences of up to four
// such values (|digit| <= 2^31 - 1) may be multiplied as they are.  Values: r^2 / 2^261 = 0.0142 r, so
// a product of |v| < 18 r is in (-1.26 r, 0.26 r); the sum of eight inputs, any 256-bit values
// below 2.21 r each, is below 17.7 r, and eight products later passes add are below 10.1 r.
struct fn {
    int32_t l[9];
};

FK20_HD void fn_add(fn &z, const fn &a, const fn &b) {
#pragma unroll
    for (int i = 0; i < 9; i++) z.l[i] = a.l[i] + b.l[i];
}

FK20_HD void fn_sub(fn &z, const fn &a, const fn &b) {
#pragma unroll
    for (int i = 0; i < 9; i++) z.l[i] = a.l[i] - b.l[i];
}

// digits within 2^28 + 4 of 0 (all but the top one), the same value
FK20_HD void fn_norm(fn &a) {
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const uint32_t t = (uint32_t)a.l[i] + (1u << 28);
        const int32_t q = ((a.l[i] >> 1) + (1 << 27)) >> 28;  // (a + 2^28) >> 29, a up to 2^31 - 1
        a.l[i] = (int32_t)(t & 0x1fffffffu) - (1 << 28) + c;
        c = q;
    }
    a.l[8] += c;
}

// z = a w / 2^261: |digits of a| < 2^31, w balanced (|digits| <= 2^28) and |w| < r
FK20_HD void fn_mul(fn &z, const fn &a, const fn &w) {
    int32_t q[9];
    fn r;
    int64_t acc = 0;
#pragma unroll
    for (int k = 0; k < 17; k++) {
#pragma unroll
        for (int i = 0; i < 9; i++)
            if (k - i >= 0 && k - i < 9) acc += (int64_t)a.l[i] * w.l[k - i];
#pragma unroll
        for (int i = 0; i < 9; i++)
            if (i < k && k - i < 9) acc += (int64_t)q[i] * FN_RT[k - i];
        const int32_t d = (int32_t)((uint32_t)acc & 0x1fffffffu);
        if (k < 9) {
            q[k] = d;  // times digit 0 of -r: removed by the shift
            FK20_OPAQUE_V(q[k]);
        } else {
            r.l[k - 9] = d;
        }
        acc >>= 29;
    }
    r.l[8] = (int32_t)acc;
    z = r;
}

// 8 words of any 256-bit value <-> digits; the words of a canonical value from non-negative digits
FK20_HD void fn_unpack(fn &z, const uint32_t *w) {
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int bit = 29 * i, wd = bit >> 5, off = bit & 31;
        const uint64_t v = ((uint64_t)(wd + 1 < 8 ? w[wd + 1] : 0u) << 32) | w[wd];
        z.l[i] = (int32_t)((uint32_t)(v >> off) & 0x1fffffffu);
    }
}

// words of the canonical value of -2 r <= a < r, |digits| as fn_mul gives them (a product is well inside)
FK20_HD void fn_canon(uint32_t *w, const fn &a) {
    fn t, u;
    int32_t c = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {  // a + r
        const int32_t v = a.l[i] - FN_RT[i] + c;
        t.l[i] = i < 8 ? (int32_t)((uint32_t)v & 0x1fffffffu) : v;
        c = v >> 29;
    }
    const bool neg = t.l[8] < 0;
    c = 0;
#pragma unroll
    for (int i = 0; i < 9; i++) {
        const int32_t v = t.l[i] + (neg ? -FN_RT[i] : FN_RT[i]) + c;
        u.l[i] = i < 8 ? (int32_t)((uint32_t)v & 0x1fffffffu) : v;
        c = v >> 29;
    }
    const bool keep = u.l[8] < 0;  // a + r was in [0, r)
#pragma unroll
    for (int i = 0; i < 9; i++) u.l[i] = keep ? t.l[i] : u.l[i];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int bit = 32 * j, li = bit / 29, off = bit % 29;
        uint32_t v = (uint32_t)u.l[li] >> off | (uint32_t)u.l[li + 1] << (29 - off);
        if (58 - off < 32 && li + 2 < 9) v |= (uint32_t)u.l[li + 2] << (58 - off);
        w[j] = v;
    }
}

// balanced digits of a value below 2^256 (8 words)
FK20_HD void fn_from_words(int32_t *z, const uint32_t *w) {
    fn t;
    fn_unpack(t, w);
    int32_t c = 0;
    for (int i = 0; i < 8; i++) {
        const int32_t v = t.l[i] + c;
        c = (v + (1 << 28)) >> 29;
        z[i] = v - (c << 29);
    }
    z[8] = t.l[8] + c;
}

}  // namespace fk20
