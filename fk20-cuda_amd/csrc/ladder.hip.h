// Fixed-scalar G1 multiplication of the column-batched transforms: x <- k * x for a scalar
// known when the library loads (a twiddle w^e or a power 2^-j), run as a precomputed program
// over the GLV + wNAF digits of k.  Shared by the HIP kernels and, compiled by g++, by the CPU
// tests (FK20_UNIFORM is then the identity).
//
// Program encoding.  A split k lambda^-t = k1 + k2 lambda (|k1|, k2 < 2^128, phi(P) =
// (beta x, y) = lambda P, t in {0, 1, 2}): k1's digits act on phi^t(P), k2's on
// phi^(t+1)(P).  One 32-bit op per non-zero digit, read wave-uniformly:
//   bits 0..7   doublings to perform before this op (for the END op: trailing doublings)
//   bit  8      apply phi to the table entry (x times beta)
//   bit  13     apply phi^2 instead (x times beta^2)
//   bits 9..11  table entry e: the odd multiple (2e + 1) P
//   bit  12     negate
//   bit  31     END
//
// Arithmetic (g1q.hip.h).  The input is converted to Jacobian coordinates and its odd multiples
// P, 3P, .., (2^(W-1) - 1) P are built with one common Z (doubling with update, then co-Z
// additions 2P + (2i - 1)P, then each entry rescaled to the last Z): on the isomorphic curve
// y^2 = x^3 + b Z^6 they are affine points, so the ladder runs Jacobian doublings (3 squares, 2
// products, a product minus square) and mixed additions (3 squares, 6 products, a pair) instead
// of complete projective formulas, and the table holds x and 2 y only.  At the end the
// accumulator's Z is multiplied by the table's Z and the point converted back to homogeneous
// coordinates.
//
// The formulas are incomplete.  For an input of prime order r that is not infinity, the
// accumulator before each addition is a P and the entry b P with a, b known scalars; the host
// checks every program (ctx.cpp) for a != 0 and a != +-b mod r, so no exceptional case
// occurs.  An input at infinity (Z = 0) is detected and returned as infinity.  Inputs outside
// the order-r subgroup are not handled here (the GLV split assumes phi(P) = lambda P): the
// transforms find such rows with g1_in_subgroup below and recompute them on another path.
#pragma once
#include "g1.hip.h"
#include "g1q.hip.h"

#ifndef FK20_UNIFORM
#define FK20_UNIFORM(x) __builtin_amdgcn_readfirstlane(x)
#endif

namespace fk20 {

static constexpr uint32_t TWOP_DBL_MASK = 0xffu;
static constexpr uint32_t TWOP_PHI = 1u << 8;
static constexpr unsigned TWOP_ENTRY_SHIFT = 9;
static constexpr uint32_t TWOP_NEG = 1u << 12;
static constexpr uint32_t TWOP_PHI2 = 1u << 13;
static constexpr uint32_t TWOP_END = 1u << 31;

// wNAF width used by the G1 transform kernels (odd multiples P, 3P, .., 15P, kept in private
// memory); the twiddle programs are built for the same width
#ifndef FK20_TW_WNAF
#define FK20_TW_WNAF 5
#endif
static constexpr int TW_WNAF = FK20_TW_WNAF;

// The ladder's table: x and 2 y of the odd multiples P, 3P, .., (2^(W-1) - 1) P of the homogeneous
// point x (coordinates < 8 p, not infinity), affine on the isomorphic curve of the common Z zt.
template <int W>
FK20_HD void tw_table(fq *TX, fq *TY, fq &zt, const g1q &x) {
    constexpr int NT = 1 << (W - 2);
    static_assert(NT >= 2, "table of at least P and 3P");
    fq MU[NT - 1];
    // homogeneous (X : Y : Z) -> Jacobian (X Z, Y Z^2, Z)
    g1j_q P, Q;                     // Q = 2P, re-scaled by every co-Z addition
    fq t;
    fq_sqr(t, x.z);
    fq_mul(P.x, x.x, x.z);
    fq_mul(P.y, x.y, t);
    P.z = x.z;
    g1q_dblu(Q, TX[0], TY[0], P);
    fq x1 = Q.x, y1 = Q.y;
#pragma unroll 1
    for (int k = 1; k < NT; k++) g1q_zaddu(TX[k], TY[k], MU[k - 1], x1, y1, TX[k - 1], TY[k - 1]);
    // entry k has Z0 * mu_0 ... mu_{k-1}; bring it to the last entry's Z by the product of
    // the later factors, y doubled on the way
    fq s = MU[NT - 2], s2, s3;
    fq_add(TY[NT - 1], TY[NT - 1], TY[NT - 1]);
#pragma unroll 1
    for (int k = NT - 2; k >= 0; k--) {
        if (k < NT - 2) fq_mul(s, s, MU[k]);   // 12 * 12 -> < 0.8
        fq_sqr(s2, s);
        fq_mul(s3, s2, s);
        fq_mul(TX[k], TX[k], s2);
        fq_addw(s3, s3, s3);                   // wide
        fq_mul(TY[k], TY[k], s3);
    }
    fq_mul(zt, Q.z, s);             // the table's common Z
}

// x <- k * x for the wave-uniform scalar whose program starts at ops[0].  x: homogeneous
// projective, coordinates < 8 p; out: < 2 p.
template <int W>
FK20_HD void tw_mul(g1q &x, const uint32_t *ops) {
    constexpr int NT = 1 << (W - 2);
    // The table lives in the lane's private memory, not in registers: each addition reads
    // one entry chosen by a wave-uniform index, so the loads are coalesced per dword and the
    // ladder's register footprint leaves room for several waves per SIMD.
    fq TX[NT], TY[NT], zt;
    const bool inf = g1q_is_inf(x);
    tw_table<W>(TX, TY, zt, x);
    fq beta, beta2;
    fq_set(beta, FQ_GLV);
    fq_set(beta2, FQ_GLV2);
    g1h acc;
    bool started = false;
#pragma unroll 1
    for (unsigned k = 0;; k++) {
        const uint32_t op = FK20_UNIFORM(ops[k]);
        const unsigned nd = op & TWOP_DBL_MASK;
#pragma unroll 1
        for (unsigned d = 0; d < nd; d++) g1h_dbl(acc, acc);
        if (op & TWOP_END) break;
        const unsigned e = (op >> TWOP_ENTRY_SHIFT) & (NT - 1);
        fq qx = TX[e], qy = TY[e];
        if (op & TWOP_PHI2) fq_mul(qx, qx, beta2);
        else if (op & TWOP_PHI) fq_mul(qx, qx, beta);
        if (op & TWOP_NEG) fq_neg(qy, qy);
        if (started) {
            g1h_madd(acc, acc, qx, qy);
        } else {
            acc.x = qx;
            acc.h = qy;
            fq_one(acc.z);
            started = true;
        }
    }
    // Jacobian with Z = acc.z * zt -> homogeneous (2 X Z : 2 Y : 2 Z^3)
    fq z, z2;
    fq_mul(z, acc.z, zt);
    fq_sqr(z2, z);
    fq_addw(z, z, z);               // wide
    fq_mul(x.z, z2, z);
    fq_mul(x.x, acc.x, z);
    x.y = acc.h;
    if (inf) g1q_inf(x);
}

// x <- [w^384] x = [w^-128] x (w128 = false) or [w^128] x (w128 = true) for x in G1.  With
// z = -0xd201000000010000 the curve parameter and lambda = z^2 - 1 the eigenvalue of phi,
// w^128 = -z^3 = |z| (lambda + 1) mod r, and 1 + lambda + lambda^2 = 0 on G1 gives
// [w^128] x = -[|z|] phi^2(x) = -phi^2([|z|] x), [w^-128] x = phi^2([|z|] x).  [|z|] x is 63
// Jacobian doublings and 5 mixed additions of x (the set bits 62, 60, 57, 48, 16 of |z| below
// the top one), x affine on the isomorphic curve of its own Z as in tw_mul; phi^2 multiplies
// the result's X by beta^2.  This replaces a program of two 64-bit halves, its 8-entry table
// and about 11 additions.  No exceptional case for x in G1 \ {O}: before each addition the
// accumulator is [m] x with m even, 2 <= m < 2^64, so m -+ 1 is not a multiple of r.
// x: homogeneous projective, coordinates < 8 p; out: < 2 p.
FK20_HD void tw_mul_z3(g1q &x, bool w128) {
    constexpr uint64_t ZABS = 0xd201000000010000ull;
    const bool inf = g1q_is_inf(x);
    fq px, ph, t;
    fq_sqr(t, x.z);
    fq_mul(px, x.x, x.z);           // Jacobian X = X Z
    fq_mul(ph, x.y, t);             // Jacobian Y = Y Z^2
    fq_add(ph, ph, ph);
    g1h acc;
    acc.x = px;
    acc.h = ph;
    fq_one(acc.z);
#pragma unroll 1
    for (int b = 62; b >= 0; b--) {
        g1h_dbl(acc, acc);
        if ((ZABS >> b) & 1) g1h_madd(acc, acc, px, ph);
    }
    // Jacobian with Z = acc.z * x.z -> homogeneous (2 X Z beta^2 : +-2 Y : 2 Z^3)
    fq z, z2, beta2;
    fq_mul(z, acc.z, x.z);
    fq_sqr(z2, z);
    fq_addw(z, z, z);               // wide
    fq_mul(x.z, z2, z);
    fq_set(beta2, FQ_GLV2);
    fq_mul(z, z, beta2);
    fq_mul(x.x, acc.x, z);
    if (w128) fq_neg(x.y, acc.h);
    else x.y = acc.h;
    if (inf) g1q_inf(x);
}

// An (x, 2 y) held in registers (the host build; the kernel keeps its copies in LDS instead, to
// leave the registers to the formulas).
struct RegSlot {
    fq x, h;
    FK20_HD void put(const fq &a, const fq &b) {
        x = a;
        h = b;
    }
    FK20_HD void get(fq &a, fq &b) const {
        a = x;
        b = h;
    }
};

// Whether p lies in the order-r subgroup G1 (infinity included): phi^2(p) = (beta^2 x, y)
// acts on G1 as lambda^2 = -z^2, and a point of E(Fp) satisfies phi^2(p) + [z^2] p = 0 only
// if it lies in G1 (Scott, "A note on group membership tests for G1, G2 and GT on BLS
// pairing-friendly curves", 2021).  [z^2] p = [|z|]([|z|] p) by double-and-add over
// |z| = 0xd201000000010000 (63 doublings and 5 additions per round) in Jacobian coordinates,
// each round's base affine on the isomorphic curve of its own Z.  The formulas are incomplete,
// which decides nothing wrongly: an addition of equal or opposite points gives Z = 0, and Z
// stays 0 from there; it cannot happen for p in G1 \ {O}, whose multiples m -+ 1 (m < 2^64) are
// not infinity, so Z = 0 in the end means that p is outside.  126 doublings of 2 600 instructions
// against 3 350 of the complete ones: 262 144 points in 3.0 ms (4.3 with complete formulas over
// fp.hip.h), 8 192 in 0.73 (1.02).
// `orig` and `base` hold p's and each round's base while the doublings run.
template <class Slot>
FK20_HD bool g1_in_subgroup(const g1q &p, Slot &orig, Slot &base) {
    constexpr uint64_t ZABS = 0xd201000000010000ull;
    const bool inf = g1q_is_inf(p);
    fq one, t, zz;
    fq_one(one);
    g1h acc;
    fq_sqr(t, p.z);
    fq_mul(acc.x, p.x, p.z);        // Jacobian (X Z, 2 Y Z^2), < 1 and < 1.4
    fq_mul(t, p.y, t);
    fq_add(acc.h, t, t);
    orig.put(acc.x, acc.h);
    zz = one;
#pragma unroll 1
    for (int round = 0; round < 2; round++) {
        fq_mul(acc.x, acc.x, one);  // < 12 -> < 0.6: the stored range
        base.put(acc.x, acc.h);
        acc.z = one;
#pragma unroll 1
        for (int b = 62; b >= 0; b--) {
            g1h_dbl(acc, acc);
            if ((ZABS >> b) & 1) {
                fq bx, bh;
                base.get(bx, bh);
                g1h_madd(acc, acc, bx, bh);
            }
        }
        fq_mul(zz, zz, acc.z);
    }
    // [z^2] p = (acc.x / zz^2, acc.h / 2 zz^3) on p's isomorphic curve against -phi^2(p)
    fq px, ph, beta2;
    orig.get(px, ph);
    fq_set(beta2, FQ_GLV2);
    fq_mul(px, px, beta2);
    fq_sqr(t, zz);
    fq_mul(px, px, t);
    fq_sub(px, px, acc.x);
    fq_mul(t, t, zz);
    fq_mul(ph, ph, t);
    fq_add(ph, ph, acc.h);
    return inf || (fq_is_zero(px) && fq_is_zero(ph) && !fq_is_zero(zz));
}

// ---------------------------------------------------------------- points over fp.hip.h
//
// The same operations on points in the unsigned Fp form, by conversion: the element-wise entry
// points and the CPU tests use that form.

FK20_HD void fq_from_fe(fq &z, const fe &a) {
    fe t, c;
    fe_set(c, FQ_FROM_FP);
    fe_mul(t, a, c);
    uint32_t w[12];
    fe_pack(w, t);
    fq_unpack_raw(z, w);
}

FK20_HD void fe_from_fq(fe &z, const fq &a) {  // |a| < 4 p
    uint32_t w[12];
    fq_pack(w, a);
    fe t, c;
    fe_unpack(t, w);
    fe_set(c, FP_FROM_FQ);
    fe_mul(z, t, c);
}

FK20_HD void g1q_from_g1p(g1q &r, const g1p &p) {
    fq_from_fe(r.x, p.x);
    fq_from_fe(r.y, p.y);
    fq_from_fe(r.z, p.z);
}

FK20_HD void g1p_from_g1q(g1p &r, const g1q &p) {
    fe_from_fq(r.x, p.x);
    fe_from_fq(r.y, p.y);
    fe_from_fq(r.z, p.z);
}

template <int W>
FK20_HD void tw_mul(g1p &x, const uint32_t *ops) {
    g1q q;
    g1q_from_g1p(q, x);
    tw_mul<W>(q, ops);
    g1p_from_g1q(x, q);
}

FK20_HD void tw_mul_z3(g1p &x, bool w128) {
    g1q q;
    g1q_from_g1p(q, x);
    tw_mul_z3(q, w128);
    g1p_from_g1q(x, q);
}

FK20_HD bool g1_in_subgroup(const g1p &p) {
    RegSlot orig, base;
    g1q q;
    g1q_from_g1p(q, p);
    return g1_in_subgroup(q, orig, base);
}

// Jacobian (X, Y, Z) with the plain Y; results as the representative (4 X, 8 Y, 2 Z).
struct g1j {
    fe x, y, z;
};

FK20_HD void g1h_from_g1j(g1h &r, const g1j &p) {
    fq_from_fe(r.x, p.x);
    fq_from_fe(r.h, p.y);
    fq_add(r.h, r.h, r.h);
    fq_from_fe(r.z, p.z);
}

FK20_HD void g1j_from_g1h(g1j &r, const g1h &p) {
    fq one;
    fq_one(one);
    fq t;
    fq_mul(t, p.x, one);
    fe_from_fq(r.x, t);
    fe_mul_small<4>(r.x, r.x);
    fe_from_fq(r.y, p.h);
    fe_mul_small<4>(r.y, r.y);
    fe_from_fq(r.z, p.z);
    fe_mul_small<2>(r.z, r.z);
}

FK20_HD void g1j_dbl(g1j &r, const g1j &p) {
    g1h t;
    g1h_from_g1j(t, p);
    g1h_dbl(t, t);
    g1j_from_g1h(r, t);
}

FK20_HD void g1j_madd(g1j &r, const g1j &p, const fe &x2, const fe &y2) {
    g1h t;
    fq x, h;
    g1h_from_g1j(t, p);
    fq_from_fe(x, x2);
    fq_from_fe(h, y2);
    fq_add(h, h, h);
    g1h_madd(t, t, x, h);
    g1j_from_g1h(r, t);
}

}  // namespace fk20
