// G1 arithmetic of BLS12-381 (y^2 = x^3 + 4) over the signed Fp form of fq.hip.h, the points of
// every kernel: the complete formulas of Renes, Costello and Batina (eprint 2015/1060, a = 0,
// b3 = 12: algorithms 7, 8, 9; the formulas of g1p_add.cu:78, g1p_dbl.cu:28) in homogeneous
// coordinates, and incomplete Jacobian formulas for the fixed-scalar ladders (ladder.hip.h).
//
// Bounds are absolute values in multiples of p.  A product of |a b| <= M p^2 is below
// 0.54 + M / 630, so inputs below 8 p and every intermediate below keep results below 1.
#pragma once
#include "fq.hip.h"
#include "fr.hip.h"

namespace fk20 {

// homogeneous (X : Y : Z); infinity is (0 : y != 0 : 0)
struct g1q {
    fq x, y, z;
};

FK20_HD void g1q_inf(g1q &p) {
    fq_zero(p.x);
    fq_one(p.y);
    fq_zero(p.z);
}

FK20_HD bool g1q_is_inf(const g1q &p) { return fq_is_zero(p.z); }

// RCB algorithm 7: r = p + q, 6 products and 3 pairs.  In < 8, out < 1.
FK20_HD void g1q_add(g1q &r, const g1q &p, const g1q &q) {
    fq t0, t1, t2, t3, t4, X3, Y3, Z3;
    fq_mul(t0, p.x, q.x);           // 64 -> < 0.7
    fq_mul(t1, p.y, q.y);
    fq_mul(t2, p.z, q.z);
    fq_addw(t3, p.x, p.y);          // wide, < 16
    fq_add(t4, q.x, q.y);
    fq_mul(t3, t3, t4);             // 256 -> < 1
    fq_sub2(t3, t3, t0, t1);        // X1 Y2 + X2 Y1 < 2.4
    fq_addw(t4, p.y, p.z);
    fq_add(X3, q.y, q.z);
    fq_mul(t4, t4, X3);
    fq_sub2(t4, t4, t1, t2);        // Y1 Z2 + Y2 Z1 < 2.4
    fq_addw(X3, p.x, p.z);
    fq_add(Y3, q.x, q.z);
    fq_mul(X3, X3, Y3);
    fq_sub2(Y3, X3, t0, t2);        // X1 Z2 + X2 Z1 < 2.4
    fq_lin<3>(t0, t0);              // < 2.1
    fq_lin<1, 12>(Z3, t1, t2);      // < 9.1
    fq_lin<1, -12>(t1, t1, t2);     // < 9.1
    fq_lin<12>(Y3, Y3);             // < 29
    fq_neg(X3, t4);
    fq_mul2(X3, t3, t1, X3, Y3);    // 92 -> < 0.7
    fq_mul2(Y3, Y3, t0, t1, Z3);    // 144 -> < 0.8
    fq_mul2(Z3, Z3, t4, t0, t3);    // 27 -> < 0.6
    r.x = X3;
    r.y = Y3;
    r.z = Z3;
}

// RCB algorithm 8: r = p + (x2, y2), the affine operand not infinity: 5 products and 3 pairs.
// In < 8 (x2, y2 < 2), out < 1.
FK20_HD void g1q_add_aff(g1q &r, const g1q &p, const fq &X2, const fq &Y2) {
    fq t0, t1, t3, t4, X3, Y3, Z3;
    fq_mul(t0, p.x, X2);            // < 0.6
    fq_mul(t1, p.y, Y2);
    fq_addw(t3, X2, Y2);            // wide, < 4
    fq_add(t4, p.x, p.y);           // < 16
    fq_mul(t3, t3, t4);             // < 0.7
    fq_sub2(t3, t3, t0, t1);        // X1 Y2 + X2 Y1 < 1.9
    fq_mul(t4, Y2, p.z);
    fq_add(t4, t4, p.y);            // Y1 + Y2 Z1 < 8.6
    fq_mul(Y3, X2, p.z);
    fq_lin<12, 12>(Y3, Y3, p.x);    // 12 (X1 + X2 Z1) < 104
    fq_lin<3>(t0, t0);              // < 1.8
    fq_lin<1, 12>(Z3, t1, p.z);     // < 97
    fq_lin<1, -12>(t1, t1, p.z);    // < 97
    fq_neg(X3, t4);
    fq_mul2(X3, t3, t1, X3, Y3);    // 184 + 895 -> < 2.3
    fq_mul2(Y3, Y3, t0, t1, Z3);    // 9600 -> < 16 for a first p < 8; < 0.8 for p < 1
    fq_mul2(Z3, Z3, t4, t0, t3);    // 840 -> < 1.9
    r.x = X3;
    r.y = Y3;
    r.z = Z3;
}

// RCB algorithm 9: r = 2p, 2 squares, 4 products and a pair.  In < 8, out < 2.
FK20_HD void g1q_dbl(g1q &r, const g1q &p) {
    fq t0, t1, t2, X3, Y3, Z3;
    fq_sqr(t0, p.y);                // < 0.7
    fq_sqr(X3, p.z);                // < 0.7
    fq_mul(t1, p.y, p.z);
    fq_lin<8>(Z3, t0);              // 8 Y^2 < 5.6
    fq_lin<12>(t2, X3);             // 12 Z^2 < 8.4
    fq_lin<1, -3>(X3, t0, t2);      // Y^2 - 36 Z^2 < 26
    fq_add(Y3, t0, t2);             // Y^2 + 12 Z^2 < 9.1
    fq_mul2(Y3, t2, Z3, X3, Y3);    // 284 -> < 1
    fq_mul(Z3, t1, Z3);
    fq_mul(t1, p.x, p.y);
    fq_mul(X3, X3, t1);
    fq_add(X3, X3, X3);
    r.x = X3;
    r.y = Y3;
    r.z = Z3;
}

FK20_HD void g1q_neg(g1q &r, const g1q &p) {
    r.x = p.x;
    fq_neg(r.y, p.y);
    r.z = p.z;
}

// ---------------------------------------------------------------- Jacobian (ladders)
//
// Jacobian coordinates (x = X / Z^2, y = Y / Z^3) held as X, H = 2 Y, Z.  With the doubled Y
// a doubling needs no multiple of Z and only two linear combinations: with A = X^2, B = H^2,
// D = X B (= 4 X Y^2):  X' = 9 A^2 - 2 D,  H' = 6 A (D - X') - B^2,  Z' = H Z, the formulas of
// dbl-2009-l (Bernstein-Lange EFD, a = 0).  They are incomplete: callers guarantee that no
// operand is infinity and no addition sees equal or opposite points (the twiddle programs are
// checked for that on the host, ctx.cpp), and none uses the curve constant b, so they also run on
// the isomorphic curve on which a co-Z table's points are affine.
struct g1h {
    fq x, h, z;
};

// 3 squares, 2 products and a product minus square: 1 885 multiply-adds in products (2 275 for
// the same formulas over fp.hip.h).  In: x < 30, h < 8, z < 8.  Out: x < 7, h < 1, z < 1.
FK20_HD void g1h_dbl(g1h &r, const g1h &p) {
    fq A, B, D, F, U;
    fq_sqr(A, p.x);                 // < 2
    fq_sqr(B, p.h);                 // < 0.7
    fq_mul(r.z, p.h, p.z);          // < 0.7
    fq_mul(D, p.x, B);              // < 0.6
    fq_sqr(F, A);                   // < 0.6
    fq_lin<9, -2>(r.x, F, D);       // < 7
    fq_subw(U, D, r.x);
    fq_lin<6>(U, U);                // < 46
    fq_mulsubsqr(r.h, A, U, B);     // 92 -> < 0.7
}

// r = p + (x2, h2 / 2): the affine operand's doubled y, on the same (possibly scaled) curve,
// neither operand infinity, not +-p.  3 squares, 6 products and a pair (3 315 multiply-adds
// in products); Z' = 2 Z (x2 Z^2 - X).
// In: x < 30, h < 8, z < 8; x2, h2 < 8.  Out: x < 12, h < 1, z < 1.2.
FK20_HD void g1h_madd(g1h &r, const g1h &p, const fq &x2, const fq &h2) {
    fq ZZ, H, R, HH, HHH, V, t;
    fq_sqr(ZZ, p.z);                // < 0.7
    fq_mul(R, h2, p.z);             // < 0.7
    fq_mul(H, x2, ZZ);              // < 0.6
    fq_mul(R, R, ZZ);               // 2 y2 Z^3 < 0.6
    fq_sub(H, H, p.x);              // < 31
    fq_sub(R, R, p.h);              // 2 (S2 - Y1) < 9
    fq_sqr(HH, H);                  // 961 -> < 2.1
    fq_mul(t, p.z, H);              // < 1
    fq_mul(V, p.x, HH);             // < 0.7
    fq_mul(HHH, H, HH);             // < 0.7
    fq_add(r.z, t, t);              // 2 Z H
    fq_sqr(t, R);                   // < 0.7
    fq_lin<1, -4, -8>(r.x, t, HHH, V);  // X' = R^2 - 4 HHH - 8 V < 10
    fq_lin<8, -2>(V, V, r.x);       // 2 (4 V - X') < 26
    fq_lin<-8>(HHH, HHH);           // < 6
    fq_mul2(r.h, R, V, p.h, HHH);   // 2 Y' = R (8 V - 2 X') - 8 H1 HHH: 234 + 48 -> < 1
}

// Doubling with update (the co-Z table start), plain y: q = 2p and (x1, y1) = p, both with
// Z = 2 Y Z.  In: x, y, z < 8.  Out: q.x < 8, q.y < 6, qz < 1.4; x1 < 3, y1 < 5.
struct g1j_q {
    fq x, y, z;
};
FK20_HD void g1q_dblu(g1j_q &q, fq &x1, fq &y1, const g1j_q &p) {
    fq A, B, C, D, E, F, t;
    fq_sqr(A, p.x);                 // < 0.7
    fq_sqr(B, p.y);
    fq_sqr(C, B);
    fq_mul(D, p.x, B);
    fq_lin<4>(D, D);                // 4 X Y^2 < 2.4
    fq_mul(t, p.y, p.z);
    fq_add(q.z, t, t);              // 2 Y Z < 1.4
    fq_lin<3>(E, A);                // < 2.1
    fq_sqr(F, E);                   // < 0.6
    fq_lin<1, -2>(q.x, F, D);       // < 5.4
    fq_subw(t, D, q.x);             // wide, < 8
    fq_mul(t, t, E);                // < 0.6
    fq_lin<8>(C, C);                // 8 Y^4 < 4.6
    fq_sub(q.y, t, C);              // < 5.2
    x1 = D;
    y1 = C;
}

// Co-Z addition with update (Meloni; Goundar-Joye-Miyaji "ZADDU"): for p1 = (x1, y1) and
// p2 = (x2, y2) sharing Z, (x3, y3) = p1 + p2 and (x1, y1) <- p1, both with Z' = Z mu,
// mu = x1 - x2 (returned).  p1 != +-p2.  2 squares, 4 products.
// In: coordinates < 6.  Out: x1, y1 < 0.8; x3 < 3, y3 < 2; mu < 12.
FK20_HD void g1q_zaddu(fq &x3, fq &y3, fq &mu, fq &x1, fq &y1, const fq &x2, const fq &y2) {
    fq C, W1, W2, D, dy, t;
    fq_sub(mu, x1, x2);             // < 12
    fq_sqr(C, mu);                  // < 0.8
    fq_mul(W1, x1, C);              // < 0.6
    fq_mul(W2, x2, C);
    fq_sub(dy, y1, y2);             // < 12
    fq_sqr(D, dy);                  // < 0.8
    fq_subw(t, W1, W2);
    fq_mul(y1, y1, t);              // Y1 (W1 - W2) < 0.6
    fq_sub2(x3, D, W1, W2);         // < 2
    fq_subw(t, W1, x3);             // wide, < 3
    fq_mul(t, t, dy);               // < 0.7
    fq_sub(y3, t, y1);              // < 1.3
    x1 = W1;
}

// (x, y) = (X / Z, Y / Z); false when Z = 0.  z_one: Z is known to be 1 (the transforms' own
// outputs are); a wave whose lanes all say so has nothing to invert.
FK20_HD bool g1q_to_affine(fq &x, fq &y, const g1q &p, bool z_one = false) {
    if (!FQ_ANY(!z_one)) {
        x = p.x;
        y = p.y;
        return true;
    }
    if (g1q_is_inf(p)) return false;
    fq zi;
    fq_inv(zi, p.z);
    fq_mul(x, p.x, zi);
    fq_mul(y, p.y, zi);
    return true;
}

// 48-byte compressed serialisation, as 12 words in memory order: big-endian canonical x, top
// byte flags 0x80 (compressed), 0x40 (infinity: 0xc0 then zeros), 0x20 (y is the larger of
// y and p - y).
FK20_HD void g1q_compress(uint32_t *w, const g1q &p, bool z_one = false) {
    fq x, y;
    if (!g1q_to_affine(x, y, p, z_one)) {
#pragma unroll
        for (int i = 0; i < 12; i++) w[i] = 0;
        w[0] = 0xc0u;
        return;
    }
    uint32_t xw[12], yw[12];
    fq_to_std(xw, x);
    fq_to_std(yw, y);
    // y > (p - 1) / 2, compared from the top word
    int cmp = 0;
#pragma unroll
    for (int i = 11; i >= 0; i--)
        if (cmp == 0) cmp = yw[i] > FP_HALF_PACKED[i] ? 1 : yw[i] < FP_HALF_PACKED[i] ? -1 : 0;
#pragma unroll
    for (int k = 0; k < 12; k++) w[k] = __builtin_bswap32(xw[11 - k]);
    w[0] |= 0x80u | (cmp > 0 ? 0x20u : 0u);
}

// ---------------------------------------------------------------- memory forms

// Standard-form g1p_t words (any representative below 2^384) -> Montgomery
FK20_HD void g1q_load_std(g1q &p, const uint32_t *w) {
    fq_from_std(p.x, w);
    fq_from_std(p.y, w + 12);
    fq_from_std(p.z, w + 24);
}

// Canonical standard form (each coordinate in [0, p))
FK20_HD void g1q_store_std(uint32_t *w, const g1q &p) {
    fq_to_std(w, p.x);
    fq_to_std(w + 12, p.y);
    fq_to_std(w + 24, p.z);
}

// The kernels' buffers: 36 words, coordinates < 4
FK20_HD void g1q_load_packed(g1q &p, const uint32_t *w) {
    fq_unpack(p.x, w);
    fq_unpack(p.y, w + 12);
    fq_unpack(p.z, w + 24);
}

FK20_HD void g1q_store_packed(uint32_t *w, const g1q &p) {
    fq_pack(w, p.x);
    fq_pack(w + 12, p.y);
    fq_pack(w + 24, p.z);
}

}  // namespace fk20
