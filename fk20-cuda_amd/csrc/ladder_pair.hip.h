// The fixed-scalar ladder (ladder.hip.h) run by two neighbouring lanes per point, for launches
// whose waves leave SIMDs idle: there a ladder's latency counts, 124 doublings after one
// another, and each formula's independent products run side by side.  Lane 0 of a pair holds X and
// lane 1 H = 2 Y, both hold Z; a doubling is a square, a product and a product minus square
// (1 630 instructions with the exchanges against 2 616), a mixed addition five products and a
// square (3 050 against 4 020).  The values go between the lanes by DPP.  A launch of single ladders
// takes 1.10 ms, of pairs 0.87 (one row of N = 4096: 3.09 -> 2.41 ms).  The two lanes' work
// is a quarter more than one lane's, so it only pays on idle SIMDs (PAIR_WAVES, fast.hip.h).
//
// pair_fq is a value of each lane: fq on the device, both lanes' values in the CPU tests.
#pragma once
#include "ladder.hip.h"

namespace fk20 {

#ifdef __HIPCC__
using pair_fq = fq;

__device__ __forceinline__ bool pair_lane1() { return threadIdx.x & 1; }
// the other lane's value
__device__ __forceinline__ void pair_swap(pair_fq &z, const pair_fq &a) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = __builtin_amdgcn_update_dpp(0, a.l[i], 0xB1, 0xf, 0xf, true);
}
// a in lane 0, b in lane 1
__device__ __forceinline__ void pair_sel(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    const bool one = pair_lane1();
#pragma unroll
    for (int i = 0; i < FQ_N; i++) z.l[i] = one ? b.l[i] : a.l[i];
}
__device__ __forceinline__ void pair_both(pair_fq &z, const fq &a) { z = a; }
#else
struct pair_fq {
    fq v[2];
};
inline void pair_swap(pair_fq &z, const pair_fq &a) {
    const pair_fq t = a;
    z.v[0] = t.v[1];
    z.v[1] = t.v[0];
}
inline void pair_sel(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    const fq x = a.v[0], y = b.v[1];
    z.v[0] = x;
    z.v[1] = y;
}
inline void pair_both(pair_fq &z, const fq &a) { z.v[0] = z.v[1] = a; }
inline void fq_mul(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    for (int i = 0; i < 2; i++) fq_mul(z.v[i], a.v[i], b.v[i]);
}
inline void fq_sqr(pair_fq &z, const pair_fq &a) {
    for (int i = 0; i < 2; i++) fq_sqr(z.v[i], a.v[i]);
}
inline void fq_mulsubsqr(pair_fq &z, const pair_fq &a, const pair_fq &b, const pair_fq &c) {
    for (int i = 0; i < 2; i++) fq_mulsubsqr(z.v[i], a.v[i], b.v[i], c.v[i]);
}
inline void fq_sub(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    for (int i = 0; i < 2; i++) fq_sub(z.v[i], a.v[i], b.v[i]);
}
inline void fq_add(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    for (int i = 0; i < 2; i++) fq_add(z.v[i], a.v[i], b.v[i]);
}
inline void fq_subw(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    for (int i = 0; i < 2; i++) fq_subw(z.v[i], a.v[i], b.v[i]);
}
inline void fq_neg(pair_fq &z, const pair_fq &a) {
    for (int i = 0; i < 2; i++) fq_neg(z.v[i], a.v[i]);
}
template <int A>
inline void fq_lin(pair_fq &z, const pair_fq &a) {
    for (int i = 0; i < 2; i++) fq_lin<A>(z.v[i], a.v[i]);
}
template <int A, int B>
inline void fq_lin(pair_fq &z, const pair_fq &a, const pair_fq &b) {
    for (int i = 0; i < 2; i++) fq_lin<A, B>(z.v[i], a.v[i], b.v[i]);
}
template <int A, int B, int C>
inline void fq_lin(pair_fq &z, const pair_fq &a, const pair_fq &b, const pair_fq &c) {
    for (int i = 0; i < 2; i++) fq_lin<A, B, C>(z.v[i], a.v[i], b.v[i], c.v[i]);
}
#endif

#ifdef __HIPCC__
#define PAIR_FN __device__ __forceinline__
#else
#define PAIR_FN inline
#endif

// p: X | H (= 2 Y); z: Z in both lanes.  Bounds as g1h (g1q.hip.h): X < 30, H, Z < 8.
struct pair_h {
    pair_fq p, z;
};

// What a lane computes that is not its own is bounded like what the other one does.
PAIR_FN void pair_dbl(pair_h &P) {
    pair_fq s, f, t, a, b, c, x, u;
    fq_sqr(s, P.p);                 // A = X^2 | B = H^2
    pair_swap(t, P.p);
    pair_sel(a, s, t);              // A | X
    fq_mul(f, a, s);                // F = A^2 | D = X B
    pair_swap(t, f);                // D | .
    fq_lin<9, -2>(x, f, t);         // X' = 9 F - 2 D | .
    fq_subw(u, t, x);
    fq_lin<6>(u, u);                // U = 6 (D - X') | .
    pair_swap(c, s);                // B | .
    pair_both(t, fq{});
    pair_sel(c, c, t);              // B | 0
    pair_sel(a, s, P.p);            // A | H
    pair_sel(b, u, P.z);            // U | Z
    fq_mulsubsqr(s, a, b, c);       // H' = A U - B^2 | Z' = H Z
    pair_swap(t, s);                // Z' | H'
    pair_sel(P.p, x, t);
    pair_sel(P.z, t, s);
}

// P + q, q = x2 | 2 y2, as g1h_madd
PAIR_FN void pair_madd(pair_h &P, const pair_fq &q) {
    pair_fq w, zz, d, s, e, a, b, v, g, x, t;
    pair_sel(b, P.z, q);
    fq_mul(w, P.z, b);              // ZZ | 2 y2 Z
    pair_swap(t, w);
    pair_sel(zz, w, t);             // ZZ | ZZ
    pair_sel(a, q, w);
    fq_mul(d, a, zz);               // x2 ZZ | 2 y2 Z^3
    fq_sub(d, d, P.p);              // H = x2 ZZ - X | R = 2 y2 Z^3 - H1
    fq_sqr(s, d);                   // HH | R^2
    pair_swap(e, d);                // R | H
    pair_sel(a, P.p, P.z);
    pair_sel(b, s, e);
    fq_mul(v, a, b);                // V = X HH | Z H
    fq_mul(g, d, s);                // HHH | .
    pair_swap(t, s);                // R^2 | .
    fq_lin<1, -4, -8>(x, t, g, v);  // X' | .
    fq_add(t, v, v);                // . | Z' = 2 Z H
    fq_lin<8, -2>(v, v, x);         // 8 V - 2 X' | .
    fq_lin<-8>(g, g);               // -8 HHH | .
    pair_swap(g, g);                // . | -8 HHH
    pair_sel(a, e, P.p);
    pair_sel(b, v, g);
    fq_mul(a, a, b);                // R (8 V - 2 X') | -8 H1 HHH
    pair_swap(b, a);
    fq_add(b, a, b);                // H' in both
    pair_sel(P.p, x, b);
    pair_swap(v, t);
    pair_sel(P.z, v, t);
}

// The point of a pair's accumulator with Z = z scale, in both lanes: (2 X Z f : 2 Y : 2 Z^3); f = 1,
// or the endomorphism's factor.
PAIR_FN void pair_finish(pair_fq &X, pair_fq &Y, pair_fq &Z, const pair_h &P, const pair_fq &scale, const pair_fq &f,
                         bool with_f) {
    pair_fq t, z, z2;
    pair_swap(t, P.p);
    pair_sel(X, P.p, t);
    pair_sel(Y, t, P.p);
    fq_mul(z, P.z, scale);
    fq_sqr(z2, z);
    fq_add(z, z, z);
    fq_mul(Z, z2, z);
    if (with_f) fq_mul(z, z, f);
    fq_mul(X, X, z);
}

// [2^n] of the homogeneous point (x : y : z) both lanes hold (coordinates < 8, z not 0): into
// Jacobian form (X Z, Y Z^2, Z), n doublings, and back.  Any point of the curve: doublings have no
// exception, as the curve's order is odd.  3 200 instructions for the two changes of form, 1 600
// a doubling against 3 270 for the complete one.
PAIR_FN void pair_dbl_n(pair_fq &x, pair_fq &y, pair_fq &z, int n) {
    pair_h P;
    pair_fq s, t, a, b;
    fq_sqr(s, z);
    pair_sel(a, x, y);
    pair_sel(b, z, s);
    fq_mul(s, a, b);                // X Z | Y Z^2
    fq_add(t, s, s);
    pair_sel(P.p, s, t);
    P.z = z;
#pragma unroll 1
    for (int i = 0; i < n; i++) pair_dbl(P);
    fq_sqr(s, P.z);
    fq_add(t, P.z, P.z);
    pair_sel(a, P.p, s);
    fq_mul(s, a, t);                // 2 X Z | 2 Z^3
    pair_swap(t, s);
    pair_sel(x, s, t);
    pair_sel(z, t, s);
    pair_swap(t, P.p);
    pair_sel(y, t, P.p);            // 2 Y
}

// The ladder's run over a table T: entry(e) gives x | 2 y of the e-th odd multiple.
template <class Entry>
PAIR_FN void pair_program(pair_h &acc, const uint32_t *ops, const Entry &entry) {
    pair_fq one, beta, beta2;
    fq c, k;
    fq_one(k);
    pair_both(one, k);
    fq_set(c, FQ_GLV);
    pair_both(beta, c);
    fq_set(c, FQ_GLV2);
    pair_both(beta2, c);
    pair_sel(beta, beta, one);
    pair_sel(beta2, beta2, one);
    bool started = false;
#pragma unroll 1
    for (unsigned i = 0;; i++) {
        const uint32_t op = FK20_UNIFORM(ops[i]);
        const unsigned nd = op & TWOP_DBL_MASK;
#pragma unroll 1
        for (unsigned d = 0; d < nd; d++) pair_dbl(acc);
        if (op & TWOP_END) break;
        pair_fq q, n;
        entry(q, (op >> TWOP_ENTRY_SHIFT) & 7);
        if (op & TWOP_PHI2) fq_mul(q, q, beta2);
        else if (op & TWOP_PHI) fq_mul(q, q, beta);
        if (op & TWOP_NEG) {
            fq_neg(n, q);
            pair_sel(q, q, n);
        }
        if (started) {
            pair_madd(acc, q);
        } else {
            acc.p = q;
            acc.z = one;
            started = true;
        }
    }
}

// [|z|] of the point x | 2 y
PAIR_FN void pair_z(pair_h &acc, const pair_fq &q) {
    constexpr uint64_t ZABS = 0xd201000000010000ull;
    fq one;
    fq_one(one);
    acc.p = q;
    pair_both(acc.z, one);
#pragma unroll 1
    for (int b = 62; b >= 0; b--) {
        pair_dbl(acc);
        if ((ZABS >> b) & 1) pair_madd(acc, q);
    }
}

// What g1_in_subgroup compares, for the point whose Jacobian (X Z | 2 Y Z^2) is `orig`: both
// lanes' residues v are 0 and zz is not if it lies in G1.
PAIR_FN void pair_subgroup(pair_fq &v, pair_fq &zz, const pair_fq &orig) {
    pair_fq one, f, t, n;
    fq k;
    fq_one(k);
    pair_both(one, k);
    pair_h acc;
    acc.p = orig;
    zz = one;
#pragma unroll 1
    for (int round = 0; round < 2; round++) {
        pair_fq base;
        fq_mul(base, acc.p, one);   // < 30 -> < 0.6
        pair_z(acc, base);
        fq_mul(zz, zz, acc.z);
    }
    // [z^2] p = (X / zz^2, H / 2 zz^3) against -phi^2(p)
    fq_set(k, FQ_GLV2);
    pair_both(f, k);
    pair_sel(f, f, one);
    fq_mul(v, orig, f);             // beta^2 x | h
    fq_sqr(f, zz);
    fq_mul(t, f, zz);
    pair_sel(f, f, t);
    fq_mul(v, v, f);                // .. zz^2 | .. zz^3
    fq_neg(n, acc.p);
    pair_sel(n, n, acc.p);
    fq_add(v, v, n);
}

#ifdef __HIPCC__
// g1_in_subgroup by a pair of lanes that both hold p, and both get the result
__device__ __forceinline__ bool g1_in_subgroup_pair(const g1q &p) {
    fq px, ph, t;
    fq_sqr(t, p.z);
    fq_mul(px, p.x, p.z);
    fq_mul(ph, p.y, t);
    fq_add(ph, ph, ph);
    pair_fq orig, v, zz;
    pair_sel(orig, px, ph);
    pair_subgroup(v, zz, orig);
    const int mine = fq_is_zero(v);
    const int other = __builtin_amdgcn_update_dpp(0, mine, 0xB1, 0xf, 0xf, true);
    return g1q_is_inf(p) || (mine && other && !fq_is_zero(zz));
}

// tw_mul and tw_mul_z3 by a pair of lanes that both hold x, and both get the result.
template <int W>
__device__ __forceinline__ void tw_mul_pair(g1q &x, const uint32_t *ops) {
    constexpr int NT = 1 << (W - 2);
    fq T[2 * NT], zt;  // x of the odd multiples, then 2 y: a lane reads its own half
    const bool inf = g1q_is_inf(x);
    tw_table<W>(T, T + NT, zt, x);
    pair_h acc;
    pair_program(acc, ops, [&](pair_fq &q, unsigned e) { q = T[(pair_lane1() ? NT : 0) + (e & (NT - 1))]; });
    pair_finish(x.x, x.y, x.z, acc, zt, zt, false);
    if (inf) g1q_inf(x);
}

__device__ __forceinline__ void tw_mul_z3_pair(g1q &x, bool w128) {
    const bool inf = g1q_is_inf(x);
    fq px, ph, t, beta2;
    fq_sqr(t, x.z);
    fq_mul(px, x.x, x.z);
    fq_mul(ph, x.y, t);
    fq_add(ph, ph, ph);
    pair_h acc;
    pair_fq q;
    pair_sel(q, px, ph);
    pair_z(acc, q);
    fq_set(beta2, FQ_GLV2);
    t = x.z;
    pair_finish(x.x, x.y, x.z, acc, t, beta2, true);
    if (w128) fq_neg(x.y, x.y);
    if (inf) g1q_inf(x);
}
#endif

}  // namespace fk20
