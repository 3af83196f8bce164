// Host build of the two-lane ladder (ladder_pair.hip.h), both lanes emulated, for CPU tests.
#define FK20_HD inline
#define __host__
#define __device__
#define FK20_UNIFORM(x) (x)
#include "../../fk20-cuda_amd/csrc/ladder_pair.hip.h"

using namespace fk20;

extern "C" {
// p (g1p_t words) <- k p by the program `ops` of wNAF width 5, the lanes' results in r0 and r1
void pair_host_tw_mul(uint32_t *r0, uint32_t *r1, const uint32_t *p, const uint32_t *ops) {
    g1q x;
    g1q_load_std(x, p);
    fq TX[8], TY[8], zt;
    tw_table<5>(TX, TY, zt, x);
    pair_h acc;
    pair_program(acc, ops, [&](pair_fq &q, unsigned e) {
        q.v[0] = TX[e];
        q.v[1] = TY[e];
    });
    pair_fq X, Y, Z, s;
    pair_both(s, zt);
    pair_finish(X, Y, Z, acc, s, s, false);
    g1q_store_std(r0, g1q{X.v[0], Y.v[0], Z.v[0]});
    g1q_store_std(r1, g1q{X.v[1], Y.v[1], Z.v[1]});
}

// whether p lies in G1, by the pair's comparison
int pair_host_in_subgroup(const uint32_t *p) {
    g1q x;
    g1q_load_std(x, p);
    fq t, px, ph;
    fq_sqr(t, x.z);
    fq_mul(px, x.x, x.z);
    fq_mul(ph, x.y, t);
    fq_add(ph, ph, ph);
    pair_fq orig, v, zz;
    orig.v[0] = px;
    orig.v[1] = ph;
    pair_subgroup(v, zz, orig);
    return g1q_is_inf(x) || (fq_is_zero(v.v[0]) && fq_is_zero(v.v[1]) && !fq_is_zero(zz.v[0]));
}

// p <- [2^n] p
void pair_host_dbl_n(uint32_t *r0, uint32_t *r1, const uint32_t *p, int n) {
    g1q x;
    g1q_load_std(x, p);
    pair_fq X, Y, Z;
    pair_both(X, x.x);
    pair_both(Y, x.y);
    pair_both(Z, x.z);
    pair_dbl_n(X, Y, Z, n);
    g1q_store_std(r0, g1q{X.v[0], Y.v[0], Z.v[0]});
    g1q_store_std(r1, g1q{X.v[1], Y.v[1], Z.v[1]});
}

// p <- [w^128] p as the kernels' short form runs it
void pair_host_z3(uint32_t *r0, uint32_t *r1, const uint32_t *p) {
    g1q x;
    g1q_load_std(x, p);
    fq t, px, ph, b2;
    fq_sqr(t, x.z);
    fq_mul(px, x.x, x.z);
    fq_mul(ph, x.y, t);
    fq_add(ph, ph, ph);
    pair_h acc;
    pair_fq q, z, f, X, Y, Z;
    q.v[0] = px;
    q.v[1] = ph;
    pair_z(acc, q);
    fq_set(b2, FQ_GLV2);
    pair_both(z, x.z);
    pair_both(f, b2);
    pair_finish(X, Y, Z, acc, z, f, true);
    fq_neg(Y, Y);
    g1q_store_std(r0, g1q{X.v[0], Y.v[0], Z.v[0]});
    g1q_store_std(r1, g1q{X.v[1], Y.v[1], Z.v[1]});
}
}
