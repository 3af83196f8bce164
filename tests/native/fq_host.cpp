// Host build of the signed Fp form and its points (fq.hip.h, g1q.hip.h) for CPU tests: the same
// source the HIP kernels inline, compiled by g++.
#define FK20_HD inline
#define __host__
#define __device__
#define FK20_UNIFORM(x) (x)
#include "../../fk20-cuda_amd/csrc/ladder.hip.h"

#include <cstring>

using namespace fk20;

static void raw(fq &z, const int32_t *d) { memcpy(z.l, d, sizeof z.l); }

extern "C" {
// digits in, digits out (13 x int32): 0 a b, 1 a^2, 2 a b + c d, 3 a b - c^2 (all / 2^390),
// 4 norm(a), 5 a + b, 6 a - b, 7 a - b - c, 8 9 a - 2 b, 9 12 a, 10 a - 4 b - 8 c, 11 1 / a
void fq_host_raw(int op, int32_t *z, const int32_t *a, const int32_t *b, const int32_t *c, const int32_t *d) {
    fq x, y, u, v, r;
    raw(x, a);
    raw(y, b);
    raw(u, c);
    raw(v, d);
    switch (op) {
    case 0: fq_mul(r, x, y); break;
    case 1: fq_sqr(r, x); break;
    case 2: fq_mul2(r, x, y, u, v); break;
    case 3: fq_mulsubsqr(r, x, y, u); break;
    case 4: fq_norm(r, x); break;
    case 5: fq_add(r, x, y); break;
    case 6: fq_sub(r, x, y); break;
    case 7: fq_sub2(r, x, y, u); break;
    case 8: fq_lin<9, -2>(r, x, y); break;
    case 9: fq_lin<12>(r, x); break;
    case 10: fq_lin<1, -4, -8>(r, x, y, u); break;
    default: fq_inv(r, x); break;
    }
    memcpy(z, r.l, sizeof r.l);
}

void fq_host_pack(uint32_t *w, const int32_t *a) {
    fq x;
    raw(x, a);
    fq_pack(w, x);
}

void fq_host_unpack(int32_t *z, const uint32_t *w) {
    fq r;
    fq_unpack(r, w);
    memcpy(z, r.l, sizeof r.l);
}

// standard form (any value below 2^384) -> Montgomery digits, and back to canonical words
void fq_host_from_std(int32_t *z, const uint32_t *w) {
    fq r;
    fq_from_std(r, w);
    memcpy(z, r.l, sizeof r.l);
}

void fq_host_to_std(uint32_t *w, const int32_t *a) {
    fq x;
    raw(x, a);
    fq_to_std(w, x);
}

void fq_host_canon(uint32_t *w, const int32_t *a) {
    fq x;
    raw(x, a);
    fq_canon_words(w, x);
}

int fq_host_is_zero(const int32_t *a) {
    fq x;
    raw(x, a);
    return fq_is_zero(x) ? 1 : 0;
}

// points as g1p_t words: 0 p + q, 1 p + (qx, qy), 2 2p, 3 -p
void g1q_host_op(int op, uint32_t *r, const uint32_t *p, const uint32_t *q) {
    g1q a, b;
    g1q_load_std(a, p);
    g1q_load_std(b, q);
    if (op == 0) g1q_add(a, a, b);
    else if (op == 1) g1q_add_aff(a, a, b.x, b.y);
    else if (op == 2) g1q_dbl(a, a);
    else g1q_neg(a, a);
    g1q_store_std(r, a);
}

void g1q_host_compress(uint32_t *w, const uint32_t *p) {
    g1q a;
    g1q_load_std(a, p);
    g1q_compress(w, a);
}
}
