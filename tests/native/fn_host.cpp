// Host build of the transforms' Fr form (fr.hip.h fn_*) for CPU tests.
#define FK20_HD inline
#define __host__
#define __device__
#include "../../fk20-cuda_amd/csrc/fr.hip.h"

#include <cstring>

using namespace fk20;

static fn raw(const int32_t *d) {
    fn z;
    memcpy(z.l, d, sizeof z.l);
    return z;
}

extern "C" {
void fn_host_mul(int32_t *z, const int32_t *a, const int32_t *w) {
    fn r;
    fn_mul(r, raw(a), raw(w));
    memcpy(z, r.l, sizeof r.l);
}
void fn_host_norm(int32_t *z, const int32_t *a) {
    fn r = raw(a);
    fn_norm(r);
    memcpy(z, r.l, sizeof r.l);
}
void fn_host_canon(uint32_t *w, const int32_t *a) { fn_canon(w, raw(a)); }
void fn_host_unpack(int32_t *z, const uint32_t *w) {
    fn r;
    fn_unpack(r, w);
    memcpy(z, r.l, sizeof r.l);
}
void fn_host_from_words(int32_t *z, const uint32_t *w) { fn_from_words(z, w); }
}
