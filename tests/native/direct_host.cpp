// Host build of the direct schedule's plans (direct.hip.h) for CPU tests.
#define FK20_HD inline
#define __host__
#define __device__
#include "../../fk20-cuda_amd/csrc/direct.hip.h"

using namespace fk20;

static std::vector<uint32_t> g_words;

extern "C" {
// Builds every plan with all exponents of one cost but w^128; returns the number of words.
unsigned direct_host_build(void) {
    int cost[256];
    for (int e = 0; e < 256; e++) cost[e] = e == 0 ? 0 : e == 128 ? 1 : 2;
    direct_build(g_words, cost);
    return (unsigned)g_words.size();
}
const uint32_t *direct_host_words(void) { return g_words.data(); }
unsigned direct_host_record(unsigned logn, unsigned kind, unsigned levels, unsigned step) {
    return direct_record(logn, kind, levels, step) * DIRECT_STEP_WORDS;
}
// waves of record `rec` (word offset) over `rows` rows, and lane `pair` of wave `local`: row, slot
unsigned direct_host_waves(unsigned rec, unsigned rows, unsigned max_lr) {
    return direct_parts(*reinterpret_cast<const DirectStep *>(&g_words[rec]), rows, max_lr).waves;
}
void direct_host_wave(unsigned rec, unsigned rows, unsigned max_lr, unsigned local, uint32_t *out) {
    const DirectStep &st = *reinterpret_cast<const DirectStep *>(&g_words[rec]);
    const DirectWave v = direct_wave(st, g_words.data(), rows, max_lr, direct_parts(st, rows, max_lr).parts, local);
    for (unsigned p = 0; p < 1u << max_lr; p++) {
        out[2 * p] = std::min(v.row0 + (p & ((1u << v.lr) - 1)), v.last);
        out[2 * p + 1] = (v.w & 0xffffu) + std::min(p >> v.lr, (v.w >> 16) - 1);
    }
}
unsigned direct_host_row_lanes(unsigned rows) { return direct_row_lanes(rows); }
}
