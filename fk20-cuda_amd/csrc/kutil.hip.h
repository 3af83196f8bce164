// Device helpers shared by the kernel translation units: vector loads and stores of words,
// points and field elements in the packed Montgomery memory form, and the per-launch item
// lookup of the batched path.
#pragma once
#include "fast.hip.h"
#include "ladder_pair.hip.h"

namespace fk20 {

// ---------------------------------------------------------------- memory helpers

__device__ __forceinline__ void ld_words(uint32_t *w, const uint32_t *g, int n4) {
#pragma unroll
    for (int i = 0; i < n4; i++) {
        uint4 v = reinterpret_cast<const uint4 *>(g)[i];
        w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
    }
}

__device__ __forceinline__ void st_words(uint32_t *g, const uint32_t *w, int n4) {
#pragma unroll
    for (int i = 0; i < n4; i++)
        reinterpret_cast<uint4 *>(g)[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
}

__device__ __forceinline__ void pt_load(g1q &p, const uint32_t *g) {
    uint32_t w[36];
    ld_words(w, g, 9);
    g1q_load_packed(p, w);
}

__device__ __forceinline__ void pt_store(uint32_t *g, const g1q &p) {
    uint32_t w[36];
    g1q_store_packed(w, p);
    st_words(g, w, 9);
}

__device__ __forceinline__ void fq_load(fq &a, const uint32_t *g) {
    uint32_t w[12];
    ld_words(w, g, 3);
    fq_unpack(a, w);
}

__device__ __forceinline__ void fq_store(uint32_t *g, const fq &a) {
    uint32_t w[12];
    fq_pack(w, a);
    st_words(g, w, 3);
}

// ---------------------------------------------------------------- sums across lanes

__device__ __forceinline__ void shfl_point(g1q &r, const g1q &p, int lane) {
#pragma unroll
    for (int i = 0; i < FQ_N; i++) {
        r.x.l[i] = __shfl(p.x.l[i], lane);
        r.y.l[i] = __shfl(p.y.l[i], lane);
        r.z.l[i] = __shfl(p.z.l[i], lane);
    }
}

// the sum of the points of the lanes t, t ^ 1, .., t ^ (span - 1) in each of them (span a power of two)
__device__ __forceinline__ void lane_sum(g1q &acc, unsigned span) {
    g1q o;
#pragma unroll 1
    for (unsigned d = 1; d < span; d *= 2) {
        shfl_point(o, acc, (int)(threadIdx.x ^ d));
        g1q_add(acc, acc, o);
    }
}

// Additions one after the other that `waves` waves of `adds` additions take on 1024 SIMDs: a wave
// alone on its SIMD needs about 1.1 times an addition's share of a busy SIMD.
inline unsigned add_rounds(size_t waves, unsigned adds) {
    const unsigned rounds = (unsigned)((waves + 1023) / 1024);
    return rounds <= 1 ? adds + adds / 8 : rounds * adds;
}

// ---------------------------------------------------------------- multi-item decoding
//
// Every launch below covers a list of items (row groups, each with its own setup, N and
// buffers).  A block finds its item from the per-item block prefix sums of the launch.

__device__ __forceinline__ unsigned find_item(const Launch &L, unsigned blk, unsigned &local) {
    unsigned k = 0, start = 0;
#pragma unroll 1
    while (k + 1 < L.nitems && blk >= L.blk_end[k]) {
        start = L.blk_end[k];
        k++;
    }
    local = blk - start;
    return k;
}

// ---------------------------------------------------------------- subgroup membership

// A lane's (x, 2 y) in LDS, packed (24 words, stride 25 to spread the lanes over the banks).
struct LdsSlot {
    uint32_t *w;
    __device__ void put(const fq &x, const fq &h) {
        uint32_t t[24];
        fq_pack(t, x);
        fq_pack(t + 12, h);
#pragma unroll
        for (int k = 0; k < 24; k++) w[k] = t[k];
    }
    __device__ void get(fq &x, fq &h) const {
        uint32_t t[24];
#pragma unroll
        for (int k = 0; k < 24; k++) t[k] = w[k];
        fq_unpack(x, t);
        fq_unpack(h, t + 12);
    }
};

// flags[i / per_group] |= 1 when pts[i] (i < count, 64 lanes a block) lies outside the order-r subgroup.
// The test's two saved points sit in LDS (`slots`), which leaves room for two waves per SIMD
// without spills.
static constexpr unsigned SUBGROUP_SLOT_WORDS = 2 * 64 * 25;
__device__ __forceinline__ void subgroup_test(uint32_t *flags, const uint32_t *pts, size_t i, size_t count,
                                              size_t per_group, uint32_t *slots) {
    if (i >= count) return;
    uint32_t w[36];
    ld_words(w, pts + i * G1P_WORDS, 9);
    g1q p;
    g1q_load_std(p, w);
    LdsSlot orig{slots + threadIdx.x * 25}, base{slots + 64 * 25 + threadIdx.x * 25};
    if (!g1_in_subgroup(p, orig, base)) atomicOr(flags + i / per_group, 1u);
}
// the same by the two lanes of a pair, 32 points a block
__device__ __forceinline__ void subgroup_test_pair(uint32_t *flags, const uint32_t *pts, size_t i, size_t count,
                                                   size_t per_group) {
    if (i >= count) return;
    uint32_t w[36];
    ld_words(w, pts + i * G1P_WORDS, 9);
    g1q p;
    g1q_load_std(p, w);
    if (!g1_in_subgroup_pair(p)) atomicOr(flags + i / per_group, 1u);
}

}  // namespace fk20
