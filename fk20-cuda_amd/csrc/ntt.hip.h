// The Fr transform of 128, 256 or 512 points as three passes of radix 8 (the last one 8, 4 or 2)
// with 8 points per lane: 64, 32 or 16 lanes per transform, so a wave runs 1, 2 or 4 of them and
// needs no barrier with others.  Points are exchanged between the passes through LDS, 9 words apart
// (an odd stride: the lanes of a step touch different banks).  39 products per 8 points, 5 inside
// each pass's transform of 8 and one per output; the last ones scale and reduce.
//
// What bounds it: the products' instructions (fr.hip.h fn_mul).  8 192 transforms of 512 points take
// 169 us, 327 with one radix-2 butterfly per thread and stage over the 8 x 32-bit form; about 50 of
// them are HBM's for 268 MB in and out.
//
// ntt_wide, for few transforms, is that radix-2 form over fn: n/2 threads per transform and one
// product per thread and stage, so 4 waves share the work that a lane of the other form does in a
// row (25 us).  It runs while those waves find idle SIMDs: up to 1 024 waves of the other form.
#pragma once
#include <type_traits>

#include "common.hip.h"

namespace fk20 {

// f(0), .., f(7) with compile-time indices: the points stay in registers (the loops are too long for
// the unroller, which would index them in scratch memory)
template <unsigned K = 0, class F>
__device__ __forceinline__ void for8(const F &f) {
    f(std::integral_constant<unsigned, K>());
    if constexpr (K < 7) for8<K + 1>(f);
}

static constexpr unsigned NTT_LDS_WORDS = 64 * 8 * 9;

// DFT of 8 in place, natural order in and out; w[k] = the order-8 root to the k (k = 1, 2, 3).
// In: digits below 2^29 in absolute value; out: below 2^31.
__device__ __forceinline__ void dft8(fn *x, const fn *w) {
    fn a[4], b[4], t;
#pragma unroll
    for (int k = 0; k < 4; k++) {
        fn_add(a[k], x[k], x[k + 4]);
        fn_sub(b[k], x[k], x[k + 4]);
        if (k) fn_mul(b[k], b[k], w[k]);
    }
    fn c0, c1, d0, d1;
    fn_add(c0, a[0], a[2]);
    fn_add(c1, a[1], a[3]);
    fn_sub(d0, a[0], a[2]);
    fn_sub(t, a[1], a[3]);
    fn_mul(d1, t, w[2]);
    fn_norm(c0);
    fn_norm(c1);
    fn_add(x[0], c0, c1);
    fn_sub(x[4], c0, c1);
    fn_add(x[2], d0, d1);
    fn_sub(x[6], d0, d1);
    fn_add(c0, b[0], b[2]);
    fn_add(c1, b[1], b[3]);
    fn_sub(d0, b[0], b[2]);
    fn_sub(t, b[1], b[3]);
    fn_mul(d1, t, w[2]);
    fn_add(x[1], c0, c1);
    fn_sub(x[5], c0, c1);
    fn_add(x[3], d0, d1);
    fn_sub(x[7], d0, d1);
}

__device__ __forceinline__ void dft4(fn *x, const fn &w4) {
    fn a0, a1, b0, b1;
    fn_add(a0, x[0], x[2]);
    fn_add(a1, x[1], x[3]);
    fn_sub(b0, x[0], x[2]);
    fn_sub(b1, x[1], x[3]);
    fn_mul(b1, b1, w4);
    fn_add(x[0], a0, a1);
    fn_sub(x[2], a0, a1);
    fn_add(x[1], b0, b1);
    fn_sub(x[3], b0, b1);
}

__device__ __forceinline__ void fn_tab(fn &z, const int32_t *t) {
#pragma unroll
    for (int i = 0; i < 9; i++) z.l[i] = t[i];
}

// One transform per 2^LOGN / 8 lanes; lane t of it.  load(i, x): the digits of input i;
// store(k, w): the canonical words of output k.  scale: index of the factor 2^-scale.
template <unsigned LOGN, bool INV, class Load, class Store>
__device__ __forceinline__ void ntt(uint32_t *lds, unsigned t, unsigned scale, const DevTables *T, const Load &load,
                                    const Store &store) {
    constexpr unsigned n = 1u << LOGN, L1 = n / 8, P = L1 / 8;
    static_assert(P == 8 || P == 4 || P == 2, "128, 256 or 512 points");
    auto root = [&](fn &z, unsigned e) { fn_tab(z, T->tw29[INV ? 512 - e : e]); };
    int32_t *s = reinterpret_cast<int32_t *>(lds);
    fn w8[4], w, x[8];
#pragma unroll
    for (unsigned k = 1; k < 4; k++) root(w8[k], 64 * k);
    // pass 1: over inputs n/8 apart
    for8([&](auto k) { load(t + L1 * k, x[k]); });
    dft8(x, w8);
    for8([&](auto j) {
        root(w, j * t * (512 / n));
        fn_mul(x[j], x[j], w);
#pragma unroll
        for (int d = 0; d < 9; d++) s[(j * L1 + t) * 9 + d] = x[j].l[d];
    });
    __syncthreads();
    // pass 2: within block j, P apart
    const unsigned j = t / P, t1 = t % P;
    for8([&](auto k) {
#pragma unroll
        for (int d = 0; d < 9; d++) x[k].l[d] = s[(j * L1 + t1 + P * k) * 9 + d];
    });
    __syncthreads();
    dft8(x, w8);
    for8([&](auto k) {
        root(w, k * t1 * (512 / L1));
        fn_mul(x[k], x[k], w);
#pragma unroll
        for (int d = 0; d < 9; d++) s[(j * L1 + k * P + t1) * 9 + d] = x[k].l[d];
    });
    __syncthreads();
    // pass 3: 8 / P groups of P neighbours
    for8([&](auto k) {
#pragma unroll
        for (int d = 0; d < 9; d++) x[k].l[d] = s[(t * 8 + k) * 9 + d];
    });
    if constexpr (P == 8) {
        dft8(x, w8);
    } else if constexpr (P == 4) {
        dft4(x, w8[2]);
        dft4(x + 4, w8[2]);
    } else {
#pragma unroll
        for (unsigned q = 0; q < 8; q += 2) {
            const fn u = x[q];
            fn_add(x[q], u, x[q + 1]);
            fn_sub(x[q + 1], u, x[q + 1]);
        }
    }
    fn_tab(w, T->scale29[scale]);
    for8([&](auto k) {
        const unsigned g = t * (8 / P) + k / P;  // block and its output: j = g / 8, j2 = g % 8
        uint32_t out[8];
        fn_mul(x[k], x[k], w);
        fn_canon(out, x[k]);
        store(g / 8 + 8 * (g % 8) + 64 * (k % P), out);
    });
}

// One transform per workgroup of n/2 threads; lds: n * 9 words.
template <unsigned LOGN, bool INV, class Load, class Store>
__device__ __forceinline__ void ntt_wide(uint32_t *lds, unsigned scale, const DevTables *T, const Load &load,
                                         const Store &store) {
    constexpr unsigned n = 1u << LOGN, half = n / 2;
    int32_t *s = reinterpret_cast<int32_t *>(lds);
    const unsigned t = threadIdx.x;
    auto get = [&](fn &z, unsigned i) {
#pragma unroll
        for (int d = 0; d < 9; d++) z.l[d] = s[i * 9 + d];
    };
    auto put = [&](unsigned i, const fn &z) {
#pragma unroll
        for (int d = 0; d < 9; d++) s[i * 9 + d] = z.l[d];
    };
    fn x, y, w;
#pragma unroll
    for (unsigned e = t; e < n; e += half) {
        load(e, x);
        put(bitrev(e, LOGN), x);
    }
    __syncthreads();
    // decimation in time; the left points gain at most 1.26 r a stage, to 13.6 r
#pragma unroll 1
    for (unsigned st = 0; st < LOGN; st++) {
        const unsigned h = 1u << st, j = t & (h - 1), l = ((t >> st) << (st + 1)) + j, r = l + h;
        const unsigned e = j << (8 - st);
        get(x, r);
        get(y, l);
        fn_tab(w, T->tw29[INV ? 512 - e : e]);
        fn_mul(x, x, w);
        fn_add(w, y, x);
        fn_sub(y, y, x);
        fn_norm(w);
        fn_norm(y);
        put(l, w);
        put(r, y);
        __syncthreads();
    }
    fn_tab(w, T->scale29[scale]);
#pragma unroll
    for (unsigned e = t; e < n; e += half) {
        uint32_t out[8];
        get(x, e);
        fn_mul(x, x, w);
        fn_canon(out, x);
        store(e, out);
    }
}

// Whether `waves` waves of the 8-per-lane form leave SIMDs idle that ntt_wide uses.
static constexpr unsigned NTT_WIDE_WAVES = 1024;

}  // namespace fk20
