// The G1 transform kernels of the column-batched path, as templates over a schedule variant
// (wNAF width W, radix-2^2 or radix-2 butterflies R22, waves per SIMD OCC).  Each variant is
// instantiated in its own translation unit (stage_variant.hip) and published as a
// StageKernels table; a context picks its variant at run time (fk20_ctx_set_schedule).
#pragma once
#include "kutil.hip.h"

namespace fk20 {

// Per item with L = log2(n2), stage schedule over the 2*Lmax - 1 launches of a batch:
//   IFFT DIT stage s (0 <= s <= L-2)  at launch Lmax-1-(L-1)+s   (right-aligned)
//   middle                            at launch Lmax-1            (shared)
//   FFT DIF stage s (1 <= s <= L-1)   at launch Lmax-1+s          (left-aligned)
// so every item of a launch runs the same kind; it.stage holds s (or -1: idle).  Within an
// item, local stage u = 0 .. 2L-2 numbers its own stages: DIT s = u (u < L-1), the middle
// (u = L-1), DIF s = u - (L-1).  Butterfly b of a stage reads and writes two positions
// (in place), given by stage_positions().

// x <- w^(+-e) x, the sign by direction (index[dir * 512 + e] is the program of w^e for TW_FWD,
// of w^-e for TW_INV): w^+-128 by tw_mul_z3, w^256 = -1 by a negation, any other exponent by
// its program.  The exponent is wave-uniform, so is the branch.
template <int W>
__device__ __forceinline__ void twiddle(g1q &x, const uint32_t *ops, const uint32_t *index, unsigned dir,
                                        unsigned e) {
    const unsigned E = (dir == TW_FWD ? e : 512u - e) & 511u;  // x <- w^E x
    if (E == 128 || E == 384) tw_mul_z3(x, E == 128);
    else if (E == 256) fq_neg(x.y, x.y);
    else if (E) tw_mul<W>(x, ops + index[dir * 512 + e]);
}

// The butterflies' twiddle: in the radix-2^2 schedule always w^+-128 (idx 128), else any.
template <int W, bool R22>
__device__ __forceinline__ void bf_twiddle(g1q &x, const uint32_t *ops, const uint32_t *index, unsigned dir,
                                           unsigned idx) {
    if constexpr (R22) tw_mul_z3(x, dir == TW_FWD);
    else twiddle<W>(x, ops, index, dir, idx);
}

// IFFT decimation in time (bit-reversed input): x = D[p1] w^-idx; D[p0], D[p1] = y + x, y - x.
template <int W, bool R22>
__device__ __forceinline__ void dit_butterfly(uint32_t *D, unsigned rows, unsigned row, const Butterfly &f,
                                              const uint32_t *ops, const uint32_t *index) {
    g1q x, y, a;
    pt_load(x, D + ((size_t)f.p1 * rows + row) * 36);
    if (f.idx) bf_twiddle<W, R22>(x, ops, index, TW_INV, f.idx);
    pt_load(y, D + ((size_t)f.p0 * rows + row) * 36);
    g1q_add(a, y, x);
    pt_store(D + ((size_t)f.p0 * rows + row) * 36, a);  // stored first: not live in the next add
    g1q_neg(x, x);
    g1q_add(x, y, x);
    pt_store(D + ((size_t)f.p1 * rows + row) * 36, x);
}

// Last IFFT stage, upper half dropped (h = first half), then the first FFT DIF stage whose
// upper input half is zero:  x = E_j + w^-idx O_j;  D[j] = x;  D[j + n2/2] = w^idx x.
template <int W, bool R22>
__device__ __forceinline__ void middle_butterfly(uint32_t *D, unsigned rows, unsigned row, const Butterfly &f,
                                                 const uint32_t *ops, const uint32_t *index) {
    g1q o, e;
    pt_load(o, D + ((size_t)f.p1 * rows + row) * 36);
    if (f.idx) bf_twiddle<W, R22>(o, ops, index, TW_INV, f.idx);
    pt_load(e, D + ((size_t)f.p0 * rows + row) * 36);
    g1q_add(e, e, o);
    pt_store(D + ((size_t)f.p0 * rows + row) * 36, e);
    if (f.idx) bf_twiddle<W, R22>(e, ops, index, TW_FWD, f.idx);
    pt_store(D + ((size_t)f.p1 * rows + row) * 36, e);
}

// FFT decimation in frequency: D[p0], D[p1] = u + v, (u - v) w^idx.  In the radix-2^2
// schedule the w^128 of a quarter stage is applied by its own launch after the butterflies
// (k_quarter_multi): in the butterfly kernel those ladders ran at 0.9 ms per launch at 512
// rows where the same ladders in a separate launch take 0.5 ms.
template <int W, bool R22>
__device__ __forceinline__ void dif_butterfly(uint32_t *D, unsigned rows, unsigned row, const Butterfly &f,
                                              const uint32_t *ops, const uint32_t *index) {
    g1q u, v, a;
    pt_load(u, D + ((size_t)f.p0 * rows + row) * 36);
    pt_load(v, D + ((size_t)f.p1 * rows + row) * 36);
    g1q_add(a, u, v);
    pt_store(D + ((size_t)f.p0 * rows + row) * 36, a);  // stored first: not live across tw_mul
    g1q_neg(v, v);
    g1q_add(v, u, v);
    if (!R22 && f.idx) bf_twiddle<W, R22>(v, ops, index, TW_FWD, f.idx);
    pt_store(D + ((size_t)f.p1 * rows + row) * 36, v);
}

// Runs local stage u's butterfly `local` of item `it` for this lane's row.  Lanes past the
// item's last row repeat the last row's work (same loads, same stores of the same values),
// so the wave never diverges: the persistent chain below relies on every lane staying
// converged around its wave-uniform steps.
template <int W>
__device__ __forceinline__ void run_butterfly(const Item &it, unsigned u, unsigned local, const uint32_t *ops,
                                              const uint32_t *index) {
    const unsigned rows = it.rows, rg = (rows + 63) / 64;
    const unsigned row = min((local % rg) * 64 + threadIdx.x, rows - 1);
    const Butterfly f = stage_positions<false>(u, it.logn2, local / rg);
    if (u + 1 < it.logn2) dit_butterfly<W, false>(it.D, rows, row, f, ops, index);
    else if (u + 1 == it.logn2) middle_butterfly<W, false>(it.D, rows, row, f, ops, index);
    else dif_butterfly<W, false>(it.D, rows, row, f, ops, index);
}

// One launch per stage: it.stage = s of this launch's kind (DIT/DIF), 0 for the middle.
// Each kernel inlines only its own butterfly (the chain kernel below needs all three).
// W: wNAF width of the twiddle programs; R22: radix-2^2 butterfly positions and twiddles
// (else radix 2, every butterfly carrying its full twiddle); OCC: waves per SIMD the
// register allocation must allow.
// Lanes past the item's last row repeat the last row's work (identical loads and stores
// within one wave) rather than leaving the wave: a ladder run by a wave with one active
// lane measured 2.3x slower than the same ladder with all 64 lanes active.
#define FK20_STAGE_KERNEL(NAME, BODY, USTAGE)                                                       \
    template <int W, bool R22, int OCC>                                                          \
    __global__ void __launch_bounds__(64, OCC) NAME(Launch L, const uint32_t *ops, const uint32_t *index) { \
        unsigned local;                                                                          \
        const Item &it = L.item[find_item(L, blockIdx.x, local)];                                \
        const unsigned rg = (it.rows + 63) / 64;                                                 \
        const unsigned row = min((local % rg) * 64 + threadIdx.x, it.rows - 1);                  \
        const Butterfly f = stage_positions<R22>((USTAGE), it.logn2, local / rg);                \
        BODY<W, R22>(it.D, it.rows, row, f, ops, index);                                         \
    }
FK20_STAGE_KERNEL(k_dit_multi, dit_butterfly, (unsigned)it.stage)
FK20_STAGE_KERNEL(k_middle_multi, middle_butterfly, it.logn2 - 1)
FK20_STAGE_KERNEL(k_dif_multi, dif_butterfly, it.logn2 - 1 + (unsigned)it.stage)
#undef FK20_STAGE_KERNEL

// The point-wise twiddle layer of odd DIF stage it.stage (radix-2^2 schedule): after that
// stage's butterflies in the FFT (dir = TW_FWD), before the butterflies of the transposed DIT
// stage in the IFFT (dir = TW_INV).  One wave per (nontrivial position, 64-row group), the
// positions taken in the cost order of the index's layer table.
template <int W, bool R22, int OCC>
__global__ void __launch_bounds__(64, OCC) k_twiddle_multi(Launch L, const uint32_t *ops, const uint32_t *index,
                                                          unsigned dir) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const unsigned rg = (it.rows + 63) / 64;
    const unsigned row = min((local % rg) * 64 + threadIdx.x, it.rows - 1);
    const uint32_t item = index[TW_LAYER + layer_table_offset(it.logn2, (unsigned)it.stage, dir) + local / rg];
    uint32_t *p = it.D + ((size_t)(item & 0xffffu) * it.rows + row) * 36;
    g1q x;
    pt_load(x, p);
    twiddle<W>(x, ops, index, dir, item >> 16);
    pt_store(p, x);
}

// The w^128 twiddles of radix-2^2 DIF quarter stage it.stage (>= 1; stage 0 is inside the
// middle), after its butterflies: one wave per (twiddled butterfly, 64-row group), the
// butterflies of the launch's second half, whose difference output D[p1] takes w^128.
template <int W, bool R22, int OCC>
__global__ void __launch_bounds__(64, OCC) k_quarter_multi(Launch L) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const unsigned rg = (it.rows + 63) / 64;
    const unsigned row = min((local % rg) * 64 + threadIdx.x, it.rows - 1);
    const unsigned b = (1u << (it.logn2 - 2)) + local / rg;
    const Butterfly f = stage_positions<true>(it.logn2 - 1 + (unsigned)it.stage, it.logn2, b);
    uint32_t *p = it.D + ((size_t)f.p1 * it.rows + row) * 36;
    g1q x;
    pt_load(x, p);
    tw_mul_z3(x, true);
    pt_store(p, x);
}

// The ladders of a direct step (direct.hip.h), record it.stage: a wave takes one product of 64
// rows, or several products of one exponent of fewer (direct_wave).
// One round of the chip's 1024 SIMDs lasts a ladder, 1.1 ms, however few of them work.
template <int W, int OCC>
__global__ void __launch_bounds__(64, OCC) k_direct_products(Launch L, const uint32_t *plan, const uint32_t *ops,
                                                            const uint32_t *index) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const DirectStep &st = reinterpret_cast<const DirectStep *>(plan)[it.stage];
    const unsigned rows = it.rows;
    const DirectWave v = direct_wave(st, plan, rows, 6, it.parts, local);
    const unsigned sub = threadIdx.x >> v.lr, count = v.w >> 16;
    const unsigned row = min(v.row0 + (threadIdx.x & ((1u << v.lr) - 1)), v.last);
    const unsigned slot = (v.w & 0xffffu) + min(sub, count - 1);  // spare lanes repeat a product
    const uint32_t pe = plan[st.prod + slot];
    const unsigned e = FK20_UNIFORM(pe >> 16);
    g1q x;
    pt_load(x, it.D + ((size_t)(pe & 0xffffu) * rows + row) * 36);
    if (e == 128) tw_mul_z3(x, true);
    else if (e) tw_mul<W>(x, ops + index[TW_FWD * 512 + e]);
    pt_store(it.P + ((size_t)slot * rows + row) * 36, x);
}

// The same ladders by two lanes each (ladder_pair.hip.h), both lanes of a pair storing the result they share.
template <int W>
__global__ void __launch_bounds__(64, 1) k_direct_products_pair(Launch L, const uint32_t *plan, const uint32_t *ops,
                                                                const uint32_t *index) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const DirectStep &st = reinterpret_cast<const DirectStep *>(plan)[it.stage];
    const unsigned rows = it.rows;
    const DirectWave v = direct_wave(st, plan, rows, 5, it.parts, local);
    const unsigned pair = threadIdx.x >> 1, sub = pair >> v.lr, count = v.w >> 16;
    const unsigned row = min(v.row0 + (pair & ((1u << v.lr) - 1)), v.last);
    const unsigned slot = (v.w & 0xffffu) + min(sub, count - 1);  // spare lanes repeat a product
    const uint32_t pe = plan[st.prod + slot];
    const unsigned e = FK20_UNIFORM(pe >> 16);
    g1q x;
    pt_load(x, it.D + ((size_t)(pe & 0xffffu) * rows + row) * 36);
    if (e == 128) tw_mul_z3_pair(x, true);
    else if (e) tw_mul_pair<W>(x, ops + index[TW_FWD * 512 + e]);
    pt_store(it.P + ((size_t)slot * rows + row) * 36, x);
}

// ---------------------------------------------------------------- persistent transform chain
//
// All 2*Lmax - 1 stages in one launch of resident waves.  Work items (one butterfly of one
// 64-row group) are numbered stage by stage; a wave takes the next number from a counter,
// waits until the two positions it reads carry the flag of the item's previous local stage,
// runs the butterfly and flags both positions with u + 1.  A wave that finishes a cheap
// (untwiddled) butterfly moves on to later stages at once instead of idling at a launch
// boundary.  Items are taken in stage order, so every item an item depends on was taken
// earlier by a running wave: the waits always end.  Each wait is bounded all the same, by
// the constant-rate wall clock (C.wait_ticks, by default about 1.3 s at the 100 MHz
// reference; a legitimate wait is at most one pass, tens of ms); on expiry the wave records
// an error in ctl[1] and proceeds, and the host turns that word into an error status.

__device__ __forceinline__ unsigned flag_load(const uint32_t *f) {
    return __hip_atomic_load(f, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

template <int W, bool R22, int OCC>
__global__ void __launch_bounds__(64, OCC) k_chain(Chain C, const uint32_t *ops, const uint32_t *index) {
    // No lane-divergent branch anywhere in this loop: the work counter is bumped by lane 0's
    // addend (every lane executes the atomic, the others add 0) and every lane stores the
    // flags, so the wave-uniform values below always come from a fully converged wave.  A
    // wave can take at most `total` items, which bounds the loop whatever happens.
#pragma unroll 1
    for (unsigned iter = 0; iter < C.total; iter++) {
        const unsigned got =
            __hip_atomic_fetch_add(C.ctl, threadIdx.x == 0 ? 1u : 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned w = __builtin_amdgcn_readfirstlane(got);  // lane 0's: the value before its add
        if (w >= C.total) break;
        unsigned t = 0;
#pragma unroll 1
        while (w >= C.t_end[t]) t++;
        unsigned local = w - (t ? C.t_end[t - 1] : 0);
        unsigned k = 0;
#pragma unroll 1
        while (local >= C.blk_end[t][k]) k++;
        if (k) local -= C.blk_end[t][k - 1];
        const Item &it = C.L.item[k];
        const unsigned u = (unsigned)C.ustage[t][k];
        const unsigned rg = (it.rows + 63) / 64, g = local % rg;
        const Butterfly f = stage_positions<false>(u, it.logn2, local / rg);
        uint32_t *fl = it.flags + (size_t)g * (1u << it.logn2);
        if (u) {
            const uint64_t t0 = wall_clock64();
            bool expired = false;
#pragma unroll 1
            while (flag_load(fl + f.p0) < u || flag_load(fl + f.p1) < u) {
                if (wall_clock64() - t0 >= C.wait_ticks) {
                    expired = true;
                    break;
                }
                __builtin_amdgcn_s_sleep(2);
            }
            if (expired) __hip_atomic_store(C.ctl + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
        }
        run_butterfly<W>(it, u, local, ops, index);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __hip_atomic_store(fl + f.p0, u + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(fl + f.p1, u + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// ---------------------------------------------------------------- drop-in entry points

// D[pos][row] = in[row][j] (standard form -> packed Montgomery), pos = bitrev(j) when brev,
// times the scalar of the program at scale_ops when given.  The blocks after these n * rg
// test the inputs, flags[row] |= 1 for a point outside G1: 126 doublings beside the scaling ladders
// instead of a launch before them (65 inverse transforms of 128, two launches of 0.74 and
// 0.77 ms: 0.79 together, the call 3.34 -> 2.57).
template <int W, int OCC>
__global__ void __launch_bounds__(64, OCC) k_plain_load(uint32_t *D, const uint32_t *in, unsigned rows,
                                                       unsigned logn, unsigned brev, const uint32_t *scale_ops,
                                                       uint32_t *flags) {
    __shared__ uint32_t slots[SUBGROUP_SLOT_WORDS];
    const unsigned rg = (rows + 63) / 64, j = blockIdx.x / rg;
    if (j >= 1u << logn) {
        const size_t i = (size_t)(blockIdx.x - (rg << logn)) * 64 + threadIdx.x;
        subgroup_test(flags, in, i, (size_t)rows << logn, (size_t)1 << logn, slots);
        return;
    }
    const unsigned row = min((blockIdx.x % rg) * 64 + threadIdx.x, rows - 1);  // spare lanes repeat the last row
    uint32_t w[36];
    ld_words(w, in + ((size_t)row * (1u << logn) + j) * G1P_WORDS, 9);
    g1q p;
    g1q_load_std(p, w);
    if (scale_ops) tw_mul<W>(p, scale_ops);
    pt_store(D + ((size_t)(brev ? bitrev(j, logn) : j) * rows + row) * 36, p);
}

// The same with two lanes per row and point (PAIR_WAVES); 65 inverse transforms of 128: 0.79 -> 0.55 ms.
template <int W>
__global__ void __launch_bounds__(64, 1) k_plain_load_pair(uint32_t *D, const uint32_t *in, unsigned rows, unsigned logn,
                                                           unsigned brev, const uint32_t *scale_ops, uint32_t *flags) {
    const unsigned rg = (rows + 31) / 32, j = blockIdx.x / rg;
    if (j >= 1u << logn) {
        const size_t i = (size_t)(blockIdx.x - (rg << logn)) * 32 + threadIdx.x / 2;
        subgroup_test_pair(flags, in, i, (size_t)rows << logn, (size_t)1 << logn);
        return;
    }
    const unsigned row = min((blockIdx.x % rg) * 32 + threadIdx.x / 2, rows - 1);
    uint32_t w[36];
    ld_words(w, in + ((size_t)row * (1u << logn) + j) * G1P_WORDS, 9);
    g1q p;
    g1q_load_std(p, w);
    if (scale_ops) tw_mul_pair<W>(p, scale_ops);
    pt_store(D + ((size_t)(brev ? bitrev(j, logn) : j) * rows + row) * 36, p);
}

// The kernel table of variant (W, R22, OCC); the persistent chain (radix 2 whatever the
// variant's butterflies) is published by the radix-2 variants only, the drop-ins' load by the default.
template <int W, bool R22, int OCC>
constexpr StageKernels make_stage_kernels() {
    StageKernels K{};
    K.dit = k_dit_multi<W, R22, OCC>;
    K.middle = k_middle_multi<W, R22, OCC>;
    K.dif = k_dif_multi<W, R22, OCC>;
    K.twiddle = k_twiddle_multi<W, R22, OCC>;
    if constexpr (!R22) K.chain = k_chain<W, R22, OCC>;
    if constexpr (R22) K.quarter = k_quarter_multi<W, R22, OCC>;
    if constexpr (R22) {
        K.direct = k_direct_products<W, OCC>;
        K.direct_pair = k_direct_products_pair<W>;
    }
    if constexpr (W == TW_WNAF && R22 && OCC == (int)DEFAULT_OCCUPANCY) {
        K.plain_load = k_plain_load<W, OCC>;
        K.plain_load_pair = k_plain_load_pair<W>;
    }
    K.wnaf = W;
    K.r22 = R22;
    K.occupancy = OCC;
    return K;
}

}  // namespace fk20
