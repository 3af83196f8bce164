// Kernels of the batched FK20 path (many rows sharing one resident setup).
//
//  1. k_scale_bases    xext_fft / n2 -> packed Montgomery bases (the IFFT's 1/n2 is folded
//                      into the setup, so the G1 IFFT below runs unscaled).
//  2. k_table_build    fixed-base signed-window tables T[b][win][d] = d * 2^(w*win) * base_b
//                      (d = 1 .. 2^(w-1)), affine, canonical Montgomery, one per base.
//  3. k_toeplitz_fft_multi  Toeplitz coefficients + NTT per (row, i), written transposed as
//                      tcT[j][i][row] so 64 rows of one column are contiguous.
//  4. k_msm_multi      hext_fft[j] of every row = sum_i tc_fft[i][j] * xext_fft[i][j] by
//                      signed fixed windows: ceil(256/w) mixed additions per term, no
//                      doublings.  Lanes = rows of one column (1, 4 or 16 lanes per row), so a
//                      wave gathers from the table region of one base.  Output goes to
//                      D[bitrev(j)][row].
//  5. the transforms   (stage_kernels.hip.h) column-batched: the G1 IFFT (DIT, bit-reversed in,
//                      natural out), the fused last IFFT stage + zero upper half + first FFT
//                      stage, and the G1 FFT (DIF, natural in, bit-reversed out), radix 2^2
//                      with point-wise twiddle layers; a wave is one butterfly or point for 64
//                      rows, so the twiddle is wave-uniform and runs as a precomputed GLV +
//                      wNAF program.  Small batches take the direct schedule instead
//                      (direct.hip.h; k_direct_split, k_direct_sums).
//  6. k_output_multi   D[pos][row] -> h_fft[row][bitrev(pos)] in the reference ABI, z = 1.
// Same mathematics as fk20_msm.cu:23-66, g1p_fft.cu:25-330 and fk20_hext_fft2h_fft.cu:27-70;
// the layout and algorithms are this library's own.
#include <cstring>

#include "common.hip.h"
#include "fast.hip.h"
#include "kutil.hip.h"
#include "ntt.hip.h"

namespace fk20 {

// ---------------------------------------------------------------- setup: scaled bases

__device__ __noinline__ void g1_mul_std(g1q &r, const g1q &p, const uint32_t *k) {
    g1q q;
    g1q_inf(q);
#pragma unroll 1
    for (int w = 7; w >= 0; w--) {
        const uint32_t kw = k[w];
#pragma unroll 1
        for (int b = 31; b >= 0; b--) {
            g1q_dbl(q, q);
            if ((kw >> b) & 1) g1q_add(q, q, p);
        }
    }
    r = q;
}

// xs[b] = scale * xext[b] (packed Montgomery); inf[b] = 1 if xext[b] is infinity.
__global__ void __launch_bounds__(64) k_scale_bases(uint32_t *xs, uint32_t *inf, const uint32_t *xext,
                                                    size_t count, const uint32_t *scale) {
    const size_t b = (size_t)blockIdx.x * 64 + threadIdx.x;
    if (b >= count) return;
    uint32_t w[36];
    ld_words(w, xext + b * G1P_WORDS, 9);
    g1q p;
    g1q_load_std(p, w);
    inf[b] = g1q_is_inf(p) ? 1u : 0u;
    uint32_t k[8];
#pragma unroll
    for (int i = 0; i < 8; i++) k[i] = scale[i];
    g1_mul_std(p, p, k);
    pt_store(xs + b * 36, p);
}

// ---------------------------------------------------------------- subgroup membership

__global__ void k_fill_u32(uint32_t *p, size_t n, uint32_t v) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// flags[i / per_group] |= 1 when pts[i] lies outside the order-r subgroup.
__global__ void __launch_bounds__(64, 2) k_subgroup_groups(uint32_t *flags, const uint32_t *pts, size_t count,
                                                           size_t per_group) {
    __shared__ uint32_t slots[SUBGROUP_SLOT_WORDS];
    subgroup_test(flags, pts, (size_t)blockIdx.x * 64 + threadIdx.x, count, per_group, slots);
}

// The same by two lanes per point (ladder_pair.hip.h), 32 points a block: 126 doublings after one
// another are the launch's time while SIMDs idle (8 192 points 0.73 -> 0.46 ms).
__global__ void __launch_bounds__(64, 1) k_subgroup_pair(uint32_t *flags, const uint32_t *pts, size_t count,
                                                         size_t per_group) {
    subgroup_test_pair(flags, pts, (size_t)blockIdx.x * 32 + threadIdx.x / 2, count, per_group);
}

// ---------------------------------------------------------------- rows outside G1
//
// On a point P outside the order-r subgroup, [a]P and [b]P differ whenever a != b as integers,
// even for a = b (mod r): a transform of such points is defined by its exact sequence of
// integer multipliers, not by the linear map mod r that the column-batched kernels compute.
// A row that holds such a point is recomputed here in the reference's order of operations:
// radix-2 decimation in time over bit-reversed positions, twiddle w^e applied to the right
// point of a butterfly as the canonical integer w^e mod r (g1p_fft.cu:25-170); the inverse
// with the butterflies transposed, w^-e applied after them and 2^-logn (and 2^-logn w^-128)
// in stage 1 (g1p_fft.cu:180-330); hext_fft -> h_fft as inverse, odd positions cleared,
// forward (fk20_hext_fft2h_fft.cu:27-70).  Products are double-and-add over complete
// formulas (g1_mul_std, as g1p_mul.cu:18).  One workgroup of 256 threads per row; the row's n
// points live in `work` (n * 36 words per row, row-contiguous); barriers order the stages.

// (a, b) <- (a + b, a - b)
__device__ __forceinline__ void addsub(g1q &a, g1q &b) {
    g1q s;
    g1q_add(s, a, b);
    g1q_neg(b, b);
    g1q_add(b, a, b);
    a = s;
}

__device__ __forceinline__ void ref_butterfly(uint32_t *Wr, unsigned s, unsigned t, bool inverse, unsigned logn,
                                              const DevTables *T) {
    const unsigned h = 1u << s, j = t & (h - 1);
    const unsigned l = ((t >> s) << (s + 1)) + j, r = l + h;
    const unsigned e = j << (8 - s);  // twiddle w^e of the order-512 root w
    g1q a, b;
    pt_load(a, Wr + (size_t)l * 36);
    pt_load(b, Wr + (size_t)r * 36);
    if (!inverse) {
        if (e) g1_mul_std(b, b, T->tw_std[e]);
        addsub(a, b);
    } else {
        addsub(a, b);
        if (s == 1) {
            g1_mul_std(a, a, T->inv2k_std[logn]);
            g1_mul_std(b, b, j ? T->inv2k_w384_std[logn] : T->inv2k_std[logn]);
        } else if (s > 1 && e) {
            g1_mul_std(b, b, T->tw_std[512 - e]);
        }
    }
    pt_store(Wr + (size_t)l * 36, a);
    pt_store(Wr + (size_t)r * 36, b);
}

// kind: 0 forward (in natural order -> out natural order), 1 inverse, 2 hext_fft -> h_fft.
// in_D != nullptr: the input is D[bitrev(j)][row] (packed Montgomery, the MSM's output layout)
// instead of in[row][j].
__global__ void __launch_bounds__(256) k_ref_rows(unsigned kind, uint32_t *out, const uint32_t *in,
                                                 const uint32_t *in_D, unsigned rows, unsigned logn, uint32_t *work,
                                                 const uint32_t *flags, unsigned flag_stride, const DevTables *T) {
    const unsigned row = blockIdx.x;
    if (!flags[(size_t)row * flag_stride]) return;  // uniform over the workgroup
    const unsigned n = 1u << logn, t = threadIdx.x;
    uint32_t *Wr = work + (size_t)row * n * 36;
    for (unsigned j = t; j < n; j += 256) {
        g1q p;
        if (in_D) {
            pt_load(p, in_D + ((size_t)bitrev(j, logn) * rows + row) * 36);
        } else {
            uint32_t w[36];
            ld_words(w, in + ((size_t)row * n + j) * G1P_WORDS, 9);
            g1q_load_std(p, w);
        }
        pt_store(Wr + (size_t)(kind == 0 ? bitrev(j, logn) : j) * 36, p);
    }
    __syncthreads();
    if (kind != 0) {
#pragma unroll 1
        for (int s = (int)logn - 1; s >= 0; s--) {
            if (t < n / 2) ref_butterfly(Wr, (unsigned)s, t, true, logn, T);
            __syncthreads();
        }
        if (kind == 2) {
            // the upper half of the inverse's natural-order output sits at the odd positions
            for (unsigned j = 2 * t + 1; j < n; j += 512) {
                g1q z;
                g1q_inf(z);
                pt_store(Wr + (size_t)j * 36, z);
            }
            __syncthreads();
        }
    }
    if (kind != 1) {
#pragma unroll 1
        for (unsigned s = 0; s < logn; s++) {
            if (t < n / 2) ref_butterfly(Wr, s, t, false, logn, T);
            __syncthreads();
        }
    }
    for (unsigned j = t; j < n; j += 256) {
        g1q p;
        pt_load(p, Wr + (size_t)(kind == 1 ? bitrev(j, logn) : j) * 36);
        uint32_t w[36];
        g1q_store_std(w, p);
        st_words(out + ((size_t)row * n + j) * G1P_WORDS, w, 9);
    }
}

// ---------------------------------------------------------------- setup: window tables

// One thread per (base, window) of the launch's bases [base0, base0 + nb): entries d * B' for
// d = 1 .. H (B' = 2^(w win) B), built as projective multiples and converted to affine by
// Montgomery's batch trick in blocks of TABLE_BLK entries (one inversion per block).  zt holds
// (z_e, prefix_{e-1}) of the current block per thread, laid out [entry][thread] so that the
// 64 lanes of a wave touch consecutive words; it is sized by the launch, not by H, so every
// (base, window) of a setup fits in one or two launches.
__global__ void __launch_bounds__(64, 2) k_table_build(uint32_t *table, uint32_t *zt, const uint32_t *xs,
                                                    const uint32_t *inf, uint32_t *err, unsigned base0,
                                                    unsigned nb, unsigned win_bits, unsigned nwin) {
    const unsigned nthreads = nb * nwin;
    const unsigned t = blockIdx.x * 64 + threadIdx.x;
    if (t >= nthreads) return;
    const unsigned b = base0 + t / nwin, win = t % nwin;
    const unsigned H = 1u << (win_bits - 1), blk = min(H, TABLE_BLK);
    uint32_t *tab = table + ((size_t)b * nwin + win) * H * TABLE_ENTRY_WORDS;
    if (inf[b]) {
        for (unsigned e = 0; e < H; e++) {
            uint32_t zero[24] = {0};
            st_words(tab + (size_t)e * TABLE_ENTRY_WORDS, zero, 6);
        }
        return;
    }
    // B' = 2^(w win) B in affine form, so each entry is one mixed addition of B' (B' is not
    // infinity: the base is not, and E(Fp) has odd order).  An entry d B' is infinity only
    // for a base of small order outside G1; the block's inversion then fails and *err says so.
    g1q E;
    fq bx, by;
    {
        g1q B;
        pt_load(B, xs + (size_t)b * 36);
#pragma unroll 1
        for (unsigned d = 0; d < win_bits * win; d++) g1q_dbl(B, B);
        g1q_to_affine(bx, by, B);
    }
    E.x = bx;
    E.y = by;
    fq_one(E.z);
#pragma unroll 1
    for (unsigned e0 = 0; e0 < H; e0 += blk) {
        fq prefix;
        fq_one(prefix);
#pragma unroll 1
        for (unsigned i = 0; i < blk; i++) {
            const unsigned e = e0 + i;
            if (e) g1q_add_aff(E, E, bx, by);
            uint32_t *z = zt + ((size_t)i * nthreads + t) * 24;
            fq_store(tab + (size_t)e * TABLE_ENTRY_WORDS, E.x);
            fq_store(tab + (size_t)e * TABLE_ENTRY_WORDS + 12, E.y);
            fq_store(z, E.z);
            fq_store(z + 12, prefix);  // prefix of z_e0 .. z_{e-1}
            fq_mul(prefix, prefix, E.z);
        }
        fq inv;
        if (fq_is_zero(prefix)) atomicOr(err, 1u);
        fq_inv(inv, prefix);
#pragma unroll 1
        for (int i = (int)blk - 1; i >= 0; i--) {
            const unsigned e = e0 + (unsigned)i;
            const uint32_t *z = zt + ((size_t)i * nthreads + t) * 24;
            fq ze, pe, zinv, x, y;
            fq_load(ze, z);
            fq_load(pe, z + 12);
            fq_mul(zinv, inv, pe);
            fq_mul(inv, inv, ze);
            fq_load(x, tab + (size_t)e * TABLE_ENTRY_WORDS);
            fq_load(y, tab + (size_t)e * TABLE_ENTRY_WORDS + 12);
            fq_mul(x, x, zinv);
            fq_mul(y, y, zinv);
            uint32_t w[24];
            fq_canon_words(w, x);
            fq_canon_words(w + 12, y);
            st_words(tab + (size_t)e * TABLE_ENTRY_WORDS, w, 6);
        }
    }
}

// ---------------------------------------------------------------- Toeplitz + NTT (transposed)

__device__ __forceinline__ int toeplitz_src_T(unsigned i, unsigned j, unsigned N) {
    const unsigned k = N / 16;
    if (j == 0) return (int)(N - 1 - i);
    if (j <= k + 1) return -1;
    return (int)(31 - i + 16 * (j - (k + 2)));
}

template <unsigned LOGN, bool WIDE>
__device__ __forceinline__ void toeplitz_fft(uint32_t *lds, const Item &it, unsigned local, const DevTables *T) {
    constexpr unsigned n = 1u << LOGN, lanes = n / 8, N = 8 * n;
    const unsigned sub = threadIdx.x / lanes, t = threadIdx.x % lanes;
    const unsigned id = WIDE ? local : local * (64 / lanes) + sub, i = id % 16;  // 16 divides into whole waves
    const size_t row = id / 16;
    const uint32_t *poly = it.poly + row * N * FR_WORDS;
    uint32_t *out = it.tcT + ((size_t)i * it.rows + row) * FR_WORDS;
    // the reference's order (k_ref_rows) applies 1/n2 inside the inverse transform
    const bool scaled = it.scale_tc && !(it.rowflag && it.rowflag[row * it.flag_stride]);
    const auto load = [&](unsigned e, fn &x) {
        const int src = toeplitz_src_T(i, e, N);
        uint32_t w[8] = {0};
        if (src >= 0) ld_words(w, poly + (size_t)src * FR_WORDS, 2);
        fn_unpack(x, w);
    };
    const auto store = [&](unsigned k, const uint32_t *w) {
        st_words(out + (size_t)k * 16 * it.rows * FR_WORDS, w, 2);
    };
    if constexpr (!WIDE) ntt<LOGN, false>(lds + sub * n * 9, t, scaled ? LOGN : 0, T, load, store);
    else if (threadIdx.x < n / 2) ntt_wide<LOGN, false>(lds, scaled ? LOGN : 0, T, load, store);
}

// The (row, i) transforms of the items, 512 / n2 per wave; WIDE: one per workgroup of 256 threads
// (whole waves of which leave before the first barrier where n2 is smaller).
template <bool WIDE>
__global__ void __launch_bounds__(WIDE ? 256 : 64, 2) k_toeplitz_fft_multi(Launch L, const DevTables *T) {
    __shared__ uint32_t lds[WIDE ? 512 * 9 : NTT_LDS_WORDS];
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    if (it.logn2 == 9) toeplitz_fft<9, WIDE>(lds, it, local, T);
    else if (it.logn2 == 8) toeplitz_fft<8, WIDE>(lds, it, local, T);
    else toeplitz_fft<7, WIDE>(lds, it, local, T);
}

// ---------------------------------------------------------------- window-table MSM

// A standard-form scalar k < r as signed fixed windows of WIN bits over a base's table
// tb[win][d - 1] = d * 2^(WIN*win) * B (affine): one mixed addition per non-zero digit, no
// doublings.  k < r < 2^255 keeps the last window's carry inside the ceil(256/WIN) windows for
// every WIN in 8..13.
//
// The entry of the next window is fetched while the current one is added: a gathered entry is a
// 128-byte line somewhere in gigabytes of tables, several microseconds away under load, and at
// two waves per SIMD (the addition's registers) nothing else covers it.
struct WindowStream {
    const uint32_t *tb;
    uint32_t k[8];
    uint32_t carry;
    unsigned win;
    __device__ void start(const uint32_t *table) {
        tb = table;
        carry = 0;
        win = 0;
    }
    // the next digit; fetches its entry (the first one for digit 0)
    __device__ int next(uint32_t *ent, unsigned WIN) {
        const unsigned H = 1u << (WIN - 1), MASK = (1u << WIN) - 1;
        const uint32_t bits = (k[0] & MASK) + carry;
        carry = bits > H ? 1u : 0u;
        const int d = (int)bits - (int)(carry << WIN);
        // shift the scalar right by WIN bits (WIN < 32)
#pragma unroll
        for (int q = 0; q < 7; q++) k[q] = (k[q] >> WIN) | (k[q + 1] << (32 - WIN));
        k[7] >>= WIN;
        const unsigned e = (unsigned)(d < 0 ? -d : d);
        ld_words(ent, tb + ((size_t)win * H + (e ? e - 1 : 0)) * TABLE_ENTRY_WORDS, 6);
        win++;
        return d;
    }
};

// acc += sum of the scalars that `fetch(t, k)` gives (t = 0 .. nterms - 1, false: skip the term)
// times their bases, term t's table at tables + t * stride words.
template <class Fetch>
__device__ __forceinline__ void window_sum(g1q &acc, const uint32_t *tables, size_t stride, unsigned nterms,
                                           unsigned WIN, const Fetch &fetch) {
    const unsigned NWIN = (256 + WIN - 1) / WIN;
    unsigned t = 0;
    WindowStream w;
    while (t < nterms && !fetch(t, w.k)) t++;
    if (t == nterms) return;
    w.start(tables + t * stride);
    uint32_t ent[24];
    int d = w.next(ent, WIN);
#pragma unroll 1
    while (true) {
        fq x, y;
        fq_unpack_raw(x, ent);
        fq_unpack_raw(y, ent + 12);
        if (d < 0) fq_neg(y, y);
        const bool add = d != 0;
        if (w.win == NWIN) {
            t++;
            while (t < nterms && !fetch(t, w.k)) t++;
            if (t < nterms) w.start(tables + t * stride);
        }
        const bool more = t < nterms;
        if (more) d = w.next(ent, WIN);
        if (add) g1q_add_aff(acc, acc, x, y);
        if (!more) break;
    }
}

// hext_fft[j] of one column j: sum over 16 terms of ceil(256/w) signed-window digits, one mixed
// addition each; output to D[bitrev(j)][row].  LP lanes share a row, each with 16 / LP of the
// terms, and add up across the wave: an addition takes 9 us in a wave alone on its SIMD and 8.3
// per wave beside others, so LP = 1 (no closing additions) is best where its waves fill the
// chip, and 4 or 16 shorten a small or ragged launch (msm_lanes picks by waves and additions:
// 64 rows of 4096 at window 8 take 4.6 ms with LP = 1 and 2.7 with 16; 512 rows 17.2 and 19.9).
template <unsigned LP>
__global__ void __launch_bounds__(64) k_msm_multi(Launch L) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const unsigned rows = it.rows, n2 = 1u << it.logn2, per_wave = 64 / LP, rg = (rows + per_wave - 1) / per_wave;
    const unsigned WIN = it.win, NWIN = (256 + WIN - 1) / WIN, H = 1u << (WIN - 1);
    const unsigned j = local / rg, i0 = threadIdx.x % LP;
    const unsigned row0 = (local % rg) * per_wave + threadIdx.x / LP;
    const unsigned row = min(row0, rows - 1);  // spare lanes repeat the last row
    const size_t per_base = (size_t)NWIN * H * TABLE_ENTRY_WORDS;
    const uint32_t *tc = it.tcT + (((size_t)j * 16 + i0) * rows + row) * FR_WORDS, *inf = it.inf + i0 * n2 + j;
    g1q acc;
    g1q_inf(acc);
    window_sum(acc, it.table + (i0 * n2 + j) * per_base, LP * n2 * per_base, 16 / LP, WIN, [&](unsigned t, uint32_t *k) {
        if (inf[t * LP * n2]) return false;
        ld_words(k, tc + (size_t)t * LP * rows * FR_WORDS, 2);
        return true;
    });
    lane_sum(acc, LP);
    if (i0 == 0 && (LP == 1 || row0 < rows)) pt_store(it.D + ((size_t)bitrev(j, it.logn2) * rows + row) * 36, acc);
}

// ---------------------------------------------------------------- KZG commitments
//
// commit[row] = sum_i poly[row][i] * srs[i] (FK20Py kzg_proofs.py:159 commit_to_poly) over
// window tables of the SRS points built like the FK20 setup's.  A lane sums `chunk` consecutive
// coefficients of one row; lp lanes share a row (a power of two: 64 / rows for small batches, so
// that no lane is idle) and add up across the wave into partial[chunk][row]; one wave per row
// then adds the row's partial sums (commit_shape picks lp and chunk).

__global__ void __launch_bounds__(64) k_commit_partial(const uint32_t *poly, const uint32_t *table,
                                                       const uint32_t *inf, uint32_t *partial, unsigned rows,
                                                       unsigned N, unsigned win_bits, unsigned chunk, unsigned lp) {
    const unsigned per_wave = 64 / lp, rg = (rows + per_wave - 1) / per_wave, c = blockIdx.x / rg;
    const unsigned row0 = (blockIdx.x % rg) * per_wave + threadIdx.x / lp;
    const unsigned row = min(row0, rows - 1);  // spare lanes repeat the last row
    const unsigned NWIN = (256 + win_bits - 1) / win_bits, H = 1u << (win_bits - 1);
    const unsigned i0 = (c * lp + threadIdx.x % lp) * chunk;  // chunk * lp divides N
    const size_t per_base = (size_t)NWIN * H * TABLE_ENTRY_WORDS;
    const uint32_t *coeff = poly + ((size_t)row * N + i0) * FR_WORDS;
    g1q acc;
    g1q_inf(acc);
    window_sum(acc, table + i0 * per_base, per_base, chunk, win_bits, [&](unsigned t, uint32_t *k) {
        if (inf[i0 + t]) return false;
        // the caller's coefficient may be any 256-bit representative: reduce it below r, so
        // the top signed window's carry stays inside the ceil(256/w) windows (at w = 8 the
        // windows end exactly at bit 256, and a value >= 2^255 would carry out of them)
        fs c;
        ld_words(c.l, coeff + (size_t)t * FR_WORDS, 2);
        fs_reduce_std(c);
#pragma unroll
        for (int q = 0; q < 8; q++) k[q] = c.l[q];
        return true;
    });
    lane_sum(acc, lp);
    if (threadIdx.x % lp == 0 && row0 < rows) pt_store(partial + ((size_t)c * rows + row) * 36, acc);
}

// out[row] = the sum of partial[0 .. nparts)[row], as a canonical standard-form g1p_t: a wave per row.
__global__ void __launch_bounds__(64) k_commit_reduce(const uint32_t *partial, uint32_t *out, unsigned rows,
                                                      unsigned nparts) {
    const unsigned row = blockIdx.x;
    g1q acc, x;
    g1q_inf(acc);
    if (threadIdx.x < nparts) pt_load(acc, partial + ((size_t)threadIdx.x * rows + row) * 36);
#pragma unroll 1
    for (unsigned p = threadIdx.x + 64; p < nparts; p += 64) {
        pt_load(x, partial + ((size_t)p * rows + row) * 36);
        g1q_add(acc, acc, x);
    }
    lane_sum(acc, 64);
    if (threadIdx.x == 0) {
        uint32_t w[36];
        g1q_store_std(w, acc);
        st_words(out + (size_t)row * G1P_WORDS, w, 9);
    }
}

// ---------------------------------------------------------------- G1 transform stages
//
// The butterfly, twiddle-layer, persistent-chain and drop-in load kernels are templates over
// a schedule variant (stage_kernels.hip.h), built once per variant (stage_variant.hip);
// launches go through the variant's StageKernels table.

extern const StageKernels stage_kernels_3_0_2, stage_kernels_3_0_3, stage_kernels_3_1_2, stage_kernels_3_1_3,
    stage_kernels_4_0_2, stage_kernels_4_0_3, stage_kernels_4_1_2, stage_kernels_4_1_3, stage_kernels_5_0_2,
    stage_kernels_5_0_3, stage_kernels_5_1_2, stage_kernels_5_1_3;

const StageKernels *stage_kernels(unsigned wnaf, bool r22, unsigned occupancy) {
    static const StageKernels *const table[3][2][2] = {
        {{&stage_kernels_3_0_2, &stage_kernels_3_0_3}, {&stage_kernels_3_1_2, &stage_kernels_3_1_3}},
        {{&stage_kernels_4_0_2, &stage_kernels_4_0_3}, {&stage_kernels_4_1_2, &stage_kernels_4_1_3}},
        {{&stage_kernels_5_0_2, &stage_kernels_5_0_3}, {&stage_kernels_5_1_2, &stage_kernels_5_1_3}}};
    if (wnaf < 3 || wnaf > 5 || occupancy < 2 || occupancy > 3) return nullptr;
    return table[wnaf - 3][r22 ? 1 : 0][occupancy - 2];
}
//
// Clears the chain's flags of every item and its work counter / error word (ctl[0..1]).
__global__ void k_chain_reset(Chain C) {
    if (blockIdx.x == 0 && threadIdx.x < 2) C.ctl[threadIdx.x] = 0;
    const Item &it = C.L.item[blockIdx.x];
    const unsigned n = ((it.rows + 63) / 64) << it.logn2;
    for (unsigned e = threadIdx.x; e < n; e += blockDim.x) it.flags[e] = 0;
}

// ---------------------------------------------------------------- direct schedule (direct.hip.h)

// The split of a direct step, in place: 2^loga lanes per (block, m, row), lane t holding point t;
// after level h the upper half [h, 2h) keeps differences and the lower one goes on with sums.
__global__ void __launch_bounds__(64) k_direct_split(Launch L, const uint32_t *plan, unsigned pass) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const DirectStep &st = reinterpret_cast<const DirectStep *>(plan)[it.stage];
    const unsigned loga = direct_split_log(st.loga, pass), logN = st.loga + st.logb;
    const unsigned logb = pass == 0 ? logN - loga : st.logb;
    const unsigned rows = it.rows, logn = it.logn2, lane = threadIdx.x, t = lane & ((1u << loga) - 1);
    const unsigned total = rows << (st.logblocks + logb);
    // spare lane groups repeat the last one's work
    const unsigned id = min((local * 64 + lane) >> loga, total - 1), row = id % rows, g = id / rows;
    const unsigned i = ((g >> logb) << logN) + (g & ((1u << logb) - 1)) + (t << logb);
    const unsigned pos = (st.in_map & 1u) ? bitrev(i, logn) : i;
    uint32_t *p = it.D + ((size_t)pos * rows + row) * 36;
    g1q x, o, u;
    g1q_inf(x);
    if (pass || !(st.in_map & 2u) || i < (1u << (logn - 1))) pt_load(x, p);
#pragma unroll 1
    for (unsigned h = 1u << (loga - 1); h; h >>= 1) {
        shfl_point(o, x, (int)(t < h ? lane + h : t < 2 * h ? lane - h : lane));
        u = x;
        if (t >= h) g1q_neg(u, x);
        g1q_add(o, o, u);
        if (t < 2 * h) x = o;
    }
    pt_store(p, x);
}

// The sums of a direct step: 2^log_lanes lanes per (output, row), each adding every so-manieth
// term, then across the lanes; D is free to be overwritten, every term is in P.
__global__ void __launch_bounds__(64) k_direct_sums(Launch L, const uint32_t *plan) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    const DirectStep &st = reinterpret_cast<const DirectStep *>(plan)[it.stage];
    const unsigned rows = it.rows, lanes = 1u << st.log_lanes, part = threadIdx.x & (lanes - 1);
    const unsigned id = min((local * 64 + threadIdx.x) >> st.log_lanes, st.nout * rows - 1), row = id % rows;
    const uint32_t *o = plan + st.sums + (size_t)(id / rows) * st.sum_words;
    g1q acc, x;
    auto term = [&](g1q &p, uint32_t c) {
        g1q_inf(p);
        if (c == DIRECT_NONE) return;
        pt_load(p, it.P + ((size_t)(c & 0x7fffffffu) * rows + row) * 36);
        if (c >> 31) g1q_neg(p, p);
    };
    term(acc, o[DIRECT_SUM_FIRST + part]);
#pragma unroll 1
    for (unsigned k = DIRECT_SUM_FIRST + lanes; k < st.sum_words; k += lanes) {
        const uint32_t c = o[k + part];
        if (!__any(c != DIRECT_NONE)) break;  // outputs come longest first
        term(x, c);
        g1q_add(acc, acc, x);
    }
    lane_sum(acc, lanes);
    if (part == 0) pt_store(it.D + ((size_t)o[0] * rows + row) * 36, acc);
}

// D[pos][row] -> the item's output format.  D is in bit-reversed order, so the natural
// index of pos is bitrev(pos) and the data-availability order (FK20Py
// list_to_reverse_bit_order of the natural list) is pos itself.
//   FK20_OUT_G1P / _DA:               g1p_t, canonical standard projective (144 bytes) with z = 1
//                                     (infinity (0 : 1 : 0)): a row's proofs are the same words
//                                     whatever batch and schedule they were computed in
//   FK20_OUT_COMPRESSED / _DA:        48-byte compressed G1 (g1_compress)
__global__ void __launch_bounds__(64) k_output_multi(Launch L) {
    unsigned local;
    const Item &it = L.item[find_item(L, blockIdx.x, local)];
    // lanes take (position, row) pairs, rows fastest, so that few rows still fill the waves that
    // run an inversion (one active lane took 146 us, 64 take 65)
    const unsigned rows = it.rows, logn2 = it.logn2, id = local * 64 + threadIdx.x;
    if (id >= rows << logn2) return;
    const unsigned pos = id / rows, row = id % rows;
    if (it.rowflag && it.rowflag[(size_t)row * it.flag_stride]) return;  // written by k_ref_rows
    g1q p;
    pt_load(p, it.D + ((size_t)pos * rows + row) * 36);
    const unsigned fmt = it.out_format;
    const size_t slot = (size_t)row * (1u << logn2) + ((fmt & 1u) ? pos : bitrev(pos, logn2));
    if (fmt & 2u) {
        uint32_t w[12];
        g1q_compress(w, p);
        st_words(it.h_fft + slot * 12, w, 3);
    } else {
        uint32_t w[36] = {0};
        fq x, y;
        if (g1q_to_affine(x, y, p)) {
            fq_to_std(w, x);
            fq_to_std(w + 12, y);
            w[24] = 1;
        } else {
            w[12] = 1;
        }
        st_words(it.h_fft + slot * G1P_WORDS, w, 9);
    }
}

// ---------------------------------------------------------------- launchers

// a fill kernel, not hipMemsetAsync: callers may capture these launches into a graph
static void launch_clear_flags(uint32_t *flags, size_t groups, hipStream_t s) {
    hipLaunchKernelGGL(k_fill_u32, dim3((unsigned)((groups + 255) / 256)), dim3(256), 0, s, flags, groups, 0u);
}

hipError_t launch_subgroup_groups(uint32_t *flags, const uint32_t *pts, size_t count, size_t per_group,
                                  hipStream_t s) {
    if (!count || !per_group) return hipSuccess;
    launch_clear_flags(flags, (count + per_group - 1) / per_group, s);
    // two lanes per point while no SIMD gets a second wave
    if (count <= 32 * PAIR_WAVES)
        hipLaunchKernelGGL(k_subgroup_pair, dim3((unsigned)((count + 31) / 32)), dim3(64), 0, s, flags, pts, count,
                           per_group);
    else
        hipLaunchKernelGGL(k_subgroup_groups, dim3((unsigned)((count + 63) / 64)), dim3(64), 0, s, flags, pts, count,
                           per_group);
    return hipGetLastError();
}

hipError_t launch_scale_bases(uint32_t *xs, uint32_t *inf, const uint32_t *xext, size_t count,
                              const uint32_t *scale, hipStream_t s) {
    hipLaunchKernelGGL(k_scale_bases, dim3((unsigned)((count + 63) / 64)), dim3(64), 0, s, xs, inf, xext, count,
                       scale);
    return hipGetLastError();
}

hipError_t launch_table_build(uint32_t *table, uint32_t *zt, const uint32_t *xs, const uint32_t *inf,
                              uint32_t *err, unsigned base0, unsigned nb, unsigned win_bits, unsigned nwin,
                              hipStream_t s) {
    const unsigned threads = nb * nwin;
    hipLaunchKernelGGL(k_table_build, dim3((threads + 63) / 64), dim3(64), 0, s, table, zt, xs, inf, err, base0,
                       nb, win_bits, nwin);
    return hipGetLastError();
}

// Lanes per row and coefficients per lane of k_commit_partial: no idle lanes below 64 rows, then
// the chunk with the fewest additions one after the other (20 windows per coefficient; larger
// chunks where it does not matter, for fewer partial sums) of those whose partial sums fit in `bytes`.
struct CommitShape {
    unsigned lp, chunk, nparts;
};
static CommitShape commit_shape(unsigned rows, unsigned N, size_t bytes) {
    CommitShape best{1, 16, N / 16};
    unsigned lp = 1, time = ~0u;
    while (lp < 64 && rows * lp * 2 <= 64) lp *= 2;
    for (unsigned chunk = 16; chunk * lp >= 4 && chunk >= 1; chunk /= 2) {
        const unsigned nparts = N / (chunk * lp), per_wave = 64 / lp;
        if ((size_t)nparts * rows * 144 > bytes) break;
        const size_t waves = (size_t)((rows + per_wave - 1) / per_wave) * nparts;
        unsigned close = (nparts + 63) / 64 + 6;
        for (unsigned l = lp; l > 1; l /= 2) close++;
        const unsigned t = add_rounds(waves, chunk * 20) + close;
        if (t < time) time = t, best = CommitShape{lp, chunk, nparts};
    }
    return best;
}

// a partial sum per 16 coefficients and per 256
size_t commit_workspace_bytes(unsigned rows, unsigned N) { return (size_t)(N / 16 + (N + 255) / 256) * rows * 144; }

// What `rows` rows, and every smaller number of them, are fastest in: rows that share lanes or a
// launch's waves want the same number of partial sums, so the last of each such range decides.
size_t commit_wanted_bytes(unsigned rows, unsigned N) {
    size_t want = commit_workspace_bytes(rows, N);
    for (unsigned r = 1;; r = r < 64 ? r + 1 : r + 64) {
        r = std::min(r, rows);
        want = std::max(want, (size_t)commit_shape(r, N, ~(size_t)0).nparts * r * 144);
        if (r >= rows) return want;
    }
}

hipError_t launch_commit(uint32_t *out, const uint32_t *poly, const uint32_t *table, const uint32_t *inf,
                         uint32_t *work, size_t work_bytes, unsigned rows, unsigned N, unsigned win_bits,
                         hipStream_t s) {
    if (!rows) return hipSuccess;
    const CommitShape c = commit_shape(rows, N, work_bytes);
    const unsigned per_wave = 64 / c.lp, rg = (rows + per_wave - 1) / per_wave;
    hipLaunchKernelGGL(k_commit_partial, dim3(c.nparts * rg), dim3(64), 0, s, poly, table, inf, work, rows, N, win_bits,
                       c.chunk, c.lp);
    hipLaunchKernelGGL(k_commit_reduce, dim3(rows), dim3(64), 0, s, work, out, rows, c.nparts);
    return hipGetLastError();
}

// Lanes per row of the MSM over the items of L (k_msm_multi): the fewest additions one after the
// other, the closing additions across the lanes included.
static unsigned msm_lanes(const Launch &L) {
    unsigned best = 1, time = ~0u;
    for (unsigned lp = 1, close = 0; lp <= 16; lp *= 4, close += 2) {
        size_t waves = 0;
        unsigned adds = 0;
        for (unsigned k = 0; k < L.nitems; k++) {
            const unsigned nwin = (256 + L.item[k].win - 1) / L.item[k].win;
            waves += ((size_t)L.item[k].rows * lp + 63) / 64 << L.item[k].logn2;
            adds = std::max(adds, 16 / lp * nwin + close + close / 4);
        }
        const unsigned t = add_rounds(waves, adds);
        if (t < time) time = t, best = lp;
    }
    return best;
}

// Fills L.blk_end from per-item block counts; returns the total.
static unsigned set_blocks(Launch &L, const unsigned *per_item) {
    unsigned total = 0;
    for (unsigned k = 0; k < L.nitems; k++) {
        total += per_item[k];
        L.blk_end[k] = total;
    }
    return total;
}

// Toeplitz coefficients and their transforms, of every item
static void launch_toeplitz_multi(Launch &L, const DevTables *T, hipStream_t s) {
    unsigned per[MAX_ITEMS];
    for (unsigned k = 0; k < L.nitems; k++) per[k] = L.item[k].rows * 16 >> (9 - L.item[k].logn2);
    unsigned total = set_blocks(L, per);
    if (total > NTT_WIDE_WAVES) {
        hipLaunchKernelGGL(k_toeplitz_fft_multi<false>, dim3(total), dim3(64), 0, s, L, T);
        return;
    }
    for (unsigned k = 0; k < L.nitems; k++) per[k] = L.item[k].rows * 16;
    total = set_blocks(L, per);
    if (total) hipLaunchKernelGGL(k_toeplitz_fft_multi<true>, dim3(total), dim3(256), 0, s, L, T);
}

// ---- direct schedule

size_t direct_product_bytes(const DirectPlan &P, unsigned rows, unsigned logn, unsigned levels) {
    size_t most = 0;
    for (unsigned kind = 0; kind < DIRECT_KINDS; kind++)
        for (unsigned s = 0; s < levels; s++)
            most = std::max<size_t>(most, P.rec[direct_record(logn, kind, levels, s)].nprod);
    return most * rows * 144;
}

// Estimated microseconds of the transforms of L's items, measured on MI355X: a round of generic
// ladders takes 870 by pairs of lanes if these need at most one wave per SIMD, else 1100 when
// each SIMD has at most one wave, 2050 per pair of waves and 1250 for an odd one after them, one
// of w^128 ladders 360, 660 and 400; a launch of additions 55 (a direct step has two), a butterfly
// launch 25.  The choice only depends on the items' sizes and rows, and the levels
// whose products the workspace holds.
unsigned direct_choose(const Launch &L, const DirectPlan &P, bool both, unsigned allowed) {
    if (!P.rec) return 0;
    unsigned lmax = 0;
    for (unsigned k = 0; k < L.nitems; k++) {
        lmax = std::max(lmax, L.item[k].logn2);
        if (L.item[k].rows > DIRECT_MAX_ROWS) return 0;
    }
    auto rounds = [](unsigned waves, unsigned one, unsigned pair, unsigned odd) {
        const unsigned c = (waves + 1023) / 1024;
        return c == 1 ? one : c / 2 * pair + c % 2 * odd;
    };
    // radix 2^2: per transform, the layers (odd stages) and the w^128 of the even ones
    unsigned best = 0, time = 0;
    for (unsigned sd = 0; sd < lmax; sd++) {
        unsigned layer = 0, quarter = 0;
        for (unsigned k = 0; k < L.nitems; k++) {
            const unsigned logn = L.item[k].logn2, rg = (L.item[k].rows + 63) / 64;
            if ((sd & 1) && sd < logn) layer += layer_count(sd, logn) * rg;
            if (!(sd & 1) && sd + 1 < logn) quarter += (1u << (logn - 2)) * rg;
        }
        time += 25 + rounds(layer, 1100, 2050, 1250) + rounds(quarter, 360, 660, 400);
    }
    if (both) time *= 2;
    for (unsigned levels = 1; levels <= DIRECT_MAX_STEPS; levels++) {
        if (!(allowed >> levels & 1)) continue;
        unsigned t = 0;
        for (unsigned half = 0; half < (both ? 2u : 1u); half++)
            for (unsigned s = 0; s < levels; s++) {
                unsigned waves = 0, pairs = 0;
                for (unsigned k = 0; k < L.nitems; k++) {
                    const DirectStep &st = P.rec[direct_record(L.item[k].logn2, both ? half : (unsigned)DIRECT_FFT, levels, s)];
                    waves += direct_parts(st, L.item[k].rows, 6).waves;
                    pairs += direct_parts(st, L.item[k].rows, 5).waves;
                }
                t += (levels == 1 ? 190 : 110) +
                     (pairs <= PAIR_WAVES ? 870 : rounds(waves, 1100, 2050, 1250));
            }
        if (t < time) time = t, best = levels;
    }
    return best;
}

// One transform of every item in the direct schedule.
static void launch_direct(Launch &L, const DirectPlan &P, unsigned levels, unsigned kind, const uint32_t *ops,
                          const uint32_t *index, const StageKernels &K, hipStream_t s, const LaunchHook &hook) {
    unsigned per[MAX_ITEMS];
    const int add = kind == DIRECT_FFT_HALF || kind == DIRECT_FFT ? LK_DIF : LK_DIT;
    for (unsigned step = 0; step < levels; step++) {
        auto blocks = [&](auto &&count) {
            for (unsigned k = 0; k < L.nitems; k++) {
                const unsigned rec = direct_record(L.item[k].logn2, kind, levels, step);
                L.item[k].stage = (int)rec;
                per[k] = count(L.item[k], P.rec[rec]);
            }
            return set_blocks(L, per);
        };
        unsigned total;
        // the items' steps are of one kind (a single step or the same number of them), so of the
        // same number of passes, but for a second pass that only radix 128 and up have
        for (unsigned pass = 0; pass < (levels == 1 ? 2u : 1u); pass++) {
            total = blocks([&](const Item &it, const DirectStep &st) {
                const unsigned loga = direct_split_log(st.loga, pass), logN = st.loga + st.logb;
                const unsigned groups = it.rows << (st.logblocks + (pass == 0 ? logN - loga : st.logb));
                return ((groups << loga) + 63) / 64;
            });
            hipLaunchKernelGGL(k_direct_split, dim3(total), dim3(64), 0, s, L, P.words, pass);
            hook(add);
        }
        unsigned max_lr = 5;
        auto waves = [&](Item &it, const DirectStep &st) {
            const DirectParts d = direct_parts(st, it.rows, max_lr);
            it.parts = d.parts;
            return d.waves;
        };
        total = blocks(waves);
        const bool pair = total <= PAIR_WAVES;
        if (!pair) {
            max_lr = 6;
            total = blocks(waves);
        }
        hipLaunchKernelGGL(pair ? K.direct_pair : K.direct, dim3(total), dim3(64), 0, s, L, P.words, ops, index);
        hook(LK_TWIDDLE);
        total = blocks([](const Item &it, const DirectStep &st) { return ((st.nout * it.rows << st.log_lanes) + 63) / 64; });
        hipLaunchKernelGGL(k_direct_sums, dim3(total), dim3(64), 0, s, L, P.words);
        hook(add);
    }
}

// Resident waves of k_chain: two per SIMD on 256 CUs.
static constexpr unsigned CHAIN_WAVES = 2048;

hipError_t launch_batch(const Launch &base, const DevTables *T, const uint32_t *ops, const uint32_t *index,
                        const StageKernels &K, hipStream_t s, LaunchHook hook, uint32_t *chain,
                        uint64_t chain_wait, const DirectPlan &direct, unsigned levels) {
    if (chain && !K.chain) return hipErrorInvalidValue;
    Launch L = base;
    unsigned per[MAX_ITEMS], lmax = 0, total;
    for (unsigned k = 0; k < L.nitems; k++) lmax = std::max(lmax, L.item[k].logn2);
    if (chain) {
        Chain C;
        memset(&C, 0, sizeof C);
        C.L = L;
        C.ctl = chain;
        hipLaunchKernelGGL(k_chain_reset, dim3(L.nitems), dim3(256), 0, s, C);
    }
    // Toeplitz + NTT
    launch_toeplitz_multi(L, T, s);
    hook(LK_TOEPLITZ_FFT);
    // MSM
    const unsigned lp = msm_lanes(L);
    for (unsigned k = 0; k < L.nitems; k++) per[k] = ((L.item[k].rows * lp + 63) / 64) << L.item[k].logn2;
    total = set_blocks(L, per);
    if (total) hipLaunchKernelGGL((lp == 1 ? k_msm_multi<1> : lp == 4 ? k_msm_multi<4> : k_msm_multi<16>), dim3(total),
                                  dim3(64), 0, s, L);
    hook(LK_MSM);
    // transform stages: global stage t = 0 .. 2*lmax - 2; item k (L = logn2) runs local stage
    // u = t - (lmax - L) while 0 <= u <= 2L - 2 (DIT right-aligned to the middle at t = lmax-1,
    // DIF left-aligned after it)
    const unsigned nt = 2 * lmax - 1;
    if (chain) {
        Chain C;
        memset(&C, 0, sizeof C);
        C.L = L;
        C.ctl = chain;
        C.wait_ticks = chain_wait;
        C.nstages = nt;
        unsigned acc = 0;
        for (unsigned t = 0; t < nt; t++) {
            unsigned in_stage = 0;
            for (unsigned k = 0; k < L.nitems; k++) {
                const Item &it = L.item[k];
                const int u = t < lmax - 1 ? (int)t - (int)(lmax - it.logn2)
                            : (int)it.logn2 - 1 + (int)(t - (lmax - 1));
                const bool live = t < lmax - 1 ? u >= 0 : u <= (int)(2 * it.logn2 - 2);
                C.ustage[t][k] = (int8_t)(live ? u : -1);
                in_stage += live ? (1u << (it.logn2 - 1)) * ((it.rows + 63) / 64) : 0;
                C.blk_end[t][k] = in_stage;
            }
            acc += in_stage;
            C.t_end[t] = acc;
        }
        C.total = acc;
        if (acc) hipLaunchKernelGGL(K.chain, dim3(std::min(acc, CHAIN_WAVES)), dim3(64), 0, s, C, ops, index);
        hook(LK_CHAIN);
    } else if (levels) {
        launch_direct(L, direct, levels, DIRECT_IFFT_HALF, ops, index, K, s, hook);
        launch_direct(L, direct, levels, DIRECT_FFT_HALF, ops, index, K, s, hook);
    } else {
        // one launch per stage; IFFT DIT stages right-aligned to the middle launch.  In the
        // radix-2^2 schedule a DIT stage whose transposed DIF stage is odd is preceded by that
        // stage's twiddle layer.
        for (unsigned t = 0; t + 1 < lmax; t++) {
            for (unsigned k = 0; k < L.nitems; k++) {
                const Item &it = L.item[k];
                const int st = (int)t - (int)(lmax - it.logn2);
                const unsigned sd = it.logn2 - 1 - (unsigned)st;
                const bool layer = K.r22 && st >= 0 && (sd & 1) && layer_count(sd, it.logn2);
                L.item[k].stage = layer ? (int)sd : -1;
                per[k] = layer ? layer_count(sd, it.logn2) * ((it.rows + 63) / 64) : 0;
            }
            total = set_blocks(L, per);
            if (total) {
                hipLaunchKernelGGL(K.twiddle, dim3(total), dim3(64), 0, s, L, ops, index, (unsigned)TW_INV);
                hook(LK_TWIDDLE);
            }
            for (unsigned k = 0; k < L.nitems; k++) {
                const int st = (int)t - (int)(lmax - L.item[k].logn2);
                L.item[k].stage = st;
                per[k] = st >= 0 ? (1u << (L.item[k].logn2 - 1)) * ((L.item[k].rows + 63) / 64) : 0;
            }
            total = set_blocks(L, per);
            if (total) hipLaunchKernelGGL(K.dit, dim3(total), dim3(64), 0, s, L, ops, index);
            hook(LK_DIT);
        }
        for (unsigned k = 0; k < L.nitems; k++) {
            L.item[k].stage = 0;
            per[k] = (1u << (L.item[k].logn2 - 1)) * ((L.item[k].rows + 63) / 64);
        }
        total = set_blocks(L, per);
        if (total) hipLaunchKernelGGL(K.middle, dim3(total), dim3(64), 0, s, L, ops, index);
        hook(LK_MIDDLE);
        // FFT DIF stages 1.., left-aligned after the middle launch
        for (unsigned t = 1; t < lmax; t++) {
            for (unsigned k = 0; k < L.nitems; k++) {
                const int st = t < L.item[k].logn2 ? (int)t : -1;
                L.item[k].stage = st;
                per[k] = st >= 0 ? (1u << (L.item[k].logn2 - 1)) * ((L.item[k].rows + 63) / 64) : 0;
            }
            total = set_blocks(L, per);
            if (total) hipLaunchKernelGGL(K.dif, dim3(total), dim3(64), 0, s, L, ops, index);
            hook(LK_DIF);
            // even DIF stages (radix-2^2): their w^128 twiddles, on the second half's outputs
            for (unsigned k = 0; k < L.nitems; k++) {
                const Item &it = L.item[k];
                const bool q = K.r22 && t + 1 < it.logn2 && (t & 1) == 0;
                L.item[k].stage = q ? (int)t : -1;
                per[k] = q ? (1u << (it.logn2 - 2)) * ((it.rows + 63) / 64) : 0;
            }
            total = set_blocks(L, per);
            if (total) {
                hipLaunchKernelGGL(K.quarter, dim3(total), dim3(64), 0, s, L);
                hook(LK_DIF);
            }
            // odd DIF stages: their twiddle layer (radix-2^2)
            for (unsigned k = 0; k < L.nitems; k++) {
                const Item &it = L.item[k];
                const bool layer = K.r22 && t < it.logn2 && (t & 1) && layer_count(t, it.logn2);
                L.item[k].stage = layer ? (int)t : -1;
                per[k] = layer ? layer_count(t, it.logn2) * ((it.rows + 63) / 64) : 0;
            }
            total = set_blocks(L, per);
            if (total) {
                hipLaunchKernelGGL(K.twiddle, dim3(total), dim3(64), 0, s, L, ops, index, (unsigned)TW_FWD);
                hook(LK_TWIDDLE);
            }
        }
    }
    // output
    for (unsigned k = 0; k < L.nitems; k++) per[k] = ((L.item[k].rows << L.item[k].logn2) + 63) / 64;
    total = set_blocks(L, per);
    if (total) hipLaunchKernelGGL(k_output_multi, dim3(total), dim3(64), 0, s, L);
    hook(LK_OUTPUT);
    return hipGetLastError();
}

// The drop-in transforms as one item of the batched launches: the DIT stage kernel runs
// IFFT stages 0 .. L-1 (the last one through the middle's positions), the DIF kernel FFT
// stages 0 .. L-1 (the first likewise), and the output kernel writes natural order from the
// DIF's bit-reversed positions (format 0) or position by position (format 1).
hipError_t launch_plain(PlainKind kind, uint32_t *out, const uint32_t *in, const uint32_t *xpk, unsigned rows,
                        unsigned logn, uint32_t *D, uint32_t *tcT, void *msm_work, size_t msm_bytes, uint32_t *flags,
                        const DevTables *T, const Programs &P, hipStream_t s, const DirectPlan &direct, uint32_t *products,
                        size_t product_bytes) {
    if (!rows) return hipSuccess;
    Launch L;
    memset(&L, 0, sizeof L);
    L.nitems = 1;
    Item &it = L.item[0];
    it.poly = in;
    it.h_fft = out;
    it.tcT = tcT;
    it.D = D;
    it.rows = rows;
    it.N = 8u << logn;
    it.logn2 = logn;
    it.scale_tc = 1;
    it.rowflag = flags;
    it.flag_stride = kind == PLAIN_POLY2H_FFT ? 0 : 1;
    const unsigned rg = (rows + 63) / 64, n = 1u << logn;
    unsigned per[MAX_ITEMS] = {};
    const uint32_t *scale = P.ops + P.scale_off[logn];
    const StageKernels &K = default_stage_kernels();  // radix-2^2, built for P's width
    // small batches: the direct schedule, as many levels as the workspace holds products for
    it.P = products;
    const bool both = kind == PLAIN_HEXT_FFT2H_FFT || kind == PLAIN_POLY2H_FFT;
    unsigned levels = 0;
    if (rows <= DIRECT_MAX_ROWS) {
        unsigned allowed = 0;
        for (unsigned l = 1; l <= DIRECT_MAX_STEPS; l++)
            if (direct_product_bytes(direct, rows, logn, l) <= product_bytes) allowed |= 1u << l;
        levels = direct_choose(L, direct, both, allowed);
    }
    // rows holding a point outside G1 are recomputed by k_ref_rows: the transform kinds check
    // their inputs as they load them, one flag per row; PLAIN_POLY2H_FFT's caller has set
    // flags[0] from the bases, which every row's MSM output combines
    auto load = [&](unsigned brev, const uint32_t *scale) {
        launch_clear_flags(flags, rows, s);
        const size_t pairs = (size_t)n * ((rows + 31) / 32) + ((size_t)rows * n + 31) / 32;
        const bool pair = pairs <= PAIR_WAVES;
        hipLaunchKernelGGL(pair ? K.plain_load_pair : K.plain_load,
                           dim3(pair ? (unsigned)pairs : n * rg + (rows * n + 63) / 64), dim3(64), 0, s, D, in, rows, logn,
                           brev, scale, flags);
    };
    auto run_direct = [&](unsigned k) {
        launch_direct(L, direct, levels, k, P.ops, P.index, K, s, LaunchHook{nullptr, nullptr});
    };
    // radix-2^2 twiddle layers (see stage_positions): DIF stage t's after its butterflies,
    // the transposed DIF stage's before DIT stage t
    auto layer = [&](unsigned sd, unsigned dir) {
        const unsigned cnt = (sd & 1) ? layer_count(sd, logn) : 0;
        if (!cnt) return;
        it.stage = (int)sd;
        per[0] = cnt * rg;
        hipLaunchKernelGGL(K.twiddle, dim3(set_blocks(L, per)), dim3(64), 0, s, L, P.ops, P.index, dir);
    };
    auto stage = [&](void (*kernel)(Launch, const uint32_t *, const uint32_t *), int st) {
        const bool dit = kernel == K.dit, dif = kernel == K.dif;
        if (dit) layer(logn - 1 - (unsigned)st, (unsigned)TW_INV);
        it.stage = st;
        per[0] = n / 2 * rg;
        const unsigned total = set_blocks(L, per);
        hipLaunchKernelGGL(kernel, dim3(total), dim3(64), 0, s, L, P.ops, P.index);
        if (dif && (st & 1) == 0 && (unsigned)st + 1 < logn) {  // its w^128 twiddles
            per[0] = (n / 4) * rg;
            hipLaunchKernelGGL(K.quarter, dim3(set_blocks(L, per)), dim3(64), 0, s, L);
        }
        if (dif) layer((unsigned)st, (unsigned)TW_FWD);
    };
    switch (kind) {
    case PLAIN_G1_FFT:
        load(0u, nullptr);
        if (levels) run_direct(DIRECT_FFT);
        else for (unsigned t = 0; t < logn; t++) stage(K.dif, (int)t);
        break;
    case PLAIN_G1_IFT:
        load(1u, scale);
        if (levels) run_direct(DIRECT_IFFT);
        else for (unsigned t = 0; t < logn; t++) stage(K.dit, (int)t);
        it.out_format = 1;
        break;
    case PLAIN_HEXT_FFT2H_FFT:
    case PLAIN_POLY2H_FFT:
        if (kind == PLAIN_HEXT_FFT2H_FFT) {
            load(1u, scale);
        } else {
            launch_toeplitz_multi(L, T, s);
            hipError_t e = launch_msm_plain_T(D, tcT, xpk, msm_work, msm_bytes, rows, n, s);
            if (e != hipSuccess) return e;
            // rows of a setup outside G1 take the reference's order from the MSM output on,
            // with tcT (no longer read) as their workspace
            hipLaunchKernelGGL(k_ref_rows, dim3(rows), dim3(256), 0, s, 2u, out, (const uint32_t *)nullptr,
                               (const uint32_t *)D, rows, logn, tcT, (const uint32_t *)flags, 0u, T);
        }
        if (levels) {
            run_direct(DIRECT_IFFT_HALF);
            run_direct(DIRECT_FFT_HALF);
            break;
        }
        for (unsigned t = 0; t + 1 < logn; t++) stage(K.dit, (int)t);
        stage(K.middle, 0);
        for (unsigned t = 1; t < logn; t++) stage(K.dif, (int)t);
        break;
    }
    per[0] = (n * rows + 63) / 64;
    hipLaunchKernelGGL(k_output_multi, dim3(set_blocks(L, per)), dim3(64), 0, s, L);
    // flagged rows of the transform kinds: their input rows are intact (the output kernel
    // skipped them, so an aliased output has not overwritten them) and D is free as workspace
    if (kind != PLAIN_POLY2H_FFT)
        hipLaunchKernelGGL(k_ref_rows, dim3(rows), dim3(256), 0, s,
                           kind == PLAIN_G1_FFT ? 0u : kind == PLAIN_G1_IFT ? 1u : 2u, out, in,
                           (const uint32_t *)nullptr, rows, logn, D, (const uint32_t *)flags, 1u, T);
    return hipGetLastError();
}

}  // namespace fk20
