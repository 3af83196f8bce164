// The direct schedule of the column-batched G1 transforms, for batches too small to fill the
// chip: fewer ladders in a row, more of them side by side.
//
// A twiddle ladder takes about as long on an idle chip as on a busy one, so a small batch's
// transform lasts the number of ladders on its longest path: four generic and four w^128 ones
// per transform of 512 in the radix-2^2 schedule (schedule.hip.h).  Here a transform is one to
// three mixed-radix steps, each of them one round of ladders.  A step of radix a on blocks of
// N = a b points computes
//     Y[j][m] = sum_t w_N^(j (m + b t)) X[m + b t],     j, t < a, m < b,
// (the twiddles of the next step included), in three launches:
//  * k_direct_split, in place: for every m the a points become the sum of all, the difference of
//    the two halves' sums, .., the a/2 differences X[t] - X[t + a/2]: log2(a) additions by a
//    lanes at once (radix above 32: two launches, the second on the sums that are left).  Output j with j = 2^v odd only needs the a / 2^(v+1) differences of level v.
//  * k_direct_products: one ladder per distinct (point, exponent) into P[slot][row]; exponents
//    are taken below 256 (w^256 = -1), and all products of one exponent are next to each other,
//    so a wave runs one program over several points times the batch's rows.
//  * k_direct_sums: every output adds its a / 2^(v+1) products.
// The blocks' size-b transforms follow with root w_N^a.  Radix 16 takes 5.3 ladders per point,
// a last step of radix 32 3.5, a single step 57 for 512 points and 14 for 128 (radix-2^2: 2.3 and
// 1.2 short ones per point, in eight rounds).
//
// Shared by the kernels, the launchers and, compiled by g++, the CPU tests.
#pragma once
#include <stdint.h>

#ifndef FK20_HD
#define FK20_HD __host__ __device__ __forceinline__
#endif

namespace fk20 {

// Which transform: the batched path's halves (hext_fft in bit-reversed order -> h, its n/2
// coefficients in natural order; h -> h_fft at bit-reversed positions) and the whole transforms
// of the drop-ins (in the positions their load and output kernels use).
enum DirectKind { DIRECT_IFFT_HALF = 0, DIRECT_FFT_HALF = 1, DIRECT_FFT = 2, DIRECT_IFFT = 3 };
static constexpr unsigned DIRECT_KINDS = 4;
// levels 1: [n]; levels 2: [16, 32], [16, 16], [8, 16] for n = 512, 256, 128; levels 3: [8, 8, 8], [4, 8, 8],
// [4, 4, 8]
static constexpr unsigned DIRECT_MAX_STEPS = 3;

// log2 of the lanes that up to 64 rows take
FK20_HD unsigned direct_row_lanes(unsigned rows) {
    unsigned lr = 0;
    while (lr < 6 && (1u << lr) < rows) lr++;
    return lr;
}

FK20_HD unsigned direct_radix_log(unsigned logn, unsigned levels, unsigned step) {
    if (levels == 1) return logn;
    if (levels == 2) return step == 0 ? (logn == 7 ? 3u : 4u) : (logn == 9 ? 5u : 4u);
    return step == 0 ? (logn == 9 ? 3u : 2u) : step == 1 ? (logn == 7 ? 2u : 3u) : 3u;
}

// A step's record in the plan words: counts, then offsets (from the plan words' start).
struct DirectStep {
    uint32_t loga, logb, logblocks;  // radix, stride, number of blocks (log2)
    uint32_t in_map;                 // bit 0: position of index i is bitrev(i); bit 1: upper half zero
    uint32_t log_lanes, sum_words;   // lanes per output of the sums (log2), words per output
    uint32_t nprod, prod;            // products: position | exponent << 16, in slot order
    uint32_t nout, sums;             // outputs
    uint32_t nwaves[7], waves[7];    // for 2^k products per wave: first slot | count << 16 (k = 0..6)
};
// How the waves of a step cover `rows` rows, 2^max_lr lanes or pairs of lanes a wave (6, or 5 with
// two lanes per ladder): groups of 2^max_lr rows of one product each, and the rows left over in
// parts of 2^lr rows, up to 2^(max_lr - lr) products of one exponent a wave.  `parts` has a bit for each
// part's lr, the largest first; the last one may be partly empty.  Of 100 rows a wave takes 64 of
// one product, 32 of two or 4 of sixteen.  With one part for all of the rest, 40 rows of N = 4096
// took 12.4 ms, now 8.5, 40 of N = 2048 6.0 and 5.2; 72 and 100 rows are the same.
struct DirectParts {
    unsigned waves, parts;
};
// The fewest waves for `rest` rows in parts below 2^limit: one part, or the largest that is full and
// the same for what is left (a part costs at least a wave per exponent).
FK20_HD DirectParts direct_rest(const DirectStep &st, unsigned rest, unsigned max_lr, unsigned limit) {
    DirectParts best{0, 0}, done{0, 0};
    bool have = rest == 0;
    while (rest) {
        const unsigned lr = direct_row_lanes(rest);
        if (lr < limit) {
            const unsigned w = done.waves + st.nwaves[max_lr - lr];
            if (!have || w < best.waves) best = DirectParts{w, done.parts | 1u << lr}, have = true;
        }
        unsigned top = lr;
        if ((1u << top) > rest) top--;
        done.waves += st.nwaves[max_lr - top];
        done.parts |= 1u << top;
        rest -= 1u << top;
        limit = top;
    }
    return best;
}
FK20_HD DirectParts direct_parts(const DirectStep &st, unsigned rows, unsigned max_lr) {
    const unsigned full = rows >> max_lr;
    DirectParts d = direct_rest(st, rows - (full << max_lr), max_lr, max_lr + 1);
    d.waves += st.nwaves[0] * full;
    return d;
}
// What wave `local` of them does: row0 + the lane's index below 2^lr, product word w
struct DirectWave {
    unsigned row0, last, lr;  // last: the last row among them
    uint32_t w;
};
FK20_HD DirectWave direct_wave(const DirectStep &st, const uint32_t *plan, unsigned rows, unsigned max_lr,
                               unsigned parts, unsigned local) {
    const unsigned full = rows >> max_lr, main = st.nwaves[0] * full;
    DirectWave r;
    if (local < main) {
        r.lr = max_lr;
        r.row0 = (local % full) << max_lr;
        r.w = plan[st.waves[0] + local / full];
    } else {
        local -= main;
        r.row0 = full << max_lr;
        r.lr = max_lr;
        while (r.lr && (!(parts >> r.lr & 1u) || local >= st.nwaves[max_lr - r.lr])) {
            if (parts >> r.lr & 1u) {
                local -= st.nwaves[max_lr - r.lr];
                r.row0 += 1u << r.lr;
            }
            r.lr--;
        }
        r.w = plan[st.waves[max_lr - r.lr] + local];
    }
    r.last = r.row0 + (1u << r.lr) - 1;
    if (r.last >= rows) r.last = rows - 1;
    return r;
}
static constexpr unsigned DIRECT_STEP_WORDS = sizeof(DirectStep) / 4;
// an output's words: its position, three unused, then its terms: slot | sign << 31, DIRECT_NONE
// past the last, to the step's longest sum rounded up to a multiple of the lanes
static constexpr unsigned DIRECT_SUM_FIRST = 4;
// The split of radix a = 2^loga and stride 2^logb in passes of at most 32 points: pass 0 takes
// up to 5 levels, pass 1 the rest on the sums it leaves, at the lowest 2^(loga + logb - 5) indices.
FK20_HD unsigned direct_split_log(unsigned loga, unsigned pass) {
    return pass == 0 ? (loga > 5 ? 5 : loga) : loga - 5;
}
static constexpr uint32_t DIRECT_NONE = 0xffffffffu;
// index of the step record of (logn, kind, levels, step) in the record table at the words' start
FK20_HD unsigned direct_record(unsigned logn, unsigned kind, unsigned levels, unsigned step) {
    return (((logn - 7) * DIRECT_KINDS + kind) * DIRECT_MAX_STEPS + (levels - 1)) * DIRECT_MAX_STEPS + step;
}
static constexpr unsigned DIRECT_RECORDS = 3 * DIRECT_KINDS * DIRECT_MAX_STEPS * DIRECT_MAX_STEPS;

}  // namespace fk20

// ---------------------------------------------------------------- host: the plans

#include <algorithm>
#include <cstring>
#include <vector>

namespace fk20 {

inline unsigned direct_bitrev(unsigned x, unsigned bits) {
    unsigned r = 0;
    for (unsigned i = 0; i < bits; i++) r |= ((x >> i) & 1u) << (bits - 1 - i);
    return r;
}

// Appends one step's tables to `words` and returns its record.  order: the exponents e < 256 as they
// are handed out.  slot: DIRECT_NONE for every (position << 8 | exponent), and left so.
inline DirectStep direct_build_step(std::vector<uint32_t> &words, unsigned logn, unsigned kind, unsigned levels,
                                    unsigned step, const unsigned *order, std::vector<uint32_t> &slot) {
    const unsigned steps = levels, n = 1u << logn;
    const bool inverse = kind == DIRECT_IFFT_HALF || kind == DIRECT_IFFT;
    unsigned logdone = 0;
    for (unsigned s = 0; s < step; s++) logdone += direct_radix_log(logn, levels, s);
    DirectStep r;
    memset(&r, 0, sizeof r);
    r.loga = direct_radix_log(logn, levels, step);
    r.logb = logn - logdone - r.loga;
    r.logblocks = logdone;
    const bool last = step + 1 == steps;
    r.in_map = step == 0 ? (inverse ? 1u : 0u) | (kind == DIRECT_FFT_HALF ? 2u : 0u) : 0u;
    const unsigned a = 1u << r.loga, b = 1u << r.logb, N = a * b;
    unsigned position[512];
    for (unsigned i = 0; i < n; i++) position[i] = (r.in_map & 1u) ? direct_bitrev(i, logn) : i;

    struct Out {
        unsigned pos, first, terms;  // terms in `terms`: position << 8 | exponent | sign << 31
    };
    std::vector<Out> outs;
    std::vector<uint32_t> terms;
    std::vector<unsigned> keys, of[256];  // the products, and by exponent
    for (unsigned blk = 0; blk < (1u << r.logblocks); blk++)
        for (unsigned j = 0; j < a; j++) {
            // output index of this block's Y[j][0]: the digits so far, least significant first
            unsigned k = 0, shift = 0;
            for (unsigned s = 0, rem = blk, left = logdone; s < step; s++) {
                const unsigned ls = direct_radix_log(logn, levels, s);
                left -= ls;
                k |= (rem >> left) << shift;
                rem &= (1u << left) - 1;
                shift += ls;
            }
            k |= j << shift;
            if (last && kind == DIRECT_IFFT_HALF && k >= n / 2) continue;
            for (unsigned m = 0; m < b; m++) {
                Out o;
                o.first = (unsigned)terms.size();
                if (!last) o.pos = ((blk << r.loga | j) << r.logb) | m;
                else o.pos = kind == DIRECT_FFT || kind == DIRECT_FFT_HALF ? direct_bitrev(k, logn) : k;
                // level v differences: positions t in [a >> (v+1), a >> v) of the split array;
                // j = 0: the total at t = 0
                unsigned lo = 0, hi = 1;
                if (j) {
                    const unsigned v = (unsigned)__builtin_ctz(j);
                    lo = a >> (v + 1);
                    hi = a >> v;
                }
                for (unsigned t = lo; t < hi; t++) {
                    unsigned e = (j * (m + b * (t - lo)) & (N - 1)) * (512 / N);
                    if (inverse) e = (512 - e) & 511u;
                    const unsigned p = position[blk * N + m + b * t];
                    const unsigned key = p << 8 | (e & 255u);
                    terms.push_back(key | (e >> 8) << 31);
                    if (slot[key] == DIRECT_NONE) {
                        slot[key] = 0;
                        of[e & 255u].push_back(key);
                    }
                }
                o.terms = (unsigned)terms.size() - o.first;
                outs.push_back(o);
            }
        }
    // slots: all products of one exponent together
    for (unsigned k = 0; k < 256; k++) {
        std::vector<unsigned> &v = of[order[k]];
        std::sort(v.begin(), v.end());
        keys.insert(keys.end(), v.begin(), v.end());
    }
    r.nprod = (uint32_t)keys.size();
    r.prod = (uint32_t)words.size();
    for (unsigned i = 0; i < keys.size(); i++) {
        slot[keys[i]] = i;
        words.push_back(keys[i] >> 8 | (keys[i] & 255u) << 16);
    }
    for (unsigned lk = 0; lk < 7; lk++) {
        r.waves[lk] = (uint32_t)words.size();
        for (unsigned i = 0; i < keys.size();) {
            unsigned c = 1;
            while (i + c < keys.size() && c < (1u << lk) && (keys[i + c] & 255u) == (keys[i] & 255u)) c++;
            words.push_back(i | c << 16);
            i += c;
        }
        r.nwaves[lk] = (uint32_t)words.size() - r.waves[lk];
    }
    r.nout = (uint32_t)outs.size();
    r.sums = (uint32_t)words.size();
    // longest sums first
    std::stable_sort(outs.begin(), outs.end(), [](const Out &x, const Out &y) { return x.terms > y.terms; });
    // 4 lanes per output for up to 16 terms, 64 for a single step's up to 256
    r.log_lanes = a > 32 ? 6 : 2;
    const unsigned lanes = 1u << r.log_lanes;
    r.sum_words = DIRECT_SUM_FIRST + ((outs[0].terms + lanes - 1) & ~(lanes - 1));
    for (const Out &o : outs) {
        const size_t at = words.size();
        words.resize(at + r.sum_words, DIRECT_NONE);
        words[at] = o.pos;
        for (unsigned t = 0; t < o.terms; t++) {
            const uint32_t k = terms[o.first + t];
            words[at + DIRECT_SUM_FIRST + t] = slot[k & 0x7fffffffu] | (k & 0x80000000u);
        }
    }
    for (unsigned k : keys) slot[k] = DIRECT_NONE;
    return r;
}

// Every plan: the record table (DIRECT_RECORDS records), then the records' tables.  cost[e]: ladder
// cost of w^e (e < 256; 0 for e = 0); the dearest are handed out first.
inline void direct_build(std::vector<uint32_t> &words, const int *cost) {
    unsigned order[256];
    for (unsigned e = 0; e < 256; e++) order[e] = e;
    std::stable_sort(order, order + 256, [&](unsigned x, unsigned y) { return cost[x] > cost[y]; });
    std::vector<uint32_t> slot((size_t)512 << 8, DIRECT_NONE);
    words.reserve((size_t)3 << 19);
    words.assign((size_t)DIRECT_RECORDS * DIRECT_STEP_WORDS, 0);
    for (unsigned logn = 7; logn <= 9; logn++)
        for (unsigned kind = 0; kind < DIRECT_KINDS; kind++)
            for (unsigned levels = 1; levels <= DIRECT_MAX_STEPS; levels++)
                for (unsigned s = 0; s < levels; s++) {
                    const DirectStep r = direct_build_step(words, logn, kind, levels, s, order, slot);
                    memcpy(&words[(size_t)direct_record(logn, kind, levels, s) * DIRECT_STEP_WORDS], &r, sizeof r);
                }
}

}  // namespace fk20
