// Fr kernels: Toeplitz coefficient layout, Fr NTT of size 128/256/512, fused Toeplitz+NTT,
// and element-wise Fr arithmetic.
//
// NTT (ntt.hip.h): the same natural-order DFT as fr_fft.cu:28-168 (forward) and
// fr_fft.cu:172-300 (inverse, scaled by 1/n).
#include "common.hip.h"
#include "ntt.hip.h"

namespace fk20 {

// ---------------------------------------------------------------- Toeplitz layout

// tc[row][i][j] from polynomial[row][N] (FK20Py fk20_multi.py:92-93; the CUDA layout of
// fk20_poly2toeplitz_coefficients.cu:40-56 for N = 4096):
//   tc[i][0] = poly[N-1-i], tc[i][1..k+1] = 0, tc[i][k+2+m] = poly[31-i+16m], m = 0..k-3.
__device__ __forceinline__ int toeplitz_src(unsigned i, unsigned j, unsigned N) {
    const unsigned k = N / 16;
    if (j == 0) return (int)(N - 1 - i);
    if (j <= k + 1) return -1;
    return (int)(31 - i + 16 * (j - (k + 2)));
}

__global__ void __launch_bounds__(256) k_toeplitz(uint4 *tc, const uint4 *poly, unsigned rows, unsigned N) {
    const unsigned n2 = N / 8;
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)rows * 16 * n2) return;
    const unsigned j = (unsigned)(e % n2), i = (unsigned)((e / n2) % 16);
    const size_t row = e / (16 * (size_t)n2);
    const int src = toeplitz_src(i, j, N);
    uint4 lo = make_uint4(0, 0, 0, 0), hi = lo;
    if (src >= 0) {
        lo = poly[2 * ((size_t)row * N + src)];
        hi = poly[2 * ((size_t)row * N + src) + 1];
    }
    tc[2 * e] = lo;
    tc[2 * e + 1] = hi;
}

// ---------------------------------------------------------------- transforms

__device__ __forceinline__ void fs_load(fs &a, const uint32_t *p) {
    const uint4 *q = reinterpret_cast<const uint4 *>(p);
    uint4 x = q[0], y = q[1];
    a.l[0] = x.x; a.l[1] = x.y; a.l[2] = x.z; a.l[3] = x.w;
    a.l[4] = y.x; a.l[5] = y.y; a.l[6] = y.z; a.l[7] = y.w;
}

__device__ __forceinline__ void fs_store(uint32_t *p, const fs &a) {
    uint4 *q = reinterpret_cast<uint4 *>(p);
    q[0] = make_uint4(a.l[0], a.l[1], a.l[2], a.l[3]);
    q[1] = make_uint4(a.l[4], a.l[5], a.l[6], a.l[7]);
}

// count transforms; the spare lanes of the last wave repeat the last one (same loads, same stores).
// A transform is read before any of it is written, so out may alias in.
template <unsigned LOGN, bool INV, bool WIDE>
__global__ void __launch_bounds__(WIDE ? (1u << LOGN) / 2 : 64) k_fr_ntt(uint32_t *out, const uint32_t *in,
                                                                        unsigned count, const DevTables *T) {
    constexpr unsigned n = 1u << LOGN, lanes = n / 8;
    __shared__ uint32_t lds[WIDE ? n * 9 : NTT_LDS_WORDS];
    const unsigned sub = threadIdx.x / lanes, t = threadIdx.x % lanes;
    const size_t id = WIDE ? blockIdx.x : min(blockIdx.x * (64 / lanes) + sub, count - 1);
    const uint32_t *src = in + id * n * FR_WORDS;
    uint32_t *dst = out + id * n * FR_WORDS;
    const auto load = [&](unsigned i, fn &x) {
        fs a;
        fs_load(a, src + (size_t)i * FR_WORDS);
        fn_unpack(x, a.l);
    };
    const auto store = [&](unsigned k, const uint32_t *w) {
        fs a;
        fs_set(a, w);
        fs_store(dst + (size_t)k * FR_WORDS, a);
    };
    if constexpr (WIDE) ntt_wide<LOGN, INV>(lds, INV ? LOGN : 0, T, load, store);
    else ntt<LOGN, INV>(lds + sub * n * 9, t, INV ? LOGN : 0, T, load, store);
}

// The Toeplitz coefficients of (row, i) straight into the transform.
template <unsigned LOGN, bool WIDE>
__global__ void __launch_bounds__(WIDE ? (1u << LOGN) / 2 : 64) k_toeplitz_fft(uint32_t *tc_fft, const uint32_t *poly,
                                                                              unsigned count, const DevTables *T) {
    constexpr unsigned n = 1u << LOGN, lanes = n / 8, N = 8 * n;
    __shared__ uint32_t lds[WIDE ? n * 9 : NTT_LDS_WORDS];
    const unsigned sub = threadIdx.x / lanes, t = threadIdx.x % lanes;
    const size_t id = WIDE ? blockIdx.x : min(blockIdx.x * (64 / lanes) + sub, count - 1);
    const unsigned i = (unsigned)(id % 16);
    const uint32_t *src = poly + id / 16 * N * FR_WORDS;
    uint32_t *dst = tc_fft + id * n * FR_WORDS;
    const auto load = [&](unsigned e, fn &x) {
        const int c = toeplitz_src(i, e, N);
        fs a;
        fs_zero(a);
        if (c >= 0) fs_load(a, src + (size_t)c * FR_WORDS);
        fn_unpack(x, a.l);
    };
    const auto store = [&](unsigned k, const uint32_t *w) {
        fs a;
        fs_set(a, w);
        fs_store(dst + (size_t)k * FR_WORDS, a);
    };
    if constexpr (WIDE) ntt_wide<LOGN, false>(lds, 0, T, load, store);
    else ntt<LOGN, false>(lds + sub * n * 9, t, 0, T, load, store);
}

// ---------------------------------------------------------------- element-wise Fr ops

__global__ void k_fr_op(int op, uint32_t *out, const uint32_t *a, const uint32_t *b, size_t count) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= count) return;
    fs x, y, z;
    fs_load(x, a + e * FR_WORDS);
    fs_to_mont(x, x);
    fs_zero(y);
    if (op <= 2 && b) {  // binary ops only: add, sub, mul
        fs_load(y, b + e * FR_WORDS);
        fs_to_mont(y, y);
    }
    switch (op) {
    case 0: fs_add(z, x, y); break;
    case 1: fs_sub(z, x, y); break;
    case 2: fs_mul(z, x, y); break;
    case 3: fs_mul(z, x, x); break;
    case 4: { fs zero; fs_zero(zero); fs_sub(z, zero, x); } break;
    case 5: {  // x^(r-2)
        fs acc;
        fs_set(acc, FR_ONE);
        for (int w = 7; w >= 0; w--) {
            const uint32_t ew = FR_RM2[w];
            for (int bit = 31; bit >= 0; bit--) {
                fs_mul(acc, acc, acc);
                if ((ew >> bit) & 1) fs_mul(acc, acc, x);
            }
        }
        z = acc;
    } break;
    default: z = x; break;
    }
    fs_from_mont(z, z);
    fs_store(out + e * FR_WORDS, z);
}

// ---------------------------------------------------------------- launchers

hipError_t launch_toeplitz(uint32_t *tc, const uint32_t *poly, unsigned rows, unsigned N, hipStream_t s) {
    const size_t total = (size_t)rows * 16 * (N / 8);
    if (!total) return hipSuccess;
    const unsigned blocks = (unsigned)((total + 255) / 256);
    hipLaunchKernelGGL(k_toeplitz, dim3(blocks), dim3(256), 0, s, reinterpret_cast<uint4 *>(tc),
                       reinterpret_cast<const uint4 *>(poly), rows, N);
    return hipGetLastError();
}

template <unsigned LOGN, bool INV>
static void ntt_launch(uint32_t *out, const uint32_t *in, unsigned count, const DevTables *T, hipStream_t s) {
    constexpr unsigned n = 1u << LOGN, per = 512 / n;
    if ((count + per - 1) / per <= NTT_WIDE_WAVES)
        hipLaunchKernelGGL((k_fr_ntt<LOGN, INV, true>), dim3(count), dim3(n / 2), 0, s, out, in, count, T);
    else
        hipLaunchKernelGGL((k_fr_ntt<LOGN, INV, false>), dim3((count + per - 1) / per), dim3(64), 0, s, out, in, count, T);
}

template <bool INV>
static hipError_t ntt_dispatch(uint32_t *out, const uint32_t *in, unsigned count, unsigned n,
                               const DevTables *T, hipStream_t s) {
    switch (n) {
    case 128: ntt_launch<7, INV>(out, in, count, T, s); break;
    case 256: ntt_launch<8, INV>(out, in, count, T, s); break;
    case 512: ntt_launch<9, INV>(out, in, count, T, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_fr_ntt(uint32_t *out, const uint32_t *in, unsigned count, unsigned n, bool inverse,
                         const DevTables *T, hipStream_t s) {
    if (!count) return hipSuccess;
    return inverse ? ntt_dispatch<true>(out, in, count, n, T, s) : ntt_dispatch<false>(out, in, count, n, T, s);
}

template <unsigned LOGN>
static void toeplitz_fft_launch(uint32_t *tc_fft, const uint32_t *poly, unsigned rows, const DevTables *T, hipStream_t s) {
    constexpr unsigned n = 1u << LOGN, per = 512 / n;
    const unsigned count = rows * 16;  // a multiple of the transforms per wave
    if (count / per <= NTT_WIDE_WAVES)
        hipLaunchKernelGGL((k_toeplitz_fft<LOGN, true>), dim3(count), dim3(n / 2), 0, s, tc_fft, poly, count, T);
    else
        hipLaunchKernelGGL((k_toeplitz_fft<LOGN, false>), dim3(count / per), dim3(64), 0, s, tc_fft, poly, count, T);
}

hipError_t launch_toeplitz_fft(uint32_t *tc_fft, const uint32_t *poly, unsigned rows, unsigned N,
                               const DevTables *T, hipStream_t s) {
    if (!rows) return hipSuccess;
    switch (N) {
    case 1024: toeplitz_fft_launch<7>(tc_fft, poly, rows, T, s); break;
    case 2048: toeplitz_fft_launch<8>(tc_fft, poly, rows, T, s); break;
    case 4096: toeplitz_fft_launch<9>(tc_fft, poly, rows, T, s); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_fr_op(int op, uint32_t *out, const uint32_t *a, const uint32_t *b, size_t count,
                        hipStream_t s) {
    if (!count) return hipSuccess;
    hipLaunchKernelGGL(k_fr_op, dim3((unsigned)((count + 63) / 64)), dim3(64), 0, s, op, out, a, b, count);
    return hipGetLastError();
}

}  // namespace fk20
